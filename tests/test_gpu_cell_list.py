"""The even-split cell-list force (k_cell_list) where it can go wrong: few
columns, groups and chunks that end inside a column, empty columns, clusters
that overflow its buffer, short memory, thin cylinders, the rounding of its
sums, and the grid it bins into."""

import contextlib
import io

import numpy as np
import pytest

from conftest import gpu_free_bytes, gpu_memory_left, say

pytestmark = pytest.mark.gpu


def _setup(N, precision, rc, rs, R=3.0, H=6.0, np_seed=2):
    from opendust_amd import workloads

    with contextlib.redirect_stdout(io.StringIO()):
        od = workloads.single_dust(N=N, n=3, precision=precision, seed=4, R=R, H=H)
        cfg, x0, v0 = workloads.prepare(od, alpha=workloads.synthetic_alpha(od), np_seed=np_seed, precision=precision)
    cfg.cutoff = rc * cfg.r_D_e
    cfg.switch_dist = 0.0 if rs is None else rs * cfg.r_D_e
    return cfg, x0, v0


def _check(oracle_lib, cfg, x0, precision):
    """Forces, cells and order of one evaluation against the oracle: the bounds
    of the other cutoff tests, FP32c on the rounded positions, a pair at the
    rounding of a hard cutoff allowed on either side."""
    from oracle.oracle import fp32c_rounded_positions

    from opendust_amd import engine

    e = engine.Engine(cfg)
    f = e.pair_forces(x0)
    cell, order, dims = e.cells()
    fc = e.force_cells()
    f2 = e.pair_forces(x0)
    e.close()
    # the device's own list: binning and radix order bit-exact on its grid
    nx, ny, nz = fc["dims"]
    w, h = fc["size"]
    ix, iy = (np.clip(np.floor((x0[:, k] + cfg.R) / w), 0, nx - 1).astype(int) for k in (0, 1))
    iz = np.clip(np.floor((x0[:, 2] + cfg.H / 2) / h), 0, nz - 1).astype(int)
    want = iz + nz * (ix + nx * iy)
    assert nx == ny == np.ceil(2 * cfg.R / w) and nz == np.ceil(cfg.H / h)
    assert np.array_equal(fc["cell"], want)
    assert np.array_equal(fc["order"], np.lexsort((np.arange(len(want)), want)))
    assert 256 ** (fc["radix_passes"] - 1) <= max(1, nx * ny * nz) < 256 ** fc["radix_passes"]
    say("  grid", fc["dims"], "radix passes", fc["radix_passes"], "units", fc["units"], "of", fc["capacity"])
    assert np.array_equal(f, f2)
    if precision == "fp64":
        ref, edge = oracle_lib.pair_forces(cfg, x0), np.zeros(len(x0))
        rel_i, rel_rms = 1e-11, 1e-13
    else:
        xr = fp32c_rounded_positions(cfg, x0)
        ref, edge = oracle_lib.pair_forces(cfg, xr), oracle_lib.cut_edge_count(cfg, xr, 1e-6)
        rel_i, rel_rms = 1e-5, 1e-6
    fn = np.linalg.norm(ref, axis=1)
    rms = np.sqrt(np.mean(fn ** 2))
    err = np.linalg.norm(f - ref, axis=1)
    f_cut = oracle_lib.cut_force_at_cutoff(cfg) if cfg.switch_dist <= 0.0 else 0.0
    bound = rel_i * fn + rel_rms * rms + edge * f_cut * 1.001
    say("  worst per-ion error / bound", float(np.max(err / np.maximum(bound, 1e-300))))
    assert np.all(err <= bound)
    want = np.array([oracle_lib.cell_of(cfg, xi)[0] for xi in x0])
    assert dims == oracle_lib.cell_of(cfg, x0[0])[1]
    assert np.array_equal(cell, want)
    assert np.array_equal(order, np.lexsort((np.arange(len(want)), want)))
    return fc


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("N,rc,rs", [(1, 2.0, None), (64, 2.0, None), (129, 3.2, 3.0), (2500, 1.0, None),
                                     (2500, 3.2, 3.0), (6001, 2.0, 1.5), (6001, 9.0, None)])
def test_cell_list_sizes_vs_oracle(oracle_lib, precision, N, rc, rs):
    cfg, x0, _ = _setup(N, precision, rc, rs)
    say("cell list", precision, "N", N, "rc", rc, "rs", rs)
    _check(oracle_lib, cfg, x0, precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
def test_sparse_cylinder_keeps_the_older_kernels(oracle_lib, precision):
    """So few ions per cutoff that every grid of the list has more cells than
    half the ions: the older kernels on columns of cutoff/4, whose memory is
    the cells' (33 million) and not the list's entries'."""
    from opendust_amd import engine

    cfg, x0, _ = _setup(16384, precision, 1.0, None, R=20.0, H=80.0)
    say("sparse cylinder", precision)
    before = gpu_free_bytes()
    e = engine.Engine(cfg)
    held = before - gpu_free_bytes()
    say("  device memory of the context, GB:", held / 1e9)
    assert held <= 0.4e9
    if precision == "fp32c":
        assert e.sym_choice() == (0, 5)
    e.close()
    fc = _check(oracle_lib, cfg, x0, precision)
    assert fc["capacity"] == 0 and fc["dims"] == (160, 160, 1280) and fc["radix_passes"] == 4


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
def test_short_memory_steps_down(precision):
    """2^20 ions at r_c = 2 in R = 10, H = 20: the list with its 4 GB of spare
    units; on a GPU with less free memory with fewer; with less still the older
    kernels on their own grid.  The same forces: to the last bit with fewer
    units, else up to rounding (FP32c: and up to pairs at the cutoff counted on
    one side, each one pair force there)."""
    from opendust_amd import engine

    cfg, x0, _ = _setup(1 << 20, precision, 2.0, None, R=10.0, H=20.0)
    say("short memory, cutoff", precision)

    def forces():
        before = gpu_free_bytes()
        with engine.Engine(cfg) as e:
            held = before - gpu_free_bytes()
            f = e.pair_forces(x0)
            fc = e.force_cells()
        say("  device memory of the context, GB:", held / 1e9, "capacity", fc["capacity"], "grid", fc["dims"])
        return f, held, fc

    f, held, full = forces()
    assert 4e9 <= held <= 5.2e9
    if precision == "fp32c":  # FP64 has no spare beyond twice the even spread
        with gpu_memory_left(int(held - 0.7e9)):
            g, _, fewer = forces()
        assert full["units"] == fewer["units"] <= fewer["capacity"] < full["capacity"]
        assert np.array_equal(f, g)
    with gpu_memory_left(int(2.3e9)):
        g, _, older = forces()
    assert older["capacity"] == 0 and older["dims"] == (40, 40, 160)
    if precision == "fp64":
        fn = np.linalg.norm(f, axis=1)
        assert np.all(np.linalg.norm(g - f, axis=1) <= 1e-11 * fn + 1e-13 * np.sqrt(np.mean(fn ** 2)))
    else:
        assert np.linalg.norm(g - f) <= 1e-5 * np.linalg.norm(f)


@pytest.mark.parametrize("N,R,H,rc,rs", [(32768, 10.0, 20.0, 2.0, None), (60000, 10.0, 20.0, 2.0, None),
                                         (130001, 10.0, 20.0, 2.0, None), (310000, 10.0, 20.0, 2.0, None),
                                         (20000, 3.0, 6.0, 3.2, 3.0), (4000, 3.0, 6.0, 3.2, 3.0)])
def test_cell_list_rounds_no_worse_than_the_older_kernels(N, R, H, rc, rs):
    """FP32c forces of the list and of the kernel on columns of cutoff/4
    (sym_tile = 5), against FP64 on the positions both see, one size for each
    length of the list's FP32 chains: its median error per ion is not larger
    (5 % for the spread of a median over N ions)."""
    from opendust_amd import engine, host
    from oracle.oracle import fp32c_rounded_positions

    cfg, x0, _ = _setup(N, "fp32c", rc, rs, R=R, H=H)
    cfg64 = engine.Config.from_buffer_copy(cfg)
    cfg64.precision = host.PREC_FP64
    say("rounding of the cell list, N", N)
    e = engine.Engine(cfg64)
    ref = e.pair_forces(fp32c_rounded_positions(cfg, x0))
    e.close()
    fn = np.linalg.norm(ref, axis=1)
    err = {}
    for tile in (0, 5):
        cfg.sym_tile = tile
        e = engine.Engine(cfg)
        err[tile] = float(np.median(np.linalg.norm(e.pair_forces(x0) - ref, axis=1)[fn > 0] / fn[fn > 0]))
        assert e.sym_choice() == (0, tile)
        e.close()
    say("  median error per ion, list and older kernel:", err[0], err[5])
    assert err[0] <= 1.05 * err[5]


def _ball(cfg, n, rng):
    """n ions in a ball of half the cutoff, away from the dust"""
    d = rng.normal(size=(n, 3))
    r = 0.5 * cfg.cutoff * rng.uniform(size=n) ** (1 / 3)
    return d / np.linalg.norm(d, axis=1)[:, None] * r[:, None] + [1.2 * cfg.r_D_e, 0.0, 3.0 * cfg.r_D_e]


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("shape", ["cluster", "two_slabs", "line"])
def test_cell_list_uneven_ions_vs_oracle(oracle_lib, precision, shape):
    """Ions far from evenly spread, within the unit buffer.  cluster: all in a
    ball of half the cutoff (every pair interacts); two_slabs: the middle of
    every column empty, so a group spans the gap; line: one column holds
    everything."""
    cfg, x0, _ = _setup(4000, precision, 1.0, None, R=3.0, H=30.0)
    rng = np.random.RandomState(5)
    lam = cfg.r_D_e
    if shape == "cluster":
        x0 = _ball(cfg, len(x0), rng)
    elif shape == "two_slabs":
        x0[:, 2] = np.where(np.arange(len(x0)) % 2, 14.0, -14.0) * lam + rng.uniform(-0.4, 0.4, len(x0)) * lam
        x0[:50, 2] = rng.uniform(-14.0, 14.0, 50) * lam
    else:
        x0[:, 0] = 0.05 * lam + 0.01 * lam * rng.uniform(size=len(x0))
        x0[:, 1] = 0.05 * lam + 0.01 * lam * rng.uniform(size=len(x0))
    say("cell list, uneven ions", shape, precision)
    fc = _check(oracle_lib, cfg, x0, precision)
    assert 0 < fc["units"] <= fc["capacity"]


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("rs", [None, 0.8])
def test_cell_list_overflow_falls_back_to_the_older_kernels(oracle_lib, precision, rs):
    """60000 ions in a ball of half the cutoff make more units than the buffer
    holds: k_pair_cell computes the force on the list's grid, hard and
    switched.  Spread out again, the same context runs the list, and a step
    from the packed state matches the oracle's."""
    from oracle.oracle import fp32c_rounded_positions

    from opendust_amd import engine

    cfg, x0, v0 = _setup(60000, precision, 1.0, rs, R=3.0, H=30.0)
    packed = _ball(cfg, len(x0), np.random.RandomState(6))
    say("cell list, overflow", precision, "rs", rs)
    fc = _check(oracle_lib, cfg, packed, precision)
    assert fc["units"] > fc["capacity"] > 0
    with engine.Engine(cfg) as e:
        e.set_ions(packed, v0)
        e.run(1)
        fc = e.force_cells()
        x, v = e.get_ions()
        fl, _, _ = e.step_info()
        assert fc["units"] > fc["capacity"]
        assert np.all(fc["cell"][fl != 0] == np.prod(fc["dims"]))  # flagged ions are left out
        e.set_ions(x0, v0)
        fc = e.force_cells()
        assert 0 < fc["units"] <= fc["capacity"]
    q0 = np.array([cfg.dust_q0[0]])
    xo, vo, _, _, flo, _ = oracle_lib.step(cfg, packed, v0, q0, 0)
    assert np.array_equal(fl, flo)
    if precision == "fp64":
        assert np.max(np.abs(x - xo)) <= 1e-11 * cfg.R and np.max(np.abs(v - vo)) <= 1e-10 * np.max(np.abs(vo))
    else:
        # kept ions: the drift of the force error, the rounding of the positions and its arithmetic
        f, fr = (oracle_lib.pair_forces(cfg, p) for p in (packed, fp32c_rounded_positions(cfg, packed)))
        fn = np.linalg.norm(f, axis=1)
        f_cut = oracle_lib.cut_force_at_cutoff(cfg) if rs is None else 0.0
        edge = oracle_lib.cut_edge_count(cfg, packed, 1e-6)
        err = np.linalg.norm(fr - f, axis=1) + 1e-5 * fn + 1e-6 * np.sqrt(np.mean(fn ** 2)) + edge * f_cut
        bound = err * cfg.dt * cfg.dt / 2 / cfg.m_s + 1e-12 * cfg.R
        keep = fl == 0
        assert np.all(np.linalg.norm(x - xo, axis=1)[keep] <= bound[keep])


def test_cells_of_every_kind_of_evaluation(oracle_lib):
    """od_get_cells, which bins on request, after forces of other positions, of
    a new state and of a step (reinjected ions left out)."""
    from opendust_amd import engine

    cfg, x0, v0 = _setup(5000, "fp32c", 1.5, None, R=3.0, H=6.0)
    x0[:9, 2] = 0.51 * cfg.H
    y = x0 * 0.7

    def want(x, left_out=None):
        cell = np.array([oracle_lib.cell_of(cfg, xi)[0] for xi in x])
        dims = oracle_lib.cell_of(cfg, x[0])[1]
        if left_out is not None:
            cell[left_out] = np.prod(dims)
        order = np.lexsort((np.arange(len(cell)), cell))
        return cell, order[: int(np.sum(cell < np.prod(dims)))], dims

    def same(got, ref):
        return np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1]) and got[2] == ref[2]

    say("cells of every kind of evaluation")
    with engine.Engine(cfg) as e:
        e.set_ions(x0, v0)
        assert same(e.cells(), want(x0))
        e.pair_forces(y)
        assert same(e.cells(), want(y))
        for flags in (0, engine.RUN_GRAPH):
            e.run(5, flags)
            fl, _, n_re = e.step_info()
            assert same(e.cells(), want(e.get_ions()[0], fl != 0))
        e.run(0)
        assert same(e.cells(), want(e.get_ions()[0], fl != 0))
        e.set_ions(x0, v0)
        assert same(e.cells(), want(x0))
        e.run(1)
        fl, _, n_re = e.step_info()
        assert n_re >= 9
        assert same(e.cells(), want(e.get_ions()[0], fl != 0))


@pytest.mark.timeout(300)
def test_cell_list_overflow_on_narrow_columns():
    """2^22 ions gathered in a quarter of the cylinder's height: columns of
    cutoff/4 and more units than the buffer holds, so k_pair32_symcol takes over
    in FP32c on the list's grid; the forces of the same kernel on its own
    (sym_tile = 5), whose slabs are higher, up to the rounding of the sums (a
    switched cutoff: no pair is counted on one side only)."""
    from opendust_amd import engine

    cfg, x0, _ = _setup(1 << 22, "fp32c", 2.0, 1.8, R=10.0, H=20.0)
    x0[:, 2] /= 4.0
    say("cell list, overflow on narrow columns")
    out = []
    for tile in (0, 5):
        cfg.sym_tile = tile
        with engine.Engine(cfg) as e:
            out.append(e.pair_forces(x0))
            fc = e.force_cells()
        say("  sym_tile", tile, "grid", fc["dims"], "units", fc["units"], "of", fc["capacity"])
        assert fc["dims"][0] == 40 and (fc["units"] > fc["capacity"] > 0 if tile == 0 else fc["capacity"] == 0)
    assert np.linalg.norm(out[0] - out[1]) <= 2e-6 * np.linalg.norm(out[1])


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("squeeze", [12, 200])
def test_squeezed_ions_are_no_slower_than_with_the_older_kernels(precision, squeeze):
    """Ions gathered in 1/12 of the cylinder, which the list's buffer holds, and
    in 1/200, which it does not: the pair stage of the automatic kernels against
    that of the FP32c kernel on columns of cutoff/4 (sym_tile = 5).  Measured
    1.1 and 2.0 times its time, FP64 3.2 and 4.6 (its law's rate is 0.36 of
    FP32's); 37 and 100 times, FP64 10, when k_pair32_symcol or k_pair_cell took
    over from a buffer of twice the even spread's units."""
    from opendust_amd import engine

    cfg, x0, v0 = _setup(131072, precision, 2.0, None, R=10.0, H=20.0)
    x0[:, 2] /= squeeze / 4 if squeeze == 12 else squeeze / 16
    x0[:, :2] /= 2.0 if squeeze == 12 else 4.0

    def pair_ms(cfg):
        with engine.Engine(cfg) as e:
            e.set_ions(x0, v0)
            best = 1e9
            for _ in range(3):
                e.stage_timing(True)
                e.set_ions(x0, v0)
                e.run(1, engine.RUN_PROFILE_STAGES)
                best = min(best, e.stage_timing(True)[0]["pair"])
            return best, e.force_cells()

    say("squeezed ions", precision, squeeze)
    ms, fc = pair_ms(cfg)
    assert (fc["units"] <= fc["capacity"]) == (squeeze == 12)
    old = engine.Config.from_buffer_copy(cfg)
    old.precision = 0
    old.sym_tile = 5
    ms_old, _ = pair_ms(old)
    say("  pair stage, ms: automatic", ms, "columns of cutoff/4, FP32c", ms_old, "units", fc["units"], fc["capacity"])
    assert ms <= ms_old * (7.0 if precision == "fp64" else 2.0 if squeeze == 12 else 4.0)


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
def test_cell_list_beyond_16_bit_ids(precision):
    """A grid of the list with more than 65536 cells: three radix passes, the
    device's binning and order bit-exact."""
    from opendust_amd import engine

    cfg, x0, _ = _setup(300000, precision, 1.0, None, R=10.0, H=40.0)
    say("cell list, many cells", precision)
    with engine.Engine(cfg) as e:
        e.pair_forces(x0)
        fc = e.force_cells()
    nx, ny, nz = fc["dims"]
    say("  grid", fc["dims"], "radix passes", fc["radix_passes"])
    assert nx * ny * nz > 65536 and fc["radix_passes"] == 3 and 0 < fc["units"] <= fc["capacity"]
    w, h = fc["size"]
    ix, iy = (np.clip(np.floor((x0[:, k] + cfg.R) / w), 0, nx - 1).astype(int) for k in (0, 1))
    want = np.clip(np.floor((x0[:, 2] + cfg.H / 2) / h), 0, nz - 1).astype(int) + nz * (ix + nx * iy)
    assert np.array_equal(fc["cell"], want)
    assert np.array_equal(fc["order"], np.lexsort((np.arange(len(want)), want)))


def test_tune_of_a_cutoff_context():
    """od_tune on a cutoff context: refused before there are ions, whatever
    kernel it runs; nothing to tune for the list, a variant for the others."""
    from opendust_amd import engine

    cfg, x0, v0 = _setup(3000, "fp32c", 2.0, None)
    for tile in (0, 2):
        cfg.sym_tile = tile
        say("tune of a cutoff context, sym_tile", tile)
        with engine.Engine(cfg) as e:
            with pytest.raises(RuntimeError, match="needs the ions"):
                e.tune(1)
            e.set_ions(x0, v0)
            chosen = e.tune(1)
            assert chosen == (0, 0) if tile == 0 else chosen[0] == 0 and 1 <= chosen[1] <= 6
            assert e.sym_choice() == chosen
            e.run(2)
