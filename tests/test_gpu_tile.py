"""The wave-tile all-pairs kernel (even split of 64-ion tiles) and the FP64
pair law's own elementary functions."""

import contextlib
import io

import numpy as np
import pytest

from conftest import gpu_free_bytes, gpu_memory_left, say

pytestmark = pytest.mark.gpu


def _setup(N, precision, np_seed=5):
    from opendust_amd import workloads

    with contextlib.redirect_stdout(io.StringIO()):
        od = workloads.single_dust(N=N, n=3, precision=precision, seed=3)
        return workloads.prepare(od, alpha=workloads.synthetic_alpha(od), np_seed=np_seed, precision=precision)


def _forces(cfg, x, mode):
    from opendust_amd import engine

    cfg = engine.Config.from_buffer_copy(cfg)
    cfg.pair_mode = mode
    e = engine.Engine(cfg)
    f = e.pair_forces(x)
    info = e.pair_info()
    e.close()
    return f, info


# edges of a 64-ion sub-block, of a target group (4 and 8 sub-blocks, 16 with
# 4 waves), the changes of shape at 2^15 (FP32) and 2^17 (FP64) ions, several
# work-groups per group and several groups per work-group
@pytest.mark.parametrize("precision,N", [(p, n) for p in ("fp64", "fp32c") for n in (
    1, 2, 63, 64, 65, 255, 256, 257, 513, 4095, 5000)] + [
    ("fp32c", 32704), ("fp32c", 32705), ("fp32c", 70001), ("fp32c", 262080), ("fp64", 40001), ("fp64", 131009)])
def test_wave_tiles_vs_oracle_or_rows(oracle_lib, precision, N):
    """Small sizes against the oracle (the bounds of the other pair kernels);
    larger ones against the row kernel in the same precision, with twice the
    arithmetic bound, since both sides carry it."""
    from opendust_amd import engine

    cfg, x0, _ = _setup(N, precision)
    say("wave tiles", precision, "N", N)
    f, info = _forces(cfg, x0, engine.PAIR_AUTO)
    assert info == (engine.PAIR_SYM, N * (N - 1))
    if N <= 5000:
        ref = oracle_lib.pair_forces(cfg, x0)
        rel_i, rel_rms, rel = (1e-11, 1e-13, 1e-11) if precision == "fp64" else (1e-4, 1e-5, 1e-5)
    else:
        ref, info = _forces(cfg, x0, engine.PAIR_ROWS)
        assert info[0] == engine.PAIR_ROWS
        rel_i, rel_rms, rel = (1e-11, 1e-13, 1e-11) if precision == "fp64" else (2e-5, 2e-6, 4e-6)
    fn = np.linalg.norm(ref, axis=1)
    rms = np.sqrt(np.mean(fn ** 2))
    err = np.linalg.norm(f - ref, axis=1)
    say("  norm-wise", np.linalg.norm(f - ref) / max(np.linalg.norm(ref), 1e-300))
    assert np.all(err <= rel_i * fn + rel_rms * rms)
    assert np.linalg.norm(f - ref) <= rel * np.linalg.norm(ref)


@pytest.mark.parametrize("N", [2000, 8000, 32704, 65536])
def test_wave_tiles_round_no_worse_than_rows(N):
    """FP32c forces of the wave tiles and of the row kernel, which adds
    compensated 64-term blocks, against FP64 on the positions both see: the
    tiles' median error per ion is not larger (5 % for the spread of a median
    over N ions)."""
    from oracle.oracle import fp32c_rounded_positions

    from opendust_amd import engine, host

    cfg, x0, _ = _setup(N, "fp32c")
    cfg64 = engine.Config.from_buffer_copy(cfg)
    cfg64.precision = host.PREC_FP64
    say("rounding of wave tiles, N", N)
    ref, _ = _forces(cfg64, fp32c_rounded_positions(cfg, x0), engine.PAIR_AUTO)
    fn = np.linalg.norm(ref, axis=1)
    err = {}
    for mode in (engine.PAIR_AUTO, engine.PAIR_ROWS):
        f, _ = _forces(cfg, x0, mode)
        err[mode] = float(np.median(np.linalg.norm(f - ref, axis=1) / fn))
    say("  median error per ion, tiles and rows:", err[engine.PAIR_AUTO], err[engine.PAIR_ROWS])
    assert err[engine.PAIR_AUTO] <= 1.05 * err[engine.PAIR_ROWS]


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
def test_wave_tiles_batch_equals_single(precision):
    """Simulations of a batch whose sizes end inside a sub-block and a group:
    the same forces as each alone (same groups, so the same sums up to where
    work-groups split them), seen through one step's velocities."""
    from opendust_amd import engine

    sizes = [1, 64, 700, 2049, 5000]
    setups = [_setup(n, precision, np_seed=20 + i) for i, n in enumerate(sizes)]
    for s, (cfg, _, _) in enumerate(setups):
        cfg.sim_id = s
    say("wave tiles, batch", precision, sizes)
    b = engine.Batch([c for c, _, _ in setups])
    for s, (_, x, v) in enumerate(setups):
        b.set_ions(s, x, v)
    b.run(2)
    for s, (cfg, x, v) in enumerate(setups):
        e = engine.Engine(cfg)
        e.set_ions(x, v)
        e.run(2)
        xs, vs = e.get_ions()
        e.close()
        xb, vb = b.get_ions(s)
        tol = 1e-12 if precision == "fp64" else 1e-6
        assert np.max(np.abs(xb - xs)) <= tol * cfg.R
        assert np.max(np.abs(vb - vs)) <= tol * np.max(np.abs(vs))
    b.close()


def test_tune_keeps_or_replaces_wave_tiles():
    """od_tune on a context that runs wave tiles: (0, 0) and the same forces
    when they stay, else a k_pair32_sym schedule within the FP32c bound."""
    from opendust_amd import engine

    cfg, x0, v0 = _setup(32768, "fp32c")
    e = engine.Engine(cfg)
    e.set_ions(x0, v0)
    f0 = e.pair_forces(x0)
    say("tune over wave tiles")
    before = gpu_free_bytes()
    chosen = e.tune(2)
    f1 = e.pair_forces(x0)
    assert e.sym_choice() == chosen
    if chosen == (0, 0):
        assert np.array_equal(f0, f1)
        assert before - gpu_free_bytes() <= 2e6  # the schedules it timed are gone
    else:
        assert np.linalg.norm(f1 - f0) <= 4e-6 * np.linalg.norm(f0)
    e.run(4, engine.RUN_GRAPH)
    e.close()


def test_batch_tune_out_of_memory_keeps_wave_tiles():
    """od_batch_tune on a GPU whose free memory does not hold the schedules it
    would time (six simulations of 2^18 ions, 3.7 GB): an error, also when
    called again, and the batch steps on with its wave tiles as if untuned."""
    from opendust_amd import engine

    cfg, x0, v0 = _setup(262080, "fp32c")
    cfgs = []
    for s in range(6):
        cfgs.append(engine.Config.from_buffer_copy(cfg))
        cfgs[s].sim_id = s

    def batch():
        b = engine.Batch(cfgs)
        for s in range(6):
            b.set_ions(s, x0, v0)
        return b

    b = batch()
    with gpu_memory_left(2500 << 20):
        for again in range(2):
            say("batch tune out of memory, call", again)
            with pytest.raises(RuntimeError, match="hipMalloc"):
                b.tune(1)
    rec = b.run(1)
    x, v = b.get_ions(5)
    b.close()
    b = batch()
    assert np.array_equal(b.run(1), rec)
    x1, v1 = b.get_ions(5)
    assert np.array_equal(x, x1) and np.array_equal(v, v1)
    b.close()


def test_short_memory_steps_down_to_rows():
    """2^19 ions in FP64 want 3.2 GB of partial sums: on a GPU with less free,
    the row kernel, with the same forces."""
    from opendust_amd import engine

    cfg, x0, _ = _setup(1 << 19, "fp64")
    say("short memory, FP64 context")
    f, info = _forces(cfg, x0, engine.PAIR_AUTO)
    assert info[0] == engine.PAIR_SYM
    with gpu_memory_left(2500 << 20):
        g, info = _forces(cfg, x0, engine.PAIR_AUTO)
    assert info[0] == engine.PAIR_ROWS
    fn = np.linalg.norm(f, axis=1)
    assert np.all(np.linalg.norm(g - f, axis=1) <= 1e-11 * fn + 1e-13 * np.sqrt(np.mean(fn ** 2)))


@pytest.mark.parametrize("precision,n_sims,left", [("fp64", 3, 2300), ("fp32c", 6, 5000)])
def test_short_memory_batch_steps_down(precision, n_sims, left):
    """Simulations of 2^18 ions whose wave tiles do not fit: FP64 the row
    items, FP32c the block schedule (whose launch leaves out the pairs inside
    a block), with the same step up to rounding."""
    from opendust_amd import engine

    cfg, x0, v0 = _setup(262080, precision)
    cfgs = []
    for s in range(n_sims):
        cfgs.append(engine.Config.from_buffer_copy(cfg))
        cfgs[s].sim_id = s

    def step():
        b = engine.Batch(cfgs)
        for s in range(n_sims):
            b.set_ions(s, x0, v0)
        b.run(1)
        x, v = b.get_ions(n_sims - 1)
        pairs = b.pair_timing()[2]
        b.close()
        return x, v, pairs

    say("short memory, batch", precision)
    x, v, pairs = step()
    with gpu_memory_left(left << 20):
        xs, vs, pairs_s = step()
    assert pairs == n_sims * 262080 * 262079
    assert pairs_s == pairs if precision == "fp64" else pairs_s < pairs
    tol = 1e-12 if precision == "fp64" else 1e-6
    assert not np.array_equal(v, vs)  # another order of the sums
    assert np.max(np.abs(x - xs)) <= tol * cfg.R and np.max(np.abs(v - vs)) <= tol * np.max(np.abs(v))


def test_fp64_pair_law_over_its_range():
    """Two ions from 1e-6 to 600 r_D_e apart, FP64 (rsqrt, exp and 1/x of the
    kernels' own), against numpy: about 10 roundings, and the rounding of the
    distance r enters exp(-r) as r times its relative error."""
    from opendust_amd import engine

    cfg, _, _ = _setup(64, "fp64")
    cfg = engine.Config.from_buffer_copy(cfg)
    cfg.n_ions = 2
    cfg.n_dust = 0
    lam, a = cfg.r_D_e, cfg.r_0 / cfg.r_D_e
    say("FP64 pair law")
    for mode in (engine.PAIR_AUTO, engine.PAIR_ROWS):
        cfg.pair_mode = mode
        e = engine.Engine(cfg)
        for d in np.geomspace(1e-6, 600.0, 60):
            x = np.array([[0.0, 0.0, 0.0], [0.6 * d * lam, -0.64 * d * lam, 0.48 * d * lam]])
            r = np.linalg.norm(x[1] / lam)
            want = cfg.kqq / lam ** 2 * np.exp(-r) / (r + a) * (1 + 1 / (r + a)) * (-x[1] / lam / r)
            f = e.pair_forces(x)
            tol = 4e-15 + 1e-15 * r
            assert np.linalg.norm(f[0] - want) <= tol * np.linalg.norm(want), d
            assert np.linalg.norm(f[1] + want) <= tol * np.linalg.norm(want), d
        e.close()


@pytest.mark.parametrize("n_r,n_h,n_mc", [(1, 1, 1), (2, 4, 255), (3, 5, 257), (2, 6, 65536), (1, 11, 65537)])
def test_trap_grid_edges_vs_oracle(oracle_lib, n_r, n_h, n_mc):
    """Heights around the tile of five, samples around a block and a chunk."""
    from opendust_amd import engine

    rho, h = np.linspace(0, 3.0, n_r), np.linspace(0, 2.5, n_h)
    say("trap grid", n_r, n_h, n_mc)
    g = engine.trap_potential_grid(3.0, 5.0, rho, h, n_mc, 17)
    o = oracle_lib.trap_grid(3.0, 5.0, rho, h, n_mc, 17)
    assert g.shape == (n_r, n_h) and np.max(np.abs(g - o) / np.abs(o)) <= 1e-12


def test_trap_grid_rounding():
    """The trap grid against 80-bit sums over the same samples: 160 points of 8
    cylinders.  A correctly rounded result is off by 0.3 to 0.6e-16 (rms of a
    rounding); 1.5e-16 leaves room for the roundings of the chunks' sums but
    not for rounded sample positions (2.1e-16)."""
    from opendust_amd import engine

    n, err = 300000, []
    say("trap grid rounding")
    for R, H, seed in ((5.0, 10.0, 1), (5.0, 10.0, 2), (2.3, 4.7, 3), (3.0, 6.0, 4), (4.4, 8.1, 5), (2.0, 10.0, 6),
                       (5.0, 5.0, 7), (3.7, 9.9, 8)):
        rho, h = np.linspace(0, R, 4), np.linspace(0, H / 2, 5)
        g = engine.trap_potential_grid(R, H, rho, h, n, seed)
        s = engine.trap_samples_host(R, H, seed, 0, n).astype(np.longdouble)
        for i, a in enumerate(rho):
            for j, b in enumerate(h):
                d = np.sqrt((a - s[:, 0]) ** 2 + s[:, 1] ** 2 + (b - s[:, 2]) ** 2)
                ref = np.sum(np.exp(-d) / (d + np.longdouble("0.001"))) / n
                err.append(float((g[i, j] - ref) / ref))
    rms = np.sqrt(np.mean(np.square(err)))
    say("  rms relative error", rms)
    assert rms <= 1.5e-16
