// od_scan.h -- addition of work counts (constexpr: the kernels and host code
// use the same function).
//
// The scans of launch_scan hold 32-bit counts.  Work-group, item and cell
// counts cannot exceed the ion count, but the units of the evenly split cell
// list grow as the square of the ions inside one cutoff (6.0e6 of them make
// 2.2e9), and a wrapped sum would pass for one that fits the unit buffer.  So
// the scans saturate: addition of numbers in [0, COUNT_MAX] clipped at
// COUNT_MAX is associative, whatever the order the result is the true sum or
// COUNT_MAX, and COUNT_MAX exceeds every capacity.
#pragma once

namespace od {

constexpr int COUNT_MAX = 0x7fffffff;

// a, b >= 0
constexpr int add_counts(int a, int b) { return a <= COUNT_MAX - b ? a + b : COUNT_MAX; }

}  // namespace od
