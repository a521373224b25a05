// jacobi_plan.hpp -- host rules of the many-sweep Jacobi launches (setup.hip),
// plain C++ so that they can be checked without a GPU.
#pragma once

namespace sp3mm {

constexpr int kGridSweeps = 64;    // sweeps of one launch of k_jacobi_grid at most
constexpr int kGridRows = 2048;    // rows it takes at most
constexpr int kGridThreads = 512;  // lanes of a workgroup

// Sweeps of the next launch when `left` (>= 2) remain.  Never one by itself,
// and never one left over: within a launch a workgroup's last sweep, which
// overwrites x, is ordered behind the other workgroups' reads of x only by the
// polls between sweeps, and a launch of one sweep has none.
inline int jacobi_chunk(int left)
{
    const int n = left < kGridSweeps ? left : kGridSweeps;
    return left - n == 1 ? n - 1 : n;
}

// Workgroups that take M rows with L lanes each, and whether `cus` CUs that hold
// per_cu of them each run them all at once (their sweeps wait for each other).
inline int jacobi_groups(int M, int L) { return (M + kGridThreads / L - 1) / (kGridThreads / L); }
inline bool jacobi_grid_resident(int M, int L, int per_cu, int cus)
{
    return (long long)jacobi_groups(M, L) <= (long long)per_cu * cus;
}

}  // namespace sp3mm
