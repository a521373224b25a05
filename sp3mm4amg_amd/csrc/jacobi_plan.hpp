// jacobi_plan.hpp -- host rules of the many-sweep Jacobi launches (setup.hip),
// plain C++ so that they can be checked without a GPU.
#pragma once

namespace sp3mm {

constexpr int kGridSweeps = 64;  // sweeps of one launch of k_jacobi_grid at most

// Sweeps of the next launch when `left` (>= 2) remain.  Never one by itself,
// and never one left over: within a launch a workgroup's last sweep, which
// overwrites x, is ordered behind the other workgroups' reads of x only by the
// polls between sweeps, and a launch of one sweep has none.
inline int jacobi_chunk(int left)
{
    const int n = left < kGridSweeps ? left : kGridSweeps;
    return left - n == 1 ? n - 1 : n;
}

}  // namespace sp3mm
