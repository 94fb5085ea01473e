// level_runs.hpp -- how the stage kernels split an element's levels: pure
// index arithmetic, for the host and the device.
#pragma once

#if defined(__HIP__) || defined(__HIPCC__)
#define NKC_HD __host__ __device__
#else
#define NKC_HD
#endif

namespace nkc {

// Runs a workgroup splits a group's levels into.
NKC_HD constexpr int level_runs(int n1) { return n1 <= 5 ? n1 : (n1 % 3 == 0 ? 3 : 2); }

// Levels of the longest run when an element has level_runs(n1) * sl of them,
// and the slab counts with an instance: those that shorten it.
NKC_HD constexpr int run_length(int n1, int sl) { return (n1 + level_runs(n1) * sl - 1) / (level_runs(n1) * sl); }
NKC_HD constexpr bool slabs_built(int n1, int sl) {
    return sl > 1 && level_runs(n1) * sl <= n1 && run_length(n1, sl) < run_length(n1, sl - 1);
}

// The level slot kk of a run from k0 of kn levels stands for (the first n1 %
// runs runs have one level more).  A short run has
// one slot fewer than the longest: its last slot repeats the last level, whose
// row of D is there to read, and what it sums is dropped (N = 8 in two slabs,
// the last run: k0 = 8, one level, two slots; level 9 would be a row past the
// table).
NKC_HD constexpr int slot_level(int n1, int runs, int k0, int kn, int kk) {
    return n1 % runs == 0 || kk < kn ? k0 + kk : n1 - 1;
}

}  // namespace nkc
