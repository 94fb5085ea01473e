// order_launch.hpp -- per-order launchers of the stage and adjoint kernels.
//
// Every polynomial order's kernel instances live in a translation unit of
// their own (order_n<N1>.hip, which includes order_inst.hpp), so the
// instances of the seven orders compile in parallel.  The host code calls
// them through these plain functions.
#pragma once
#include <hip/hip_runtime.h>

#include "adjoint_kernel.hpp"
#include "box_kernel.hpp"

namespace nkc {

// Waves per SIMD the register allocator of the stage kernel keeps to (0:
// free): 128 VGPRs from N = 6 on, where the 8-wave workgroups of N = 8, 9
// then fit twice on a CU and the 4-wave ones of N = 6, 7 four times; 168 at
// N = 7 with a PML, an incident field or a sheet, which would spill at 128 (its swizzled LDS
// addresses take a register each).
constexpr int box_waves(int n1, int feat) { return n1 < 7 ? 0 : (n1 == 8 && feat >= 2) ? 3 : 4; }

// Waves per SIMD of the instances with a sheet, as built: 129 and 152 VGPRs at
// N = 5, 161 and 167 at N = 7, below 128 at the other orders.
constexpr int sheet_waves(int n1) { return n1 == 6 || n1 == 8 ? 3 : 4; }

// nt: k and the outputs past the caches (see stage_nt)
#define NKC_DECL_ORDER(n)                                                                          \
    void launch_stage_n##n(const StageArgs &a, int mat, int mode, bool nt, int sl, int grid, hipStream_t s); \
    void launch_adjoint_n##n(const AdjArgs &a, int mat, bool nt, int grid, hipStream_t s);
NKC_DECL_ORDER(4)
NKC_DECL_ORDER(5)
NKC_DECL_ORDER(6)
NKC_DECL_ORDER(7)
NKC_DECL_ORDER(8)
NKC_DECL_ORDER(9)
NKC_DECL_ORDER(10)
#undef NKC_DECL_ORDER

}  // namespace nkc
