// order_inst.hpp -- the stage and adjoint kernel instances of one polynomial
// order.  Included by order_n<N1>.hip with NKC_N1 = N + 1 defined.
#pragma once
#ifndef NKC_N1
#error "define NKC_N1 before including order_inst.hpp"
#endif
#include "order_launch.hpp"

namespace nkc {
namespace {

template <int N1, int MAT, int MODE, int FEAT>
void launch_f(const StageArgs &a, bool nt, int grid, hipStream_t s) {
    constexpr int OCC = box_waves(N1, FEAT);
    const dim3 bs(BoxShape<N1>::BS);
    if (MODE != MODE_RESIDUAL && nt)
        hipLaunchKernelGGL((box_kernel<N1, MAT, MODE, FEAT, MODE != MODE_RESIDUAL, OCC>), dim3(grid), bs, 0, s, a);
    else
        hipLaunchKernelGGL((box_kernel<N1, MAT, MODE, FEAT, false, OCC>), dim3(grid), bs, 0, s, a);
}

// Kernel instance by feature set: FEAT = 3 with a graphene sheet, 2 with a
// PML or an incident field, 1 with a source, Drude or Lorentz region, 0
// otherwise.  The residual test entry has the plain and the full instance.
// The slab instances (see stage_slabs); whether one was launched.
template <int N1, int MAT, int SL>
bool launch_s(const StageArgs &a, int sl, int feat, int grid, hipStream_t s) {
    if constexpr (slabs_built(N1, SL)) {
        if (sl != SL || feat > 2) return false;
        const dim3 g(grid * SL), bs(BoxShape<N1>::BS);
        constexpr int O0 = box_waves(N1, 0), O1 = box_waves(N1, 1), O2 = box_waves(N1, 2);
        if (feat == 0) hipLaunchKernelGGL((box_kernel<N1, MAT, MODE_RK, 0, false, O0, SL>), g, bs, 0, s, a);
        else if (feat == 1) hipLaunchKernelGGL((box_kernel<N1, MAT, MODE_RK, 1, false, O1, SL>), g, bs, 0, s, a);
        else hipLaunchKernelGGL((box_kernel<N1, MAT, MODE_RK, 2, false, O2, SL>), g, bs, 0, s, a);
        return true;
    }
    return false;
}

template <int N1, int MAT>
void launch_m(const StageArgs &a, int mode, bool nt, int sl, int grid, hipStream_t s) {
    const int feat = a.gr_off ? 3 : (a.pml_off || a.inc_mask) ? 2 : (a.src_off || a.drude_off || a.lor_off) ? 1 : 0;
    if (sl > 1 && (launch_s<N1, MAT, 2>(a, sl, feat, grid, s) || launch_s<N1, MAT, 3>(a, sl, feat, grid, s) ||
                   launch_s<N1, MAT, 4>(a, sl, feat, grid, s) || launch_s<N1, MAT, 5>(a, sl, feat, grid, s)))
        return;
    if (mode == MODE_RESIDUAL) {
        if (feat) launch_f<N1, MAT, MODE_RESIDUAL, 3>(a, false, grid, s);
        else launch_f<N1, MAT, MODE_RESIDUAL, 0>(a, false, grid, s);
    } else if (a.st_r || a.st_J) {
        // the adjoint's recompute: sources and Drude regions only
        if (feat) launch_f<N1, MAT, MODE_RK_STORE, 1>(a, nt, grid, s);
        else launch_f<N1, MAT, MODE_RK_STORE, 0>(a, nt, grid, s);
    } else if (feat == 3) {
        launch_f<N1, MAT, MODE_RK, 3>(a, nt, grid, s);
    } else if (feat == 2) {
        launch_f<N1, MAT, MODE_RK, 2>(a, nt, grid, s);
    } else if (feat == 1) {
        launch_f<N1, MAT, MODE_RK, 1>(a, nt, grid, s);
    } else {
        launch_f<N1, MAT, MODE_RK, 0>(a, nt, grid, s);
    }
}

template <int N1, int MAT, bool GM>
void launch_adj_g(const AdjArgs &a, bool nt, int grid, hipStream_t s) {
    const dim3 bs(BoxShape<N1>::BS);
    if (nt) hipLaunchKernelGGL((adjoint_kernel<N1, MAT, GM, true>), dim3(grid), bs, 0, s, a);
    else hipLaunchKernelGGL((adjoint_kernel<N1, MAT, GM, false>), dim3(grid), bs, 0, s, a);
}

template <int N1, int MAT>
void launch_adj_t(const AdjArgs &a, bool nt, int grid, hipStream_t s) {
    if (a.rs) launch_adj_g<N1, MAT, true>(a, nt, grid, s);
    else launch_adj_g<N1, MAT, false>(a, nt, grid, s);
}

}  // namespace

#define NKC_CAT2(a, b) a##b
#define NKC_CAT(a, b) NKC_CAT2(a, b)

void NKC_CAT(launch_stage_n, NKC_N1)(const StageArgs &a, int mat, int mode, bool nt, int sl, int grid, hipStream_t s) {
    if (mat == MAT_ELEM) launch_m<NKC_N1, MAT_ELEM>(a, mode, nt, sl, grid, s);
    else launch_m<NKC_N1, MAT_NODE>(a, mode, nt, sl, grid, s);
}

void NKC_CAT(launch_adjoint_n, NKC_N1)(const AdjArgs &a, int mat, bool nt, int grid, hipStream_t s) {
    if (mat == MAT_ELEM) launch_adj_t<NKC_N1, MAT_ELEM>(a, nt, grid, s);
    else launch_adj_t<NKC_N1, MAT_NODE>(a, nt, grid, s);
}

#undef NKC_CAT
#undef NKC_CAT2

}  // namespace nkc
