// stage_args.hpp -- arguments of the stage kernels and the small device
// helpers the stage, adjoint and general-hexahedra kernels share.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nkc {

template <bool NT, class T>
__device__ __forceinline__ void st_stream(T *p, T v) {
    if constexpr (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}

template <bool NT, class T>
__device__ __forceinline__ T ld_stream(const T *p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}

// Kernel face order (symmetric): 0 x-, 1 x+, 2 y-, 3 y+, 4 z-, 5 z+.
enum FaceType : int32_t { FACE_PEC = -1, FACE_NONE = -2 };

enum StageMode : int { MODE_RK = 0, MODE_RESIDUAL = 1, MODE_RK_STORE = 2 };
enum MatMode : int { MAT_ELEM = 0, MAT_NODE = 1 };

struct StageArgs {
    const double *__restrict__ uin;   // 6 fields, stride fs
    double *__restrict__ uout;        // MODE_RK: updated fields
    double *__restrict__ kbuf;        // MODE_RK: RK register, in place
    double *__restrict__ res;         // MODE_RESIDUAL: residual out
    const double *__restrict__ D;     // n1*n1, D(i,l) at D[i + n1*l]
    const double *__restrict__ geo;   // per element: gx gy gz L0..L5 (9)
    const int32_t *__restrict__ nbr;  // per element: 6 neighbour ids / FaceType
    const double *__restrict__ fco;   // ELEM: e*6*4 ; NODE: (e*6+f)*n2*4
    const double *__restrict__ ieps;  // ELEM: per element ; NODE: per node
    const double *__restrict__ imu;
    int64_t fs;                       // field stride (doubles)
    int32_t nelt;
    int32_t per_xcd;                  // elements per XCD slice (grid remap)
    double rka, rkb, dt;
    // MODE_RK: bit 0 reads the RK register, bit 1 writes it.  The first
    // stage's a_1 = 0 makes the read moot and the next step's first stage
    // ignores what the last stage would write, so a step's first stage
    // skips the read and its last stage the write (10 % of a step's bytes).
    int32_t kflags;
    const double *__restrict__ dt_e;  // per-element dt (batched cavities) or null
    // the stage's time and the source's factor g at that time (written on
    // the device at the start of the step)
    const double *__restrict__ tst;
    // usersrc-style source on E: src_amp (un-weighted, per node of the
    // elements with src_off[e] >= 0) * dir * g(t)
    const int32_t *__restrict__ src_off;
    const double *__restrict__ src_amp;
    double src_dir[3];
    // Drude ADE (cem_maxwell_drude): elements with drude_off[e] >= 0 carry
    // J, kJ ([3][n1^3] each) and (a, b) per node
    const int32_t *__restrict__ drude_off;
    double *__restrict__ dJ;
    double *__restrict__ dkJ;
    const double *__restrict__ dpar;
    double *__restrict__ dresJ;       // MODE_RESIDUAL: resJ out (same layout as J)
    // Lorentz ADE (cem_maxwell_lorentz): elements with lor_off[e] >= 0 carry
    // J then P (6 n1^3 doubles at lor_off[e] 6 n1^3) and their RK register,
    // per-node (a, b, c) at (lor_off[e] n1^3 + vloc) 3
    const int32_t *__restrict__ lor_off;
    double *__restrict__ lL;
    double *__restrict__ lkL;
    const double *__restrict__ lpar;
    double *__restrict__ lresL;       // MODE_RESIDUAL: (resJ, resP) out
    // MODE_RK, adjoint recompute: keep the stage residual (6 fields, stride
    // fs) and the stage-input Drude current (layout of dJ) when non-null
    double *__restrict__ st_r;
    double *__restrict__ st_J;
    // PML (pml_step): elements with pml_off[e] >= 0 carry sigma x, y, z
    // (3 n1^3 doubles at pml_off[e] 3 n1^3) and the auxiliary fields B then
    // D (6 n1^3 at pml_off[e] 6 n1^3) with their RK register
    const int32_t *__restrict__ pml_off;
    const double *__restrict__ psig;
    double *__restrict__ pP;
    double *__restrict__ pkP;
    double *__restrict__ presP;       // MODE_RESIDUAL: (resB, resD) out
    // userinc-style incident plane wave: inc_mask[e] bit f (kernel face
    // order) adds it to the element's own trace on face f, bit 8 + f to the
    // neighbour's trace seen across face f; u = cos(inc_k . x - inc_om t)
    // at the trace's node (coordinates xyz, 3 x fs)
    const int32_t *__restrict__ inc_mask;
    const double *__restrict__ xyz;
    double inc_k[3], inc_om, inc_h[3], inc_e[3];
    // graphene sheet current (userfsrc + cem_3d_graphene_current):
    // gr_off[e*6 + f] = the sheet block of face f (kernel order) or -1.  Per
    // block and face node q (the flux's in-face index, the same on both
    // sides of a face): 14 doubles at gpar[(b*14 + c)*n2 + q] (the twelve
    // sheet parameters, Yfac = 0.5/Y_0, yconduc) and the state (fjn slots
    // 2..6 x 3 components) at [(b*15 + c)*n2 + q], read from gA and written
    // to gAn (both sides of a face read each other's state, so the stages
    // alternate two copies), the RK register gK in place.
    const int32_t *__restrict__ gr_off;
    const double *__restrict__ gpar;
    const double *__restrict__ gA;
    double *__restrict__ gAn;
    double *__restrict__ gK;
    // xcd_bal: XCD x takes elements xcd_lo[x] .. xcd_lo[x + 1] - 1 (ranges
    // of equal work when some elements cost more, e.g. a Drude region)
    // instead of equal runs of per_xcd elements
    int32_t xcd_bal;
    int32_t xcd_lo[9];
};

__device__ __forceinline__ int remap_element(int b, int nelt, int per_xcd) {
    // Workgroups are dealt round-robin to the 8 XCDs; give each XCD a
    // contiguous run of elements so x/y neighbours share its L2.
    int xcd = b & 7;
    int slot = b >> 3;
    return xcd * per_xcd + slot;
}

// n x v for a general n.
__device__ __forceinline__ void gcross(const double n[3], const double v[3], double o[3]) {
    o[0] = n[1] * v[2] - n[2] * v[1];
    o[1] = n[2] * v[0] - n[0] * v[2];
    o[2] = n[0] * v[1] - n[1] * v[0];
}

// n x v for n = sg * e_AX.
template <int AX>
__device__ __forceinline__ void ncross(double sg, const double v[3], double o[3]) {
    if (AX == 0) { o[0] = 0.0;        o[1] = -sg * v[2]; o[2] = sg * v[1]; }
    if (AX == 1) { o[0] = sg * v[2];  o[1] = 0.0;        o[2] = -sg * v[0]; }
    if (AX == 2) { o[0] = -sg * v[1]; o[1] = sg * v[0];  o[2] = 0.0; }
}

}  // namespace nkc
