// box_kernel.hpp -- the fused DG-SEM Maxwell RK stage on axis-aligned
// elements, for gfx950.
//
// One launch = one stage of cem_maxwell_op_rk (src/cem_maxwell.F:327-345):
// volume curl (maxwell_wght_curl :1428-1497 over local_grad3,
// src/nek5_grad.F:2-19), face restriction (:604-652), on-device face exchange
// (replaces gs_op_fields(gsh_face,...) :962), PEC mirror (:1368-1426),
// upwind/central flux (:922-1002), lift (:654-756), inverse mass
// (:1833-1904) and the 2N-storage RK update (rk4_upd,
// src/cem_common.F:18-76), fused so every field value crosses HBM once per
// stage in each direction.
//
// Mapping: one workgroup per element.  Each update group (0: H from -curl E,
// 1: E from curl H) owns whole waves, so the fields a wave touches and the
// bases of their addresses are scalar; a lane adds one 32-bit byte offset.
// Within a group a lane owns column (i, j) of one run of levels.  The stage
// goes through LDS in this order:
//   0  the element (64-node chunks), the tangential neighbour traces, the
//      lane's RK register and per-node data: every load up front, one HBM
//      round trip; the element into LDS;
//   1  each wave forms the flux of whole faces (at N = 3 of face nodes packed
//      over the lanes) into LDS: four tangential components, a face's flux has
//      none along its normal;
//   2  t derivatives of all the lane's levels from one read of its column,
//      lifts, then per level the r and s derivatives, physics, k update;
//   3  k and then u back into the element's place in LDS and out in the
//      order of memory, whole 128-byte lines.
//
// What bounds it: HBM, about 28.8 B per node and field; what used to cost
// more at every order but N = 7 is how the bytes left: a level's (N+1)^2
// doubles straddle cache lines, and a store that covers part of a line costs
// about a whole one (the N = 7 kernel with its arrays shifted by 8 bytes: 555
// -> 719 us at 32^3; only the stores matter, shifted element loads 547 -> 555).
// With phase 3's line-aligned stores, the 32-bit addressing and the single column read a stage takes, against the
// kernel before on the same card, N = 3 (44^3) 241 -> 208 us (per-node
// materials 282 -> 256), N = 4 (40^3) 408 -> 343, N = 5 (36^3) 474 -> 378, N = 6
// (32^3) 509 -> 412, N = 7 (32^3) 577 -> 544, N = 8 (22^3) 354 -> 279, N = 9
// (24^3) 600 -> 507 (per-node materials, 20^3, 405 -> 346).
//
// Field order in HBM: 0 Hx, 1 Hy, 2 Hz, 3 Ex, 4 Ey, 5 Ez, each a contiguous
// array of npts doubles at stride fs, volume index i + n1*j + n1^2*k +
// n1^3*e as in the reference.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "level_runs.hpp"
#include "stage_args.hpp"

namespace nkc {

// Launch shape and LDS layout for polynomial order N1 - 1.
//   A group's levels are split into KS runs of (N+1)^2 lanes: padded to
//   whole waves (PAD) when two runs fill them well (N = 7: 64 of 64 lanes,
//   N = 9: 100 of 128, N = 6: 49 of 64), packed back to back otherwise (N =
//   8: three runs, 243 of 256 lanes; N = 5: 108 of 128; N = 3, 4: a run per
//   level, 64 of 64 and 125 of 128).
//   At N = 9 five packed runs (500 of 512 lanes, 16 waves) measured 732 us
//   and three or four 810-830 against 507: they need more registers or LDS
//   reads than two workgroups per CU leave.
template <int N1>
struct BoxShape {
    static constexpr int N2 = N1 * N1, N3 = N2 * N1;
    static constexpr int KS = level_runs(N1);
    static constexpr bool PAD = KS == 2;
    static constexpr int PL = PAD ? (N2 + 63) / 64 * 64 : N2;        // lanes per run of levels
    static constexpr int GL = (KS * PL + 63) / 64 * 64;              // lanes per group
    static constexpr int BS = 2 * GL, WG = GL / 64;                  // WG: waves per group
    static constexpr int KL = (N1 + KS - 1) / KS;                    // levels of the longest run
    // 64-node chunks of a field per wave of its group: loads from the
    // element's first node, stores from the 128-byte line it lies in (G
    // divides the element's distance from a line; at most 16 - G doubles)
    static constexpr int CH = (N3 + 63) / 64, NLD = (CH + WG - 1) / WG;
    static constexpr int G = N3 % 16 == 0 ? 16 : N3 % 8 == 0 ? 8 : N3 % 4 == 0 ? 4 : N3 % 2 == 0 ? 2 : 1;
    static constexpr int CHS = (N3 + 16 - G + 63) / 64, NST = (CHS + WG - 1) / WG;
    static constexpr int FC = (N2 + 63) / 64;                        // wave chunks per face
    static constexpr int NF = (6 * FC + 2 * WG - 1) / (2 * WG);      // face chunks per wave
    // u(i,j,k) of field f at f*N3 + idx: XOR swizzle for power-of-two n1
    // (rows, columns and z-columns bank-conflict free), plain order
    // otherwise (at most 2-way conflicted)
    static constexpr bool SWZ = (N1 & (N1 - 1)) == 0;
    __device__ static __forceinline__ int idx(int i, int j, int k) { return (SWZ ? (i ^ j) : i) + N1 * j + N2 * k; }
    static constexpr int LDS_BYTES(int feat) { return 8 * (6 * N3 + (feat == 3 ? 30 : 24) * N2 + N2); }
};

// A wave-uniform base plus a lane's byte offset below 2^32 (scalar base and
// one VGPR: no 64-bit address arithmetic per lane); imm: constant bytes.
__device__ __forceinline__ const double *at(const double *b, unsigned off, int imm = 0) {
    return reinterpret_cast<const double *>(reinterpret_cast<const char *>(b) + off + imm);
}
__device__ __forceinline__ double *at(double *b, unsigned off, int imm = 0) {
    return reinterpret_cast<double *>(reinterpret_cast<char *>(b) + off + imm);
}

template <class T>
__device__ __forceinline__ T pick3(int s, T a, T b, T c) { return s == 0 ? a : s == 1 ? b : c; }

// Value of v in lane `lane` of the wave (lane a compile-time constant or
// wave-uniform), for every lane: two v_readlane_b32 into a scalar pair.
__device__ __forceinline__ double bcast_lane(double v, int lane) {
    const long long b = __builtin_bit_cast(long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __builtin_bit_cast(double, (long long)(((unsigned long long)hi << 32) | lo));
}

// Incident plane wave u at volume node p (global index), time t.
__device__ __forceinline__ double incident(const StageArgs &a, int64_t p, double t) {
    return cos(a.inc_k[0] * a.xyz[p] + a.inc_k[1] * a.xyz[a.fs + p] + a.inc_k[2] * a.xyz[2 * a.fs + p] - a.inc_om * t);
}

// Sheet current J (components along ax, t1, t2) at node q of sheet block b
// for the side whose outward normal is sg e_ax, from that side's tangential
// traces tr = (H t1, H t2, E t1, E t2) (the incident wave included) and the
// stage-input state (cem_3d_graphene_current, src/cem_maxwell.F:2860-2886):
//   tmp = Yfac (-n x H + yconduc n x (E x n)),
//   J = (s2 + s3 + s5 - (b_cp1 + b_cp2) tmp) / (1 - (b_cp1 + b_cp2) Yfac).
// With upd the side's state takes this stage's RK update (:2887-2929):
// f = tmp - Yfac J drives the Drude slot 2 and the critical-point pairs
// (3, 4) and (5, 6).
template <int N2>
__device__ __forceinline__ void sheet_current(const StageArgs &a, int b, int q, int ax, int t1, int t2, double sg,
                                              const double tr[4], bool upd, double dt, double J[3]) {
    const double *p = a.gpar + (int64_t)b * 14 * N2 + q;
    const double *A = a.gA + (int64_t)b * 15 * N2 + q;
    const double nH[3] = {0.0, sg * tr[1], -sg * tr[0]};
    const double nEn[3] = {0.0, tr[2], tr[3]};
    const double Yfac = p[12 * N2], yc = p[13 * N2];
    const double cpf = p[2 * N2] + p[7 * N2];
    const double jnf = 1.0 - cpf * Yfac;
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        const int c = s == 0 ? ax : s == 1 ? t1 : t2;
        const double A0 = A[c * N2], A1 = A[(3 + c) * N2], A3 = A[(9 + c) * N2];
        const double tmp = Yfac * (nH[s] + yc * nEn[s]);
        J[s] = (A0 + A1 + A3 - cpf * tmp) / jnf;
        if (upd) {
            const double A2 = A[(6 + c) * N2], A4 = A[(12 + c) * N2];
            const double f = tmp - Yfac * J[s];
            double r[5];
            r[0] = -p[0] * A0 + p[N2] * f;
            r[1] = A2 + p[5 * N2] * f;
            r[2] = -p[3 * N2] * A1 - p[4 * N2] * A2 + p[6 * N2] * f;
            r[3] = A4 + p[10 * N2] * f;
            r[4] = -p[8 * N2] * A3 - p[9 * N2] * A4 + p[11 * N2] * f;
            const double Ao[5] = {A0, A1, A2, A3, A4};
            const int64_t o = (int64_t)b * 15 * N2 + q;
#pragma unroll
            for (int sl = 0; sl < 5; ++sl) {
                const int64_t x = o + (3 * sl + c) * N2;
                const double kn = a.rka * a.gK[x] + dt * r[sl];
                a.gK[x] = kn;
                a.gAn[x] = Ao[sl] + a.rkb * kn;
            }
        }
    }
}

// The element of workgroup b (nelt when the workgroup has none).  BAL: the
// instance reads the equal-work ranges (those with in-stage physics, whose
// elements differ in cost; the plain instances keep the registers the table
// would take).
template <bool BAL, class Args>
__device__ __forceinline__ int stage_element(const Args &a, int b, int nelt) {
    if (BAL && a.xcd_bal) {
        const int x = b & 7, e = a.xcd_lo[x] + (b >> 3);
        return e < a.xcd_lo[x + 1] ? e : nelt;
    }
    return remap_element(b, nelt, a.per_xcd);
}

template <int N1, int MAT>
__device__ __forceinline__ void load_coef(const StageArgs &a, int e, int f, int q, double c4[4]) {
    const double *p = (MAT == MAT_ELEM) ? a.fco + ((int64_t)e * 6 + f) * 4
                                        : a.fco + (((int64_t)e * 6 + f) * (N1 * N1) + q) * 4;
    c4[0] = p[0]; c4[1] = p[1]; c4[2] = p[2]; c4[3] = p[3];
}

// MODE: the RK update, the residual alone, or the RK update keeping the
// stage residual (st_r) and the stage-input Drude current (st_J) for the
// adjoint.
// FEAT = 1 compiles the in-stage source, Drude and Lorentz terms, FEAT = 2
// the PML and the incident field as well, FEAT = 3 the graphene sheet too;
// FEAT = 0 leaves them all out, so the plain step carries none of their
// registers or instructions.
// NT: non-temporal k loads and output stores (chosen by the launcher from
// the mesh's size).
// OCC > 0: waves per SIMD the register allocator keeps to.
// SL > 1: an element in SL workgroups, each with a slab of its levels (small
// meshes without a sheet, whose state a face's one workgroup updates; see
// stage_slabs).
template <int N1, int MAT, int MODE, int FEAT, bool NT, int OCC, int SL = 1>
__global__ void __launch_bounds__(BoxShape<N1>::BS) __attribute__((amdgpu_waves_per_eu(OCC > 0 ? OCC : 1)))
box_kernel(StageArgs a) {
    using S = BoxShape<N1>;
    constexpr int RUNS = S::KS * SL;         // runs of levels of an element
    constexpr int N2 = S::N2, N3 = S::N3, KL = (N1 + RUNS - 1) / RUNS, WG = S::WG;
    constexpr bool RK = MODE != MODE_RESIDUAL;
    static_assert(SL == 1 || (FEAT <= 2 && RUNS <= N1), "slabs");
    // N = 9: the misaligned level loads of k measured 507 us plain, 518
    // non-temporal (24^3); every other order 3-4 % faster non-temporal
    constexpr bool NTK = NT && N1 != 10;
    constexpr int FS = FEAT == 3 ? 5 : 4;   // flux components kept per face (a sheet's FE has one along the normal)
    __shared__ double s_u[6 * N3];
    __shared__ double s_f[6 * FS * N2];     // [face][FH t1, FH t2, FE t1, FE t2 (, FE n)][a + n1 b]
    __shared__ double s_D[N2];              // D(i,l) at [i + n1 l]

    // an element's slabs follow each other on its XCD
    const int slab = SL > 1 ? (blockIdx.x >> 3) % SL : 0;
    const int e = stage_element<(FEAT >= 1)>(a, SL > 1 ? (blockIdx.x & 7) + 8 * ((blockIdx.x >> 3) / SL) : blockIdx.x,
                                             a.nelt);
    if (e >= a.nelt) return;
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int grp = w >= WG ? 1 : 0;
    const int wg = w - grp * WG;
    const int rl = t - grp * S::GL;
    // lanes past the last node repeat it, in the same wave: they read what
    // the node's own lane reads, in the same instructions, and write the same
    // values to the same places (no execution masks to keep)
    int part, q;
    if (S::PAD) {
        part = __builtin_amdgcn_readfirstlane(rl / S::PL);
        q = min(rl - part * S::PL, N2 - 1);
    } else {
        const int r2 = min(rl, S::KS * N2 - 1);
        part = r2 / N2;
        q = r2 - part * N2;
    }
    const int j = q / N1, i = q - j * N1;
    constexpr int BASE = N1 / RUNS, REM = N1 % RUNS;
    const int run = slab * S::KS + part;
    const int k0 = run * BASE + (run < REM ? run : REM);
    const int kn = BASE + (run < REM ? 1 : 0);
    const int64_t eo = (int64_t)e * N3, fs = a.fs;
    // the slab's nodes, x0 to x1
    const int ra = slab * S::KS, rb = ra + S::KS;
    const int x0 = SL > 1 ? N2 * (ra * BASE + min(ra, REM)) : 0, x1 = SL > 1 ? N2 * (rb * BASE + min(rb, REM)) : N3;
    constexpr int NX = SL > 1 ? N2 * S::KS * KL : N3;    // at most

    // ---- phase 0: every global load of the element, issued up front ----
    const double *ug = a.uin + 3 * grp * fs + eo;
    double ld[3][S::NLD];
    unsigned ldo[S::NLD];
#pragma unroll
    for (int n = 0; n < S::NLD; ++n) {
        ldo[n] = (unsigned)((wg + WG * n) * 64 + lane);
        if ((n + 1) * WG * 64 > N3) ldo[n] = min(ldo[n], (unsigned)(N3 - 1));
        ldo[n] *= 8;
    }
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int n = 0; n < S::NLD; ++n) ld[c][n] = *at(ug + c * fs, ldo[n]);
    // neighbour traces (a wall reads the element itself, unused), flux
    // coefficients and lift factors of this wave's face chunks
    // PACKF: face nodes back to back over the workgroup's lanes (96 of 128 at N
    // = 3) instead of a face a wave pass (three passes of 16 of 64 lanes, with
    // three sets of traces and coefficients held: 81 VGPRs against 63 with
    // per-node materials; us per stage 3.1e6 nodes 154 -> 142, 1e7 510 -> 474;
    // per element 1e7 396 -> 387, 1e5 7.3 -> 6.8).  From N = 4 on a face fills
    // the better part of a wave and the face stays uniform across it.
    constexpr bool PACKF = N1 == 4;
    constexpr int NF = PACKF ? 1 : S::NF;
    // face and in-face node of the wave's chunk n
    auto face_at = [&](int n, int &fq) {
        if (PACKF) {
            const int x = min(t, 6 * N2 - 1), f = x / N2;
            fq = x - f * N2;
            return f;
        }
        const int id = min(w + 2 * WG * n, 6 * S::FC - 1), f = id / S::FC;
        fq = (id - f * S::FC) * 64 + lane;
        if (N2 % 64 != 0) fq = min(fq, N2 - 1);
        return f;
    };
    double up[NF][4], cf[NF][4], fL[NF];
    int fown[NF], ftype[NF];
    [[maybe_unused]] int64_t fnb[NF];
    // sheet blocks on the own and on the far side, asked for with the traces:
    // at the flux they were another round trip of every element (N = 3, 3.1e6
    // nodes 213 -> 204 us per stage)
    [[maybe_unused]] int sho[NF], shn[NF];
#pragma unroll
    for (int n = 0; n < NF; ++n) {
        int fq;
        const int f = face_at(n, fq), ax = f >> 1, side = f & 1;
        const int fb = fq / N1, fa = fq - fb * N1;
        ftype[n] = a.nbr[e * 6 + f];
        const int M = side ? N1 - 1 : 0;
        const int on = pick3(ax, N1 * fa + N2 * fb, fa + N2 * fb, fa + N1 * fb);
        const int st = pick3(ax, 1, N1, N2);
        const int opp = on + (N1 - 1 - M) * st;
        if (S::SWZ) fown[n] = ax == 0 ? S::idx(M, fa, fb) : ax == 1 ? S::idx(fa, M, fb) : S::idx(fa, fb, M);
        else fown[n] = on + M * st;
        const int64_t po = (int64_t)(ftype[n] >= 0 ? ftype[n] : e) * N3;
        if (FEAT >= 2) fnb[n] = po + opp;
        const double *p1 = a.uin + po + pick3(ax, fs, 2 * fs, (int64_t)0);
        const double *p2 = a.uin + po + pick3(ax, 2 * fs, (int64_t)0, fs);
        up[n][0] = *at(p1, 8u * (unsigned)opp);
        up[n][1] = *at(p2, 8u * (unsigned)opp);
        up[n][2] = *at(p1 + 3 * fs, 8u * (unsigned)opp);
        up[n][3] = *at(p2 + 3 * fs, 8u * (unsigned)opp);
        load_coef<N1, MAT>(a, e, f, fq, cf[n]);
        if (FEAT == 3) {
            sho[n] = a.gr_off ? a.gr_off[e * 6 + f] : -1;
            shn[n] = a.gr_off && ftype[n] >= 0 ? a.gr_off[ftype[n] * 6 + (f ^ 1)] : -1;
        }
        fL[n] = a.geo[(int64_t)e * 9 + 3 + f];
    }
    // this lane's nodes: RK register, inverse materials, source amplitude
    const unsigned node0 = 8u * (unsigned)(k0 * N2 + q);
    auto run_has = [&](int kk) { return REM == 0 || kk < kn; };   // a short run skips its last slot
    // KLATE: the RK register level by level instead of up front, in the
    // instances whose 128 VGPRs it would overflow: a level ahead with a source
    // or a dispersive region at N = 8 (22^3: 351 -> 310 us; at N = 9 the
    // up-front loads are the faster ones, 24^3: 535 against 554), at the level
    // (KHERE) with a PML or an incident wave, where the level ahead would spill
    // more (PML, N = 6 at 24^3 297 -> 264 us, N = 8 at 20^3 327 -> 318, N = 9 at
    // 16^3 328 -> 300; what still spills: N = 6 12 B a lane, 44 with per-node
    // materials, N = 9 28 and 20 B), and in the stages kept for the adjoint at N =
    // 7 and 9, whose stage residual's addresses come on top: up front they
    // spilled 12 to 56 B and were up to 13 per cent slower than the kernel before
    // (2e6 nodes, that kernel / up front / a level ahead / here: N = 7 per node
    // 102 / 115 / 102 / 98, with a Drude region 108 / 116 / 94 / 93, N = 9 per node
    // 156 / 146 / 132 / 126; 8e5: N = 9 per element with a Drude region 46.4 / 50.3
    // / 43.3 / 42.0)
    constexpr bool KHERE = (FEAT >= 2 && N1 >= 7) || (MODE == MODE_RK_STORE && (N1 == 8 || N1 == 10));
    constexpr bool KLATE = KHERE || (N1 == 9 && FEAT == 1);
    double kp[3][KLATE ? 1 : KL];
    const bool rdk = RK && (a.kflags & 1);
    const double *kb = a.kbuf + 3 * grp * fs + eo;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int kk = 0; kk < (KLATE ? 1 : KL); ++kk) kp[c][kk] = 0.0;
    if (rdk && !KHERE) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int kk = 0; kk < (KLATE ? 1 : KL); ++kk)
                if (run_has(kk)) kp[c][kk] = ld_stream<NTK>(at(kb + c * fs, node0, 8 * kk * N2));
    }
    const double *geo = a.geo + (int64_t)e * 9;
    const double sgn = grp ? 1.0 : -1.0;
    const double gx = sgn * geo[0], gy = sgn * geo[1], gz = sgn * geo[2];
    const double dt = a.dt_e ? a.dt_e[e] : a.dt;
    // N = 8 and 9 in whole elements, whose 8-wave workgroups live on 128 VGPRs
    // with three and five levels a lane: what a level alone needs is loaded at the level
    // instead of held from here (MHERE 1/m of per-node materials, SHERE the
    // source's amplitude beside a PML, an incident wave or a sheet), and DRREG
    // the row of D stays in LDS there.  Held, they spilled 20 to 84 B a lane: us
    // per stage, per-node materials at 9.9e5 nodes 44.3 -> 40.1 (2.9e6: 131 ->
    // 123), with a Drude region 55.0 -> 50.3, with a PML 89.8 -> 68.1 (per
    // element 70.0 -> 62.7; 2.9e6: 218 -> 188); N = 8 with a dispersive region and
    // per-node materials, 28 B: 1.25e6 64.8 -> 57.5, 3.0e6 171 -> 156.
    constexpr bool MHERE = MAT == MAT_NODE && (N1 == 10 || (N1 == 9 && FEAT == 1)) && SL == 1;
    double minv[MAT == MAT_NODE && !MHERE ? KL : 1];
    const double *mp = (grp ? a.ieps : a.imu) + eo;
    if (MAT == MAT_ELEM) {
        minv[0] = grp ? a.ieps[e] : a.imu[e];
    } else if (!MHERE) {
#pragma unroll
        for (int kk = 0; kk < KL; ++kk) minv[kk] = run_has(kk) ? *at(mp, node0, 8 * kk * N2) : 0.0;
    }
    const int so = (FEAT >= 1 && grp == 1 && a.src_off) ? a.src_off[e] : -1;
    constexpr bool SHERE = FEAT >= 2 && N1 == 10 && SL == 1;
    [[maybe_unused]] double samp[SHERE ? 1 : KL];
    [[maybe_unused]] const double *sp = a.src_amp + (int64_t)so * N3;
    if constexpr (FEAT >= 1 && !SHERE) {
#pragma unroll
        for (int kk = 0; kk < KL; ++kk) samp[kk] = 0.0;
        if (so >= 0) {
#pragma unroll
            for (int kk = 0; kk < KL; ++kk)
                if (run_has(kk)) samp[kk] = *at(sp, node0, 8 * kk * N2);
        }
    }
    const double sgt = (FEAT >= 1 && so >= 0) ? a.tst[1] : 0.0;   // usersrc time factor
    if (t < N2) s_D[t] = a.D[t];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int n = 0; n < S::NLD; ++n) {
            double *x = s_u + (3 * grp + c) * N3;
            if (S::SWZ) x[(wg + WG * n) * 64 + S::idx(lane % N1, (lane / N1) % N1, lane / N2)] = ld[c][n];
            else *at(x, ldo[n]) = ld[c][n];
        }
    const int imask = (FEAT >= 2 && a.inc_mask) ? a.inc_mask[e] : 0;
    const double tinc = (FEAT >= 2 && imask) ? a.tst[0] : 0.0;
    __syncthreads();

    // dispersive currents: resE -= J bm1 takes the stage-input J of the
    // lane's nodes; the currents' own update follows the levels
    const int dd = (FEAT >= 1 && grp == 1 && a.drude_off) ? a.drude_off[e] : -1;
    const int lo = (FEAT >= 1 && grp == 1 && a.lor_off) ? a.lor_off[e] : -1;
    [[maybe_unused]] const double *dJe = a.dJ + (int64_t)dd * 3 * N3, *lJe = a.lL + (int64_t)lo * 6 * N3;

    // ---- phase 1: each wave takes whole faces (or halves of one) ----
#pragma unroll
    for (int n = 0; n < NF; ++n) {
        if (PACKF ? 64 * w >= 6 * N2 : 6 * S::FC % (2 * WG) != 0 && w + 2 * WG * n >= 6 * S::FC) break;
        int fq;
        const int f = face_at(n, fq), ax = f >> 1, side = f & 1;
        const int t1 = pick3(ax, 1, 2, 0), t2 = pick3(ax, 2, 0, 1);
        const double *s1 = s_u + t1 * N3 + fown[n], *s2 = s_u + t2 * N3 + fown[n];
        double um[4] = {s1[0], s2[0], s1[3 * N3], s2[3 * N3]};
        const double sg = side ? 1.0 : -1.0, L = fL[n];
        if constexpr (FEAT >= 2) {
            // userinc: the wave on the own and on the neighbour's trace
            const double ih[2] = {pick3(ax, a.inc_h[1], a.inc_h[2], a.inc_h[0]), pick3(ax, a.inc_h[2], a.inc_h[0], a.inc_h[1])};
            const double ie[2] = {pick3(ax, a.inc_e[1], a.inc_e[2], a.inc_e[0]), pick3(ax, a.inc_e[2], a.inc_e[0], a.inc_e[1])};
            if ((imask >> f) & 1) {
                const int fb = fq / N1, fa = fq - fb * N1, M = side ? N1 - 1 : 0;
                const int on = pick3(ax, M + N1 * fa + N2 * fb, fa + N1 * M + N2 * fb, fa + N1 * fb + N2 * M);
                const double u = incident(a, eo + on, tinc);
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    um[c] += ih[c] * u;
                    um[2 + c] += ie[c] * u;
                }
            }
            if ((imask >> (8 + f)) & 1) {
                const double u = incident(a, fnb[n], tinc);
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    up[n][c] += ih[c] * u;
                    up[n][2 + c] += ie[c] * u;
                }
            }
        }
        // d: the jumps, n x [.] = sg (-d t2, d t1); no partner: gs leaves
        // -n x E-, -n x H-; PEC doubles E, zeroes H
        double d[4];
        if (ftype[n] >= 0) {
#pragma unroll
            for (int c = 0; c < 4; ++c) d[c] = up[n][c] - um[c];
        } else {
            const double fe = ftype[n] == FACE_PEC ? -2.0 : -1.0, fh = ftype[n] == FACE_PEC ? 0.0 : -1.0;
            d[0] = fh * um[0];
            d[1] = fh * um[1];
            d[2] = fe * um[2];
            d[3] = fe * um[3];
        }
        // cf = (Y02, C02Y, Z02, C02Z): FH = L (Y02 n x [E] - C02Y n x (n x [H])), FE alike
        double *o = s_f + f * FS * N2 + fq;
        const double a0 = sg * cf[n][0], a2 = sg * cf[n][2];
        if constexpr (FEAT == 3) {
            // the sheet adds -(J own + J neighbour), what userfsrc subtracts
            // on each side, to the gathered -n x H (none on a PEC wall); the
            // own side's state advances
            double g[3] = {0.0, 0.0, 0.0}, J[3];
            if (a.gr_off) {
                const int b = sho[n];
                if (b >= 0) {
                    sheet_current<N2>(a, b, fq, ax, t1, t2, sg, um, RK, dt, J);
                    g[0] -= J[0]; g[1] -= J[1]; g[2] -= J[2];
                }
                const int bn = shn[n];
                if (bn >= 0) {
                    sheet_current<N2>(a, bn, fq, ax, t1, t2, -sg, up[n], false, dt, J);
                    g[0] -= J[0]; g[1] -= J[1]; g[2] -= J[2];
                }
                if (ftype[n] == FACE_PEC) g[0] = g[1] = g[2] = 0.0;
            }
            const double sH1 = g[1] - sg * d[1], sH2 = g[2] + sg * d[0];
            o[0] = L * (cf[n][1] * (sg * sH2) - a0 * d[3]);
            o[N2] = L * (a0 * d[2] - cf[n][1] * (sg * sH1));
            o[2 * N2] = L * (cf[n][3] * d[2] + cf[n][2] * sH1);
            o[3 * N2] = L * (cf[n][3] * d[3] + cf[n][2] * sH2);
            o[4 * N2] = L * (cf[n][2] * g[0]);
        } else {
            o[0] = L * (cf[n][1] * d[0] - a0 * d[3]);
            o[N2] = L * (cf[n][1] * d[1] + a0 * d[2]);
            o[2 * N2] = L * (cf[n][3] * d[2] - a2 * d[1]);
            o[3 * N2] = L * (cf[n][3] * d[3] + a2 * d[0]);
        }
    }
    __syncthreads();

    // ---- phase 2: this lane's levels; group 0 updates H from -curl E,
    // group 1 updates E from curl H ----
    const double *S0 = s_u + (grp ? 0 : 3) * N3, *S1 = S0 + N3, *S2 = S1 + N3;
    double *const own = s_u + 3 * grp * N3;
    // residuals of the lane's levels: the t derivatives of every level from
    // one read of the lane's column.  In padded runs the level is the same
    // across the wave: lane l holds D(k, l) and readlane spreads it.
    double R0[KL], R1[KL], R2[KL];
#pragma unroll
    for (int kk = 0; kk < KL; ++kk) R0[kk] = R1[kk] = R2[kk] = 0.0;
    {
        double dk[S::PAD ? KL : 1];
        if constexpr (S::PAD) {
            const int wl = lane < N1 ? lane : 0;
#pragma unroll
            for (int kk = 0; kk < KL; ++kk) dk[kk] = s_D[(run_has(kk) ? k0 + kk : N1 - 1) + N1 * wl];
        }
#pragma unroll
        for (int l = 0; l < N1; ++l) {
            const double v0 = S0[S::idx(i, j, l)], v1 = S1[S::idx(i, j, l)];
#pragma unroll
            for (int kk = 0; kk < KL; ++kk) {
                const double d = S::PAD ? bcast_lane(dk[S::PAD ? kk : 0], l) : s_D[slot_level(N1, RUNS, k0, kn, kk) + N1 * l];
                R0[kk] += d * v1;
                R1[kk] += d * v0;
            }
        }
    }
#pragma unroll
    for (int kk = 0; kk < KL; ++kk) {
        R0[kk] *= -gz;
        R1[kk] *= gz;
    }
    // lifted fluxes: along x and y every level, along z the first and last
    if (i == 0 || i == N1 - 1) {
        const double *fx = s_f + ((i == 0 ? 0 : FS) + 2 * grp) * N2 + j + N1 * k0;
#pragma unroll
        for (int kk = 0; kk < KL; ++kk)
            if (run_has(kk)) {
                R1[kk] += fx[N1 * kk];
                R2[kk] += fx[N2 + N1 * kk];
                if (FEAT == 3 && grp) R0[kk] += fx[2 * N2 + N1 * kk];
            }
    }
    if (j == 0 || j == N1 - 1) {
        const double *fy = s_f + ((j == 0 ? 2 * FS : 3 * FS) + 2 * grp) * N2 + i + N1 * k0;
#pragma unroll
        for (int kk = 0; kk < KL; ++kk)
            if (run_has(kk)) {
                R2[kk] += fy[N1 * kk];
                R0[kk] += fy[N2 + N1 * kk];
                if (FEAT == 3 && grp) R1[kk] += fy[2 * N2 + N1 * kk];
            }
    }
    if (k0 == 0) {
        const double *fz = s_f + (4 * FS + 2 * grp) * N2 + q;
        R0[0] += fz[0];
        R1[0] += fz[N2];
        if (FEAT == 3 && grp) R2[0] += fz[2 * N2];
    }
    if (k0 + kn == N1) {
        const double *fz = s_f + (5 * FS + 2 * grp) * N2 + q;
        constexpr int KE = BASE - 1;     // the last run is a short one
        R0[KE] += fz[0];
        R1[KE] += fz[N2];
        if (FEAT == 3 && grp) R2[KE] += fz[2 * N2];
    }
    if constexpr (FEAT >= 1) {
        // usersrc: resE += amp * bm1 * dir * g(t) before the inverse mass;
        // with a PML after its step, which takes the residual without it
        if (FEAT == 1 && so >= 0) {
#pragma unroll
            for (int kk = 0; kk < KL; ++kk) {
                const double am = samp[SHERE ? 0 : kk] * sgt;
                R0[kk] += am * a.src_dir[0];
                R1[kk] += am * a.src_dir[1];
                R2[kk] += am * a.src_dir[2];
            }
        }
        auto take = [&](const double *Je) {
#pragma unroll
            for (int kk = 0; kk < KL; ++kk)
                if (run_has(kk)) {
                    R0[kk] -= *at(Je, node0, 8 * kk * N2);
                    R1[kk] -= *at(Je + N3, node0, 8 * kk * N2);
                    R2[kk] -= *at(Je + 2 * N3, node0, 8 * kk * N2);
                }
        };
        if (FEAT == 1 && dd >= 0) take(dJe);
        if (FEAT == 1 && lo >= 0) take(lJe);
    }
    // keep the sums here: the compiler would sink them into the levels and
    // hold every value they read instead (N = 8: 172 VGPRs against 112)
#pragma unroll
    for (int kk = 0; kk < KL; ++kk) asm volatile("" : "+v"(R0[kk]), "+v"(R1[kk]), "+v"(R2[kk]));
    const int po = (FEAT >= 2 && a.pml_off) ? a.pml_off[e] : -1;
    // D rows of the lane's column; at N = 9 the s row stays in LDS (its 20
    // VGPRs would spill at two 8-wave workgroups per CU)
    constexpr bool DSREG = N1 < 9 || (N1 == 9 && FEAT <= 1);
    constexpr bool DRREG = !(N1 == 10 && FEAT >= 2 && SL == 1);
    double Dr[DRREG ? N1 : 1], Ds[DSREG ? N1 : 1];
    if constexpr (DRREG) {
#pragma unroll
        for (int l = 0; l < N1; ++l) Dr[l] = s_D[i + N1 * l];
    }
    if constexpr (DSREG) {
#pragma unroll
        for (int l = 0; l < N1; ++l) Ds[l] = s_D[j + N1 * l];
    }
#pragma unroll
    for (int kk = 0; kk < KL; ++kk) {
        if (!run_has(kk)) break;
        const int k = k0 + kk;
        const unsigned vloc = (unsigned)(k * N2 + q);
        if (KHERE && rdk) {
#pragma unroll
            for (int c = 0; c < 3; ++c) kp[c][0] = ld_stream<NTK>(at(kb + c * fs, node0, 8 * kk * N2));
        }
        const double ko[3] = {kp[0][KLATE ? 0 : kk], kp[1][KLATE ? 0 : kk], kp[2][KLATE ? 0 : kk]};
        if (KLATE && !KHERE && rdk && kk + 1 < kn) {
#pragma unroll
            for (int c = 0; c < 3; ++c) kp[c][0] = ld_stream<NTK>(at(kb + c * fs, node0, 8 * (kk + 1) * N2));
        }
        [[maybe_unused]] double pl[3], pk[3], sig[3];
        auto load_aux = [&] {
            const double *sb = a.psig + (int64_t)po * 3 * N3, *pb = a.pP + (int64_t)po * 6 * N3 + 3 * grp * N3;
            const double *qb = a.pkP + (int64_t)po * 6 * N3 + 3 * grp * N3;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                sig[c] = *at(sb, node0, 8 * (c * N3 + kk * N2));
                pl[c] = *at(pb, node0, 8 * (c * N3 + kk * N2));
                pk[c] = RK ? *at(qb, node0, 8 * (c * N3 + kk * N2)) : 0.0;
            }
        };
        // requested before the level's derivatives where the registers hold
        // them (PML, N = 5 at 20^3 107 -> 102 us, N = 7 at 16^3 110 -> 108; at N =
        // 8 they spill, 12^3 69 -> 81)
        constexpr bool PEARLY = FEAT >= 2 && (N1 == 6 || N1 == 8);
        if constexpr (PEARLY) {
            if (po >= 0) load_aux();
        }
        double S1_r = 0, S2_r = 0, S0_s = 0, S2_s = 0;
#pragma unroll
        for (int l = 0; l < N1; ++l) {
            const int pr = S::idx(l, j, k), ps = S::idx(i, l, k);
            const double dsl = DSREG ? Ds[DSREG ? l : 0] : s_D[j + N1 * l];
            const double drl = DRREG ? Dr[DRREG ? l : 0] : s_D[i + N1 * l];
            S1_r += drl * S1[pr];
            S2_r += drl * S2[pr];
            S0_s += dsl * S0[ps];
            S2_s += dsl * S2[ps];
        }
        double r[3];
        r[0] = R0[kk] + gy * S2_s;
        r[1] = R1[kk] - gx * S2_r;
        r[2] = R2[kk] + (gx * S1_r - gy * S0_s);
        const double mi = MHERE ? *at(mp, node0, 8 * kk * N2) : minv[MAT == MAT_NODE && !MHERE ? kk : 0];
        [[maybe_unused]] const double *uo = own + S::idx(i, j, k);   // the group's own fields at this node
        if (FEAT >= 2 && po >= 0) {
            // pml_step: with sa, sb, sd = sigma/eps of the component's own,
            // next and last axis, the auxiliary field P (B for H, D for E)
            //   resP = res - sb P,  res += (sa - sb) P - sd mu H  (H)
            //                       res += (sa - sb) P - sigma_d E (E)
            if constexpr (!PEARLY) load_aux();
            const int64_t pb = (int64_t)po * 6 * N3 + 3 * grp * N3 + vloc;
            const double iep = grp ? mi : (MAT == MAT_NODE) ? (a.ieps + eo)[vloc] : a.ieps[e];
            const double mu = grp ? 0.0 : 1.0 / mi;
            const double sp[3] = {sig[0] * iep, sig[1] * iep, sig[2] * iep};
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int cb = (c + 1) % 3, cd = (c + 2) % 3;
                const double P = pl[c];
                const double rP = r[c] - sp[cb] * P;
                const double drive = grp ? sig[cd] * uo[c * N3] : sp[cd] * mu * uo[c * N3];
                r[c] += -sp[cb] * P + sp[c] * P - drive;
                if (!RK) {
                    a.presP[pb + c * N3] = rP;
                } else {
                    const double kq = a.rka * pk[c] + dt * rP;
                    a.pkP[pb + c * N3] = kq;
                    a.pP[pb + c * N3] = P + a.rkb * kq;
                }
            }
        }
        if (FEAT >= 2) {
            if (so >= 0) {
                const double am = (SHERE ? *at(sp, node0, 8 * kk * N2) : samp[SHERE ? 0 : kk]) * sgt;
#pragma unroll
                for (int c = 0; c < 3; ++c) r[c] += am * a.src_dir[c];
            }
            if (dd >= 0) {
#pragma unroll
                for (int c = 0; c < 3; ++c) r[c] -= *at(dJe + c * N3, node0, 8 * kk * N2);
            }
            if (lo >= 0) {
#pragma unroll
                for (int c = 0; c < 3; ++c) r[c] -= *at(lJe + c * N3, node0, 8 * kk * N2);
            }
        }
        // inverse mass (the J w3 of hbm1/ebm1 is already divided out) and
        // the RK register
        if (!RK || (MODE == MODE_RK_STORE && a.st_r)) {
            double *rp = (RK ? a.st_r : a.res) + 3 * grp * fs + eo;
#pragma unroll
            for (int c = 0; c < 3; ++c) *at(rp + c * fs, node0, 8 * kk * N2) = mi * r[c];
        }
        if (RK) {
            const double s = dt * mi;
#pragma unroll
            for (int c = 0; c < 3; ++c) r[c] = a.rka * ko[c] + s * r[c];
        }
        R0[kk] = r[0];   // RK: the new register
        R1[kk] = r[1];
        R2[kk] = r[2];
        asm volatile("" : "+v"(R0[kk]), "+v"(R1[kk]), "+v"(R2[kk]));
    }
    if constexpr (FEAT >= 1) {
        // cem_maxwell_drude: resJ = -a J + b E; cem_maxwell_lorentz: resJ =
        // -a J - b P + c E, resP = J; the RK update from the stage-start E
        // (still in LDS), in the order of memory: every load of an element
        // at once instead of a round trip per level.  Each node by one lane,
        // once every wave has read the currents its levels take
        if ((a.drude_off && a.drude_off[e] >= 0) || (a.lor_off && a.lor_off[e] >= 0)) __syncthreads();
        constexpr int NLX = SL > 1 ? ((NX + 63) / 64 + WG - 1) / WG : S::NLD;
        auto place = [&](int v) {
            if (SL > 1) return S::idx(v % N1, v / N1 % N1, v / N2);
            return S::SWZ ? (v - lane) + S::idx(lane % N1, (lane / N1) % N1, lane / N2) : v;
        };
        if (dd >= 0) {
            const int64_t jb = (int64_t)dd * 3 * N3;
#pragma unroll
            for (int n = 0; n < NLX; ++n) {
                const int v = x0 + (wg + WG * n) * 64 + lane;
                if (v >= x1) continue;
                const double *uo = own + place(v);
                const double pa = a.dpar[((int64_t)dd * N3 + v) * 2], pb = a.dpar[((int64_t)dd * N3 + v) * 2 + 1];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const int64_t x = jb + c * N3 + v;
                    const double Jc = a.dJ[x];
                    const double rJ = -pa * Jc + pb * uo[c * N3];
                    if (!RK) {
                        a.dresJ[x] = rJ;
                    } else {
                        if (MODE == MODE_RK_STORE) a.st_J[x] = Jc;
                        const double kj = a.rka * a.dkJ[x] + dt * rJ;
                        a.dkJ[x] = kj;
                        a.dJ[x] = Jc + a.rkb * kj;
                    }
                }
            }
        }
        if (lo >= 0) {
            const int64_t lb = (int64_t)lo * 6 * N3;
#pragma unroll
            for (int n = 0; n < NLX; ++n) {
                const int v = x0 + (wg + WG * n) * 64 + lane;
                if (v >= x1) continue;
                const double *uo = own + place(v);
                const double *lp = a.lpar + ((int64_t)lo * N3 + v) * 3;
                const double la = lp[0], lbp = lp[1], lc = lp[2];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const int64_t x = lb + c * N3 + v, y = x + 3 * N3;
                    const double Jc = a.lL[x], Pc = a.lL[y];
                    const double rJ = -la * Jc - lbp * Pc + lc * uo[c * N3];
                    if (!RK) {
                        a.lresL[x] = rJ;
                        a.lresL[y] = Jc;
                    } else {
                        const double kj = a.rka * a.lkL[x] + dt * rJ;
                        const double kp2 = a.rka * a.lkL[y] + dt * Jc;
                        a.lkL[x] = kj;
                        a.lkL[y] = kp2;
                        a.lL[x] = Jc + a.rkb * kj;
                        a.lL[y] = Pc + a.rkb * kp2;
                    }
                }
            }
        }
    }
    if constexpr (RK) {
        // ---- phase 3: the outputs leave in the order of memory, 64-node
        // chunks that start on 128-byte lines, first k, then u ----
        constexpr bool LINE = S::G == 16 && (SL == 1 || (N2 * S::KS * BASE % 16 == 0 && REM == 0));
        constexpr int NST = SL > 1 ? ((NX + (LINE ? 0 : 15) + 63) / 64 + WG - 1) / WG : S::NST;
        const int m = LINE ? 0 : (int)((eo + x0) & 15);
        unsigned sto[NST];
#pragma unroll
        for (int n = 0; n < NST; ++n) {
            int x = x0 + (wg + WG * n) * 64 + lane - m;
            if (!LINE && n == 0) x = max(x, x0);
            if (SL > 1 || (n + 1) * WG * 64 > N3) x = min(x, x1 - 1);
            sto[n] = 8u * (unsigned)x;
        }
        auto flush = [&](double *dst) {
            double *p = dst + 3 * grp * fs + eo;
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int n = 0; n < NST; ++n) {
                    // a chunk past the end (N = 4, and slabs)
                    if (SL > 1 ? x0 + (wg + WG * n) * 64 - m >= x1
                               : S::WG * NST * 64 - N3 >= 64 && (wg + WG * n) * 64 - m >= N3)
                        break;
                    const double *x = own + c * N3;
                    if (SL > 1 && S::SWZ) {
                        const int v = (int)(sto[n] / 8);
                        st_stream<NT>(at(p + c * fs, sto[n]), x[S::idx(v % N1, v / N1 % N1, v / N2)]);
                        continue;
                    }
                    const double v = S::SWZ ? x[(wg + WG * n) * 64 + S::idx(lane % N1, (lane / N1) % N1, lane / N2)] : *at(x, sto[n]);
                    st_stream<NT>(at(p + c * fs, sto[n]), v);
                }
        };
        double un[3][KL];
        __syncthreads();   // every read of the element's fields is done
        auto knew = [&](int c, int kk) { return c == 0 ? R0[kk] : c == 1 ? R1[kk] : R2[kk]; };
#pragma unroll
        for (int kk = 0; kk < KL; ++kk) {
            if (!run_has(kk)) break;
#pragma unroll
            for (int c = 0; c < 3; ++c) un[c][kk] = own[c * N3 + S::idx(i, j, k0 + kk)] + a.rkb * knew(c, kk);
        }
        // MODE_RK: bit 1 of kflags writes k
        if (a.kflags & 2) {
#pragma unroll
            for (int kk = 0; kk < KL; ++kk) {
                if (!run_has(kk)) break;
#pragma unroll
                for (int c = 0; c < 3; ++c) own[c * N3 + S::idx(i, j, k0 + kk)] = knew(c, kk);
            }
            __syncthreads();
            flush(a.kbuf);
            __syncthreads();
        }
#pragma unroll
        for (int kk = 0; kk < KL; ++kk) {
            if (!run_has(kk)) break;
#pragma unroll
            for (int c = 0; c < 3; ++c) own[c * N3 + S::idx(i, j, k0 + kk)] = un[c][kk];
        }
        __syncthreads();
        flush(a.uout);
    }
}

}  // namespace nkc
