// geo_kernel.hpp -- the RK stage on general hexahedra (curved, rotated,
// sheared elements; any conforming face pairing), for gfx950.
//
// The same stage as box_kernel.hpp (cem_maxwell_op + rk_maxwell_ab,
// src/cem_maxwell.F:484-508, 1906-1968), with the geometry per node instead
// of per element: maxwell_wght_curl's full cofactor combine
// (src/cem_maxwell.F:1464-1495) in strong form, curl u = sum_a G_a x du/dr_a
// with G_ab = (cofactor ab)/J, the flux of cem_maxwell_flux3d
// (:922-1002) with each face node's own unit normal and partner (any
// in-face orientation), the lift area/(J w3) of add_flux_to_res and
// invqmass (:654-756, 1833-1904).
//
// Mapping: a workgroup takes an element, or on meshes too small to fill the
// chip a slab of its levels (GeoArgs::nslab slabs per element; every one
// stages the whole element, the r, s, t lines of its nodes).  Half of the
// waves update H, half E (nine derivative sums a lane instead of eighteen:
// 254 -> under 128 VGPRs, twice the workgroups per CU), each lane one node
// after another in the order of memory.
//   0  every load of the element and of the slab's face nodes (geometry,
//      partner traces) up front; the element into LDS;
//   1  the flux of the slab's face nodes into LDS;
//   2  per node: metrics, RK register and inverse material requested first,
//      then the derivatives from LDS, the curl, the lifted fluxes of the
//      faces the node lies on, inverse mass and the low-storage RK update.
// Bound: on small meshes one workgroup's chain of phases (5 x 5 x 2 elements
// at N = 11: 41 -> 12.3 us per stage), on large ones the bytes (10^3
// elements at N = 7, in the Infinity Cache: 36 -> 28 us).
// Up to N = 11 (12^3 nodes: 125 KB of LDS, one workgroup per CU).  Materials
// per node, flux coefficients per face node.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "stage_args.hpp"

namespace nkc {

enum GeoMode : int { GMODE_RK = 0, GMODE_RESIDUAL = 1, GMODE_CURL = 2 };

struct GeoArgs {
    const double *__restrict__ uin;    // 6 fields, stride fs
    double *__restrict__ uout;         // GMODE_RK
    double *__restrict__ kbuf;         // GMODE_RK: RK register in place
    double *__restrict__ res;          // GMODE_RESIDUAL / GMODE_CURL
    const double *__restrict__ D;      // D(i,l) at D[i + n1 l]
    const double *__restrict__ gmet;   // 9 x npts metric quotients (component major)
    const double *__restrict__ bmw;    // npts: bm1 = J w3 (GMODE_CURL)
    const double *__restrict__ fgeo;   // 4 per face node: n_x, n_y, n_z, area/bm1
    const int32_t *__restrict__ fnb;   // per face node: partner volume node / FaceType
    const double *__restrict__ fco;    // 4 per face node: Y02, C02Y, Z02, C02Z
    const double *__restrict__ ieps;   // per node
    const double *__restrict__ imu;
    int64_t fs;
    int64_t npts;
    int32_t nelt;
    int32_t per_xcd;
    int32_t nslab;                     // workgroups per element, each a run of levels
    double rka, rkb, dt;
    int32_t kflags;                    // bit 0 read k, bit 1 write k
};

// Lanes of a workgroup: 16 waves per CU at one (N = 11) or two (N = 8, 9)
// workgroups per CU, 8 at N = 10, whose 100 KB of LDS leave one of 512 lanes,
// and three to four workgroups of four waves below, what their LDS allows.  At
// N = 7 the three 4-wave workgroups on a CU serve meshes whose stages stream
// (nt), two of 8 waves with one face node a lane those in the caches: 6^3
// 10.1 / 9.5 us, 8^3 18.4 / 16.7, 10^3 31.2 / 29.6, 12^3 48.4 / 47.2, 16^3
// 134.9 / 141.5.
constexpr int geo_block(int n1, bool nt) { return n1 >= 12 ? 1024 : n1 >= 9 || (n1 == 8 && !nt) ? 512 : 256; }

// In-element volume index of in-face node q = a + n1 b on the reference's
// face ef0 + 1 (0: y-, 1: x+, 2: y+, 3: x-, 4: z-, 5: z+), skpdat order
// (src/nek5_connect11.F:1483-1528).
template <int N1>
__device__ __forceinline__ int ed_face_node(int ef0, int q) {
    constexpr int N2 = N1 * N1, M = N1 - 1;
    const int a = q % N1, b = q / N1;
    switch (ef0) {
    case 0: return a + N2 * b;
    case 1: return M + N1 * a + N2 * b;
    case 2: return a + N1 * M + N2 * b;
    case 3: return N1 * a + N2 * b;
    case 4: return a + N1 * b;
    default: return a + N1 * b + N2 * M;
    }
}

template <int N1, int MODE, bool NT>
__global__ void __launch_bounds__(geo_block(N1, NT)) __attribute__((amdgpu_waves_per_eu(4)))
geo_stage_kernel(GeoArgs a) {
    constexpr int N2 = N1 * N1, N3 = N2 * N1, BS = geo_block(N1, NT), W = BS / 64, GL = BS / 2, NFN = 6 * N2;
    constexpr int CH = (N3 + 63) / 64, NLD = (6 * CH + W - 1) / W, NFL = (NFN + BS - 1) / BS;
    __shared__ double s_u[6 * N3];
    __shared__ double s_f[6 * NFN];      // [FH 0..2, FE 0..2][face node of the slab]
    __shared__ double s_D[N2];
    // the slabs of an element follow each other on one XCD
    const int slot = blockIdx.x >> 3;
    const int e = (blockIdx.x & 7) * a.per_xcd + slot / a.nslab;
    const int slab = slot % a.nslab;
    if (e >= a.nelt || slot / a.nslab >= a.per_xcd) return;
    const int kb = slab * N1 / a.nslab, ks = (slab + 1) * N1 / a.nslab - kb;   // levels kb .. kb + ks - 1
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int64_t eo = (int64_t)e * N3, fs = a.fs;

    // ---- phase 0 ----
    double ld[NLD];
#pragma unroll
    for (int n = 0; n < NLD; ++n) {
        const int id = min(w + W * n, 6 * CH - 1), f = id / CH;
        const int off = min((id - f * CH) * 64 + lane, N3 - 1);
        ld[n] = (a.uin + f * fs + eo)[(unsigned)off];
    }
    // the slab's face nodes: its rows of the four side faces (reference
    // order y-, x+, y+, x-), then z- and z+ where the slab touches them
    const int side = 4 * N1 * ks, zlo = kb == 0 ? N2 : 0, zhi = kb + ks == N1 ? N2 : 0;
    const int nf = MODE == GMODE_CURL ? 0 : side + zlo + zhi;
    double up[NFL][6], fg[NFL][4], cf[NFL][4];
    int32_t nb[NFL];
    int own[NFL];
    int64_t sl[NFL];
#pragma unroll
    for (int n = 0; n < NFL; ++n) {
        const int x = t + BS * n;
        int ef = 0, q = 0;
        if (x < side) {
            const int row = x / N1;
            ef = (row >= ks) + (row >= 2 * ks) + (row >= 3 * ks);
            q = x - row * N1 + N1 * (kb + row - ef * ks);
        } else if (x < nf) {
            const int z = x - side;
            ef = z < zlo ? 4 : 5;
            q = z < zlo ? z : z - zlo;
        }
        own[n] = ed_face_node<N1>(ef, q);
        sl[n] = ((int64_t)e * 6 + ef) * N2 + q;
        nb[n] = x < nf ? a.fnb[sl[n]] : FACE_NONE;
    }
#pragma unroll
    for (int n = 0; n < NFL; ++n) {
        const bool on = t + BS * n < nf;
#pragma unroll
        for (int c = 0; c < 6; ++c) up[n][c] = nb[n] >= 0 ? a.uin[c * fs + nb[n]] : 0.0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            fg[n][c] = on ? a.fgeo[4 * sl[n] + c] : 0.0;
            cf[n][c] = on ? a.fco[4 * sl[n] + c] : 0.0;
        }
    }
    for (int v = t; v < N2; v += BS) s_D[v] = a.D[v];
#pragma unroll
    for (int n = 0; n < NLD; ++n) {
        const int id = min(w + W * n, 6 * CH - 1), f = id / CH;
        s_u[f * N3 + min((id - f * CH) * 64 + lane, N3 - 1)] = ld[n];
    }
    __syncthreads();

    // ---- phase 1: the flux at the slab's face nodes ----
#pragma unroll
    for (int n = 0; n < NFL; ++n) {
        const int x = t + BS * n;
        if (x >= nf) break;
        const double nv[3] = {fg[n][0], fg[n][1], fg[n][2]};
        const double L = fg[n][3];
        double um[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) um[c] = s_u[c * N3 + own[n]];
        double sE[3], sH[3];
        if (nb[n] >= 0) {
            // n x [E] = (-n x E-) + (-n' x E+), n' = -n
            const double dH[3] = {up[n][0] - um[0], up[n][1] - um[1], up[n][2] - um[2]};
            const double dE[3] = {up[n][3] - um[3], up[n][4] - um[4], up[n][5] - um[5]};
            gcross(nv, dE, sE);
            gcross(nv, dH, sH);
        } else {
            // no partner: gs leaves -n x E-, -n x H-; PEC doubles E, zeroes H
            const double Em[3] = {-um[3], -um[4], -um[5]};
            gcross(nv, Em, sE);
            if (nb[n] == FACE_PEC) {
                sE[0] *= 2.0; sE[1] *= 2.0; sE[2] *= 2.0;
                sH[0] = sH[1] = sH[2] = 0.0;
            } else {
                const double Hm[3] = {-um[0], -um[1], -um[2]};
                gcross(nv, Hm, sH);
            }
        }
        double fu[3], fw[3];
        gcross(nv, sH, fu);
        gcross(nv, sE, fw);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            s_f[c * NFN + x] = L * (cf[n][0] * sE[c] - cf[n][1] * fu[c]);
            s_f[(3 + c) * NFN + x] = L * (cf[n][2] * sH[c] - cf[n][3] * fw[c]);
        }
    }
    if (MODE != GMODE_CURL) __syncthreads();

    // ---- phase 2: this half's fields at the slab's nodes, in the order of
    // memory from the 128-byte line the slab starts in ----
    const int grp = w >= W / 2 ? 1 : 0;
    const int64_t so = eo + kb * N2;                       // the slab's first node
    const int m = (int)(so & 15), nn = ks * N2;
    const double *S0 = s_u + (grp ? 0 : 3) * N3, *S1 = S0 + N3, *S2 = S1 + N3;
    const double sgn = grp ? 1.0 : -1.0;
    const double *mp = (grp ? a.ieps : a.imu) + so;
    for (int v = t - grp * GL - m; v < nn; v += GL) {
        if (v < 0) continue;
        const unsigned uv = (unsigned)v;
        double G[9], ko[3] = {0.0, 0.0, 0.0}, mi = 0.0;
#pragma unroll
        for (int c = 0; c < 9; ++c) G[c] = (a.gmet + c * a.npts + so)[uv];
        if (MODE == GMODE_RK && (a.kflags & 1)) {
#pragma unroll
            for (int c = 0; c < 3; ++c) ko[c] = ld_stream<NT>(a.kbuf + (3 * grp + c) * fs + so + uv);
        }
        if (MODE != GMODE_CURL) mi = mp[uv];
        const int k = kb + v / N2, q = v % N2, j = q / N1, i = q % N1;
        // d/dr, d/ds, d/dt of the other group's three fields
        double dr[3] = {0.0, 0.0, 0.0}, ds[3] = {0.0, 0.0, 0.0}, dt_[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int l = 0; l < N1; ++l) {
            const double di = s_D[i + N1 * l], dj = s_D[j + N1 * l], dk = s_D[k + N1 * l];
            const int pr = l + N1 * j + N2 * k, ps = i + N1 * l + N2 * k, pt = i + N1 * j + N2 * l;
            dr[0] += di * S0[pr]; dr[1] += di * S1[pr]; dr[2] += di * S2[pr];
            ds[0] += dj * S0[ps]; ds[1] += dj * S1[ps]; ds[2] += dj * S2[ps];
            dt_[0] += dk * S0[pt]; dt_[1] += dk * S1[pt]; dt_[2] += dk * S2[pt];
        }
        // gradient component b of field c: dr G[0 + b] + ds G[3 + b] + dt G[6 + b]
        auto dx = [&](int c, int b) { return dr[c] * G[b] + ds[c] * G[3 + b] + dt_[c] * G[6 + b]; };
        double r[3];
        r[0] = sgn * (dx(2, 1) - dx(1, 2));
        r[1] = sgn * (dx(0, 2) - dx(2, 0));
        r[2] = sgn * (dx(1, 0) - dx(0, 1));
        if (MODE == GMODE_CURL) {
            const double wt = a.bmw[so + v];
#pragma unroll
            for (int c = 0; c < 3; ++c) a.res[(3 * grp + c) * fs + so + v] = wt * r[c];
            continue;
        }
        // lifted fluxes of the faces through this node (reference face order)
        const double *fl = s_f + 3 * grp * NFN;
        auto lift = [&](int x) {
#pragma unroll
            for (int c = 0; c < 3; ++c) r[c] += fl[c * NFN + x];
        };
        const int kr = (k - kb) * N1, fr = N1 * ks;
        if (j == 0) lift(kr + i);
        if (i == N1 - 1) lift(fr + kr + j);
        if (j == N1 - 1) lift(2 * fr + kr + i);
        if (i == 0) lift(3 * fr + kr + j);
        if (k == 0) lift(side + q);
        if (k == N1 - 1) lift(side + zlo + q);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const int64_t x = (3 * grp + c) * fs + so;
            r[c] *= mi;
            if (MODE == GMODE_RESIDUAL) {
                (a.res + x)[uv] = r[c];
            } else {
                const double kn = a.rka * ko[c] + a.dt * r[c];
                if (a.kflags & 2) st_stream<NT>(a.kbuf + x + uv, kn);
                st_stream<NT>(a.uout + x + uv, s_u[(3 * grp + c) * N3 + kb * N2 + v] + a.rkb * kn);
            }
        }
    }
}

}  // namespace nkc
