// adjoint_kernel.hpp -- one reversed RK stage of the discrete adjoint.
//
// Forward stage i (box_kernel.hpp): r = P B(u) + P s, k <- a_i k + dt r,
// u <- u + b_i k, with P = diag(1/mu, 1/eps) per node, B the strong-form DG
// operator (volume curl + lifted upwind/central flux) and s the source.
// Reversing it, with lambda the adjoint of u and kappa the adjoint of k:
//   kt = kappa + b_i lambda,  v = P kt
//   lambda <- lambda + dt B^T v          (B^T: Dt-curl + transposed flux/lift)
//   kappa  <- a_i kt
//   g_eps  += dt (d r/d eps)^T kt,  g_mu += dt (d r/d mu)^T kt
// where r depends on eps/mu through P (d r_E/d eps = -r_E/eps) and through
// the impedance averages of the face coefficients (Y = sqrt(eps/mu),
// Z = sqrt(mu/eps), as cem_maxwell_materials forms them, src/cem_maxwell.F:
// 262-325).  The stage input state u and the stage residual r come from the
// forward recompute.  Each face node gathers both halves of the transposed
// flux of its face: its own flux and the neighbour's flux on the shared face,
// so every output has a single owner (no atomics).
//
// The workgroup's shape and phases are the forward stage's (BoxShape):
//   0  lambda, kappa, the stage residual, the gradient and the inverse
//      material in the order of memory, 64-node chunks that start on
//      128-byte lines; v = P kt into LDS, kappa out at once from the same
//      lanes, lambda kept in registers;
//   1  each wave takes whole faces: the transposed flux (four tangential
//      components) and the face's part of the material gradient into LDS;
//   2  per lane a column's run of levels: the transposed curl and the faces;
//   3  the sums through the element's place in LDS back to the lanes that
//      hold lambda and the gradient, and out in whole lines.
//
// What bounds it: HBM.  With the gradients at N = 7, 16^3, a stage moves 0.83
// GB (140 us at the card's four-stream rate) for 0.67 GB of algorithmic
// bytes: the x-face reads of the stage state touch one node per 64-byte row
// and so every line of the element and of its x-neighbours.  Whole-line stores from the lanes that loaded, tangential
// traces, a split of the levels as the stage's and equal-work ranges under a
// Drude region took, per stage with the gradients, N = 4 (28^3) 469 -> 350
// us, N = 5 (24^3) 364 -> 285, N = 6 (20^3) 304 -> 260, N = 7 (16^3) 190 ->
// 165, N = 8 (16^3) 380 -> 280, N = 9 (12^3) 213 -> 155; without them, with a
// Drude region, N = 7 (16^3) 173 -> 118, N = 9 (12^3) 216 -> 110.
#pragma once
#include "box_kernel.hpp"

namespace nkc {

struct AdjArgs {
    const double *__restrict__ lam_in;  // 6 fields, stride fs
    const double *__restrict__ kap_in;
    double *__restrict__ lam_out;
    double *__restrict__ kap_out;
    const double *__restrict__ us;      // stage input state
    const double *__restrict__ rs;      // stage residual (inverse-mass scaled)
    double *__restrict__ geps;          // npts, accumulated
    double *__restrict__ gmu;
    const double *__restrict__ D;
    const double *__restrict__ geo;
    const int32_t *__restrict__ nbr;
    const double *__restrict__ ieps;
    const double *__restrict__ imu;
    int64_t fs;
    int32_t nelt;
    int32_t per_xcd;
    double rka, rkb, dt, C0;
    // Drude region (cem_maxwell_drude): per element offset into the compact
    // per-element blocks (-1: none), per-node (a, b); the adjoint current
    // and its RK register (in place), the stage-input current, and the
    // per-node gradients with respect to a and b (accumulated)
    const int32_t *__restrict__ drude_off;
    const double *__restrict__ dpar;
    double *__restrict__ lamJ;
    double *__restrict__ kapJ;
    const double *__restrict__ stJ;
    double *__restrict__ gA;
    double *__restrict__ gB;
    int32_t xcd_bal;                    // equal-work element ranges, as in StageArgs
    int32_t xcd_lo[9];
};

// Flux coefficients of one side of a face, (Y02, C02Y, Z02, C02Z) =
// (-Y1/(2Y0), C0/(2Y0), Z1/(2Z0), C0/(2Z0)), from hy = 1/(2Y0) and
// hz = 1/(2Z0); the same products the host tables hold.
__device__ __forceinline__ void side_coef(double hy, double hz, double Y1, double Z1, double C0, double c[4]) {
    c[0] = -hy * Y1;
    c[1] = hy * C0;
    c[2] = hz * Z1;
    c[3] = hz * C0;
}

// Gradient of <a, F(coef)> with respect to (Y0, Y1, Z0, Z1) through the
// coefficients above (d(1/(2Y0))/dY0 = -2 hy^2).
__device__ __forceinline__ void coef_bar(double gY02, double gC02Y, double gZ02, double gC02Z,
                                         double hy, double hz, double Y1, double Z1, double C0,
                                         double &Yb0, double &Yb1, double &Zb0, double &Zb1) {
    Yb0 = (gY02 * Y1 - gC02Y * C0) * (2.0 * hy * hy);
    Yb1 = -gY02 * hy;
    Zb0 = -(gZ02 * Z1 + gC02Z * C0) * (2.0 * hz * hz);
    Zb1 = gZ02 * hz;
}

// Transposed flux at one face node of this element (normal sg along the
// face's axis), both halves of the shared face, plus the material gradient's
// factor at the own node.  Every vector is (H t1, H t2, E t1, E t2): a face's
// flux and its transpose have no component along the normal, and n x (v1, v2)
// = sg (-v2, v1).
//   vo: own v = P kt; vn: the neighbour's at the paired node (interior faces)
//   d: the jumps the stage's flux saw (PEC: E doubled, H zero; no partner:
//      minus the own traces)
//   L, Ln: own / neighbour lift factors
//   Yo, Zo, Yn, Zn: own and neighbour admittance and impedance
// The flux coefficients are formed here from the admittances/impedances as
// cem_maxwell_materials averages them (src/cem_maxwell.F:262-325): interior
// Y0 = (Y- + Y+)/2, Y1 = Y+; PEC Y0 = Y1 = Y-; no partner Y0 = Y-/2, Y1 = 0.
// Out: adj added to B^T v at the own node; dq with g_eps = dq/eps, g_mu =
// -dq/mu (Y = sqrt(eps/mu), Z = sqrt(mu/eps): dY/deps = Y/(2 eps), dZ/deps =
// -Z/(2 eps)).
template <bool GM>
__device__ __forceinline__ void adj_face(double sg, int type, const double vo[4], const double vn[4],
                                         const double d[4], double L, double Ln, double C0,
                                         double Yo, double Zo, double Yn, double Zn, double adj[4], double &dq) {
    double Ys, Zs;                       // twice the averages
    if (type >= 0) { Ys = Yo + Yn; Zs = Zo + Zn; }
    else if (type == FACE_PEC) { Ys = 2.0 * Yo; Zs = 2.0 * Zo; }
    else { Ys = Yo; Zs = Zo; }
    const double hy = 0.5 / (0.5 * Ys), hz = 0.5 / (0.5 * Zs);
    double cf[4], cfn[4];
    side_coef(hy, hz, Ys - Yo, Zs - Zo, C0, cf);
    double av[4], bv[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) { av[c] = L * vo[c]; bv[c] = Ln * vn[c]; }
    // own half: F_H = Y02 sE - C02Y n x sH, F_E = Z02 sH - C02Z n x sE, sE = n x d_E, sH = n x d_H
    if (type == FACE_PEC) {
        adj[0] = 0.0;
        adj[1] = 0.0;
        adj[2] = -2.0 * cf[0] * (sg * av[1]) - 2.0 * cf[3] * av[2];
        adj[3] = 2.0 * cf[0] * (sg * av[0]) - 2.0 * cf[3] * av[3];
    } else {
        // the own traces enter the jumps with a minus sign
        adj[0] = -cf[1] * av[0] - cf[2] * (sg * av[3]);
        adj[1] = -cf[1] * av[1] + cf[2] * (sg * av[2]);
        adj[2] = -cf[0] * (sg * av[1]) - cf[3] * av[2];
        adj[3] = cf[0] * (sg * av[0]) - cf[3] * av[3];
    }
    if (type >= 0) {
        // neighbour half: its normal is -n, its jump vectors equal ours
        side_coef(hy, hz, Ys - Yn, Zs - Zn, C0, cfn);
        adj[0] += cfn[1] * bv[0] - cfn[2] * (sg * bv[3]);
        adj[1] += cfn[1] * bv[1] + cfn[2] * (sg * bv[2]);
        adj[2] += cfn[3] * bv[2] - cfn[0] * (sg * bv[1]);
        adj[3] += cfn[3] * bv[3] + cfn[0] * (sg * bv[0]);
    }
    if constexpr (GM) {
        const double sE[2] = {-sg * d[3], sg * d[2]}, sH[2] = {-sg * d[1], sg * d[0]};
        double Yb0, Yb1, Zb0, Zb1, dY, dZ;
        const double Y1 = type >= 0 ? Ys - Yo : type == FACE_PEC ? Yo : 0.0;
        const double Z1 = type >= 0 ? Zs - Zo : type == FACE_PEC ? Zo : 0.0;
        coef_bar(av[0] * sE[0] + av[1] * sE[1], av[0] * d[0] + av[1] * d[1], av[2] * sH[0] + av[3] * sH[1],
                 av[2] * d[2] + av[3] * d[3], hy, hz, Y1, Z1, C0, Yb0, Yb1, Zb0, Zb1);
        if (type == FACE_PEC) {
            dY = Yb0 + Yb1;
            dZ = Zb0 + Zb1;
        } else {
            dY = 0.5 * Yb0;
            dZ = 0.5 * Zb0;
        }
        if (type >= 0) {
            coef_bar(bv[0] * sE[0] + bv[1] * sE[1], -(bv[0] * d[0] + bv[1] * d[1]), bv[2] * sH[0] + bv[3] * sH[1],
                     -(bv[2] * d[2] + bv[3] * d[3]), hy, hz, Ys - Yn, Zs - Zn, C0, Yb0, Yb1, Zb0, Zb1);
            dY += 0.5 * Yb0 + Yb1;
            dZ += 0.5 * Zb0 + Zb1;
        }
        dq = 0.5 * (dY * Yo - dZ * Zo);
    }
}

// Waves per SIMD the register allocator keeps to (0: free), as box_waves.
// At N = 7 with the gradients 128 VGPRs would spill 50 bytes a lane, which
// costs more than the fourth workgroup on a CU gives (16^3: 180 us a stage
// against 162); at N = 8 and 9 168 VGPRs would leave one 8-wave workgroup.
constexpr int adjoint_waves(int n1, bool gm) { return n1 < 7 ? 0 : (n1 == 8 && gm) ? 3 : 4; }

// GM: also the eps/mu gradients (needs the stage residual); otherwise the
// adjoint state and the Drude gradients only (no residual store is read).
// NT: non-temporal residual loads and output stores.
template <int N1, int MAT, bool GM, bool NT>
__global__ void __launch_bounds__(BoxShape<N1>::BS)
    __attribute__((amdgpu_waves_per_eu(adjoint_waves(N1, GM) ? adjoint_waves(N1, GM) : 1)))
adjoint_kernel(AdjArgs a) {
    using S = BoxShape<N1>;
    constexpr int N2 = S::N2, N3 = S::N3, KL = S::KL, WG = S::WG;
    constexpr int FS = GM ? 5 : 4;          // per face: H t1, H t2, E t1, E t2 (, dq)
    __shared__ double s_v[6 * N3];          // v = P kt, then the sums of phase 2
    __shared__ double s_f[6 * FS * N2];     // [face][component][a + n1 b]
    __shared__ double s_D[N2];              // D(l,i) at [i + n1 l]

    const int e = stage_element<true>(a, blockIdx.x, a.nelt);
    if (e >= a.nelt) return;
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int grp = w >= WG ? 1 : 0;        // 0: H fields, 1: E fields
    const int wg = w - grp * WG;
    const int rl = t - grp * S::GL;
    // lanes past the last node repeat it, in the same wave (see box_kernel)
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
    constexpr int BASE = N1 / S::KS, REM = N1 % S::KS;
    static_assert(S::PAD || REM == 0, "a short run's last slot would read a row of D past the table");
    const int k0 = part * BASE + (part < REM ? part : REM);
    const int kn = BASE + (part < REM ? 1 : 0);
    auto run_has = [&](int kk) { return REM == 0 || kk < kn; };
    const int64_t eo = (int64_t)e * N3, fs = a.fs;
    if (t < N2) s_D[t % N1 * N1 + t / N1] = a.D[t];

    // ---- phase 0: this wave's chunks of its group's fields ----
    const int m = S::G == 16 ? 0 : (int)(eo & 15);
    unsigned sto[S::NST];
#pragma unroll
    for (int n = 0; n < S::NST; ++n) {
        int x = (wg + WG * n) * 64 + lane - m;
        if (S::G != 16 && n == 0) x = max(x, 0);
        if ((n + 1) * WG * 64 > N3) x = min(x, N3 - 1);
        sto[n] = 8u * (unsigned)x;
    }
    // offsets zero-extended where they are used, so that the addresses stay
    // a scalar base and 32 bits
    auto here = [&] {
#pragma unroll
        for (int n = 0; n < S::NST; ++n) asm volatile("" : "+v"(sto[n]));
    };
    here();
    // a chunk past the element's end (N = 4 only)
    auto past = [&](int n) { return S::WG * S::NST * 64 - N3 >= 64 && (wg + WG * n) * 64 - m >= N3; };
    // chunk n's place in an LDS field
    auto place = [&](double *f, int n) -> double * {
        return S::SWZ ? f + (wg + WG * n) * 64 + S::idx(lane % N1, (lane / N1) % N1, lane / N2) : at(f, sto[n]);
    };
    double *const own = s_v + 3 * grp * N3;
    const int64_t go = 3 * grp * fs + eo;
    // neighbour traces of this wave's faces (a wall reads the element
    // itself, unused): v = P kt, the stage's jumps, the materials
    double vn[S::NF][4], fd[S::NF][4], fm[S::NF][2], fL[S::NF][2], fk[S::NF][4], fl[S::NF][4], fi[S::NF][2];
    [[maybe_unused]] double fo[S::NF][4], fn[S::NF][4];
    int fown[S::NF], ftype[S::NF];
    auto load_face = [&](int n) {
        const int id = min(w + 2 * WG * n, 6 * S::FC - 1), f = id / S::FC;
        const int ax = f >> 1, side = f & 1;
        int fq = (id - f * S::FC) * 64 + lane;
        if (N2 % 64 != 0) fq = min(fq, N2 - 1);
        const int fb = fq / N1, fa = fq - fb * N1;
        ftype[n] = a.nbr[e * 6 + f];
        const int M = side ? N1 - 1 : 0;
        const int on = pick3(ax, N1 * fa + N2 * fb, fa + N2 * fb, fa + N1 * fb);
        const int st = pick3(ax, 1, N1, N2);
        const unsigned opp = 8u * (unsigned)(on + (N1 - 1 - M) * st), mine = 8u * (unsigned)(on + M * st);
        if (S::SWZ) fown[n] = ax == 0 ? S::idx(M, fa, fb) : ax == 1 ? S::idx(fa, M, fb) : S::idx(fa, fb, M);
        else fown[n] = on + M * st;
        const int ne = ftype[n] >= 0 ? ftype[n] : e;
        const int64_t po = (int64_t)ne * N3;
        const int64_t c1 = pick3(ax, fs, 2 * fs, (int64_t)0), c2 = pick3(ax, 2 * fs, (int64_t)0, fs);
        const int64_t off[4] = {c1, c2, c1 + 3 * fs, c2 + 3 * fs};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            fk[n][c] = *at(a.kap_in + po + off[c], opp);
            fl[n][c] = *at(a.lam_in + po + off[c], opp);
            if constexpr (GM) {
                fo[n][c] = *at(a.us + eo + off[c], mine);
                fn[n][c] = *at(a.us + po + off[c], opp);
            }
        }
        if (MAT == MAT_ELEM) {
            fi[n][0] = a.imu[ne];
            fi[n][1] = a.ieps[ne];
            fm[n][0] = a.imu[e];
            fm[n][1] = a.ieps[e];
        } else {
            fi[n][0] = *at(a.imu + po, opp);
            fi[n][1] = *at(a.ieps + po, opp);
            fm[n][0] = *at(a.imu + eo, mine);
            fm[n][1] = *at(a.ieps + eo, mine);
        }
        fL[n][0] = a.geo[(int64_t)e * 9 + 3 + f];
        fL[n][1] = a.geo[(int64_t)ne * 9 + 3 + (f ^ 1)];
    };
    // a face's loads reduced to what its flux needs
    auto settle = [&](int n) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            vn[n][c] = fi[n][c < 2 ? 0 : 1] * (fk[n][c] + a.rkb * fl[n][c]);
            fd[n][c] = 0.0;
            if constexpr (GM) {
                const double wall = ftype[n] == FACE_PEC ? (c < 2 ? 0.0 : -2.0) : -1.0;
                fd[n][c] = ftype[n] >= 0 ? fn[n][c] - fo[n][c] : wall * fo[n][c];
                asm volatile("" : "+v"(vn[n][c]), "+v"(fd[n][c]));
            }
        }
    };
    // what the registers hold: the first face's loads in flight with the
    // chunks' (N = 7 with the gradients: 180 -> 162 us), one face's loads at a
    // time, lambda from its load to the update (read again at N = 9 with the
    // gradients, 12^3: 165 -> 150 us)
    constexpr bool EARLY = GM == (N1 == 8), ONE = GM && N1 != 8, HOLD = !(GM && N1 == 10);

    // kept to the end: lambda and, with GM, kt.r
    double lm[3][S::NST];
    [[maybe_unused]] double kr[GM ? S::NST : 1];
    const double *const mp = (grp ? a.ieps : a.imu);
    double *const g = (grp ? a.geps : a.gmu) + eo;
    {
        double kt[3][S::NST], pm[S::NST];
        [[maybe_unused]] double rr[3][GM ? S::NST : 1];
#pragma unroll
        for (int n = 0; n < S::NST; ++n) pm[n] = MAT == MAT_ELEM ? mp[e] : *at(mp + eo, sto[n]);
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int n = 0; n < S::NST; ++n) {
                lm[c][n] = *at(a.lam_in + go + c * fs, sto[n]);
                kt[c][n] = *at(a.kap_in + go + c * fs, sto[n]);
                if constexpr (GM) rr[c][n] = ld_stream<NT>(at(a.rs + go + c * fs, sto[n]));
            }
        if (EARLY) load_face(0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < S::NST; ++n) {
            if constexpr (GM) kr[n] = 0.0;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                kt[c][n] = kt[c][n] + a.rkb * lm[c][n];
                if constexpr (GM) kr[n] += kt[c][n] * rr[c][n];
                *place(own + c * N3, n) = pm[n] * kt[c][n];
            }
            // summed here, not where it is used with every value it reads held until then
            if constexpr (GM) asm volatile("" : "+v"(kr[n]));
        }
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int n = 0; n < S::NST; ++n)
                if (!past(n)) st_stream<NT>(at(a.kap_out + go + c * fs, sto[n]), a.rka * kt[c][n]);
    }
    // the other faces behind the chunks'
    if (!EARLY) {
        __builtin_amdgcn_sched_barrier(0);
        load_face(0);
    }
    if (ONE) settle(0);
#pragma unroll
    for (int n = 1; n < S::NF; ++n) {
        __builtin_amdgcn_sched_barrier(0);
        load_face(n);
        if (ONE) settle(n);
    }
    if constexpr (!ONE) {
#pragma unroll
        for (int n = 0; n < S::NF; ++n) settle(n);
    }
    __syncthreads();

    // ---- phase 1: each wave takes whole faces (or halves of one) ----
#pragma unroll
    for (int n = 0; n < S::NF; ++n) {
        const int id = w + 2 * WG * n, f = id / S::FC;
        if (6 * S::FC % (2 * WG) != 0 && id >= 6 * S::FC) break;
        const int ax = f >> 1;
        int fq = (id - f * S::FC) * 64 + lane;
        if (N2 % 64 != 0) fq = min(fq, N2 - 1);
        const double *s1 = s_v + pick3(ax, 1, 2, 0) * N3 + fown[n], *s2 = s_v + pick3(ax, 2, 0, 1) * N3 + fown[n];
        const double vo[4] = {s1[0], s2[0], s1[3 * N3], s2[3 * N3]};
        double adj[4], dq = 0.0;
        // admittance and impedance of both sides from 1/mu and 1/eps (a table
        // of the pairs read here: 0.90 GB a stage at 16^3, N = 7, instead of
        // 0.83, 172-182 us against 162-169)
        const double Yo = sqrt(fm[n][0] / fm[n][1]), Zo = sqrt(fm[n][1] / fm[n][0]);
        const double Yn = sqrt(fi[n][0] / fi[n][1]), Zn = sqrt(fi[n][1] / fi[n][0]);
        adj_face<GM>(f & 1 ? 1.0 : -1.0, ftype[n], vo, vn[n], fd[n], fL[n][0], fL[n][1], a.C0, Yo, Zo, Yn, Zn, adj, dq);
        double *o = s_f + f * FS * N2 + fq;
#pragma unroll
        for (int c = 0; c < 4; ++c) o[c * N2] = adj[c];
        if constexpr (GM) o[4 * N2] = dq;
    }
    __syncthreads();

    // ---- phase 2: this lane's levels, the transposed curl: sums over l
    // with D(l, .) of the other group's v ----
    const double *geo = a.geo + (int64_t)e * 9;
    const double sgn = grp ? 1.0 : -1.0;
    const double gx = sgn * geo[0], gy = sgn * geo[1], gz = sgn * geo[2];
    const double *S0 = s_v + (grp ? 0 : 3) * N3, *S1 = S0 + N3, *S2 = S1 + N3;
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
                const double d = S::PAD ? bcast_lane(dk[S::PAD ? kk : 0], l) : s_D[k0 + kk + N1 * l];
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
    // the faces: along x and y every level, along z the first and last
    if (i == 0 || i == N1 - 1) {
        const double *fx = s_f + (i == 0 ? 0 : FS) * N2 + j + N1 * k0;
#pragma unroll
        for (int kk = 0; kk < KL; ++kk)
            if (run_has(kk)) {
                R1[kk] += fx[2 * grp * N2 + N1 * kk];
                R2[kk] += fx[(2 * grp + 1) * N2 + N1 * kk];
            }
    }
    if (j == 0 || j == N1 - 1) {
        const double *fy2 = s_f + (j == 0 ? 2 * FS : 3 * FS) * N2 + i + N1 * k0;
#pragma unroll
        for (int kk = 0; kk < KL; ++kk)
            if (run_has(kk)) {
                R2[kk] += fy2[2 * grp * N2 + N1 * kk];
                R0[kk] += fy2[(2 * grp + 1) * N2 + N1 * kk];
            }
    }
    if (k0 == 0) {
        const double *fz = s_f + 4 * FS * N2 + q;
        R0[0] += fz[2 * grp * N2];
        R1[0] += fz[(2 * grp + 1) * N2];
    }
    if (k0 + kn == N1) {
        const double *fz = s_f + 5 * FS * N2 + q;
        constexpr int KE = BASE - 1;     // the last run is a short one
        R0[KE] += fz[2 * grp * N2];
        R1[KE] += fz[(2 * grp + 1) * N2];
    }
    // keep the sums here (see box_kernel)
#pragma unroll
    for (int kk = 0; kk < KL; ++kk) {
        asm volatile("" : "+v"(R0[kk]), "+v"(R1[kk]), "+v"(R2[kk]));
    }
    constexpr bool DSREG = N1 < 10;
    double Dr[N1], Ds[DSREG ? N1 : 1];
#pragma unroll
    for (int l = 0; l < N1; ++l) Dr[l] = s_D[i + N1 * l];
    if constexpr (DSREG) {
#pragma unroll
        for (int l = 0; l < N1; ++l) Ds[l] = s_D[j + N1 * l];
    }
#pragma unroll
    for (int kk = 0; kk < KL; ++kk) {
        if (!run_has(kk)) break;
        const int k = k0 + kk;
        double S1_r = 0, S2_r = 0, S0_s = 0, S2_s = 0;
#pragma unroll
        for (int l = 0; l < N1; ++l) {
            const int pr = S::idx(l, j, k), ps = S::idx(i, l, k);
            const double dsl = DSREG ? Ds[DSREG ? l : 0] : s_D[j + N1 * l];
            S1_r += Dr[l] * S1[pr];
            S2_r += Dr[l] * S2[pr];
            S0_s += dsl * S0[ps];
            S2_s += dsl * S2[ps];
        }
        R0[kk] += gy * S2_s;
        R1[kk] -= gx * S2_r;
        R2[kk] += gx * S1_r - gy * S0_s;
        asm volatile("" : "+v"(R0[kk]), "+v"(R1[kk]), "+v"(R2[kk]));
    }
    if constexpr (!HOLD) {
        here();
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int n = 0; n < S::NST; ++n) lm[c][n] = *at(a.lam_in + go + c * fs, sto[n]);
    }
    if (grp == 1 && a.drude_off) {
        // r_J = -a J + b E, r_E -= J/eps: lambda_E += dt b ktJ,
        // lambda_J += dt (-v_E - a ktJ), kappa_J = a_i ktJ;
        // d/da = -ktJ.J, d/db = ktJ.E at the stage input.  In place: the
        // lanes that repeat a node read it in the same instruction as its own
        // lane, which alone writes
        const int dd = a.drude_off[e];
        if (dd >= 0) {
            here();
            double *const lJ = a.lamJ + (int64_t)dd * 3 * N3, *const kJ = a.kapJ + (int64_t)dd * 3 * N3;
            const double *const sJ = a.stJ + (int64_t)dd * 3 * N3, *const uE = a.us + 3 * fs + eo;
            double *const gA = a.gA + (int64_t)dd * N3, *const gB = a.gB + (int64_t)dd * N3;
#pragma unroll
            for (int n = 0; n < S::NST; ++n) {
                if (past(n)) break;
                const bool mine = (wg + WG * n) * 64 + lane - m == (int)(sto[n] / 8);
                const double2 ab = *reinterpret_cast<const double2 *>(at(a.dpar + (int64_t)dd * 2 * N3, 2 * sto[n]));
                double lj[3], kt[3], tA = 0.0, tB = 0.0;
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    lj[c] = *at(lJ, sto[n], 8 * c * N3);
                    kt[c] = *at(kJ, sto[n], 8 * c * N3) + a.rkb * lj[c];
                    tA += kt[c] * *at(sJ, sto[n], 8 * c * N3);
                    tB += kt[c] * *at(uE + c * fs, sto[n]);
                }
                const double ga = *at(gA, sto[n]) - a.dt * tA, gbn = *at(gB, sto[n]) + a.dt * tB;
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    lm[c][n] += a.dt * (ab.y * kt[c]);
                    lj[c] += a.dt * (-*place(own + c * N3, n) - ab.x * kt[c]);
                }
                if (mine) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        *at(lJ, sto[n], 8 * c * N3) = lj[c];
                        *at(kJ, sto[n], 8 * c * N3) = a.rka * kt[c];
                    }
                    *at(gA, sto[n]) = ga;
                    *at(gB, sto[n]) = gbn;
                }
            }
        }
    }

    // ---- phase 3 ----
    __syncthreads();   // every read of v is done
#pragma unroll
    for (int kk = 0; kk < KL; ++kk) {
        if (!run_has(kk)) break;
        const int x = S::idx(i, j, k0 + kk);
        own[x] = R0[kk];
        own[N3 + x] = R1[kk];
        own[2 * N3 + x] = R2[kk];
    }
    __syncthreads();
    here();
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int n = 0; n < S::NST; ++n)
            if (!past(n)) st_stream<NT>(at(a.lam_out + go + c * fs, sto[n]), lm[c][n] + a.dt * *place(own + c * N3, n));
    if constexpr (GM) {
        // g_m = dt/m (+- dq of the node's faces - kt.r), dq from LDS
        double gv[S::NST], pm[S::NST];
#pragma unroll
        for (int n = 0; n < S::NST; ++n) {
            gv[n] = *at(g, sto[n]);
            pm[n] = MAT == MAT_ELEM ? mp[e] : *at(mp + eo, sto[n]);
        }
#pragma unroll
        for (int n = 0; n < S::NST; ++n) {
            const int v = (int)(sto[n] / 8), vk = v / N2, vj = v / N1 - N1 * vk, vi = v - N1 * (v / N1);
            const double *f = s_f + 4 * N2;
            double dq = 0.0;
            if (vi == 0 || vi == N1 - 1) dq += f[(vi ? FS : 0) * N2 + vj + N1 * vk];
            if (vj == 0 || vj == N1 - 1) dq += f[(vj ? 3 * FS : 2 * FS) * N2 + vi + N1 * vk];
            if (vk == 0 || vk == N1 - 1) dq += f[(vk ? 5 * FS : 4 * FS) * N2 + vi + N1 * vj];
            if (!past(n)) *at(g, sto[n]) = gv[n] + a.dt * pm[n] * ((grp ? dq : -dq) - kr[n]);
        }
    }
}

}  // namespace nkc
