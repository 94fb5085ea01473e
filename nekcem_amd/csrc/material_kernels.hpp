// material_kernels.hpp -- the material tables of a mesh from per-node
// permittivity and permeability, and the fields at a list of nodes.
//
// An optimisation replaces the materials before every pass.  The tables were
// formed on one host core from a host copy of the parameters and uploaded
// (16^3, N = 7: 46 ms, of a pass of 165 ms); here one lane forms the
// coefficients of one face node, whose 32 bytes are stored side by side, and
// the neighbour's material comes from L2 (1.4 ms for the whole call, nearly
// all of it the copy of the parameters).  Every value is the one the host
// formed: the same IEEE divisions and square roots in the same order.
// Probe losses read and seed a few nodes: their fields are gathered and
// their seeds added here, where whole states went through host memory (20 ms
// and 20 ms of the same pass; 0.1 ms each now).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace nkc {

// Smallest node of a workgroup's share whose eps or mu is not positive (NaN
// included), or ~0, into out[blockIdx.x] (pinned host memory).
__global__ void bad_material(const double *__restrict__ eps, const double *__restrict__ mu, int64_t npts,
                             unsigned long long *out) {
    __shared__ unsigned long long sm;
    if (threadIdx.x == 0) sm = ~0ull;
    __syncthreads();
    unsigned long long bad = ~0ull;
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < npts; p += (int64_t)gridDim.x * blockDim.x)
        if ((!(eps[p] > 0.0) || !(mu[p] > 0.0)) && bad == ~0ull) bad = (unsigned long long)p;
    if (bad != ~0ull) atomicMin(&sm, bad);
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = sm;
}

// In-element node of face kf (faces in mesh order: x-, x+, y-, y+, z-, z+)
// under face coordinate q.
__device__ __forceinline__ int face_volume_node(int n1, int kf, int q) {
    const int a = q % n1, b = q / n1, n2 = n1 * n1, far = (kf & 1) ? n1 - 1 : 0;
    return kf < 2 ? far + n1 * a + n2 * b : kf < 4 ? a + n1 * far + n2 * b : a + n1 * b + n2 * far;
}

// The four flux coefficients of every face node, as cem_maxwell_materials
// averages the impedances (src/cem_maxwell.F:262-325): the gs sum with the
// partner's, PEC doubled, alone otherwise; Z_1 = Z_0' - Z-, Z_0 = Z_0'/2.
__global__ void face_coefs(const double *__restrict__ eps, const double *__restrict__ mu,
                           const int32_t *__restrict__ nbr, int n1, int64_t nelt, int pec, double C0,
                           double *__restrict__ fco) {
    const int n2 = n1 * n1, n3 = n2 * n1;
    const int64_t n = nelt * 6 * n2;
    for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < n; s += (int64_t)gridDim.x * blockDim.x) {
        const int64_t f = s / n2, e = f / 6;
        const int q = (int)(s - f * n2), kf = (int)(f - e * 6);
        const int32_t nb = nbr[f];
        const int64_t v = e * n3 + face_volume_node(n1, kf, q);
        const double Zm = sqrt(mu[v] / eps[v]), Ym = sqrt(eps[v] / mu[v]);
        double Z0 = Zm, Y0 = Ym;
        if (nb >= 0) {
            const int64_t w = (int64_t)nb * n3 + face_volume_node(n1, kf ^ 1, q);
            Z0 += sqrt(mu[w] / eps[w]);
            Y0 += sqrt(eps[w] / mu[w]);
        } else if (nb == pec) {
            Z0 *= 2.0;
            Y0 *= 2.0;
        }
        const double Y1 = Y0 - Ym, Z1 = Z0 - Zm, hy = 0.5 / (0.5 * Y0), hz = 0.5 / (0.5 * Z0);
        double2 *c = reinterpret_cast<double2 *>(fco + 4 * s);
        c[0] = make_double2(-hy * Y1, hy * C0);
        c[1] = make_double2(hz * Z1, hz * C0);
    }
}

// eps, mu -> 1/eps, 1/mu in place.
__global__ void invert_pair(double *__restrict__ a, double *__restrict__ b, int64_t n) {
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
        a[p] = 1.0 / a[p];
        b[p] = 1.0 / b[p];
    }
}

// The six fields at n listed nodes, out[6][n].
__global__ void gather_nodes(const double *__restrict__ u, int64_t fs, const int64_t *__restrict__ node, int64_t n,
                             double *__restrict__ out) {
    const int c = blockIdx.y;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        out[c * n + i] = u[c * fs + node[i]];
}

// in[6][n] added to the six fields at n listed nodes.
__global__ void scatter_nodes(double *__restrict__ u, int64_t fs, const int64_t *__restrict__ node, int64_t n,
                              const double *__restrict__ in) {
    const int c = blockIdx.y;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        atomicAdd(u + c * fs + node[i], in[c * n + i]);
}

}  // namespace nkc
