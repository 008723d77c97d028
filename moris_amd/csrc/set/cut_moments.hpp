// cut_moments.hpp -- moments of the linear (HEX8 / QUAD4) cells, shared by the lattice and the generic
// element kernels, and the wavefront reductions of the moment kernels.
//
// The moment integrand of a box cell, dN_a/dx_i dN_b/dx_j with N_a = prod_d l_{a_d}(x_d), l_0 = (1 - x) / 2,
// l_1 = (1 + x) / 2, is a quadratic in each axis, so its sum over a cut cell's integration points (TET_11 /
// TRI_7 on the sub-cells, w* = w detJ, points with detJ < -1e-6 skipped, cl_FEM_Element_Bulk.cpp:258-355) is
// a fixed function of the cell's 3^DIM moments
//   m[x][y](z) = sum_ip w* p_x p_y (p_z),   p_0 = l_0^2, p_1 = l_0 l_1, p_2 = l_1^2.
// Every entry is a sum of such moments with one sign (l_a l_b = p_{a+b}, l_a = p_a + p_{a+1}, 1 = p_0 + 2 p_1 +
// p_2), so that no entry, however small, loses digits to cancellation between moments.
#pragma once
#include <hip/hip_runtime.h>

#include "set_device.hpp"

namespace mgpu {

// a + b over the two halves of the wavefront (SWAP 32) or of each half (16): lanes of the first get the
// sum of a, lanes of the second that of b
template <int SWAP>
__device__ __forceinline__ double swap_add(double a, double b) {
    const uint64_t ua = __double_as_longlong(a), ub = __double_as_longlong(b);
    uint32_t r[4];
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const uint32_t x = (uint32_t)(ua >> (32 * w)), y = (uint32_t)(ub >> (32 * w));
        const auto s = SWAP == 32 ? __builtin_amdgcn_permlane32_swap(x, y, false, false)
                                  : __builtin_amdgcn_permlane16_swap(x, y, false, false);
        r[w] = s[0];
        r[2 + w] = s[1];
    }
    return __longlong_as_double(((uint64_t)r[1] << 32) | r[0]) + __longlong_as_double(((uint64_t)r[3] << 32) | r[2]);
}

// 64 lanes' sums of NV values: afterwards quarter c of the wavefront holds, in register r < NP, the 16
// remaining partial sums of value r + NP (c & 1) + 2 NP (c >> 1), which go to LDS (red, 68 NP doubles).
template <int NV>
struct WaveSums {
    static constexpr int NP = (NV + 3) / 4;
    __device__ static __forceinline__ void store(const double* acc, double* red, int lane) {
        double h[2 * NP];
#pragma unroll
        for (int v = 0; v < 2 * NP; ++v)
            h[v] = swap_add<32>(v < NV ? acc[v < NV ? v : 0] : 0.0, v + 2 * NP < NV ? acc[v + 2 * NP < NV ? v + 2 * NP : 0] : 0.0);
#pragma unroll
        for (int r = 0; r < NP; ++r) red[r * 68 + (lane >> 4) * 17 + (lane & 15)] = swap_add<16>(h[r], h[r + NP]);
    }
    // slot t < 4 NP: the value it holds (>= NV: none) and its sum
    __device__ static __forceinline__ int value(int t) { return (t >> 2) + ((t & 1) ? NP : 0) + ((t & 2) ? 2 * NP : 0); }
    __device__ static __forceinline__ double sum(const double* red, int t) {
        const double* p = red + (t >> 2) * 68 + (t & 3) * 17;
        double s = 0.0;
#pragma unroll
        for (int l = 0; l < 16; ++l) s += p[l];
        return s;
    }
};

// A sub-cell (simplex, vertices X) as the affine map of its rule: per axis vertex 2 and the edges to the
// others, in the coordinate (x - lo) sc; then the factor of the rule's weights (0 where the sub-cell's
// detJ < -1e-6).  vol: product of the half extents of the cell over DIM!.
template <int DIM>
__device__ __forceinline__ void stage_simplex(const double* X, const double* lo, const double* sc, double vol, double* T) {
    double J[DIM][DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d)
#pragma unroll
        for (int r = 0; r < DIM; ++r) J[r][d] = X[(r < 2 ? r : 3) * DIM + d] - X[2 * DIM + d];
    double detJ;
    if constexpr (DIM == 3)
        detJ = (J[0][0] * (J[1][1] * J[2][2] - J[2][1] * J[1][2]) - J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0])) * vol;
    else
        detJ = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * vol;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        T[(DIM + 1) * d] = (X[2 * DIM + d] - lo[d]) * sc[d];
#pragma unroll
        for (int r = 0; r < DIM; ++r) T[(DIM + 1) * d + 1 + r] = J[r][d] * sc[d];
    }
    T[(DIM + 1) * DIM] = detJ < kDetJLowerLimit ? 0.0 : detJ;
}

template <int DIM>
struct LinearMoments {
    static constexpr int N = DIM == 3 ? 27 : 9;
    static constexpr int NQ = DIM == 3 ? kTet11Points : kTri7Points;
    static constexpr int BATCH = 64;                          // sub-cells staged at a time
    static constexpr int TET = DIM == 3 ? 14 : 8;             // staged doubles of one (even)
    static constexpr int RULE = BATCH * TET;                  // [q][xi.., w]
    static constexpr int LDS = RULE + NQ * (DIM + 1) > 68 * WaveSums<N>::NP ? RULE + NQ * (DIM + 1) : 68 * WaveSums<N>::NP;
};

// The moments of a cut cell, one wavefront: a lane a point, the sums in registers.  lds: LDS doubles
// of scratch; the result in m (LDS, N doubles), valid after the call.
template <int DIM>
__device__ __forceinline__ void cut_moments(const double* ig_xi, int ig0, int nsub, const double* hh, double* lds, double* m) {
    using LM = LinearMoments<DIM>;
    constexpr int NQ = LM::NQ, NX = (DIM + 1) * DIM;
    const int lane = threadIdx.x;
    double vol = DIM == 3 ? 1.0 / 6.0 : 0.5;
    for (int d = 0; d < DIM; ++d) vol *= 0.5 * hh[d];
    for (int t = lane; t < NQ * (DIM + 1); t += 64) {
        const int q = t / (DIM + 1), c = t - (DIM + 1) * q;
        if constexpr (DIM == 3) lds[LM::RULE + t] = c < 3 ? kTet11Xi[q][c] : kTet11W[q];
        else lds[LM::RULE + t] = c < 2 ? kTri7Xi[q][c] : kTri7W[q];
    }
    double acc[LM::N];
#pragma unroll
    for (int k = 0; k < LM::N; ++k) acc[k] = 0.0;
    for (int t0 = 0; t0 < nsub; t0 += LM::BATCH) {
        const int nt = min(LM::BATCH, nsub - t0), npts = nt * NQ;
        if (t0 > 0) __syncthreads();   // the previous batch is read
        if (lane < nt) {
            const double2* X2 = reinterpret_cast<const double2*>(ig_xi + (size_t)(ig0 + t0 + lane) * NX);
            double X[NX];
#pragma unroll
            for (int n = 0; n < NX / 2; ++n) {
                const double2 v = X2[n];
                X[2 * n] = v.x;
                X[2 * n + 1] = v.y;
            }
            const double lo[3] = {-1.0, -1.0, -1.0}, sc[3] = {0.5, 0.5, 0.5};   // [-1, 1] to [0, 1]
            stage_simplex<DIM>(X, lo, sc, vol, lds + lane * LM::TET);
        }
        __syncthreads();
        for (int p0 = 0; p0 < npts; p0 += 64) {
            const int ip = p0 + lane, ipc = ip < npts ? ip : 0;   // lanes past the end: point 0, weight 0
            const int t = ipc / NQ, q = ipc - NQ * t;
            const double* T = lds + t * LM::TET;
            const double* b = lds + LM::RULE + (DIM + 1) * q;
            double p[DIM][3];
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                double x = T[(DIM + 1) * d];
#pragma unroll
                for (int r = 0; r < DIM; ++r) x += b[r] * T[(DIM + 1) * d + 1 + r];
                const double y = 1.0 - x;
                p[d][0] = y * y;
                p[d][1] = x * y;
                p[d][2] = x * x;
            }
            const double w = ip < npts ? b[DIM] * T[NX] : 0.0;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double wi = w * p[0][i];
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    if constexpr (DIM == 3) {
                        const double wij = wi * p[1][j];
#pragma unroll
                        for (int k = 0; k < 3; ++k) acc[(i * 3 + j) * 3 + k] += wij * p[2][k];
                    } else {
                        acc[i * 3 + j] += wi * p[1][j];
                    }
                }
            }
        }
    }
    using WS = WaveSums<LM::N>;
    __syncthreads();
    WS::store(acc, lds, lane);
    __syncthreads();
    if (lane < 4 * WS::NP) {
        const int v = WS::value(lane);
        const double s = WS::sum(lds, lane);
        if (v < LM::N) m[v] = s;
    }
    __syncthreads();
}

// The moments of a whole cell: the integrals of p_0, p_1, p_2 over [-1, 1] are 2/3, 1/3, 2/3 (HEX_2x2x2 and
// QUAD_2x2 integrate them exactly).
template <int DIM>
__device__ __forceinline__ void whole_moments(const double* hh, double* m) {
    double vol = 1.0;
    for (int d = 0; d < DIM; ++d) vol *= 0.5 * hh[d];
    if (threadIdx.x < LinearMoments<DIM>::N) {
        int t = threadIdx.x, k = 1;
        for (int d = 0; d < DIM; ++d) {
            k *= t % 3 == 1 ? 1 : 2;
            t /= 3;
        }
        m[threadIdx.x] = vol * (double)k / (DIM == 3 ? 27.0 : 9.0);
    }
    __syncthreads();
}

// M[(i,a),(j,b)] of vertices a, b from the moments: s_a^i s_b^j / (h_i h_j) times the sum of the moments that
// make up [l_b on axis i] [l_a on axis j] prod_(other d) l_a l_b (i != j), prod_(d != i) l_a l_b (i == j).
template <int DIM>
__device__ __forceinline__ void moment_block(const double* m, int a, int b, const double* hh, double (*M)[DIM]) {
    constexpr int ST[3] = {DIM == 3 ? 9 : 3, DIM == 3 ? 3 : 1, 1};
    int ab[DIM], bb[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        // vertex signs of the HEX8 / QUAD4 order as bits
        ab[d] = d == 0 ? (a ^ (a >> 1)) & 1 : (d == 1 ? (a >> 1) & 1 : a >> 2);
        bb[d] = d == 0 ? (b ^ (b >> 1)) & 1 : (d == 1 ? (b >> 1) & 1 : b >> 2);
    }
#pragma unroll
    for (int i = 0; i < DIM; ++i)
#pragma unroll
        for (int j = 0; j < DIM; ++j) {
            int at = 0;
#pragma unroll
            for (int d = 0; d < DIM; ++d)
                if (d != i && d != j) at += (ab[d] + bb[d]) * ST[d];
            double v;
            if (i == j) {
                v = m[at] + 2.0 * m[at + ST[i]] + m[at + 2 * ST[i]];
            } else {
                at += bb[i] * ST[i] + ab[j] * ST[j];
                v = (m[at] + m[at + ST[i]]) + (m[at + ST[j]] + m[at + ST[i] + ST[j]]);
            }
            M[i][j] = (ab[i] == bb[j] ? v : -v) / (hh[i] * hh[j]);
        }
}

// Entry (al, a), (be, b) of B^T D B from the moment block of (a, b).
template <int DIM>
__device__ __forceinline__ double elastic_entry(const double (*D)[DIM == 3 ? 6 : 3], const double (*M)[DIM], int al, int be) {
    double v = 0.0;
#pragma unroll
    for (int i = 0; i < DIM; ++i)
#pragma unroll
        for (int j = 0; j < DIM; ++j)
            if (d_nonzero<DIM>(voigt<DIM>(al, i), voigt<DIM>(be, j))) v += D[voigt<DIM>(al, i)][voigt<DIM>(be, j)] * M[i][j];
    return v;
}

}  // namespace mgpu
