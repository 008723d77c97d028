// hex27.hip -- element matrices of HEX27 IP cells on the generic path.
//
// The moment integrand of a box HEX27 cell, dN_a/dx_i dN_b/dx_j (two triquadratic factors, one
// differentiated each), is a polynomial of degree <= 4 in each axis.  Its sum over a cell's
// integration points (TET_35 on the XTK sub-tets, w* = w detJ, points with detJ < -1e-6 skipped,
// cl_FEM_Element_Bulk.cpp:258-355; HEX_3x3x3 on whole cells) is therefore a fixed linear function of
// the cell's 125 moments of degree <= 4 per axis, and factorises over the axes.
// Both quadrature options take this route, in FP64 at either precision option: it is the point sum in
// another order, K (as a whole) within 1.2e-16 .. 2.8e-16 of sums in 80-bit long double, against 7.8e-16 ..
// 2.1e-15 with M accumulated point by point; for its small entries see the basis below.  32^3 cut cells,
// elasticity, p = 2 (1.1M sub-tets, 37.8M points): element kernels 11.8 ms with M accumulated point by point
// on 21 FP64 MFMA tiles, 0.98 ms here.
//
//   k_hex27_moments    two wavefronts per element: the 125 moments of a cut cell, a lane a point (whole
//                      cells: closed form).
//   k_hex27_tensor     elements whose T is a tensor product of one 1D matrix per axis (nodal rows,
//                      untruncated p = 2 B-splines): T folded into the 1D factor tables, so that K_e
//                      comes straight from the moments; one block of 4 wavefronts per element.
//   k_hex27_general    any other T (truncated hierarchical rows): K_p from the moments with the
//                      Lagrange tables, K_e = T^T K_p T on FP64 MFMA.
// K_e goes to the element's slot of the pool, or (scatter mode) is added into the CSR values.
#include <hip/hip_runtime.h>

#include <cmath>

#include "../common/fem_tables.hpp"
#include "cut_moments.hpp"
#include "set_state.hpp"

namespace mgpu {

namespace {

typedef double doublex4_t __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------------------------------------
// The moments are taken in the Bernstein basis of the box that holds the cell's material: on each axis
// the sub-cells' vertices span [lo, hi], t = (x - lo) / (hi - lo), s = 1 - t, and the basis is
// g_m = t^m s^(4 - m), m <= 4, so that every moment is a sum of terms of one sign.  The 1D functions (and
// their derivatives) are f_0 s^2 + f_1 t s + f_2 t^2 with coefficients of the box (axis_coefficient), a
// product F_a F_b is sum_kl f_ak f_bl g_(k+l).  Because t spans [0, 1] over the material itself, the terms of a
// product are of the size of the product: small entries (a basis function that a sliver in a corner,
// along an edge or around the cell's centre barely touches) keep their digits as in the sum over the
// points.  Relative error of the worst diagonal entry, slivers of edge 0.1 .. 1e-5 at a corner: 4e-16 ..
// 6e-15, summed point by point 3e-15 .. 2e-11; a fixed basis on [-1, 1] fails either at the corners (Lagrange
// functions and multiples of x^3 - x: 2e-12 .. 1e-4) or at the centre (Bernstein: 1e-10 .. all digits).
//
// A record of kHex27MomStride doubles per element: the moments, a factor of all of them, then from kHex27MomTab
// the coefficients [axis][function, derivative][alpha][k].
// ------------------------------------------------------------------------------------------------
static_assert(kHex27MomTab + 54 <= kHex27MomStride && kHex27MomTab > kHex27Moments, "the tables follow the moments and their factor");

// Coefficient k of 1D function alpha (0 .. 2) or its derivative on [lo, hi].  Every function is p q + c with
// linear p, q, its coefficients p q, p q' + p' q, p' q' of their values at the ends; with u = (1 + x) / 2,
// v = (1 - x) / 2: Lagrange -v x, 4 u v, u x; uniform quadratic B-splines (the T rows, vertex rows 1/2 1/2, mid
// rows 1/8 3/4 1/8, times those) v v / 2, 1/2 + u v, u u / 2.
__device__ __forceinline__ double axis_coefficient(bool spline, bool deriv, int alpha, int k, double lo, double hi) {
    double p[2], q[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        const double x = n ? hi : lo, u = 0.5 * (1.0 + x), v = 0.5 * (1.0 - x);
        if (deriv) {
            p[n] = spline ? (alpha == 0 ? -0.5 * v : (alpha == 1 ? -0.5 * x : 0.5 * u))
                          : (alpha == 0 ? x - 0.5 : (alpha == 1 ? -2.0 * x : x + 0.5));
            q[n] = 1.0;
        } else {
            p[n] = spline ? (alpha == 0 ? 0.5 * v : (alpha == 1 ? u : 0.5 * u))
                          : (alpha == 0 ? -v : (alpha == 1 ? 4.0 * u : u));
            q[n] = spline ? (alpha == 2 ? u : v) : (alpha == 1 ? v : x);
        }
    }
    const double c = spline && !deriv && alpha == 1 ? 0.5 : 0.0;
    return k == 0 ? p[0] * q[0] + c : (k == 2 ? p[1] * q[1] + c : p[0] * q[1] + p[1] * q[0] + 2.0 * c);
}
__device__ __forceinline__ void write_tables(bool spline, const double* lo, const double* hi, double* tab) {
    const int t = threadIdx.x;
    if (t >= 54) return;
    const int d = t / 18, r = t - 18 * d;
    tab[t] = axis_coefficient(spline, r >= 9, (r % 9) / 3, r % 3, d == 0 ? lo[0] : (d == 1 ? lo[1] : lo[2]),
                              d == 0 ? hi[0] : (d == 1 ? hi[1] : hi[2]));
}

// ------------------------------------------------------------------------------------------------
// k_hex27_moments: mom[e][(i 5 + j) 5 + k] = sum_ip w* g_i(x) g_j(y) g_k(z), and the element's tables.  Two
// wavefronts per element, each with 13 or 12 of the 25 pairs (i, j) as 65 or 60 sums per lane in registers;
// 64 points at a time, a lane a point.  A batch of 64 sub-tets is staged in LDS as vertex 2, the three
// edges and the volume factor.  The lanes' sums are added pairwise by half and quarter wavefront
// (gfx950's lane swaps reduce two registers at once), the last 16 in LDS.
// Bound by FP64 arithmetic, 112 operations a point and wavefront: 32^3 cut cells (37.8M points) 0.50 ms
// (0.56 with two wavefronts a SIMD instead of three, the weight read under a branch); a
// 16 x 16 x 4 FP64 MFMA tile per 4 points took 0.69 ms: its operands pass through LDS (25 doubles a point),
// half the tile is padding, and FP64 MFMA runs at the rate of the vector unit.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ void hex27_basis(double t, double* v) {
    const double s = 1.0 - t, t2 = t * t, ts = t * s, s2 = s * s;
    v[0] = s2 * s2;
    v[1] = ts * s2;
    v[2] = ts * ts;
    v[3] = ts * t2;
    v[4] = t2 * t2;
}

constexpr int kMomBatch = 64;                          // sub-tets staged at a time
constexpr int kMomTet = 14;                            // x_2, edges, volume factor (even: 16-byte reads)
constexpr int kMomRule = kMomBatch * kMomTet;          // LDS offset of TET_35 [q][xi_0, xi_1, xi_2, w]
constexpr int kMomLds = 17 * 68;                       // the reduction's space
static_assert(kMomRule + 4 * kTet35Points <= kMomLds, "staged sub-tets and the rule fit the reduction's space");

// min over the lanes of equal lane % 8
__device__ __forceinline__ double min_mod8(double v) {
    auto both = [](double x, auto f) {
        const uint64_t u = __double_as_longlong(x);
        uint32_t r[4];
        f((uint32_t)u, r[0], r[2]);
        f((uint32_t)(u >> 32), r[1], r[3]);
        return fmin(__longlong_as_double(((uint64_t)r[1] << 32) | r[0]), __longlong_as_double(((uint64_t)r[3] << 32) | r[2]));
    };
    v = both(v, [](uint32_t w, uint32_t& x, uint32_t& y) {
        x = w;
        y = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0x128, 0xf, 0xf, true);   // lane + 8 within 16
    });
    v = both(v, [](uint32_t w, uint32_t& x, uint32_t& y) {
        const auto s = __builtin_amdgcn_permlane16_swap(w, w, false, false);
        x = s[0];
        y = s[1];
    });
    return both(v, [](uint32_t w, uint32_t& x, uint32_t& y) {
        const auto s = __builtin_amdgcn_permlane32_swap(w, w, false, false);
        x = s[0];
        y = s[1];
    });
}
__device__ __forceinline__ double read_lane(double v, int lane) {
    const uint64_t u = __double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, lane), hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), lane);
    return __longlong_as_double(((uint64_t)hi << 32) | lo);
}

__device__ __forceinline__ void load_tet(const GenView& g, int tet, double* X) {
    const double2* X2 = reinterpret_cast<const double2*>(g.ig_xi + (size_t)tet * 12);
#pragma unroll
    for (int n = 0; n < 6; ++n) {
        const double2 v = X2[n];
        X[2 * n] = v.x;
        X[2 * n + 1] = v.y;
    }
}

// The box of the sub-tets' vertices and the factors to [0, 1] (0 for an axis without extent: t = 0, the
// functions' values at lo), the same in every lane.  X: the lane's sub-tet of the first batch.
__device__ __forceinline__ void hex27_box(const GenView& g, int ig0, int nsub, const double* X, double* lds, double* lo,
                                          double* hi, double* sc) {
    const int lane = threadIdx.x;
    double b[6];   // the least of x, y, z and of -x, -y, -z
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        b[d] = fmin(fmin(X[d], X[3 + d]), fmin(X[6 + d], X[9 + d]));
        b[3 + d] = fmin(fmin(-X[d], -X[3 + d]), fmin(-X[6 + d], -X[9 + d]));
    }
    for (int t = kMomBatch + lane; t < nsub; t += 64) {
        double Y[12];
        load_tet(g, ig0 + t, Y);
#pragma unroll
        for (int n = 0; n < 12; ++n) {
            b[n % 3] = fmin(b[n % 3], Y[n]);
            b[3 + n % 3] = fmin(b[3 + n % 3], -Y[n]);
        }
    }
#pragma unroll
    for (int d = 0; d < 6; ++d) lds[d * 65 + lane] = b[d];
    __syncthreads();
    const double* col = lds + min(lane & 7, 5) * 65 + (lane >> 3) * 8;
    double v = col[0];
#pragma unroll
    for (int n = 1; n < 8; ++n) v = fmin(v, col[n]);
    v = min_mod8(v);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        lo[d] = read_lane(v, d);
        hi[d] = -read_lane(v, 3 + d);
    }
    const double ext = lane == 0 ? hi[0] - lo[0] : (lane == 1 ? hi[1] - lo[1] : hi[2] - lo[2]);
    const double inv = ext > 1e-290 ? 1.0 / ext : 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d) sc[d] = read_lane(inv, d);
    __syncthreads();   // the space is free again
}

template <int ROLE>
__device__ __forceinline__ void hex27_cut_moments(const GenView& g, int ig0, int nsub, double vol6, const double* lo,
                                                  const double* sc, double* lds, double* out) {
    constexpr int P0 = ROLE == 0 ? 0 : 13, NP = ROLE == 0 ? 13 : 12, I0 = P0 / 5;
    const int lane = threadIdx.x;
    double acc[NP][5];
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int k = 0; k < 5; ++k) acc[p][k] = 0.0;
    for (int t = lane; t < 4 * kTet35Points; t += 64) {
        const int q = t >> 2, c = t & 3;
        lds[kMomRule + t] = c < 3 ? kTet35Xi[q][c] : kTet35W[q];
    }
    for (int t0 = 0; t0 < nsub; t0 += kMomBatch) {
        const int nt = min(kMomBatch, nsub - t0), npts = nt * kTet35Points;
        if (t0 > 0) {   // (the first batch is staged)
            __syncthreads();   // the previous batch is read
            if (lane < nt) {
                double X[12];
                load_tet(g, ig0 + t0 + lane, X);
                stage_simplex<3>(X, lo, sc, vol6, lds + lane * kMomTet);
            }
        }
        __syncthreads();
        for (int p0 = 0; p0 < npts; p0 += 64) {
            // lanes past the end: point 0 with weight 0.  The point is vertex 2 plus the rule's
            // coordinates along the edges (the same affine map as the vertex weights (xi0, xi1,
            // 1 - xi0 - xi1 - xi2, xi2))
            const int ip = p0 + lane, ipc = ip < npts ? ip : 0;
            const int t = ipc / kTet35Points, q = ipc - kTet35Points * t;
            const double* T = lds + t * kMomTet;
            const double* b = lds + kMomRule + 4 * q;
            double x[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) x[d] = T[4 * d] + b[0] * T[4 * d + 1] + b[1] * T[4 * d + 2] + b[2] * T[4 * d + 3];
            const double wt = b[3] * T[12], w = ip < npts ? wt : 0.0;
            double gx[5], gy[5], gz[5];
            hex27_basis(x[0], gx);
            hex27_basis(x[1], gy);
            hex27_basis(x[2], gz);
#pragma unroll
            for (int i = I0; i < 5; ++i) gx[i] *= w;
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                const double v = gx[(P0 + p) / 5] * gy[(P0 + p) % 5];
#pragma unroll
                for (int k = 0; k < 5; ++k) acc[p][k] += v * gz[k];
            }
        }
    }
    using WS = WaveSums<NP * 5>;
    __syncthreads();
    WS::store(&acc[0][0], lds, lane);
    __syncthreads();
    for (int t = lane; t < 4 * WS::NP; t += 64) {
        const int v = WS::value(t);
        const double s = WS::sum(lds, t);
        if (v < NP * 5) out[P0 * 5 + v] = s;
    }
}

__global__ __launch_bounds__(64, 3) void k_hex27_moments(GenView g, double* mom) {
    __shared__ __align__(16) double lds[kMomLds];
    // 16 blocks in a row hold 8 elements, the role changing after 8: the round robin over the 8 XCDs
    // gives each both roles in turn
    const int b = blockIdx.x, role = (b >> 3) & 1, be = (b >> 4) * 8 + (b & 7);
    if (be >= g.n_el) return;
    const int e = __builtin_amdgcn_readfirstlane(g.order ? g.order[be] : be);
    double hh[3];
    for (int d = 0; d < 3; ++d) hh[d] = g.ip_box[(size_t)e * 6 + 3 + d];
    const double detJ = (0.5 * hh[0]) * (0.5 * hh[1]) * (0.5 * hh[2]);
    const double vol6 = read_lane(detJ / 6.0, 0);   // (in scalar registers)
    const int ig0 = __builtin_amdgcn_readfirstlane(g.ig_ptr[e]), nsub = __builtin_amdgcn_readfirstlane(g.ig_ptr[e + 1]) - ig0;
    double* out = mom + (size_t)e * kHex27MomStride;
    double lo[3] = {-1.0, -1.0, -1.0}, hi[3] = {1.0, 1.0, 1.0}, sc[3];
    if (nsub > 0) {
        double X[12];
        load_tet(g, ig0 + min((int)threadIdx.x, nsub - 1), X);   // (lanes past the end: the last one again)
        hex27_box(g, ig0, nsub, X, lds, lo, hi, sc);
        if ((int)threadIdx.x < nsub) stage_simplex<3>(X, lo, sc, vol6, lds + threadIdx.x * kMomTet);
    }
    if (role == 0 && threadIdx.x == 0) out[kHex27Moments] = nsub == 0 ? detJ / 27000.0 : 1.0;
    if (role == 0) write_tables(g.t_perm[(size_t)e * kHex27PermStride + 27] == 2, lo, hi, out + kHex27MomTab);
    if (nsub == 0) {
        // whole cell: products of the 1D integrals 2/5, 1/10, 1/15, 1/10, 2/5 (HEX_3x3x3 is exact for them), as
        // integers: the contraction is exact until the record's factor is applied.  (Rounded here, the
        // same error in every whole cell put K of a set with many of them 3.6e-16 off instead of 2.7e-16.)
        auto n30 = [](int m) { return m == 2 ? 2 : (m == 0 || m == 4 ? 12 : 3); };
        for (int t = threadIdx.x; t < kHex27Moments && role == 0; t += 64)
            out[t] = (double)(n30(t / 25) * n30((t / 5) % 5) * n30(t % 5));
    } else if (role == 0) {
        hex27_cut_moments<0>(g, ig0, nsub, vol6, lo, sc, lds, out);
    } else {
        hex27_cut_moments<1>(g, ig0, nsub, vol6, lo, sc, lds, out);
    }
}

// ------------------------------------------------------------------------------------------------
// M from the moments, by sum factorisation over the axes: block p = (i, j), i <= j, of
//   M[(i,a),(j,b)] = s_i s_j sum_{x,y,z <= 4} mom_xyz P_0(a_0,b_0; x) P_1(a_1,b_1; y) P_2(a_2,b_2; z),
// s_i = 2 / h_i, P_d(alpha,beta; m) = sum_(k + l = m) f_alpha,k f_beta,l of the element's tables, contracted over z,
// y, x.  Wavefronts take whole tasks, so that the tables are scalar loads.  Result G[p][a][b] in LDS,
// a = (a_0 3 + a_1) 3 + a_2; NF == 1: the sum of the three diagonal blocks only.  The diagonal blocks are
// symmetric bit for bit.  LDS: mom, Z[zt][x 5 + y][ab_2], Y[block][x][ab_1][ab_2], then G over Z and Y.
// ------------------------------------------------------------------------------------------------
typedef const __attribute__((address_space(4))) double* scalar_table;   // memory that this kernel only reads

// o[3 alpha + beta] = sum_kl A[alpha][k] B[beta][l] T[k + l], A == B where SYM
template <bool SYM>
__device__ __forceinline__ void axis_contract(const double* T, scalar_table A, scalar_table B, double* o) {
#pragma unroll
    for (int al = 0; al < 3; ++al) {
        double v[3];
#pragma unroll
        for (int l = 0; l < 3; ++l) v[l] = A[3 * al] * T[l] + A[3 * al + 1] * T[l + 1] + A[3 * al + 2] * T[l + 2];
#pragma unroll
        for (int be = 0; be < 3; ++be) {
            if (SYM && be < al) continue;
            const double w = v[0] * B[3 * be] + v[1] * B[3 * be + 1] + v[2] * B[3 * be + 2];
            o[3 * al + be] = w;
            if (SYM) o[3 * be + al] = w;
        }
    }
}
// tau = 2 [alpha differentiated] + [beta differentiated] (the same for the wavefront); tab: the axis' tables
__device__ __forceinline__ void axis_contract(const double* T, scalar_table tab, int tau, double* o) {
    scalar_table A = tab + (tau & 2 ? 9 : 0), B = tab + (tau & 1 ? 9 : 0);
    if (tau == 0 || tau == 3) axis_contract<true>(T, A, A, o);
    else axis_contract<false>(T, A, B, o);
}

template <int NF> struct Hex27Blocks;
template <> struct Hex27Blocks<1> {
    static constexpr int n = 3;
    static constexpr int i[3] = {0, 1, 2}, j[3] = {0, 1, 2};
};
template <> struct Hex27Blocks<3> {
    static constexpr int n = 6;
    static constexpr int i[6] = {0, 0, 0, 1, 1, 2}, j[6] = {0, 1, 2, 1, 2, 2};
};
constexpr int kSfZ = 128, kSfY = kSfZ + 3 * 225;
template <int NF>
constexpr int sf_lds() {   // doubles
    return NF == 3 ? 6 * 729 : kSfY + 3 * 405;
}
static_assert(kSfY + 6 * 405 <= 6 * 729, "the contraction stages fit the space of G");

template <int NF>
__device__ __forceinline__ void sf_moments(const GenView& g, const double* mom, int e, double* lds) {
    using B = Hex27Blocks<NF>;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    double* Z = lds + kSfZ;
    double* Y = lds + kSfY;
    const double* rec = mom + (size_t)__builtin_amdgcn_readfirstlane(e) * kHex27MomStride;
    const scalar_table tab = (scalar_table)(rec + kHex27MomTab);
    if (tid < kHex27Moments) lds[tid] = rec[tid];
    // the tables' lines are requested here: a stage that asked for its own would wait for memory each time
    double line[7];
#pragma unroll
    for (int n = 0; n < 7; ++n) line[n] = tab[8 * n < 54 ? 8 * n : 53];
    const double factor = rec[kHex27Moments];
    double sc[3];
    for (int d = 0; d < 3; ++d) sc[d] = 2.0 / g.ip_box[(size_t)e * 6 + 3 + d];
    __syncthreads();
#pragma unroll
    for (int n = 0; n < 7; ++n) asm volatile("" ::"s"(line[n]));   // (used here: not dropped, not moved down)
    // z: task zt = wave, tau_2 = 0, 1, 3 (alpha alone is differentiated on axis 2 in no block i <= j)
    if (wave < 3 && lane < 25) {
        double m[5], o[9];
#pragma unroll
        for (int k = 0; k < 5; ++k) m[k] = lds[lane * 5 + k];
        axis_contract(m, tab + 36, wave == 2 ? 3 : wave, o);
#pragma unroll
        for (int ab = 0; ab < 9; ++ab) Z[wave * 225 + lane * 9 + ab] = o[ab];
    }
    __syncthreads();
    // y: task block p, lane (x, ab_2)
    for (int p = wave; p < B::n; p += 4) {
        const int i = NF == 1 ? p : (p >= 3) + (p >= 5), j = NF == 1 ? p : (p < 3 ? p : (p < 5 ? p - 2 : 2));
        const int tau1 = 2 * (i == 1) + (j == 1), tau2 = 2 * (i == 2) + (j == 2);
        if (lane < 45) {
            const int x = lane / 9, ab2 = lane - 9 * x;
            const double* Zp = Z + (tau2 == 3 ? 2 : tau2) * 225 + x * 45 + ab2;
            double z[5], o[9];
#pragma unroll
            for (int y = 0; y < 5; ++y) z[y] = Zp[9 * y];
            axis_contract(z, tab + 18, tau1, o);
#pragma unroll
            for (int ab1 = 0; ab1 < 9; ++ab1) Y[p * 405 + x * 81 + ab1 * 9 + ab2] = o[ab1];
        }
    }
    __syncthreads();
    // x: task (p, half), lane ab_12; the results stay in registers until Y is read by every task
    constexpr int NT = NF == 3 ? 3 : 1;
    double r[NT][9];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
#pragma unroll
        for (int q = 0; q < 9; ++q) r[n][q] = 0.0;
        const int task = wave + 4 * n;
        if (NF == 1 && task >= 2) continue;
        const int ab12 = (task & 1) * 64 + lane;
        if (ab12 >= 81) continue;
#pragma unroll
        for (int pp = 0; pp < (NF == 3 ? 1 : 3); ++pp) {
            const int p = NF == 3 ? task >> 1 : pp;
            const int i = NF == 1 ? p : (p >= 3) + (p >= 5), j = NF == 1 ? p : (p < 3 ? p : (p < 5 ? p - 2 : 2));
            const double s2 = factor * (i == 0 ? sc[0] : (i == 1 ? sc[1] : sc[2])) * (j == 0 ? sc[0] : (j == 1 ? sc[1] : sc[2]));
            double y[5], o[9];
#pragma unroll
            for (int x = 0; x < 5; ++x) y[x] = s2 * Y[p * 405 + x * 81 + ab12];
            axis_contract(y, tab, 2 * (i == 0) + (j == 0), o);
#pragma unroll
            for (int ab0 = 0; ab0 < 9; ++ab0) r[n][ab0] += o[ab0];
        }
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int task = wave + 4 * n;
        if (NF == 1 && task >= 2) continue;
        const int ab12 = (task & 1) * 64 + lane;
        if (ab12 >= 81) continue;
        const int p = NF == 3 ? task >> 1 : 0;
        const int a12 = (ab12 / 27) * 3 + (ab12 / 3) % 3, b12 = ((ab12 / 9) % 3) * 3 + ab12 % 3;
#pragma unroll
        for (int ab0 = 0; ab0 < 9; ++ab0) lds[p * 729 + ((ab0 / 3) * 9 + a12) * 27 + (ab0 % 3) * 9 + b12] = r[n][ab0];
    }
    __syncthreads();
}

// Entry (f, a), (h, b) of K as a sum of three coefficients times entries of G:
//   f == h: c0 M_ff[a,b] + cs (M_ii + M_jj)[a,b];  f != h: c1 M_fh[a,b] + cs M_hf[a,b], M_hf[a,b] = M_fh[b,a]
// (isotropic D, block (f, h) of B^T D B; diffusion: the material times the summed diagonal blocks).
// The three entries sit at base[n] + a sa[n] + b sb[n].
struct KTerms {
    double c[3];
    int base[3], sa[3], sb[3];
};
template <int NF>
__device__ __forceinline__ KTerms k_terms(int f, int h, double c0, double c1, double cs) {
    KTerms k;
    if (NF == 1) {
        k.c[0] = c0;
        k.c[1] = k.c[2] = 0.0;
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            k.base[n] = 0;
            k.sa[n] = 27;
            k.sb[n] = 1;
        }
        return k;
    }
    // block index of (i, j), i <= j: 0 (0,0) 1 (0,1) 2 (0,2) 3 (1,1) 4 (1,2) 5 (2,2)
    const int lo = min(f, h), hi = max(f, h);
    const int pf = f == 0 ? 0 : (f == 1 ? 3 : 5);
    const int pfh = lo == 0 ? hi : (lo == 1 ? hi + 2 : 5);
    const bool dg = f == h, up = f < h;
    k.c[0] = dg ? c0 : c1;
    k.c[1] = cs;
    k.c[2] = dg ? cs : 0.0;
    k.base[0] = 729 * (dg ? pf : pfh);
    k.base[1] = 729 * (dg ? (f == 0 ? 3 : 0) : pfh);
    k.base[2] = 729 * (dg ? (f == 2 ? 3 : 5) : pfh);
    k.sa[0] = dg || up ? 27 : 1;
    k.sb[0] = dg || up ? 1 : 27;
    k.sa[1] = dg || !up ? 27 : 1;
    k.sb[1] = dg || !up ? 1 : 27;
    k.sa[2] = k.sa[0];
    k.sb[2] = k.sb[0];
    return k;
}

template <int NF>
__device__ __forceinline__ void hex27_material(const GenView& g, int e, double& c0, double& c1, double& cs) {
    if (NF == 1) {
        c0 = g.material[e];
        c1 = cs = 0.0;
    } else {
        double D[6][6];
        elastic_D<3>(g.material[2 * e], g.material[2 * e + 1], D);
        c0 = D[0][0];
        c1 = D[0][1];
        cs = D[5][5];
    }
}

// ------------------------------------------------------------------------------------------------
// k_hex27_tensor: K_e of elements whose T is a tensor product (t_perm[e][27] = 1 nodal, 2 B-spline, 3 B-spline on
// a HEX8 cell; t_perm[e][y] the tensor index of the element's adof y).  Threads 0 .. 3 NA - 1 hold a column of K_e and
// write NF rows' worth of consecutive values per step (stores of whole lines).  Without the products by T
// and their LDS space four blocks instead of two fit a CU: 0.48 ms for 32^3 elements of 81 x 81 (1.7 GB
// written, 3.5 TB/s), against 1.7 ms on the general path.
// ------------------------------------------------------------------------------------------------
template <int NF, bool SCATTER>
__global__ __launch_bounds__(256) void k_hex27_tensor(GenView g, const int32_t* els, const double* mom, double* vals) {
    constexpr int NA = NF * 27;
    constexpr int RPS = NF == 3 ? 3 : 9;   // rows per step; divides 27
    static_assert(RPS * NA <= 256 && 27 % RPS == 0, "a step's rows lie in one field block");
    __shared__ double lds[sf_lds<NF>()];
    __shared__ int perm[27];
    const int e = els[blockIdx.x];
    const int tid = threadIdx.x;
    const uint8_t* pm = g.t_perm + (size_t)e * kHex27PermStride;
    if (tid < 27) perm[tid] = pm[tid];
    sf_moments<NF>(g, mom, e, lds);
    double c0, c1, cs;
    hex27_material<NF>(g, e, c0, c1, cs);
    if (tid >= RPS * NA) return;
    const int rs = tid / NA, col = tid - NA * rs, h = col / 27, y = col - 27 * h;
    const int b = perm[y];
    double* ke = SCATTER ? nullptr : g.ke + g.ke_off[e];
    const int32_t* rows = SCATTER ? g.topo + g.topo_ptr[e] : nullptr;
    const uint16_t* rk = SCATTER ? g.rank + g.rank_off[e] : nullptr;
    for (int f = 0; f < NF; ++f) {
        const KTerms k = k_terms<NF>(f, h, c0, c1, cs);
        const double* G0 = lds + k.base[0] + b * k.sb[0];
        const double* G1 = lds + k.base[1] + b * k.sb[1];
        const double* G2 = lds + k.base[2] + b * k.sb[2];
#pragma unroll 3
        for (int n = 0; n < 27 / RPS; ++n) {
            const int x = RPS * n + rs, a = perm[x];
            double v = k.c[0] * G0[a * k.sa[0]];
            if (NF > 1) v += k.c[1] * G1[a * k.sa[1]] + k.c[2] * G2[a * k.sa[2]];
            if constexpr (SCATTER) {
                const int32_t row = rows[f * 27 + x], r0 = g.row_ptr[row], len = (g.row_ptr[row + 1] - r0) / NF;
                unsafeAtomicAdd(vals + r0 + h * len + rk[x * 27 + y], v);
            } else {
                ke[(f * 27 + RPS * n) * NA + tid] = v;
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// k_hex27_general: K_e = T^T K_p T per (f, h) block on FP64 MFMA (16 x 16 tiles, k in steps of 4, operands
// from LDS; A: row lane % 16, k = lane / 16; B: k = lane / 16, column lane % 16; result register j of a
// lane: row lane / 16 + 4 j, column lane % 16): W = K_p[f][h] T (27 x na_t), its K_p operand formed
// from G, then T^T W.  K_e being symmetric only the blocks h >= f are computed, block (h, f) is their
// mirror image.
// In scatter mode entry (x, y) of block (f, h) sits in row topo[f na_t + x], field block h of that row,
// at the rank of adof y among the row adof's neighbours.  No other element of the colour touches
// the row, so the adds are hardware FP64 atomics without return (no old value travels to the CU)
// that still reach every value in colour order: the same sums on every call.
// ------------------------------------------------------------------------------------------------
template <int NF, bool SCATTER>
__global__ __launch_bounds__(256) void k_hex27_general(GenView g, const int32_t* els, const double* mom, double* vals) {
    constexpr int NB = 27;
    constexpr int SF = sf_lds<NF>();
    __shared__ double lds[SF + 2 * NB * kHex27MaxAdofsPerType];
    const int e = els[blockIdx.x];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int col16 = lane & 15, kq = lane >> 4;
    // dense element-local T (27 x na_t, the same for every dof type)
    double* Tt = lds + SF;
    double* W = Tt + NB * kHex27MaxAdofsPerType;
    const int na_t = g.na_t[e];
    const int NA = NF * na_t;
    for (int idx = tid; idx < NB * na_t; idx += 256) Tt[idx] = 0.0;
    __syncthreads();
    if (tid < NB)
        for (int q = g.t_ptr[e * NB + tid]; q < g.t_ptr[e * NB + tid + 1]; ++q) Tt[tid * na_t + g.t_col[q]] += g.t_w[q];
    sf_moments<NF>(g, mom, e, lds);
    double c0, c1, cs;
    hex27_material<NF>(g, e, c0, c1, cs);
    // HEX27 basis of row / column operand n of a tile -> its tensor index in G
    auto half = [&](int a) { return (kHex27Half[a][0] * 3 + kHex27Half[a][1]) * 3 + kHex27Half[a][2]; };
    int ah[2], bh[(NB + 3) / 4];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) ah[mt] = half(min(mt * 16 + col16, NB - 1));
#pragma unroll
    for (int ks = 0; ks < (NB + 3) / 4; ++ks) bh[ks] = half(min(4 * ks + kq, NB - 1));
    double* ke = SCATTER ? nullptr : g.ke + g.ke_off[e];
    const int32_t* rows = SCATTER ? g.topo + g.topo_ptr[e] : nullptr;
    const uint16_t* rk = SCATTER ? g.rank + g.rank_off[e] : nullptr;
    const int n_nt = (na_t + 15) / 16;   // 16-column tiles of T, W and K_e
    for (int f = 0; f < NF; ++f)
        for (int hb = f; hb < NF; ++hb) {
            const KTerms kt = k_terms<NF>(f, hb, c0, c1, cs);
            for (int tile = wave; tile < 2 * n_nt; tile += 4) {
                const int mt = tile / n_nt, nt = tile - n_nt * (tile / n_nt);
                const int arow = mt * 16 + col16, bcol = nt * 16 + col16;   // a; y
                const int a = mt ? ah[1] : ah[0];
                doublex4_t c4 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int ks = 0; ks < (NB + 3) / 4; ++ks) {
                    const int k = 4 * ks + kq;   // b
                    double av = kt.c[0] * lds[kt.base[0] + a * kt.sa[0] + bh[ks] * kt.sb[0]];
                    if (NF > 1)
                        av += kt.c[1] * lds[kt.base[1] + a * kt.sa[1] + bh[ks] * kt.sb[1]] +
                              kt.c[2] * lds[kt.base[2] + a * kt.sa[2] + bh[ks] * kt.sb[2]];
                    av = (arow < NB && k < NB) ? av : 0.0;
                    const double bv = (k < NB && bcol < na_t) ? Tt[k * na_t + bcol] : 0.0;
                    c4 = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, c4, 0, 0, 0);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int r = mt * 16 + kq + 4 * j;
                    if (r < NB && bcol < na_t) W[r * na_t + bcol] = c4[j];
                }
            }
            __syncthreads();
            for (int tile = wave; tile < n_nt * n_nt; tile += 4) {
                const int mt = tile / n_nt, nt = tile - n_nt * (tile / n_nt);
                const int xrow = mt * 16 + col16, ycol = nt * 16 + col16;   // x; y
                // scatter mode: the tile's CSR positions (and those of its mirror image in block
                // (h, f)) are requested before its MFMA work, which hides their chain of dependent
                // loads
                [[maybe_unused]] int pos[4], pos2[4];
                if constexpr (SCATTER) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int x = mt * 16 + kq + 4 * j;
                        pos[j] = pos2[j] = -1;
                        if (x < na_t && ycol < na_t) {
                            const int32_t row = rows[f * na_t + x];
                            const int32_t r0 = g.row_ptr[row], len = (g.row_ptr[row + 1] - r0) / NF;
                            pos[j] = r0 + hb * len + rk[x * na_t + ycol];
                            if (hb != f) {
                                const int32_t row2 = rows[hb * na_t + ycol];
                                const int32_t r2 = g.row_ptr[row2], len2 = (g.row_ptr[row2 + 1] - r2) / NF;
                                pos2[j] = r2 + f * len2 + rk[ycol * na_t + x];
                            }
                        }
                    }
                }
                doublex4_t c4 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int ks = 0; ks < (NB + 3) / 4; ++ks) {
                    const int k = 4 * ks + kq;   // a
                    const double av = (k < NB && xrow < na_t) ? Tt[k * na_t + xrow] : 0.0;
                    const double bv = (k < NB && ycol < na_t) ? W[k * na_t + ycol] : 0.0;
                    c4 = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, c4, 0, 0, 0);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int x = mt * 16 + kq + 4 * j;
                    if constexpr (SCATTER) {
                        if (pos[j] >= 0) unsafeAtomicAdd(vals + pos[j], c4[j]);
                        if (pos2[j] >= 0) unsafeAtomicAdd(vals + pos2[j], c4[j]);
                    } else if (x < na_t && ycol < na_t) {
                        ke[(size_t)(f * na_t + x) * NA + hb * na_t + ycol] = c4[j];
                        if (hb != f) ke[(size_t)(hb * na_t + ycol) * NA + f * na_t + x] = c4[j];
                    }
                }
            }
            __syncthreads();
        }
}

template <int NF, bool SCATTER>
void launch_elements_t(const GenView& g, int32_t n_tensor, int32_t n_general, const int32_t* els, const double* mom,
                       double* vals, hipStream_t s) {
    if (n_tensor > 0)
        hipLaunchKernelGGL((k_hex27_tensor<NF, SCATTER>), dim3((unsigned)n_tensor), dim3(256), 0, s, g, els, mom, vals);
    if (n_general > 0)
        hipLaunchKernelGGL((k_hex27_general<NF, SCATTER>), dim3((unsigned)n_general), dim3(256), 0, s, g,
                           els + n_tensor, mom, vals);
}

}  // namespace

void launch_hex27_moments(const GenView& g, double* mom, hipStream_t s) {
    hipLaunchKernelGGL(k_hex27_moments, dim3((unsigned)((g.n_el + 7) / 8 * 16)), dim3(64), 0, s, g, mom);
}

void launch_hex27_elements(const GenView& g, int nf, bool scatter, int32_t n_tensor, int32_t n_general,
                           const int32_t* els, const double* mom, double* vals, hipStream_t s) {
    if (nf == 1) {
        if (scatter) launch_elements_t<1, true>(g, n_tensor, n_general, els, mom, vals, s);
        else launch_elements_t<1, false>(g, n_tensor, n_general, els, mom, vals, s);
    } else {
        if (scatter) launch_elements_t<3, true>(g, n_tensor, n_general, els, mom, vals, s);
        else launch_elements_t<3, false>(g, n_tensor, n_general, els, mom, vals, s);
    }
}

}  // namespace mgpu
