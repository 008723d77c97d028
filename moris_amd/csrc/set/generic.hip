// generic.hip -- the generic element path of an mgpu_set: any T rows (B-spline p = 2, THB-like
// rows with several weighted entries) and sets without a lattice.
//
//   k_generic_element   one wavefront per element.  The moments
//                         M[(i,a),(j,b)] = sum_ip w* dN_a/dx_i dN_b/dx_j
//                       over the element's integration points (HEX_2x2x2 / QUAD_2x2 on the IP box
//                       when uncut, TET_11 / TRI_7 on the XTK sub-cells when cut; w* = w detJ,
//                       points with detJ < -1e-6 skipped, cl_FEM_Element_Bulk.cpp:258-355) are
//                       staged 64 points at a time in LDS; lane (a, b) owns the DIM x DIM block.
//                       K_p = B^T D B from M (IWG compute_jacobian,
//                       cl_FEM_IWG_Isotropic_Struc_Linear_Bulk.cpp:200, cl_FEM_IWG_Diffusion_Bulk.cpp
//                       :280), then K_e = T^T K_p T with the element's dense T built from its rows
//                       (Equation_Object::build_PADofMap / get_egn_obj_jacobian_and_residual,
//                       cl_MSI_Equation_Object.cpp:426-493, :789-842), in FP64 through LDS, written
//                       to the element's slot of the K_e pool.
//   hex27.hip           HEX27 IP cells (HEX_3x3x3 / TET_35): K_e from the element's moments.  In scatter
//                       mode (sets too large for a K_e pool) colour by colour, each element adding its
//                       K_e into the CSR values after k_generic_zero.
//   k_generic_rows      rows mode: one group of lanes per CSR row, the rows of the K_e holding it summed
//                       in LDS in ascending element order (deterministic SumIntoGlobalValues,
//                       cl_Sparse_Matrix_EpetraFECrs.cpp:103-133), then the row of R = K u (R_e = K_e u_e
//                       for these linear IWGs).
//   k_generic_gather    sets with rows too long for that: one thread per CSR value, the sum of its K_e
//                       entries in the same order.
//   k_generic_rhs       R = K u after k_generic_gather or scatter mode: one wavefront per row.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <numeric>
#include <type_traits>
#include <vector>

#include "../common/fem_tables.hpp"
#include "set_state.hpp"

namespace mgpu {

namespace {

template <class T>
mgpu_status gupload(mgpu_set* S, const T* src, size_t n, T** dst);

// the gather sources in 32 bits when every K_e entry index fits, else in 64 bits
mgpu_status upload_gather_src(mgpu_set* S, const std::vector<int64_t>& src, GenView& g) {
    g.gather_src = nullptr;
    g.gather_src32 = nullptr;
    const size_t n_ke = S->h.ke_off.empty() ? 0 : (size_t)S->h.ke_off.back();
    if (n_ke < ((size_t)1 << 31)) {
        std::vector<int32_t> s32(src.begin(), src.end());
        return gupload(S, s32.data(), s32.size(), const_cast<int32_t**>(&g.gather_src32));
    }
    return gupload(S, src.data(), src.size(), const_cast<int64_t**>(&g.gather_src));
}

template <class T>
mgpu_status gupload(mgpu_set* S, const T* src, size_t n, T** dst) {
    *dst = nullptr;
    if (n == 0) return MGPU_OK;
    void* p = nullptr;
    HIP_TRY(hipMalloc(&p, n * sizeof(T)));
    S->allocs.push_back(p);
    HIP_TRY(hipMemcpy(p, src, n * sizeof(T), hipMemcpyHostToDevice));
    *dst = static_cast<T*>(p);
    return MGPU_OK;
}

// Integration point ip of element e: w* and the physical gradients g[i][a] of the IP cell.
template <int DIM>
__device__ inline double generic_point(const GenView& g, int e, bool cut, int ip, const double* hh,
                                       double (*grad)[DIM == 3 ? 8 : 4]) {
    constexpr int NB = DIM == 3 ? 8 : 4;
    double xi[DIM];
    double w;
    if (!cut) {
        // IG cell = IP cell: HEX_2x2x2 / QUAD_2x2, detJ = prod(h / 2)
        for (int d = 0; d < DIM; ++d) xi[d] = DIM == 3 ? kHex2Xi[ip][d] : kQuad2Xi[ip][d];
        double detJ = 1.0;
        for (int d = 0; d < DIM; ++d) detJ *= 0.5 * hh[d];
        w = (DIM == 3 ? kHex2W[ip] : kQuad2W[ip]) * detJ;
    } else {
        constexpr int NV = DIM + 1;
        constexpr int NQ = DIM == 3 ? kTet11Points : kTri7Points;
        const int sc = g.ig_ptr[e] + ip / NQ;
        const int q = ip % NQ;
        const double* X = g.ig_xi + (size_t)sc * NV * DIM;
        double N[NV];
        if constexpr (DIM == 3) {
            N[0] = kTet11Xi[q][0];
            N[1] = kTet11Xi[q][1];
            N[2] = 1.0 - kTet11Xi[q][0] - kTet11Xi[q][1] - kTet11Xi[q][2];
            N[3] = kTet11Xi[q][2];
        } else {
            N[0] = kTri7Xi[q][0];
            N[1] = kTri7Xi[q][1];
            N[2] = 1.0 - kTri7Xi[q][0] - kTri7Xi[q][1];
        }
        for (int d = 0; d < DIM; ++d) {
            double v = 0.0;
            for (int k = 0; k < NV; ++k) v += N[k] * X[k * DIM + d];
            xi[d] = v;
        }
        double detJ;
        if constexpr (DIM == 3) {
            double J[3][3];
            const int rr[3] = {0, 1, 3};
            for (int r = 0; r < 3; ++r)
                for (int d = 0; d < 3; ++d) J[r][d] = (X[rr[r] * 3 + d] - X[2 * 3 + d]) * (0.5 * hh[d]);
            detJ = (J[0][0] * (J[1][1] * J[2][2] - J[2][1] * J[1][2]) -
                    J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                    J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0])) / 6.0;
        } else {
            double J[2][2];
            for (int r = 0; r < 2; ++r)
                for (int d = 0; d < 2; ++d) J[r][d] = (X[r * 2 + d] - X[2 * 2 + d]) * (0.5 * hh[d]);
            detJ = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) / 2.0;
        }
        w = detJ < kDetJLowerLimit ? 0.0 : (DIM == 3 ? kTet11W[q] : kTri7W[q]) * detJ;
    }
    lagrange_dNdxi<DIM>(xi, grad);
    for (int i = 0; i < DIM; ++i)
        for (int a = 0; a < NB; ++a) grad[i][a] *= 2.0 / hh[i];
    return w;
}

constexpr int kGenLds = 24 * 24 + 8 * kGenericMaxAdofsPerType + 24 * 3 * kGenericMaxAdofsPerType;

// Moment-fitted rule of a cut HEX8 / QUAD4 cell (MGPU_QUAD_MOMENT_FIT on the generic path): the
// 3^DIM tensor points of the 3-point Gauss rule with weights W_g = sum_q w*_q L_i(x_q) L_j(y_q)
// (L_k(z_q)) over the cell's TET_11 / TRI_7 points, L the quadratics through the nodes -s, 0, s.
// The (bi)trilinear moment integrand has degree <= 2 per axis, so the rule gives the subdivision's
// sum.  One wavefront: lanes over the points, then a reduction in lane order into Wg.
constexpr int kGenFitW = kGenLds - 32;   // LDS offset of the fitted weights (doubles)
template <int DIM>
__device__ inline void gen_mfit_weights(const GenView& g, int e, const double* hh, double* lds, int lane) {
    constexpr int NV = DIM + 1;
    constexpr int NQ = DIM == 3 ? kTet11Points : kTri7Points;
    constexpr int NW = DIM == 3 ? 27 : 9;
    static_assert(NW * 65 <= kGenFitW, "reduction rows and the fitted weights fit the LDS");
    const double sg = kHex3Xi[1][0];   // the 3-point Gauss node (the rule's literal)
    const int npts = (g.ig_ptr[e + 1] - g.ig_ptr[e]) * NQ;
    double acc[NW];
#pragma unroll
    for (int k = 0; k < NW; ++k) acc[k] = 0.0;
    for (int ip = lane; ip < npts; ip += 64) {
        const int sc = g.ig_ptr[e] + ip / NQ, q = ip % NQ;
        const double* X = g.ig_xi + (size_t)sc * NV * DIM;
        double N[NV];
        if constexpr (DIM == 3) {
            N[0] = kTet11Xi[q][0];
            N[1] = kTet11Xi[q][1];
            N[2] = 1.0 - kTet11Xi[q][0] - kTet11Xi[q][1] - kTet11Xi[q][2];
            N[3] = kTet11Xi[q][2];
        } else {
            N[0] = kTri7Xi[q][0];
            N[1] = kTri7Xi[q][1];
            N[2] = 1.0 - kTri7Xi[q][0] - kTri7Xi[q][1];
        }
        double L[DIM][3];
        for (int d = 0; d < DIM; ++d) {
            double x = 0.0;
            for (int k = 0; k < NV; ++k) x += N[k] * X[k * DIM + d];
            L[d][0] = x * (x - sg) / (2.0 * sg * sg);
            L[d][1] = 1.0 - x * x / (sg * sg);
            L[d][2] = x * (x + sg) / (2.0 * sg * sg);
        }
        double detJ;
        if constexpr (DIM == 3) {
            double J[3][3];
            const int rr[3] = {0, 1, 3};
            for (int r = 0; r < 3; ++r)
                for (int d = 0; d < 3; ++d) J[r][d] = (X[rr[r] * 3 + d] - X[2 * 3 + d]) * (0.5 * hh[d]);
            detJ = (J[0][0] * (J[1][1] * J[2][2] - J[2][1] * J[1][2]) -
                    J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                    J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0])) / 6.0;
        } else {
            double J[2][2];
            for (int r = 0; r < 2; ++r)
                for (int d = 0; d < 2; ++d) J[r][d] = (X[r * 2 + d] - X[2 * 2 + d]) * (0.5 * hh[d]);
            detJ = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) / 2.0;
        }
        const double w = detJ < kDetJLowerLimit ? 0.0 : (DIM == 3 ? kTet11W[q] : kTri7W[q]) * detJ;
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            const int ix = k % 3, iy = (k / 3) % 3, iz = k / 9;
            double v = w * L[0][ix] * L[1][iy];
            if constexpr (DIM == 3) v *= L[2][iz];
            acc[k] += v;
        }
    }
#pragma unroll
    for (int k = 0; k < NW; ++k) lds[k * 65 + lane] = acc[k];
    __syncthreads();
    if (lane < NW) {
        double v = 0.0;
        for (int l = 0; l < 64; ++l) v += lds[lane * 65 + l];
        lds[kGenFitW + lane] = v;
    }
    __syncthreads();
}

template <int DIM, int NF, typename T, bool MFIT>
__global__ __launch_bounds__(64) void k_generic_element(GenView g) {
    constexpr int NB = DIM == 3 ? 8 : 4;
    constexpr int NG = DIM * NB;
    constexpr int NP = NF * NB;
    constexpr int GP = NG + 1;
    static_assert(2 * 64 * GP * sizeof(T) <= kGenLds * sizeof(double), "LDS phases");
    __shared__ double lds[kGenLds];
    const int e = g.order ? g.order[blockIdx.x] : (int)blockIdx.x;
    const int lane = threadIdx.x;
    double hh[DIM];
    for (int d = 0; d < DIM; ++d) hh[d] = g.ip_box[(size_t)e * 2 * DIM + DIM + d];
    const bool cut = g.ig_ptr[e + 1] > g.ig_ptr[e];
    const bool fit = MFIT && cut;
    const int npts = fit ? (DIM == 3 ? 27 : 9)
                         : (cut ? (g.ig_ptr[e + 1] - g.ig_ptr[e]) * (DIM == 3 ? kTet11Points : kTri7Points)
                                : (DIM == 3 ? kHex2Points : kQuad2Points));
    if constexpr (MFIT)
        if (fit) gen_mfit_weights<DIM>(g, e, hh, lds, lane);

    // phase 1: moments, lane (a, b) owns M[(i,a),(j,b)], i, j < DIM
    T* sgw = reinterpret_cast<T*>(lds);
    T* sg = sgw + 64 * GP;
    const int a = (lane / NB) % NB, b = lane % NB;
    const bool owner = lane < NB * NB;
    T M[DIM][DIM];
    for (int i = 0; i < DIM; ++i)
        for (int j = 0; j < DIM; ++j) M[i][j] = T(0);
    for (int p0 = 0; p0 < npts; p0 += 64) {
        const int ip = p0 + lane;
        if (ip < npts) {
            double grad[DIM][NB];
            double w;
            if (fit) {
                // tensor point ip of the 3-point Gauss rule, x fastest, and its fitted weight
                const double nd[3] = {-kHex3Xi[1][0], 0.0, kHex3Xi[1][0]};
                double xi[DIM];
                xi[0] = nd[ip % 3];
                xi[1] = nd[(ip / 3) % 3];
                if constexpr (DIM == 3) xi[2] = nd[ip / 9];
                lagrange_dNdxi<DIM>(xi, grad);
                for (int i = 0; i < DIM; ++i)
                    for (int c = 0; c < NB; ++c) grad[i][c] *= 2.0 / hh[i];
                w = lds[kGenFitW + ip];
            } else {
                w = generic_point<DIM>(g, e, cut, ip, hh, grad);
            }
            for (int i = 0; i < DIM; ++i)
                for (int c = 0; c < NB; ++c) {
                    sgw[lane * GP + i * NB + c] = (T)(w * grad[i][c]);
                    sg[lane * GP + i * NB + c] = (T)grad[i][c];
                }
        }
        __syncthreads();
        const int np = min(64, npts - p0);
        if (owner)
            for (int p = 0; p < np; ++p)
                for (int i = 0; i < DIM; ++i)
                    for (int j = 0; j < DIM; ++j) M[i][j] += sgw[p * GP + i * NB + a] * sg[p * GP + j * NB + b];
        __syncthreads();
    }

    // phase 2: K_p (NP x NP) from M and the material
    double* Kp = lds;
    double* Tt = Kp + NP * NP;                        // [NB][na_t]
    double* W = Tt + NB * kGenericMaxAdofsPerType;     // [NP][NF * na_t]
    const int na_t = g.na_t[e];
    const int NA = NF * na_t;
    if (owner) {
        if (NF == 1) {
            double v = 0.0;
            for (int i = 0; i < DIM; ++i) v += (double)M[i][i];
            Kp[a * NP + b] = g.material[e] * v;
        } else {
            constexpr int NS = DIM == 3 ? 6 : 3;
            double D[NS][NS];
            elastic_D<DIM>(g.material[2 * e], g.material[2 * e + 1], D);
            for (int al = 0; al < DIM; ++al)
                for (int be = 0; be < DIM; ++be) {
                    double v = 0.0;
                    for (int i = 0; i < DIM; ++i)
                        for (int j = 0; j < DIM; ++j)
                            if (d_nonzero<DIM>(voigt<DIM>(al, i), voigt<DIM>(be, j)))
                                v += D[voigt<DIM>(al, i)][voigt<DIM>(be, j)] * (double)M[i][j];
                    Kp[(al * NB + a) * NP + be * NB + b] = v;
                }
        }
    }
    // phase 3: dense element-local T (per dof type; the same rows serve every type)
    for (int idx = lane; idx < NB * na_t; idx += 64) Tt[idx] = 0.0;
    __syncthreads();
    if (lane < NB)
        for (int q = g.t_ptr[e * NB + lane]; q < g.t_ptr[e * NB + lane + 1]; ++q) Tt[lane * na_t + g.t_col[q]] += g.t_w[q];
    __syncthreads();
    // phase 4: W = K_p T (block diagonal T over dof types)
    for (int idx = lane; idx < NP * NA; idx += 64) {
        const int r = idx / NA, cy = idx % NA;
        const int gg = cy / na_t, y = cy % na_t;
        double v = 0.0;
        for (int b2 = 0; b2 < NB; ++b2) v += Kp[r * NP + gg * NB + b2] * Tt[b2 * na_t + y];
        W[idx] = v;
    }
    __syncthreads();
    // phase 5: K_e = T^T W
    double* ke = g.ke + g.ke_off[e];
    for (int idx = lane; idx < NA * NA; idx += 64) {
        const int X = idx / NA, Y = idx % NA;
        const int f = X / na_t, x = X % na_t;
        double v = 0.0;
        for (int b1 = 0; b1 < NB; ++b1) v += Tt[b1 * na_t + x] * W[(f * NB + b1) * NA + Y];
        ke[idx] = v;
    }
}

__global__ void k_generic_zero(double* vals, int64_t n) {
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x)
        __builtin_nontemporal_store(0.0, vals + p);   // an output: nothing reads it back here
}

// L lanes per row (f, a): the K_e rows of the elements holding adof a, na_t NF consecutive pool values
// each, added into the row's values in LDS at the columns of the element's rank table (one table per
// element serves its NF x NF blocks).  Within an element every column is distinct, and LDS operations of
// a wavefront complete in order, so the adds (without return) reach each value in ascending element
// order: the same sums on every call.  The lanes fetch the addresses of L elements at a time.  Bound by
// the pool reads: 32^3 elements of 81 x 81 (1.7 GB) with the values and R 0.71 ms, against 1.57 + 0.12 ms
// for one thread per value with a list of its entries (12 more bytes an entry) and R after it.
template <int L, int NF>
__global__ __launch_bounds__(256) void k_generic_rows(GenView g, int max_nbr, const double* u, double* vals, double* rhs) {
    extern __shared__ double acc_all[];
    const int grp = threadIdx.x / L, lane = threadIdx.x % L;
    const int64_t gr = (int64_t)blockIdx.x * (blockDim.x / L) + grp;
    const int a = (int)(gr / NF), f = (int)(gr - (int64_t)a * NF);
    const bool live = a < g.N;
    const int row = live ? f * g.N + a : 0;
    const int r0 = live ? g.row_ptr[row] : 0, n = live ? g.row_ptr[row + 1] - r0 : 0, len = n / NF;
    double* acc = acc_all + (size_t)grp * NF * max_nbr;
    for (int q = lane; q < n; q += L) acc[q] = 0.0;
    __syncthreads();
    const int64_t q0 = live ? g.adof_ptr[a] : 0, q1 = live ? g.adof_ptr[a + 1] : 0;
    for (int64_t qb = q0; qb < q1; qb += L) {
        // the lane's element: start of its K_e row, of its rank row, its adofs per type
        int64_t ko = 0, ro = 0;
        int nt = 0;
        if (qb + lane < q1) {
            const int e = g.adof_el[qb + lane], x = g.adof_x[qb + lane];
            nt = g.na_t[e];
            ko = g.ke_off[e] + (int64_t)(f * nt + x) * (NF * nt);
            ro = g.rank_off[e] + (int64_t)x * nt;
        }
        const int cnt = (int)min((int64_t)L, q1 - qb);
#pragma unroll 4
        for (int k = 0; k < cnt; ++k) {
            const double* ke = g.ke + __shfl(ko, k, L);
            const uint16_t* rk = g.rank + __shfl(ro, k, L);
            const int na_t = __shfl(nt, k, L);
            for (int idx = lane; idx < NF * na_t; idx += L) {
                const int h = NF == 1 ? 0 : (idx >= na_t) + (NF == 3 && idx >= 2 * na_t);
                __hip_atomic_fetch_add(acc + h * len + rk[idx - h * na_t], ke[idx], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
    }
    __syncthreads();
    double v = 0.0;
    for (int q = lane; q < n; q += L) {
        const double w = acc[q];
        __builtin_nontemporal_store(w, vals + r0 + q);   // an output: nothing reads it back here
        v += w * u[g.col_idx[r0 + q]];
    }
#pragma unroll
    for (int off = L / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, L);
    if (live && lane == 0) rhs[row] = v;
}

template <typename I>
__global__ void k_generic_gather(GenView g, const I* src, double* vals) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= g.nnz) return;
    double v = 0.0;
    for (int64_t k = g.gather_ptr[p]; k < g.gather_ptr[p + 1]; ++k) v += g.ke[src[k]];
    __builtin_nontemporal_store(v, vals + p);   // an output: nothing reads it back here
}

// one wavefront per row: lanes stride over the row's values, then a butterfly reduction (a fixed
// order, so R is the same on every call)
__global__ __launch_bounds__(256) void k_generic_rhs(GenView g, const double* vals, const double* u, double* rhs) {
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r >= g.n_rows) return;
    double v = 0.0;
    for (int p = g.row_ptr[r] + lane; p < g.row_ptr[r + 1]; p += 64) v += vals[p] * u[g.col_idx[p]];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    if (lane == 0) rhs[r] = v;
}

}  // namespace

mgpu_status generic_upload(mgpu_set* S, const mgpu_set_desc& d) {
    const SetHost& h = S->h;
    GenView& g = S->g;
    g.n_el = h.n_el;
    g.N = h.n_adofs_type;
    g.n_rows = h.n_rows;
    g.nnz = (int64_t)h.col_idx.size();
    const size_t n_ig = (size_t)d.ig_ptr[h.n_el];
    const size_t n_t = (size_t)d.t_ptr[(size_t)h.n_el * h.nb];
    mgpu_status rc;
    if ((rc = gupload(S, d.ip_box, (size_t)h.n_el * 2 * h.dim, const_cast<double**>(&g.ip_box))) ||
        (rc = gupload(S, d.material, (size_t)h.n_el * h.nm, const_cast<double**>(&g.material))) ||
        (rc = gupload(S, d.ig_ptr, (size_t)h.n_el + 1, const_cast<int32_t**>(&g.ig_ptr))) ||
        (rc = gupload(S, d.ig_xi, n_ig * (h.dim + 1) * h.dim, const_cast<double**>(&g.ig_xi))) ||
        (rc = gupload(S, d.t_ptr, (size_t)h.n_el * h.nb + 1, const_cast<int32_t**>(&g.t_ptr))) ||
        (rc = gupload(S, h.t_col.data(), n_t, const_cast<int32_t**>(&g.t_col))) ||
        (rc = gupload(S, d.t_weight, n_t, const_cast<double**>(&g.t_w))) ||
        (rc = gupload(S, h.na_t.data(), h.na_t.size(), const_cast<int32_t**>(&g.na_t))) ||
        (rc = gupload(S, h.ke_off.data(), h.ke_off.size(), const_cast<int64_t**>(&g.ke_off))) ||
        (rc = gupload(S, h.row_ptr.data(), h.row_ptr.size(), const_cast<int32_t**>(&g.row_ptr))) ||
        (rc = gupload(S, h.col_idx.data(), h.col_idx.size(), const_cast<int32_t**>(&g.col_idx))))
        return rc;
    if (h.rows || h.scatter) {
        if ((rc = gupload(S, h.rank_off.data(), h.rank_off.size(), const_cast<int64_t**>(&g.rank_off))) ||
            (rc = gupload(S, h.rank.data(), h.rank.size(), const_cast<uint16_t**>(&g.rank))))
            return rc;
    }
    if (h.rows) {
        if ((rc = gupload(S, h.adof_ptr.data(), h.adof_ptr.size(), const_cast<int64_t**>(&g.adof_ptr))) ||
            (rc = gupload(S, h.adof_el.data(), h.adof_el.size(), const_cast<int32_t**>(&g.adof_el))) ||
            (rc = gupload(S, h.adof_x.data(), h.adof_x.size(), const_cast<int32_t**>(&g.adof_x))))
            return rc;
    } else if (!h.scatter) {
        if ((rc = gupload(S, h.gather_ptr.data(), h.gather_ptr.size(), const_cast<int64_t**>(&g.gather_ptr))) ||
            (rc = upload_gather_src(S, h.gather_src, g)))
            return rc;
    }
    if (h.nb == 27 && h.n_el > 0) {
        // the elements with tensor T first, within each colour (scatter mode) or over the set
        std::vector<int32_t> els(h.colour_el), cp(h.colour_ptr);
        if (!h.scatter) {
            els.resize((size_t)h.n_el);
            std::iota(els.begin(), els.end(), 0);
            cp = {0, h.n_el};
        }
        S->n_tensor.clear();
        for (size_t c = 0; c + 1 < cp.size(); ++c) {
            auto mid = std::stable_partition(els.begin() + cp[c], els.begin() + cp[c + 1], [&](int32_t e) {
                return h.t_perm[(size_t)e * kHex27PermStride + 27] != 0;
            });
            S->n_tensor.push_back((int32_t)(mid - els.begin()) - cp[c]);
        }
        void* p = nullptr;
        HIP_TRY(hipMalloc(&p, (size_t)h.n_el * kHex27Moments * sizeof(double)));
        S->allocs.push_back(p);
        S->d_mom = static_cast<double*>(p);
        if ((rc = gupload(S, els.data(), els.size(), const_cast<int32_t**>(&S->d_hex_els))) ||
            (rc = gupload(S, h.t_perm.data(), h.t_perm.size(), const_cast<uint8_t**>(&g.t_perm))))
            return rc;
    }
    if (h.scatter) {
        if ((rc = gupload(S, h.topo.data(), h.topo.size(), const_cast<int32_t**>(&g.topo))) ||
            (rc = gupload(S, h.topo_ptr.data(), h.topo_ptr.size(), const_cast<int64_t**>(&g.topo_ptr))))
            return rc;
        return MGPU_OK;   // no K_e pool
    }
    // the elements with most sub-cells first (stable), so that a launch does not end on one long
    // element; used when the tuning selects it
    {
        std::vector<int32_t> order((size_t)h.n_el);
        for (int32_t e = 0; e < h.n_el; ++e) order[(size_t)e] = e;
        std::stable_sort(order.begin(), order.end(), [&](int32_t x, int32_t y) {
            return d.ig_ptr[x + 1] - d.ig_ptr[x] > d.ig_ptr[y + 1] - d.ig_ptr[y];
        });
        if (h.n_el > 0 && (rc = gupload(S, order.data(), order.size(), const_cast<int32_t**>(&S->d_gen_order))))
            return rc;
    }
    const size_t n_ke = h.ke_off.empty() ? 0 : (size_t)h.ke_off.back();
    if (n_ke > 0) {
        void* p = nullptr;
        HIP_TRY(hipMalloc(&p, n_ke * sizeof(double)));
        S->allocs.push_back(p);
        g.ke = static_cast<double*>(p);
    }
    return MGPU_OK;
}

namespace {
template <bool MFIT>
void launch_generic_element(mgpu_set* S, bool f32, dim3 gr, dim3 bl) {
    const SetHost& h = S->h;
    if (h.dim == 3 && h.nf == 1) {
        if (f32) hipLaunchKernelGGL((k_generic_element<3, 1, float, MFIT>), gr, bl, 0, S->stream, S->g);
        else hipLaunchKernelGGL((k_generic_element<3, 1, double, MFIT>), gr, bl, 0, S->stream, S->g);
    } else if (h.dim == 3) {
        if (f32) hipLaunchKernelGGL((k_generic_element<3, 3, float, MFIT>), gr, bl, 0, S->stream, S->g);
        else hipLaunchKernelGGL((k_generic_element<3, 3, double, MFIT>), gr, bl, 0, S->stream, S->g);
    } else if (h.nf == 1) {
        if (f32) hipLaunchKernelGGL((k_generic_element<2, 1, float, MFIT>), gr, bl, 0, S->stream, S->g);
        else hipLaunchKernelGGL((k_generic_element<2, 1, double, MFIT>), gr, bl, 0, S->stream, S->g);
    } else {
        if (f32) hipLaunchKernelGGL((k_generic_element<2, 2, float, MFIT>), gr, bl, 0, S->stream, S->g);
        else hipLaunchKernelGGL((k_generic_element<2, 2, double, MFIT>), gr, bl, 0, S->stream, S->g);
    }
}


// Lanes per row: 16, 32 or 64, the least that holds the longest K_e row (64 at most) and lets a
// wavefront's rows fit kRowsMaxLds; as many rows a block as that space and 256 threads allow.
template <int L, int NF>
void launch_rows_t(mgpu_set* S, const double* u, double* vals, double* rhs) {
    const int row_bytes = NF * std::max(S->h.max_nbr, 1) * (int)sizeof(double);
    int groups = 256 / L;
    while (groups * L > 64 && groups * row_bytes > kRowsMaxLds) groups /= 2;
    const int64_t n = (int64_t)NF * S->g.N;
    hipLaunchKernelGGL((k_generic_rows<L, NF>), dim3((unsigned)((n + groups - 1) / groups)), dim3((unsigned)(groups * L)),
                       (size_t)groups * row_bytes, S->stream, S->g, std::max(S->h.max_nbr, 1), u, vals, rhs);
}
void launch_rows(mgpu_set* S, const double* u, double* vals, double* rhs) {
    const int nf = S->h.nf, na = nf * S->h.na_t_max;
    if (S->h.n_rows == 0) return;
    auto go = [&](auto nfc) {
        constexpr int NF = decltype(nfc)::value;
        const int row_bytes = NF * S->h.max_nbr * (int)sizeof(double);
        if (na <= 16 && 4 * row_bytes <= kRowsMaxLds) launch_rows_t<16, NF>(S, u, vals, rhs);
        else if (na <= 32 && 2 * row_bytes <= kRowsMaxLds) launch_rows_t<32, NF>(S, u, vals, rhs);
        else launch_rows_t<64, NF>(S, u, vals, rhs);
    };
    if (nf == 1) go(std::integral_constant<int, 1>{});
    else if (nf == 2) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 3>{});
}
}  // namespace

mgpu_status launch_generic(mgpu_set* S, const double* u, double* vals, double* rhs, hipEvent_t* ev) {
    const SetHost& h = S->h;
    if (ev)
        for (int k = 0; k < 3; ++k) HIP_TRY(hipEventRecord(ev[k], S->stream));
    if (h.n_el > 0) {
        const bool f32 = S->precision == MGPU_PREC_MIXED;
        const dim3 gr((unsigned)h.n_el), bl(64);
        if (h.nb == 27 && h.scatter) {
            // zero the values, then the elements colour by colour
            launch_hex27_moments(S->g, S->d_mom, S->stream);
            if (S->g.nnz > 0)
                hipLaunchKernelGGL(k_generic_zero, dim3((unsigned)std::min<int64_t>((S->g.nnz + 255) / 256, 65536)),
                                   dim3(256), 0, S->stream, vals, S->g.nnz);
            for (size_t c = 0; c + 1 < h.colour_ptr.size(); ++c) {
                const int32_t c0 = h.colour_ptr[c], cnt = h.colour_ptr[c + 1] - c0;
                if (cnt > 0)
                    launch_hex27_elements(S->g, h.nf, true, S->n_tensor[c], cnt - S->n_tensor[c], S->d_hex_els + c0,
                                          S->d_mom, vals, S->stream);
            }
        } else if (h.nb == 27) {
            launch_hex27_moments(S->g, S->d_mom, S->stream);
            launch_hex27_elements(S->g, h.nf, false, S->n_tensor[0], h.n_el - S->n_tensor[0], S->d_hex_els, S->d_mom,
                                  vals, S->stream);
        } else if (S->quadrature == MGPU_QUAD_MOMENT_FIT) {
            launch_generic_element<true>(S, f32, gr, bl);
        } else {
            launch_generic_element<false>(S, f32, gr, bl);
        }
        HIP_TRY(hipGetLastError());
    }
    if (ev) HIP_TRY(hipEventRecord(ev[3], S->stream));
    if (h.rows) {
        launch_rows(S, u, vals, rhs);
    } else if (S->g.nnz > 0 && !h.scatter) {
        const dim3 gg((unsigned)((S->g.nnz + 255) / 256));
        if (S->g.gather_src32)
            hipLaunchKernelGGL(k_generic_gather<int32_t>, gg, dim3(256), 0, S->stream, S->g, S->g.gather_src32, vals);
        else
            hipLaunchKernelGGL(k_generic_gather<int64_t>, gg, dim3(256), 0, S->stream, S->g, S->g.gather_src, vals);
    }
    HIP_TRY(hipGetLastError());
    if (ev) HIP_TRY(hipEventRecord(ev[4], S->stream));
    if (h.n_rows > 0 && !h.rows)
        hipLaunchKernelGGL(k_generic_rhs, dim3((unsigned)((h.n_rows + 3) / 4)), dim3(256), 0, S->stream, S->g,
                           vals, u, rhs);
    HIP_TRY(hipGetLastError());
    if (ev) HIP_TRY(hipEventRecord(ev[5], S->stream));
    return MGPU_OK;
}

}  // namespace mgpu
