// generic.hip -- the generic element path of an mgpu_set: any T rows (B-spline p = 2, THB-like
// rows with several weighted entries) and sets without a lattice.
//
//   k_generic_nodal, k_generic_element
//                       HEX8 / QUAD4 IP cells, one wavefront per element.  The moments
//                         M[(i,a),(j,b)] = sum_ip w* dN_a/dx_i dN_b/dx_j
//                       over the element's integration points (HEX_2x2x2 / QUAD_2x2 on the IP box
//                       when uncut, TET_11 / TRI_7 on the XTK sub-cells when cut; w* = w detJ,
//                       points with detJ < -1e-6 skipped, cl_FEM_Element_Bulk.cpp:258-355) come
//                       from the cell's 3^dim moments (cut_moments.hpp), in FP64 with either
//                       quadrature and at either precision option.  K_p = B^T D B from M (IWG
//                       compute_jacobian, cl_FEM_IWG_Isotropic_Struc_Linear_Bulk.cpp:200,
//                       cl_FEM_IWG_Diffusion_Bulk.cpp:280), then K_e = T^T K_p T with the element's
//                       dense T built from its rows (Equation_Object::build_PADofMap /
//                       get_egn_obj_jacobian_and_residual, cl_MSI_Equation_Object.cpp:426-493,
//                       :789-842), in FP64 through LDS, written to the element's slot of the K_e
//                       pool; with nodal rows K_e is K_p in adof order.  HEX8 elements with uniform
//                       p = 2 rows: k_hex8_moments, then k_hex27_tensor.
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
#include "cut_moments.hpp"
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

// The element's moments in m (LDS): of the cut cell's points, or of the whole cell.  scratch: LDS.
template <int DIM>
__device__ __forceinline__ void generic_moments(const GenView& g, int e, double* scratch, double* m, double* hh) {
    for (int d = 0; d < DIM; ++d) hh[d] = g.ip_box[(size_t)e * 2 * DIM + DIM + d];
    const int ig0 = g.ig_ptr[e], nsub = g.ig_ptr[e + 1] - ig0;
    if (nsub > 0) cut_moments<DIM>(g.ig_xi, ig0, nsub, hh, scratch, m);
    else whole_moments<DIM>(hh, m);
}

// K_p's entries of the vertex pair (a, b): kv[al DIM + be] (elasticity) or kv[0].
template <int DIM, int NF>
__device__ __forceinline__ void generic_kp(const GenView& g, int e, const double* m, const double* hh, int a, int b, double* kv) {
    double M[DIM][DIM];
    moment_block<DIM>(m, a, b, hh, M);
    if constexpr (NF == 1) {
        double v = 0.0;
#pragma unroll
        for (int i = 0; i < DIM; ++i) v += M[i][i];
        kv[0] = g.material[e] * v;
    } else {
        constexpr int NS = DIM == 3 ? 6 : 3;
        double D[NS][NS];
        elastic_D<DIM>(g.material[2 * e], g.material[2 * e + 1], D);
#pragma unroll
        for (int al = 0; al < DIM; ++al)
#pragma unroll
            for (int be = 0; be < DIM; ++be) kv[al * DIM + be] = elastic_entry<DIM>(D, M, al, be);
    }
}

// Elements with nodal T rows (a permutation): K_e is K_p with rows and columns in adof order, each lane (a, b)
// storing its entries; no T products and no LDS for them, so that six times as many wavefronts fit
// a CU as with the general kernel below.  62120 elements, elasticity (40^3 cells): 0.09 ms, 0.81 ms
// with the point-wise moments and the dense T products.
template <int DIM, int NF>
__global__ __launch_bounds__(64) void k_generic_nodal(GenView g, const int32_t* els) {
    constexpr int NB = DIM == 3 ? 8 : 4, NA = NF * NB;
    __shared__ __align__(16) double lds[LinearMoments<DIM>::LDS];
    __shared__ double m[LinearMoments<DIM>::N];
    const int e = els[blockIdx.x], lane = threadIdx.x;
    double hh[DIM], kv[NF * NF];
    generic_moments<DIM>(g, e, lds, m, hh);
    if (lane >= NB * NB) return;
    const int a = lane / NB, b = lane % NB;
    generic_kp<DIM, NF>(g, e, m, hh, a, b, kv);
    const int x = g.t_col[g.t_ptr[e * NB + a]], y = g.t_col[g.t_ptr[e * NB + b]];
    double* ke = g.ke + g.ke_off[e];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int h = 0; h < NF; ++h) ke[(f * NB + x) * NA + h * NB + y] = kv[f * NF + h];
}

// HEX8 elements with the 27 adofs of uniform quadratic B-splines: their moments in the layout that
// k_hex27_tensor contracts (5 per axis, the last two zero), T folded into its tables: on the cell the B-splines
// are their linear interpolants l_0 / 2, 1 / 2, l_1 / 2 = f_0 l_0 + f_1 l_1, the derivatives constant.
__global__ __launch_bounds__(64) void k_hex8_moments(GenView g, const int32_t* els, double* mom) {
    __shared__ __align__(16) double lds[LinearMoments<3>::LDS];
    __shared__ double m[LinearMoments<3>::N];
    const int e = els[blockIdx.x];
    double hh[3];
    generic_moments<3>(g, e, lds, m, hh);
    double* out = mom + (size_t)e * kHex27MomStride;
    for (int t = threadIdx.x; t < kHex27Moments; t += 64) {
        const int i = t / 25, j = (t / 5) % 5, k = t % 5;
        out[t] = i < 3 && j < 3 && k < 3 ? m[(i * 3 + j) * 3 + k] : 0.0;
    }
    if (threadIdx.x == 0) out[kHex27Moments] = 1.0;
    if (threadIdx.x < 54) {
        const int r = threadIdx.x % 18, al = (r % 9) / 3, k = r % 3;
        out[kHex27MomTab + threadIdx.x] =
            k == 2 ? 0.0 : (r >= 9 ? 0.25 * (al - 1) : (al == 1 || al == 2 * k ? 0.5 : 0.0));
    }
}

// Any other T rows: K_p in LDS, then K_e = T^T K_p T with dense T, one column block (dof type) at a time.
template <int DIM, int NF>
__global__ __launch_bounds__(64) void k_generic_element(GenView g, const int32_t* els) {
    constexpr int NB = DIM == 3 ? 8 : 4;
    constexpr int NP = NF * NB;
    constexpr int MX = kGenericMaxAdofsPerType;
    constexpr int kT = NP * NP, kW = kT + NB * MX;
    // (the moments' scratch is dead once m is formed)
    constexpr int kLds = kW + NP * MX > LinearMoments<DIM>::LDS ? kW + NP * MX : LinearMoments<DIM>::LDS;
    __shared__ __align__(16) double lds[kLds];
    __shared__ double m[LinearMoments<DIM>::N];
    const int e = els[blockIdx.x], lane = threadIdx.x;
    double hh[DIM];
    generic_moments<DIM>(g, e, lds, m, hh);
    double* Kp = lds;
    double* Tt = lds + kT;   // [NB][na_t]
    double* W = lds + kW;    // [NP][na_t]
    const int na_t = g.na_t[e];
    const int NA = NF * na_t;
    if (lane < NB * NB) {
        const int a = lane / NB, b = lane % NB;
        double kv[NF * NF];
        generic_kp<DIM, NF>(g, e, m, hh, a, b, kv);
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int h = 0; h < NF; ++h) Kp[(f * NB + a) * NP + h * NB + b] = kv[f * NF + h];
    }
    // dense element-local T (per dof type; the same rows serve every type)
    for (int idx = lane; idx < NB * na_t; idx += 64) Tt[idx] = 0.0;
    __syncthreads();
    if (lane < NB)
        for (int q = g.t_ptr[e * NB + lane]; q < g.t_ptr[e * NB + lane + 1]; ++q) Tt[lane * na_t + g.t_col[q]] += g.t_w[q];
    __syncthreads();
    double* ke = g.ke + g.ke_off[e];
    for (int h = 0; h < NF; ++h) {
        // W = K_p(:, h) T
        for (int idx = lane; idx < NP * na_t; idx += 64) {
            const int r = idx / na_t, y = idx - na_t * r;
            double v = 0.0;
#pragma unroll
            for (int b = 0; b < NB; ++b) v += Kp[r * NP + h * NB + b] * Tt[b * na_t + y];
            W[idx] = v;
        }
        __syncthreads();
        // K_e(:, h) = T^T W
        for (int idx = lane; idx < NA * na_t; idx += 64) {
            const int X = idx / na_t, y = idx - na_t * X;
            const int f = X / na_t, x = X - na_t * f;
            double v = 0.0;
#pragma unroll
            for (int b = 0; b < NB; ++b) v += Tt[b * na_t + x] * W[(f * NB + b) * na_t + y];
            ke[(size_t)X * NA + h * na_t + y] = v;
        }
        __syncthreads();
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
// the pool reads (28672 elements of 81 x 81: 2.04 GB fetched, 0.34 GB written by the counters, 0.62 ms, 3.8 TB/s):
// 32768 elements (1.7 GB of pool) with the values and R 0.71 ms, against 1.57 + 0.12 ms for one thread
// per value with a list of its entries (12 more bytes an entry) and R after it.
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
    // the K_e pool first: large HEX27 sets do without where the memory is short
    const size_t n_ke = h.ke_off.empty() ? 0 : (size_t)h.ke_off.back();
    if (n_ke > 0 && !h.scatter) {
        void* p = nullptr;
        const bool optional = h.nb == 27 && h.rows && (int64_t)n_ke > kGatherMaxEntries;
        bool pool = true;
        if (optional) {
            size_t free_bytes = 0, total = 0;
            pool = hipMemGetInfo(&free_bytes, &total) == hipSuccess &&
                   !scatter_by_memory(h.nb, h.rows, (int64_t)n_ke, free_bytes) &&
                   hipMalloc(&p, n_ke * sizeof(double)) == hipSuccess;
            if (!pool) (void)hipGetLastError();
        } else {
            HIP_TRY(hipMalloc(&p, n_ke * sizeof(double)));
        }
        if (pool) {
            S->allocs.push_back(p);
            g.ke = static_cast<double*>(p);
        } else {
            rows_to_scatter(d, S->h);
        }
    }
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
    auto tensor = [&](int32_t e) { return !h.t_perm.empty() && h.t_perm[(size_t)e * kHex27PermStride + 27] != 0; };
    bool any_tensor = false;
    for (int32_t e = 0; e < h.n_el && !any_tensor; ++e) any_tensor = tensor(e);
    if (h.n_el > 0 && (h.nb == 27 || any_tensor)) {
        void* p = nullptr;
        HIP_TRY(hipMalloc(&p, (size_t)h.n_el * kHex27MomStride * sizeof(double)));
        S->allocs.push_back(p);
        S->d_mom = static_cast<double*>(p);
        if ((rc = gupload(S, h.t_perm.data(), h.t_perm.size(), const_cast<uint8_t**>(&g.t_perm)))) return rc;
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
            auto mid = std::stable_partition(els.begin() + cp[c], els.begin() + cp[c + 1], tensor);
            S->n_tensor.push_back((int32_t)(mid - els.begin()) - cp[c]);
        }
        if ((rc = gupload(S, els.data(), els.size(), const_cast<int32_t**>(&S->d_els)))) return rc;
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
        if (h.nb != 27 && h.n_el > 0) {
            // HEX8 / QUAD4 elements by class (nodal rows, tensor rows, any other), in element order and
            // most sub-cells first
            std::vector<uint8_t> cls((size_t)h.n_el, 2);
            for (int32_t e = 0; e < h.n_el; ++e) {
                bool nodal = h.na_t[(size_t)e] == h.nb;
                for (int64_t q = (int64_t)e * h.nb; q < (int64_t)(e + 1) * h.nb && nodal; ++q)
                    nodal = d.t_ptr[q + 1] - d.t_ptr[q] == 1 && d.t_weight[d.t_ptr[q]] == 1.0;
                cls[(size_t)e] = nodal ? 0 : (tensor(e) ? 1 : 2);
            }
            std::vector<int32_t> els((size_t)h.n_el);
            std::iota(els.begin(), els.end(), 0);
            for (int c = 0; c < 3; ++c) S->n_class[c] = (int32_t)std::count(cls.begin(), cls.end(), (uint8_t)c);
            auto by_class = [&](int32_t x, int32_t y) { return cls[(size_t)x] < cls[(size_t)y]; };
            std::stable_sort(els.begin(), els.end(), by_class);
            std::stable_sort(order.begin(), order.end(), by_class);
            if ((rc = gupload(S, els.data(), els.size(), const_cast<int32_t**>(&S->d_els))) ||
                (rc = gupload(S, order.data(), order.size(), const_cast<int32_t**>(&S->d_els_order))))
                return rc;
        }
    }
    return MGPU_OK;
}

namespace {
template <int DIM, int NF>
void launch_linear_elements(mgpu_set* S, double* vals) {
    const int32_t* els = S->g.order ? S->d_els_order : S->d_els;
    const int32_t n0 = S->n_class[0], n1 = S->n_class[1], n2 = S->n_class[2];
    if (n0 > 0) hipLaunchKernelGGL((k_generic_nodal<DIM, NF>), dim3((unsigned)n0), dim3(64), 0, S->stream, S->g, els);
    if (n1 > 0) {
        hipLaunchKernelGGL(k_hex8_moments, dim3((unsigned)n1), dim3(64), 0, S->stream, S->g, els + n0, S->d_mom);
        launch_hex27_elements(S->g, NF, false, n1, 0, els + n0, S->d_mom, vals, S->stream);
    }
    if (n2 > 0)
        hipLaunchKernelGGL((k_generic_element<DIM, NF>), dim3((unsigned)n2), dim3(64), 0, S->stream, S->g, els + n0 + n1);
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
        if (h.nb == 27 && h.scatter) {
            // zero the values, then the elements colour by colour
            launch_hex27_moments(S->g, S->d_mom, S->stream);
            if (S->g.nnz > 0)
                hipLaunchKernelGGL(k_generic_zero, dim3((unsigned)std::min<int64_t>((S->g.nnz + 255) / 256, 65536)),
                                   dim3(256), 0, S->stream, vals, S->g.nnz);
            for (size_t c = 0; c + 1 < h.colour_ptr.size(); ++c) {
                const int32_t c0 = h.colour_ptr[c], cnt = h.colour_ptr[c + 1] - c0;
                if (cnt > 0)
                    launch_hex27_elements(S->g, h.nf, true, S->n_tensor[c], cnt - S->n_tensor[c], S->d_els + c0,
                                          S->d_mom, vals, S->stream);
            }
        } else if (h.nb == 27) {
            launch_hex27_moments(S->g, S->d_mom, S->stream);
            launch_hex27_elements(S->g, h.nf, false, S->n_tensor[0], h.n_el - S->n_tensor[0], S->d_els, S->d_mom,
                                  vals, S->stream);
        } else if (h.dim == 3) {
            if (h.nf == 1) launch_linear_elements<3, 1>(S, vals);
            else launch_linear_elements<3, 3>(S, vals);
        } else {
            if (h.nf == 1) launch_linear_elements<2, 1>(S, vals);
            else launch_linear_elements<2, 2>(S, vals);
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
