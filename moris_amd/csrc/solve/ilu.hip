// ilu.hip -- incomplete LU preconditioner ILU(k) on the GPU, for the GMRES solve of assembled
// systems.  Target: gfx950 (MI355X), 64-wide wavefronts.
//
// The reference's solver pairs AztecOO GMRES with an incomplete factorisation of each subdomain
// (AZ_precond = AZ_dom_decomp, AZ_subdomain_solve = AZ_ilu, AZ_graph_fill = k: ILU(k),
// projects/SOL/DLA/src/cl_DLA_Linear_Solver_Aztec.cpp:353-380; UT_MDL_XTK_HMR_Linear_Struc_2D.cpp
// :990-993 solves with AZ_gmres + AZ_ilu).  Aztec itself is a Trilinos package that is not part of
// the reference sources; the algorithm restated here is the published ILU(k) (Saad, Iterative
// Methods for Sparse Linear Systems, 2nd ed., Algorithm 10.4 (ILU(0), IKJ order) and Algorithm
// 10.5 / eq. 10.14 (level of fill: lev(a_ij) = min(lev(a_ij), lev(a_ik) + lev(a_kj) + 1), fill
// kept up to level k)).
//
//   symbolic (host, once per pattern)   the factor pattern (the matrix pattern plus the fill of level
//                                       <= k, every diagonal present), the diagonal positions and
//                                       two level schedules: row i's forward level is one more than
//                                       the largest of the rows k < i in its pattern, its backward
//                                       level one more than the largest of the rows j > i
//                                       and, per lower entry, the entries of its row that it updates
//   numeric (device, per matrix)        k_ilu_fill / k_ilu_scatter copy K into the factor pattern;
//                                       one launch per forward level of k_ilu_row, one workgroup of
//                                       one wavefront per row: the row in LDS, for each k < i in
//                                       order a_ik /= u_kk, then the lanes update the entries j > k
//                                       of the row by the listed entries of row k's upper part
//   apply (device)                      z = U^-1 L^-1 v: k_ilu_tri, one workgroup with the vector in
//                                       LDS and a barrier per level; long vectors and wide levels one
//                                       launch per forward level of k_ilu_lower (one wavefront per
//                                       row, butterfly sum in a fixed order), then per backward level
//                                       of k_ilu_upper
// Every value is FP64, every sum in a fixed order: the factors and the applied vectors are the
// same on every call.
#include "ilu.hpp"

#include <algorithm>
#include <cstring>
#include <map>
#include <memory>
#include <string>
#include <type_traits>

#include "../../../include/moris_gpu_solve.h"
#include "../setup/internal.hpp"

#define ILU_TRY(expr)                                                                              \
    do {                                                                                           \
        hipError_t _e = (expr);                                                                    \
        if (_e != hipSuccess)                                                                      \
            return mgpu::set_error(MGPU_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(_e)); \
    } while (0)

namespace mgpu {
namespace ilu {

constexpr int kMaxRow = 5000;   // longest factor row the numeric kernel keeps in LDS (60 KB)
constexpr size_t kMaxUpdates = (size_t)1 << 25;   // elimination lists up to 256 MiB; beyond, the rows are searched
// Stream of k_ilu_tri (24 bytes a slot) up to 512 MiB; beyond, a launch per level.  A level takes a step's 512
// slots however few rows it has: 16383 rows of one level each 0.40 GB (5.6 ms a solve against 80 launched),
// rows of 1000 entries each side would take 6.4 GB beside 0.4 GB of factor.
constexpr size_t kMaxTriBytes = (size_t)1 << 29;
// A step of k_ilu_tri and a level launched on its own, in microseconds: 0.17 .. 0.21 (8825, 8000 and 15625 rows,
// 1264, 672 and 1184 steps: 0.22, 0.15 and 0.26 ms a call) and 3.2 .. 3.5 (8825 rows, 400 levels: 1.4 ms; 216k
// and 729k rows, 828 and 1248 levels: 2.6 and 4.1 ms).
constexpr double kTriStepUs = 0.17, kLevelUs = 3.5;

__global__ void k_ilu_clear(int32_t* err) {
    if (threadIdx.x == 0) err[0] = 0;
}

__global__ __launch_bounds__(256) void k_ilu_fill(int64_t n, double* lu) {
    for (int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x; p < n; p += (int64_t)gridDim.x * 256) lu[p] = 0.0;
}

__global__ __launch_bounds__(256) void k_ilu_scatter(int64_t n, const int32_t* pos, const double* vals, double* lu) {
    for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (int64_t)gridDim.x * 256) lu[pos[k]] = vals[k];
}

// One row of the numeric factorisation (IKJ order); rows of earlier levels are final.  LIST: the entries
// updated by each lower entry come from the elimination lists, those of kRowAhead lower entries requested
// at a time (the loads of a row would otherwise wait for each other: 8.8k rows of about 30, 200 levels,
// 7.3 ms per factorisation with binary searches, 3.1 ms with the lists).
constexpr int kRowAhead = 16;
template <bool LIST>
__global__ __launch_bounds__(64) void k_ilu_row(const int32_t* rows, const int32_t* rp, const int32_t* ci,
                                                const int32_t* diag, const int64_t* upd_ptr, const int2* upd,
                                                double* lu, int32_t* err, int max_row) {
    extern __shared__ double sm[];
    double* v = sm;
    int32_t* c = reinterpret_cast<int32_t*>(sm + max_row);
    const int i = rows[blockIdx.x];
    const int lane = threadIdx.x;
    const int r0 = rp[i], len = rp[i + 1] - r0, dpos = diag[i] - r0;
    for (int q = lane; q < len; q += 64) {
        v[q] = lu[r0 + q];
        c[q] = ci[r0 + q];
    }
    __syncthreads();
    if constexpr (LIST) {
        for (int pb = 0; pb < dpos; pb += kRowAhead) {
            // the pivots and the first 64 updates of the coming lower entries
            const int np = min(kRowAhead, dpos - pb);
            // (without branches around the loads: each would wait for its own)
            double piv[kRowAhead], uu[kRowAhead];
            int64_t a0[kRowAhead + 1];
            int2 t[kRowAhead];
#pragma unroll
            for (int k = 0; k <= kRowAhead; ++k) a0[k] = upd_ptr[r0 + pb + min(k, np)];
#pragma unroll
            for (int k = 0; k < kRowAhead; ++k) {
                t[k] = upd[a0[k] + lane < a0[k + 1] ? a0[k] + lane : 0];
                piv[k] = lu[diag[c[pb + min(k, np - 1)]]];
            }
#pragma unroll
            for (int k = 0; k < kRowAhead; ++k) uu[k] = lu[t[k].y];
#pragma unroll
            for (int k = 0; k < kRowAhead; ++k) {
                if (k >= np) break;
                const double lik = v[pb + k] / piv[k];
                if (piv[k] == 0.0 && lane == 0) err[0] = 1;
                __syncthreads();   // every lane has read v[pb + k]
                if (lane == 0) v[pb + k] = lik;
                if (a0[k] + lane < a0[k + 1]) v[t[k].x] -= lik * uu[k];
                for (int64_t j = a0[k] + 64 + lane; j < a0[k + 1]; j += 64) v[upd[j].x] -= lik * lu[upd[j].y];
                __syncthreads();
            }
        }
    } else {
        for (int p = 0; p < dpos; ++p) {
            const int k = c[p];
            const double piv = lu[diag[k]];
            const double lik = v[p] / piv;
            if (piv == 0.0 && lane == 0) err[0] = 1;
            __syncthreads();   // every lane has read v[p]
            if (lane == 0) v[p] = lik;
            const int u0 = diag[k] + 1, u1 = rp[k + 1];
            for (int q = p + 1 + lane; q < len; q += 64) {
                const int j = c[q];
                int lo = u0, hi = u1;
                while (lo < hi) {
                    const int mid = lo + ((hi - lo) >> 1);
                    if (ci[mid] < j) lo = mid + 1;
                    else hi = mid;
                }
                if (lo < u1 && ci[lo] == j) v[q] -= lik * lu[lo];
            }
            __syncthreads();
        }
    }
    for (int q = lane; q < len; q += 64) lu[r0 + q] = v[q];
    if (lane == 0 && v[dpos] == 0.0) err[0] = 1;
}

// ------------------------------------------------------------------------------------------------
// k_ilu_tri: both triangular solves in one workgroup, the vector in LDS.  A level costs a barrier instead
// of a launch.  The factor is streamed in level order, kTriThreads slots a step, L lanes per row and
// kTriThreads / L rows a step (rows with more entries take several steps); a step's loads do not
// depend on the vector and are requested kTriAhead steps before their use.  A slot's word holds its
// column, its row, and whether the step ends its rows (the lanes' sums are added and the row is
// finished) and its level (barrier).  Empty slots and rows point at an element beyond the vector that
// stays 0.  Every sum is taken in a fixed order.  Bound by the slots in flight to one CU (16 bytes a slot,
// 512 threads x 16 steps ahead; 256 x 32 took 0.24, 1024 x 16 0.28 ms): 8825 rows, 400 levels 0.2 ms, 1.4 ms with
// a launch per level.
// ------------------------------------------------------------------------------------------------
constexpr int kTriThreads = 512, kTriAhead = 16;
constexpr int kTriMaxRows = 16383;   // 14-bit indices, the last one the empty slots'; 128 KB of LDS
constexpr uint32_t kTriRowEnd = 1u << 30, kTriLevelEnd = 1u << 31;

// sum over each run of L lanes, the same in all of them
template <int L>
__device__ __forceinline__ double lanes_sum(double s) {
    auto dpp = [](double x, auto ctrl) {
        constexpr int C = decltype(ctrl)::value;
        const uint64_t u = __double_as_longlong(x);
        const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, C, 0xf, 0xf, true);
        const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), C, 0xf, 0xf, true);
        return __longlong_as_double(((uint64_t)hi << 32) | lo);
    };
    s += dpp(s, std::integral_constant<int, 0xB1>{});    // lane ^ 1
    s += dpp(s, std::integral_constant<int, 0x4E>{});    // lane ^ 2
    if constexpr (L >= 8) s += dpp(s, std::integral_constant<int, 0x141>{});    // mirrored in 8
    if constexpr (L >= 16) s += dpp(s, std::integral_constant<int, 0x140>{});   // mirrored in 16
    if constexpr (L >= 32) s += __shfl_xor(s, 16);
    if constexpr (L >= 64) s += __shfl_xor(s, 32);
    return s;
}

struct __align__(16) TriSlot {
    double a;        // the factor entry (0: none)
    uint32_t meta;   // column, row, flags
    uint32_t dword;  // backward, last step of a row: lanes 0 and 1 of the row hold its diagonal's words
};

constexpr size_t kTriSlotBytes = sizeof(TriSlot) + 2 * sizeof(int32_t);   // with its factor and diagonal entry

template <int L>
__global__ __launch_bounds__(kTriThreads) void k_ilu_tri(int32_t n, int32_t n_fwd, int32_t n_bwd, const TriSlot* slots,
                                                         const double* src, double* dst, const int32_t* skip) {
    __shared__ double y[kTriMaxRows + 1];
    if (skip && *skip) return;
    const unsigned tid = threadIdx.x;
    for (int r = (int)tid; r < n; r += kTriThreads) y[r] = src[r];
    if (tid == 0) y[n] = 0.0;
    typedef uint32_t word4 __attribute__((ext_vector_type(4)));
    word4 sl[kTriAhead];
    auto request = [&](int k, int t) { sl[k] = reinterpret_cast<const word4*>(slots + (size_t)t * kTriThreads)[tid]; };
    auto solve = [&](int t0, int t1, auto bwd) {
        constexpr bool BWD = decltype(bwd)::value;
#pragma unroll
        for (int k = 0; k < kTriAhead; ++k) request(k, t0 + k);   // (the steps come in multiples of kTriAhead)
        double s = 0.0, yv = y[sl[0][2] & 16383];
        for (int t = t0; t < t1; t += kTriAhead) {
#pragma unroll
            for (int k = 0; k < kTriAhead; ++k) {
                const word4 w = sl[k];
                const uint32_t wn = sl[(k + 1) % kTriAhead][2], flags = __builtin_amdgcn_readfirstlane(w[2]);
                request(k, min(t + kTriAhead, t1 - kTriAhead) + k);   // (past the end: repeated, unused)
                // the next step's elements, now unless this step ends their level
                double yn = 0.0;
                if (!(flags & kTriLevelEnd)) yn = y[wn & 16383];
                s += __longlong_as_double(((uint64_t)w[1] << 32) | w[0]) * yv;
                if (flags & kTriRowEnd) {
                    const int row = (w[2] >> 14) & 16383;
                    double v = y[row] - lanes_sum<L>(s);
                    if constexpr (BWD) {
                        const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)w[3], 0xB1, 0xf, 0xf, true);   // lane ^ 1
                        v /= __longlong_as_double(((uint64_t)hi << 32) | w[3]);
                    }
                    if (tid % L == 0) y[row] = v;
                    s = 0.0;
                }
                if (flags & kTriLevelEnd) {
                    __syncthreads();
                    yn = y[wn & 16383];
                }
                yv = yn;
            }
        }
    };
    __syncthreads();
    if (n_fwd > 0) solve(0, n_fwd, std::false_type{});
    if (n_bwd > 0) solve(n_fwd, n_fwd + n_bwd, std::true_type{});
    __syncthreads();
    for (int r = (int)tid; r < n; r += kTriThreads) dst[r] = y[r];
}

// The factor's values into the stream: dpos[k] >= 0: slot k holds the low word of that diagonal entry, its
// neighbour the high word (-2: the pair of an empty row, 1.0; -1: neither).
__global__ __launch_bounds__(256) void k_ilu_pack(int64_t n, const int32_t* pos, const int32_t* dpos, const double* lu,
                                                  TriSlot* slots) {
    for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (int64_t)gridDim.x * 256) {
        slots[k].a = pos[k] >= 0 ? lu[pos[k]] : 0.0;
        if (dpos[k] != -1) {
            const uint64_t d = __double_as_longlong(dpos[k] >= 0 ? lu[dpos[k]] : 1.0);
            slots[k].dword = (uint32_t)d;
            slots[k + 1].dword = (uint32_t)(d >> 32);
        }
    }
}

// y_i -= sum_{k < i} l_ik y_k for the rows of one forward level (one wavefront per row).
__global__ __launch_bounds__(256) void k_ilu_lower(int32_t cnt, const int32_t* rows, const int32_t* rp,
                                                   const int32_t* ci, const int32_t* diag, const double* lu,
                                                   double* y, const int32_t* skip) {
    if (skip && *skip) return;
    const int w = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (w >= cnt) return;
    const int i = rows[w];
    double s = 0.0;
    for (int p = rp[i] + lane; p < diag[i]; p += 64) s += lu[p] * y[ci[p]];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (lane == 0) y[i] -= s;
}

// z_i = (z_i - sum_{j > i} u_ij z_j) / u_ii for the rows of one backward level.
__global__ __launch_bounds__(256) void k_ilu_upper(int32_t cnt, const int32_t* rows, const int32_t* rp,
                                                   const int32_t* ci, const int32_t* diag, const double* lu,
                                                   double* z, const int32_t* skip) {
    if (skip && *skip) return;
    const int w = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (w >= cnt) return;
    const int i = rows[w];
    double s = 0.0;
    for (int p = diag[i] + 1 + lane; p < rp[i + 1]; p += 64) s += lu[p] * z[ci[p]];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (lane == 0) z[i] = (z[i] - s) / lu[diag[i]];
}

__global__ __launch_bounds__(256) void k_ilu_copy(int32_t n, const double* src, double* dst, const int32_t* skip) {
    if (skip && *skip) return;
    for (int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x; r < n; r += (int64_t)gridDim.x * 256) dst[r] = src[r];
}

template <class T>
mgpu_status dev_upload(mgpu_ilu* f, const std::vector<T>& h, T** d) {
    *d = nullptr;
    if (h.empty()) return MGPU_OK;
    void* p = nullptr;
    ILU_TRY(hipMalloc(&p, h.size() * sizeof(T)));
    f->allocs.push_back(p);
    ILU_TRY(hipMemcpy(p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
    *d = static_cast<T*>(p);
    return MGPU_OK;
}

// The same for an array that the solve can do without: false, and no allocation kept, where it does not fit.
template <class T>
bool dev_upload_optional(mgpu_ilu* f, const std::vector<T>& h, T** d) {
    *d = nullptr;
    void* p = nullptr;
    if (hipMalloc(&p, h.size() * sizeof(T)) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    if (hipMemcpy(p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipGetLastError();
        (void)hipFree(p);
        return false;
    }
    f->allocs.push_back(p);
    *d = static_cast<T*>(p);
    return true;
}
template <class T>
void dev_drop(mgpu_ilu* f, T** d) {
    if (!*d) return;
    f->allocs.erase(std::find(f->allocs.begin(), f->allocs.end(), static_cast<void*>(*d)));
    (void)hipFree(*d);
    *d = nullptr;
}

// One triangular solve as a stream with L lanes per row: the rows of each level (order: most entries first),
// kTriThreads / L at a time; range: the entries of a row that the solve uses.
template <class Range>
int tri_chunks(int L, int32_t row, Range range) {
    return std::max(1, (int)((range(row).second - range(row).first + L - 1) / L));
}
// its steps (whole multiples of kTriAhead, the last ones doing nothing)
template <class Range>
int64_t tri_steps(int L, const std::vector<int32_t>& order, const std::vector<int32_t>& off, Range range) {
    int64_t steps = 0;
    for (size_t l = 0; l + 1 < off.size(); ++l)
        for (int32_t g = off[l]; g < off[l + 1]; g += kTriThreads / L) steps += tri_chunks(L, order[(size_t)g], range);
    return (steps + kTriAhead - 1) / kTriAhead * kTriAhead;
}
struct TriStream {
    std::vector<TriSlot> slots;
    std::vector<int32_t> pos, dpos;
};
// and its slots, from slot `at` of the stream on (all empty before); diag: the rows' diagonals (backward) or null
template <class Range>
void tri_fill(int L, int32_t n, const std::vector<int32_t>& order, const std::vector<int32_t>& off, Range range,
              const std::vector<int32_t>& fci, const std::vector<int32_t>* diag, size_t at, TriStream& out) {
    const int RPS = kTriThreads / L;
    for (size_t l = 0; l + 1 < off.size(); ++l) {
        for (int32_t g = off[l]; g < off[l + 1]; g += RPS) {
            const int32_t g1 = std::min(g + RPS, off[l + 1]);
            const int chunks = tri_chunks(L, order[(size_t)g], range);
            for (int c = 0; c < chunks; ++c) {
                const uint32_t flags = (c + 1 == chunks ? kTriRowEnd : 0u) |
                                       (c + 1 == chunks && g1 == off[l + 1] ? kTriLevelEnd : 0u);
                for (int k = 0; k < RPS; ++k) {
                    const int32_t i = g + k < g1 ? order[(size_t)(g + k)] : n;
                    const auto r = i < n ? range(i) : std::make_pair(0, 0);
                    if (diag && c + 1 == chunks) out.dpos[at] = i < n ? (*diag)[(size_t)i] : -2;
                    for (int lane = 0; lane < L; ++lane, ++at) {
                        const int32_t p = r.first + c * L + lane;
                        const bool some = p < r.second;
                        if (some) out.pos[at] = p;
                        out.slots[at].meta = (uint32_t)(some ? fci[(size_t)p] : n) | ((uint32_t)i << 14) | flags;
                    }
                }
            }
        }
    }
}

// Rows ordered by level (counting sort, ascending row within a level); offsets per level.
void schedule(const std::vector<int32_t>& level, std::vector<int32_t>& rows, std::vector<int32_t>& off) {
    const int32_t n = (int32_t)level.size();
    int32_t n_lev = 0;
    for (int32_t v : level) n_lev = std::max(n_lev, v + 1);
    off.assign((size_t)n_lev + 1, 0);
    for (int32_t v : level) off[(size_t)v + 1]++;
    for (int32_t l = 0; l < n_lev; ++l) off[(size_t)l + 1] += off[(size_t)l];
    rows.assign((size_t)n, 0);
    std::vector<int32_t> fill(off.begin(), off.end() - 1);
    for (int32_t i = 0; i < n; ++i) rows[(size_t)fill[(size_t)level[(size_t)i]]++] = i;
}

}  // namespace ilu

void ilu_apply_launch(const mgpu_ilu* f, const double* v, double* z, const int32_t* skip, hipStream_t s) {
    if (f->tri_lanes > 0) {
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(1), dim3(ilu::kTriThreads), 0, s, f->n, f->n_steps[0], f->n_steps[1],
                               static_cast<const ilu::TriSlot*>(f->tri_slots), v, z, skip);
        };
        if (f->tri_lanes == 4) go(ilu::k_ilu_tri<4>);
        else if (f->tri_lanes == 8) go(ilu::k_ilu_tri<8>);
        else if (f->tri_lanes == 16) go(ilu::k_ilu_tri<16>);
        else if (f->tri_lanes == 32) go(ilu::k_ilu_tri<32>);
        else go(ilu::k_ilu_tri<64>);
        return;
    }
    const dim3 t(256);
    if (v != z) hipLaunchKernelGGL(ilu::k_ilu_copy, dim3(1024), t, 0, s, f->n, v, z, skip);
    for (size_t l = 0; l + 1 < f->lev_f.size(); ++l) {
        const int32_t cnt = f->lev_f[l + 1] - f->lev_f[l];
        hipLaunchKernelGGL(ilu::k_ilu_lower, dim3((unsigned)((cnt + 3) / 4)), t, 0, s, cnt, f->rows_f + f->lev_f[l],
                           f->rp, f->ci, f->diag, f->lu, z, skip);
    }
    for (size_t l = 0; l + 1 < f->lev_b.size(); ++l) {
        const int32_t cnt = f->lev_b[l + 1] - f->lev_b[l];
        hipLaunchKernelGGL(ilu::k_ilu_upper, dim3((unsigned)((cnt + 3) / 4)), t, 0, s, cnt, f->rows_b + f->lev_b[l],
                           f->rp, f->ci, f->diag, f->lu, z, skip);
    }
}

}  // namespace mgpu

using namespace mgpu;

extern "C" mgpu_status mgpu_ilu_create(int32_t n, const int32_t* row_ptr, const int32_t* col_idx, int32_t fill_level,
                                       void* stream, mgpu_ilu** out) {
    MGPU_GUARD_BEGIN
    if (!out) return set_error(MGPU_ERR_INVALID_ARG, "null argument");
    *out = nullptr;
    if (n < 0 || fill_level < 0) return set_error(MGPU_ERR_INVALID_ARG, "negative size or fill level");
    if (n > 0 && (!row_ptr || !col_idx)) return set_error(MGPU_ERR_INVALID_ARG, "null device pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    // the matrix pattern on the host
    std::vector<int32_t> rp((size_t)n + 1, 0);
    if (n > 0) {
        ILU_TRY(hipMemcpyAsync(rp.data(), row_ptr, ((size_t)n + 1) * sizeof(int32_t), hipMemcpyDeviceToHost, s));
        ILU_TRY(hipStreamSynchronize(s));
    }
    if (rp[0] != 0) return set_error(MGPU_ERR_INVALID_ARG, "row_ptr[0] must be 0");
    for (int32_t i = 0; i < n; ++i)
        if (rp[(size_t)i + 1] < rp[(size_t)i]) return set_error(MGPU_ERR_INVALID_ARG, "row_ptr not monotone");
    const int64_t nnz_in = rp[(size_t)n];
    std::vector<int32_t> ci((size_t)nnz_in);
    if (nnz_in > 0) {
        ILU_TRY(hipMemcpyAsync(ci.data(), col_idx, (size_t)nnz_in * sizeof(int32_t), hipMemcpyDeviceToHost, s));
        ILU_TRY(hipStreamSynchronize(s));
    }
    for (int32_t i = 0; i < n; ++i)
        for (int32_t p = rp[(size_t)i]; p < rp[(size_t)i + 1]; ++p) {
            if (ci[(size_t)p] < 0 || ci[(size_t)p] >= n) return set_error(MGPU_ERR_INVALID_ARG, "column out of range");
            if (p > rp[(size_t)i] && ci[(size_t)p] <= ci[(size_t)p - 1])
                return set_error(MGPU_ERR_INVALID_ARG, "columns not sorted ascending");
        }
    // factor pattern: ILU(k) fill by levels, row by row; a missing diagonal is added
    std::vector<int32_t> frp((size_t)n + 1, 0), fci;
    fci.reserve((size_t)nnz_in + (size_t)n);
    std::vector<std::vector<std::pair<int32_t, int32_t>>> upper(fill_level > 0 ? (size_t)n : 0);
    std::map<int32_t, int32_t> row;
    for (int32_t i = 0; i < n; ++i) {
        if (fill_level == 0) {
            bool has_diag = false;
            for (int32_t p = rp[(size_t)i]; p < rp[(size_t)i + 1]; ++p) {
                const int32_t c = ci[(size_t)p];
                if (!has_diag && c > i) {
                    fci.push_back(i);
                    has_diag = true;
                }
                if (c == i) has_diag = true;
                fci.push_back(c);
            }
            if (!has_diag) fci.push_back(i);
        } else {
            row.clear();
            for (int32_t p = rp[(size_t)i]; p < rp[(size_t)i + 1]; ++p) row[ci[(size_t)p]] = 0;
            row.emplace(i, 0);
            for (auto it = row.begin(); it != row.end() && it->first < i; ++it) {
                const int32_t lik = it->second;
                for (const auto& kj : upper[(size_t)it->first]) {
                    const int32_t lev = lik + kj.second + 1;
                    if (lev > fill_level) continue;
                    auto f = row.find(kj.first);
                    if (f == row.end()) row.emplace(kj.first, lev);
                    else f->second = std::min(f->second, lev);
                }
            }
            for (const auto& e : row) {
                fci.push_back(e.first);
                if (e.first > i) upper[(size_t)i].push_back(e);
            }
        }
        if (fci.size() >= (size_t)INT32_MAX) return set_error(MGPU_ERR_INVALID_ARG, "factor pattern exceeds int32");
        frp[(size_t)i + 1] = (int32_t)fci.size();
    }
    upper.clear();
    auto F = std::make_unique<mgpu_ilu>();
    struct Cleanup {
        mgpu_ilu* f;
        ~Cleanup() {
            if (f)
                for (void* p : f->allocs) (void)hipFree(p);
        }
    } cleanup{F.get()};
    F->n = n;
    F->nnz = (int64_t)fci.size();
    F->nnz_in = nnz_in;
    F->fill_level = fill_level;
    std::vector<int32_t> diag((size_t)n), pos((size_t)nnz_in), lev_f((size_t)n, 0), lev_b((size_t)n, 0);
    for (int32_t i = 0; i < n; ++i) {
        const int32_t a = frp[(size_t)i], b = frp[(size_t)i + 1];
        F->max_row = std::max(F->max_row, b - a);
        diag[(size_t)i] = (int32_t)(std::lower_bound(fci.begin() + a, fci.begin() + b, i) - fci.begin());
        // matrix entries into the factor row (both sorted)
        int32_t q = a;
        for (int32_t p = rp[(size_t)i]; p < rp[(size_t)i + 1]; ++p) {
            while (fci[(size_t)q] < ci[(size_t)p]) ++q;
            pos[(size_t)p] = q;
        }
        int32_t lf = 0;
        for (int32_t p = a; p < diag[(size_t)i]; ++p) lf = std::max(lf, lev_f[(size_t)fci[(size_t)p]] + 1);
        lev_f[(size_t)i] = lf;
    }
    for (int32_t i = n - 1; i >= 0; --i) {
        int32_t lb = 0;
        for (int32_t p = diag[(size_t)i] + 1; p < frp[(size_t)i + 1]; ++p) lb = std::max(lb, lev_b[(size_t)fci[(size_t)p]] + 1);
        lev_b[(size_t)i] = lb;
    }
    if (F->max_row > ilu::kMaxRow)
        return set_error(MGPU_ERR_UNSUPPORTED, "a factor row has more than " + std::to_string(ilu::kMaxRow) + " entries");
    std::vector<int32_t> rows_f, rows_b;
    ilu::schedule(lev_f, rows_f, F->lev_f);
    ilu::schedule(lev_b, rows_b, F->lev_b);
    mgpu_status rc;
    if ((rc = ilu::dev_upload(F.get(), frp, &F->rp)) || (rc = ilu::dev_upload(F.get(), fci, &F->ci)) ||
        (rc = ilu::dev_upload(F.get(), diag, &F->diag)) || (rc = ilu::dev_upload(F.get(), pos, &F->pos)) ||
        (rc = ilu::dev_upload(F.get(), rows_f, &F->rows_f)) || (rc = ilu::dev_upload(F.get(), rows_b, &F->rows_b)))
        return rc;
    // elimination lists: the entries of row i that row k's upper part updates, for every lower entry (i, k).
    // Their number is estimated first, from every 64th row: patterns far beyond the limit pay for no list.
    try {
        std::vector<int32_t> at((size_t)n, -1);   // position of each column in the current row
        auto row_updates = [&](int32_t i, auto hit, auto entry) {
            const int32_t r0 = frp[(size_t)i], r1 = frp[(size_t)i + 1];
            for (int32_t t = r0; t < r1; ++t) at[(size_t)fci[(size_t)t]] = t - r0;
            for (int32_t q = r0; q < r1; ++q) {
                if (q < diag[(size_t)i]) {
                    const int32_t k = fci[(size_t)q];
                    for (int32_t u = diag[(size_t)k] + 1; u < frp[(size_t)k + 1]; ++u)
                        if (at[(size_t)fci[(size_t)u]] >= 0) hit(at[(size_t)fci[(size_t)u]], u);
                }
                entry(q);
            }
            for (int32_t t = r0; t < r1; ++t) at[(size_t)fci[(size_t)t]] = -1;
        };
        size_t expected = 0;
        for (int32_t i = 0; i < n; i += 64) row_updates(i, [&](int32_t, int32_t) { expected += 64; }, [](int32_t) {});
        bool fits = expected <= ilu::kMaxUpdates;
        std::vector<int64_t> up;
        std::vector<int2> upd;
        if (fits) {
            up.assign((size_t)F->nnz + 1, 0);
            upd.reserve(expected + expected / 8);
        }
        for (int32_t i = 0; i < n && fits; ++i) {
            row_updates(i, [&](int32_t x, int32_t u) { upd.push_back(make_int2(x, u)); },
                        [&](int32_t q) { up[(size_t)q + 1] = (int64_t)upd.size(); });
            fits = upd.size() <= ilu::kMaxUpdates;
        }
        if (fits && !upd.empty() && ilu::dev_upload_optional(F.get(), up, &F->upd_ptr) &&
            !ilu::dev_upload_optional(F.get(), upd, &F->upd))
            ilu::dev_drop(F.get(), &F->upd_ptr);
    } catch (const std::bad_alloc&) {   // (the rows are searched)
    }
    // one workgroup for the triangular solves where its steps take less time than the levels' launches
    if (n > 0 && n <= ilu::kTriMaxRows) {
        auto low = [&](int32_t i) { return std::make_pair(frp[(size_t)i], diag[(size_t)i]); };
        auto upp = [&](int32_t i) { return std::make_pair(diag[(size_t)i] + 1, frp[(size_t)i + 1]); };
        // most entries first within a level
        std::vector<int32_t> ord_f(rows_f), ord_b(rows_b);
        auto sort_levels = [&](std::vector<int32_t>& ord, const std::vector<int32_t>& off, auto range) {
            auto more = [&](int32_t x, int32_t y) {
                return range(x).second - range(x).first > range(y).second - range(y).first;
            };
            for (size_t l = 0; l + 1 < off.size(); ++l)
                std::stable_sort(ord.begin() + off[l], ord.begin() + off[l + 1], more);
        };
        sort_levels(ord_f, F->lev_f, low);
        sort_levels(ord_b, F->lev_b, upp);
        // more lanes per row only where they save a quarter of the steps: fewer lanes, fewer
        // additions across them (8825 rows of 30: 8 lanes 0.19 ms, 16 lanes 0.22 ms, 4 lanes 0.31 ms)
        int best = 0;
        int64_t steps[2] = {0, 0};
        for (int L = 4; L <= 64; L *= 2) {
            const int64_t sf = ilu::tri_steps(L, ord_f, F->lev_f, low), sb = ilu::tri_steps(L, ord_b, F->lev_b, upp);
            if (best == 0 || 4 * (sf + sb) < 3 * (steps[0] + steps[1])) {
                best = L;
                steps[0] = sf;
                steps[1] = sb;
            }
        }
        const int64_t all = steps[0] + steps[1];
        const size_t slots = (size_t)all * ilu::kTriThreads;
        const double launches = (double)(F->lev_f.size() + F->lev_b.size() - 2);
        if (all * ilu::kTriStepUs < launches * ilu::kLevelUs && slots * ilu::kTriSlotBytes <= ilu::kMaxTriBytes) {
            try {
                ilu::TriStream st;
                st.slots.assign(slots, ilu::TriSlot{0.0, (uint32_t)n | ((uint32_t)n << 14), 0u});
                st.pos.assign(slots, -1);
                st.dpos.assign(slots, -1);
                ilu::tri_fill(best, n, ord_f, F->lev_f, low, fci, nullptr, 0, st);
                ilu::tri_fill(best, n, ord_b, F->lev_b, upp, fci, &diag, (size_t)steps[0] * ilu::kTriThreads, st);
                ilu::TriSlot* sl = nullptr;
                if (ilu::dev_upload_optional(F.get(), st.slots, &sl) &&
                    ilu::dev_upload_optional(F.get(), st.pos, &F->tri_pos) &&
                    ilu::dev_upload_optional(F.get(), st.dpos, &F->tri_dpos)) {
                    F->tri_slots = sl;
                    F->tri_lanes = best;
                    F->n_steps[0] = (int32_t)steps[0];
                    F->n_steps[1] = (int32_t)steps[1];
                } else {
                    ilu::dev_drop(F.get(), &sl);
                    ilu::dev_drop(F.get(), &F->tri_pos);
                }
            } catch (const std::bad_alloc&) {   // (a launch per level)
            }
        }
    }
    void* p = nullptr;
    if (F->nnz > 0) {
        ILU_TRY(hipMalloc(&p, (size_t)F->nnz * sizeof(double)));
        F->allocs.push_back(p);
        F->lu = static_cast<double*>(p);
    }
    ILU_TRY(hipMalloc(&p, sizeof(int32_t)));
    F->allocs.push_back(p);
    F->err = static_cast<int32_t*>(p);
    cleanup.f = nullptr;
    *out = F.release();
    return MGPU_OK;
    MGPU_GUARD_END
}

extern "C" mgpu_status mgpu_ilu_factor(mgpu_ilu* f, const double* vals, void* stream) {
    MGPU_GUARD_BEGIN
    if (!f) return set_error(MGPU_ERR_INVALID_ARG, "null factor");
    if (f->nnz_in > 0 && !vals) return set_error(MGPU_ERR_INVALID_ARG, "null device pointer");
    f->factored = false;
    if (f->n == 0) {
        f->factored = true;
        return MGPU_OK;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 t(256), g(1024);
    hipLaunchKernelGGL(ilu::k_ilu_clear, dim3(1), dim3(64), 0, s, f->err);
    hipLaunchKernelGGL(ilu::k_ilu_fill, g, t, 0, s, f->nnz, f->lu);
    if (f->nnz_in > 0) hipLaunchKernelGGL(ilu::k_ilu_scatter, g, t, 0, s, f->nnz_in, f->pos, vals, f->lu);
    const size_t lds = (size_t)f->max_row * (sizeof(double) + sizeof(int32_t));
    for (size_t l = 0; l + 1 < f->lev_f.size(); ++l) {
        const int32_t cnt = f->lev_f[l + 1] - f->lev_f[l];
        hipLaunchKernelGGL(f->upd_ptr ? ilu::k_ilu_row<true> : ilu::k_ilu_row<false>, dim3((unsigned)cnt), dim3(64), lds,
                           s, f->rows_f + f->lev_f[l], f->rp, f->ci, f->diag, f->upd_ptr, f->upd, f->lu, f->err,
                           f->max_row);
    }
    if (f->tri_lanes > 0) {
        const int64_t steps = (int64_t)f->n_steps[0] + f->n_steps[1];
        hipLaunchKernelGGL(ilu::k_ilu_pack, g, t, 0, s, steps * ilu::kTriThreads, f->tri_pos, f->tri_dpos, f->lu,
                           static_cast<ilu::TriSlot*>(f->tri_slots));
    }
    ILU_TRY(hipGetLastError());
    int32_t err = 0;
    ILU_TRY(hipMemcpyAsync(&err, f->err, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    ILU_TRY(hipStreamSynchronize(s));
    if (err) return set_error(MGPU_ERR_INVALID_ARG, "zero pivot in the incomplete factorisation");
    f->factored = true;
    return MGPU_OK;
    MGPU_GUARD_END
}

extern "C" mgpu_status mgpu_ilu_apply(const mgpu_ilu* f, const double* v, double* z, void* stream) {
    MGPU_GUARD_BEGIN
    if (!f) return set_error(MGPU_ERR_INVALID_ARG, "null factor");
    if (!f->factored) return set_error(MGPU_ERR_STATE, "the factor has not been computed");
    if (f->n == 0) return MGPU_OK;
    if (!v || !z) return set_error(MGPU_ERR_INVALID_ARG, "null device pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    ilu_apply_launch(f, v, z, nullptr, s);
    ILU_TRY(hipGetLastError());
    return MGPU_OK;
    MGPU_GUARD_END
}

extern "C" mgpu_status mgpu_ilu_factors(const mgpu_ilu* f, int32_t* n, int64_t* nnz, const int32_t** row_ptr,
                                        const int32_t** col_idx, const double** lu, int32_t* n_levels) {
    if (!f) return set_error(MGPU_ERR_INVALID_ARG, "null factor");
    if (n) *n = f->n;
    if (nnz) *nnz = f->nnz;
    if (row_ptr) *row_ptr = f->rp;
    if (col_idx) *col_idx = f->ci;
    if (lu) *lu = f->lu;
    if (n_levels) {
        n_levels[0] = f->lev_f.empty() ? 0 : (int32_t)f->lev_f.size() - 1;
        n_levels[1] = f->lev_b.empty() ? 0 : (int32_t)f->lev_b.size() - 1;
    }
    return MGPU_OK;
}

extern "C" mgpu_status mgpu_ilu_destroy(mgpu_ilu* f) {
    if (!f) return MGPU_OK;
    (void)hipDeviceSynchronize();
    for (void* p : f->allocs) (void)hipFree(p);
    delete f;
    return MGPU_OK;
}
