// Host check of the choice between the forms of a large HEX27 set (no GPU): the limits of the K_e pool,
// and a set in rows mode turned into one in scatter mode equal to one built so.
// Usage: mode_check N REFINE   (N^3 lattice, gyroid cut, p = 2 B-splines, HEX27 cells).
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <string>
#include "moris_gpu.h"
#include "set_internal.hpp"
using namespace mgpu;
static_assert(!scatter_by_size(27, true, (int64_t)1 << 30) && scatter_by_size(27, true, ((int64_t)1 << 30) + 1),
              "rows mode: a pool of up to 8 GiB");
static_assert(!scatter_by_size(27, false, (int64_t)1 << 28) && scatter_by_size(27, false, ((int64_t)1 << 28) + 1),
              "gather lists: a pool of up to 2 GiB");
static_assert(!scatter_by_size(8, true, (int64_t)1 << 40) && !scatter_by_size(8, false, (int64_t)1 << 40), "HEX27 only");
static_assert(!scatter_by_memory(27, true, (int64_t)1 << 28, 0), "up to 2 GiB: the pool, whatever is free");
static_assert(!scatter_by_memory(27, true, (int64_t)1 << 29, (size_t)32 << 30) &&
                  scatter_by_memory(27, true, ((int64_t)1 << 29) + 1, (size_t)32 << 30),
              "beyond: an eighth of the free memory");
static_assert(!scatter_by_memory(27, false, (int64_t)1 << 29, 0) && !scatter_by_memory(8, true, (int64_t)1 << 40, 0),
              "only sets in rows mode can do without");
int main(int argc, char** argv) {
    const int n = atoi(argv[1]), refine = atoi(argv[2]);
    mgpu_problem_spec s{};
    s.dim = 3; s.n[0] = s.n[1] = s.n[2] = n;
    s.hi[0] = s.hi[1] = s.hi[2] = 1.0;
    s.iwg = MGPU_IWG_STRUC_LINEAR_BULK; s.ls_kind = MGPU_LS_GYROID; s.gyroid_scale = 2 * M_PI * n / 4.0;
    s.material_phase = 1; s.E = 1.0; s.nu = 0.3; s.seed = 20261202;
    s.bspline_order = 2; s.lagrange_order = 2; s.refine_levels = refine;
    mgpu_problem* p = nullptr;
    if (mgpu_problem_build(&s, &p)) { printf("build failed\n"); return 1; }
    mgpu_set_desc d;
    mgpu_problem_desc(p, &d);
    SetHost a, b;
    std::string err;
    if (build_set_host(d, a, &err) != MGPU_OK) { printf("set: %s\n", err.c_str()); return 1; }
    if (!a.rows || a.scatter || a.adof_el.empty()) { printf("not in rows mode\n"); return 1; }
    rows_to_scatter(d, a);
    setenv("MGPU_GENERIC_SCATTER", "1", 1);
    if (build_set_host(d, b, &err) != MGPU_OK) { printf("set: %s\n", err.c_str()); return 1; }
    const bool same = a.scatter == b.scatter && a.rows == b.rows && a.colour_ptr == b.colour_ptr &&
                      a.colour_el == b.colour_el && a.rank_off == b.rank_off && a.rank == b.rank && a.topo == b.topo &&
                      a.topo_ptr == b.topo_ptr && a.ke_off == b.ke_off && a.row_ptr == b.row_ptr &&
                      a.col_idx == b.col_idx && a.t_perm == b.t_perm && a.adof_ptr == b.adof_ptr && a.adof_el == b.adof_el;
    if (!same || b.colour_ptr.size() < 9) { printf("the sets differ\n"); return 1; }
    printf("OK: %d elements, %zu colours\n", a.n_el, a.colour_ptr.size() - 1);
    mgpu_problem_destroy(p);
    return 0;
}
