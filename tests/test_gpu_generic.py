"""GPU tests of the generic element path (T rows with several weighted entries, sets without a
lattice): element K_p on the GPU, K_e = T^T K_p T in FP64, deterministic sums into the CSR
values, R = K u.

* quadratic B-spline T rows (bspline_order 2: every Lagrange node carries 2^dim splines of weight
  2^-dim) against the oracle's dense T^T K T: CSR pattern and element topology bit-exact, K and R
  within 1e-12, the mixed precision option bit for bit the same (generic sets are FP64 at either);
* HEX27 IP cells (lagrange_order 2: HEX_3x3x3 on whole cells, TET_35 on XTK sub-tets, p = 2
  B-spline rows of 8 to 27 entries or nodal rows) to the same bars;
* one THB refinement level (refine_levels 1) on HEX8 and HEX27 cells, up to 38 adofs per type and
  element, to the same bars;
* a nodal set with its lattice hint removed runs the generic path and reproduces the lattice
  stencil path to 1e-12;
* graph replays of generic sets are bit-identical to eager calls; learned quadrature is refused.
"""
import ctypes

import numpy as np
import pytest

import moris_amd as M
from helpers import SEED, rel, two_bodies
from moris_amd import learned as L
from oracle import py as O

pytestmark = pytest.mark.gpu

CASES = {
    "p2_sphere_8_elasticity": lambda: M.make_spec(3, (8, 8, 8), iwg=M.IWG_STRUC_LINEAR_BULK,
                                                  spheres=[[0.5, 0.5, 0.5, 0.3]], bspline_order=2),
    "p2_sphere_10_diffusion": lambda: M.make_spec(3, (10, 10, 10), spheres=[[0.45, 0.5, 0.55, 0.33]],
                                                  k_sigma=0.5, bspline_order=2),
    "p2_circle_16x12_plane_stress": lambda: M.make_spec(2, (16, 12), iwg=M.IWG_STRUC_LINEAR_BULK,
                                                        spheres=[[0.5, 0.5, 0.0, 0.3]], bspline_order=2),
    "p2_plane_2d_diffusion_phase0": lambda: M.make_spec(2, (9, 7), ls_kind=M.LS_PLANE, plane=[0.6, 0.8, 0.0, -0.55],
                                                        material_phase=0, bspline_order=2),
    "p2_uncut_elasticity": lambda: M.make_spec(3, (3, 4, 2), iwg=M.IWG_STRUC_LINEAR_BULK, bspline_order=2),
    # HEX27 IP cells (HEX_3x3x3 uncut, TET_35 on the sub-tets): p = 2 B-splines and nodal Lagrange rows
    "hex27_p2_gyroid_6_elasticity": lambda: M.make_spec(3, (6, 6, 6), iwg=M.IWG_STRUC_LINEAR_BULK,
                                                        ls_kind=M.LS_GYROID, gyroid_scale=2 * np.pi * 1.5,
                                                        bspline_order=2, lagrange_order=2),
    "hex27_p2_sphere_6_diffusion": lambda: M.make_spec(3, (6, 5, 4), spheres=[[0.5, 0.5, 0.5, 0.3]], k_sigma=0.5,
                                                       bspline_order=2, lagrange_order=2),
    "hex27_lagrange_sphere_5_elasticity": lambda: M.make_spec(3, (5, 5, 5), iwg=M.IWG_STRUC_LINEAR_BULK,
                                                              spheres=[[0.4, 0.5, 0.6, 0.35]], lagrange_order=2),
    "hex27_p2_uncut_elasticity": lambda: M.make_spec(3, (3, 4, 2), iwg=M.IWG_STRUC_LINEAR_BULK, bspline_order=2,
                                                     lagrange_order=2),
    # one THB level (truncated hierarchical quadratic B-splines, up to 38 adofs per type and element)
    "thb_sphere_6_hex8_elasticity": lambda: M.make_spec(3, (6, 6, 6), iwg=M.IWG_STRUC_LINEAR_BULK,
                                                        spheres=[[0.5, 0.5, 0.5, 0.3]], bspline_order=2,
                                                        refine_levels=1),
    "thb_plane_6_hex8_elasticity": lambda: M.make_spec(3, (6, 6, 6), iwg=M.IWG_STRUC_LINEAR_BULK, ls_kind=M.LS_PLANE,
                                                       plane=[0.3, 0.5, 0.8, -0.6], bspline_order=2, refine_levels=1),
    "thb_plane_5_hex27_elasticity": lambda: M.make_spec(3, (5, 5, 5), iwg=M.IWG_STRUC_LINEAR_BULK, ls_kind=M.LS_PLANE,
                                                        plane=[0.3, 0.5, 0.8, -0.6], bspline_order=2,
                                                        lagrange_order=2, refine_levels=1),
    "thb_sphere_4_hex27_diffusion": lambda: M.make_spec(3, (4, 4, 4), spheres=[[0.5, 0.5, 0.5, 0.3]], k_sigma=0.4,
                                                        bspline_order=2, lagrange_order=2, refine_levels=1),
    # XTK enrichment: a cell split into two subphase elements, bases replicated per level; nodal
    # p = 1 rows that leave the lattice stencil for the generic path
    "enriched_two_spheres_p1_elasticity": lambda: M.make_spec(3, (10, 10, 10), iwg=M.IWG_STRUC_LINEAR_BULK,
                                                              spheres=two_bodies(3, 10), material_phase=0, enrich=1),
    "enriched_two_circles_p1_plane_stress": lambda: M.make_spec(2, (16, 16), iwg=M.IWG_STRUC_LINEAR_BULK,
                                                                spheres=two_bodies(2, 16), material_phase=0,
                                                                enrich=1),
    "enriched_gyroid_7_p1_diffusion": lambda: M.make_spec(3, (7, 7, 7), ls_kind=M.LS_GYROID, gyroid_scale=9.0,
                                                          k_sigma=0.5, enrich=1),
    "enriched_gyroid_6_p2_hex27_elasticity": lambda: M.make_spec(3, (6, 6, 6), iwg=M.IWG_STRUC_LINEAR_BULK,
                                                                 ls_kind=M.LS_GYROID, gyroid_scale=2 * np.pi * 1.6,
                                                                 bspline_order=2, lagrange_order=2, enrich=1),
}


def _oracle_topology(s, nb, nf, N):
    rows = []
    for e in range(len(s["elem_cell"])):
        q0, q1 = s["t_ptr"][e * nb], s["t_ptr"][(e + 1) * nb]
        u = np.unique(s["t_adof"][q0:q1])
        rows.append(np.concatenate([u + f * N for f in range(nf)]))
    return rows


@pytest.mark.parametrize("case", sorted(CASES))
def test_generic_path_matches_oracle(case):
    print("case", case, flush=True)
    spec, keep = CASES[case]()
    P = M.Problem(spec, keep)
    S = M.Set(P.desc, keepalive=P)
    Q = O.OracleProblem(spec)
    s = Q.setup()
    rp, ci = S.pattern()
    assert np.array_equal(rp, s["row_ptr"]) and np.array_equal(ci, s["col_idx"])
    nb = P.desc.n_bases
    nf = spec.dim if spec.iwg == M.IWG_STRUC_LINEAR_BULK else 1
    topo, want = S.topology_lists(), _oracle_topology(s, nb, nf, Q.n_adofs_per_type)
    assert len(topo) == len(want) and all(np.array_equal(a, b) for a, b in zip(topo, want))
    u = np.random.default_rng(SEED + 11).uniform(-1.0, 1.0, S.n_rows)
    vo, Ro = Q.assemble(u)
    vals, R = S.compute_jacobian_and_residual(u)
    assert rel(vals, vo) <= 1e-12 and rel(R, Ro) <= 1e-12, (rel(vals, vo), rel(R, Ro))
    # generic sets are FP64 at either precision option
    S.options(M.PREC_MIXED, M.QUAD_SUBDIVISION)
    vm, Rm = S.compute_jacobian_and_residual(u)
    assert np.array_equal(vm.view(np.uint64), vals.view(np.uint64)) and np.array_equal(Rm.view(np.uint64), R.view(np.uint64))


def _without_lattice(desc):
    d = M.SetDesc()
    ctypes.memmove(ctypes.byref(d), ctypes.byref(desc), ctypes.sizeof(M.SetDesc))
    d.lattice.n[0] = 0
    d.elem_cell = None
    return d


@pytest.mark.parametrize("iwg", [M.IWG_SPATIALDIFF_BULK, M.IWG_STRUC_LINEAR_BULK])
def test_generic_path_reproduces_lattice_stencil(iwg):
    spec, keep = M.make_spec(3, (9, 9, 9), iwg=iwg, spheres=[[0.5, 0.5, 0.5, 0.33]], k_sigma=0.4)
    P = M.Problem(spec, keep)
    S_lat = M.Set(P.desc, keepalive=P)
    S_gen = M.Set(_without_lattice(P.desc), keepalive=P)
    assert np.array_equal(S_lat.pattern()[0], S_gen.pattern()[0])
    assert np.array_equal(S_lat.pattern()[1], S_gen.pattern()[1])
    u = np.random.default_rng(3).uniform(-1.0, 1.0, S_lat.n_rows)
    v1, R1 = S_lat.compute_jacobian_and_residual(u)
    v2, R2 = S_gen.compute_jacobian_and_residual(u)
    assert rel(v2, v1) <= 1e-12 and rel(R2, R1) <= 1e-12


@pytest.mark.parametrize("lagrange_order", [1, 2])
def test_generic_element_order_and_autotune(lagrange_order):
    """Generic sets in gather mode have two launch shapes: element workgroups in element order, or
    most sub-cells first.  Both give bit-identical K and R (each K_e has its own pool slot and the
    gather sums in a fixed order); the autotuner times both, keeps the faster, and the result still
    matches the oracle."""
    spec, keep = M.make_spec(3, (6, 6, 6), iwg=M.IWG_STRUC_LINEAR_BULK, ls_kind=M.LS_GYROID,
                             gyroid_scale=2 * np.pi * 1.5, bspline_order=2, lagrange_order=lagrange_order)
    P = M.Problem(spec, keep)
    S = M.Set(P.desc, keepalive=P)
    u = np.random.default_rng(SEED + 5).uniform(-1.0, 1.0, S.n_rows)
    ub, vb, rb = M.DeviceBuffer.from_array(u), M.DeviceBuffer(8 * S.nnz), M.DeviceBuffer(8 * S.n_rows)
    out = []
    for order in (0, 1):
        S.tuning(cut_order=order)
        S.assemble_device(ub, vb, rb)
        M.synchronize()
        out.append((vb.to_array(np.float64, S.nnz), rb.to_array(np.float64, S.n_rows)))
    assert np.array_equal(out[0][0].view(np.uint64), out[1][0].view(np.uint64))
    assert np.array_equal(out[0][1].view(np.uint64), out[1][1].view(np.uint64))
    ms = S.autotune(ub, vb, rb, iters=2, ignore_cache=True)
    assert set(ms) == {(0, 0), (0, 1)} and all(t > 0 for t in ms.values()), ms
    _, order = S.tuning()
    assert ms[(0, order)] == min(ms.values())
    S.assemble_device(ub, vb, rb)
    M.synchronize()
    assert np.array_equal(vb.to_array(np.float64, S.nnz).view(np.uint64), out[0][0].view(np.uint64))
    Q = O.OracleProblem(spec)
    s = Q.setup()
    vo, Ro, _ = O.assemble_desc(P.desc, s["row_ptr"], s["col_idx"], u)
    assert rel(out[0][0], vo) <= 1e-12 and rel(out[0][1], Ro) <= 1e-12


def test_generic_batch_replays_and_learned_refused():
    sets, bufs, eager = [], [], []
    for k, r in enumerate((0.28, 0.31)):
        spec, keep = M.make_spec(3, (6, 6, 6), iwg=M.IWG_STRUC_LINEAR_BULK, spheres=[[0.5, 0.5, 0.5, r]],
                                 bspline_order=2)
        P = M.Problem(spec, keep)
        S = M.Set(P.desc, keepalive=P)
        u = np.random.default_rng(k).uniform(-1.0, 1.0, S.n_rows)
        ub, vb, rb = M.DeviceBuffer.from_array(u), M.DeviceBuffer(8 * S.nnz), M.DeviceBuffer(8 * S.n_rows)
        S.assemble_device(ub, vb, rb)
        M.synchronize()
        eager.append((vb.to_array(np.float64, S.nnz), rb.to_array(np.float64, S.n_rows)))
        sets.append(S)
        bufs.append((ub, vb, rb))
    B = M.Batch(sets, [b[0] for b in bufs], [b[1] for b in bufs], [b[2] for b in bufs], n_branches=2)
    for _ in range(3):
        for S, (_, vb, rb) in zip(sets, bufs):
            z = np.zeros(S.nnz)
            M.load_library().mgpu_memcpy_htod(vb.ptr, z.ctypes.data, z.nbytes)
        M.synchronize()
        B.launch()
        B.synchronize()
        for S, (_, vb, rb), (ve, re) in zip(sets, bufs, eager):
            assert np.array_equal(vb.to_array(np.float64, S.nnz), ve)
            assert np.array_equal(rb.to_array(np.float64, S.n_rows), re)
    B.close()
    with pytest.raises(M.MgpuError, match="learned quadrature"):
        L.attach(sets[0], L.MLP(seed=1))


def test_quadratic_thb_gyroid_size_independent_properties():
    """The quadratic configuration at a size the oracle does not reach in seconds (12^3 base, one THB
    level on the intersected cells, HEX27 cells, gyroid of period 4 cells, elasticity): K is
    symmetric, rigid translations (partition of unity) are in its null space, u^T K u >= 0, R = K u,
    and the mixed path stays within 1e-6 of FP64."""
    n = 12
    spec, keep = M.make_spec(3, (n, n, n), iwg=M.IWG_STRUC_LINEAR_BULK, ls_kind=M.LS_GYROID,
                             gyroid_scale=2 * np.pi * n / 4.0, bspline_order=2, lagrange_order=2, refine_levels=1)
    P = M.Problem(spec, keep)
    S = M.Set(P.desc, keepalive=P)
    print("elements", P.n_elements, "cut", P.n_cut, "rows", S.n_rows, "nnz", S.nnz, flush=True)
    rp, ci = S.pattern()
    N = S.n_rows // 3
    u = np.random.default_rng(SEED + 41).uniform(-1.0, 1.0, S.n_rows)
    vals, R = S.compute_jacobian_and_residual(u)
    import scipy.sparse as sp
    K = sp.csr_matrix((vals, ci, rp), shape=(S.n_rows, S.n_rows))
    kmax = np.abs(vals).max()
    assert abs(K - K.T).max() <= 1e-13 * kmax
    for f in range(3):
        t = np.zeros(S.n_rows)
        t[f * N:(f + 1) * N] = 1.0
        assert np.abs(K @ t).max() <= 1e-12 * kmax * np.sqrt(S.n_rows)
    assert u @ (K @ u) >= -1e-12 * kmax * S.n_rows
    assert rel(R, K @ u) <= 1e-12
    S.options(M.PREC_MIXED, M.QUAD_SUBDIVISION)
    vm, Rm = S.compute_jacobian_and_residual(u)
    assert np.array_equal(vm.view(np.uint64), vals.view(np.uint64)) and np.array_equal(Rm.view(np.uint64), R.view(np.uint64))


HEX27_CASES = sorted(c for c in CASES if "hex27" in c)


@pytest.mark.parametrize("case", HEX27_CASES)
def test_hex27_scatter_mode_matches_oracle_and_gather(case, monkeypatch):
    """Scatter mode of the HEX27 kernel (colour classes adding K_e into the CSR values, the mode of
    sets too large for a K_e pool), forced on small sets: the same pattern, K and R within 1e-12 of
    the oracle and of the gather mode (only the order of summation differs), 1e-6 on the mixed path,
    and bit-identical repeated calls."""
    print("case", case, flush=True)
    spec, keep = CASES[case]()
    P = M.Problem(spec, keep)
    S_gather = M.Set(P.desc, keepalive=P)
    monkeypatch.setenv("MGPU_GENERIC_SCATTER", "1")
    S = M.Set(P.desc, keepalive=P)
    monkeypatch.delenv("MGPU_GENERIC_SCATTER")
    Q = O.OracleProblem(spec)
    s = Q.setup()
    rp, ci = S.pattern()
    assert np.array_equal(rp, s["row_ptr"]) and np.array_equal(ci, s["col_idx"])
    u = np.random.default_rng(SEED + 12).uniform(-1.0, 1.0, S.n_rows)
    vo, Ro = Q.assemble(u)
    vals, R = S.compute_jacobian_and_residual(u)
    vg, Rg = S_gather.compute_jacobian_and_residual(u)
    assert rel(vals, vo) <= 1e-12 and rel(R, Ro) <= 1e-12, (rel(vals, vo), rel(R, Ro))
    assert rel(vals, vg) <= 1e-12 and rel(R, Rg) <= 1e-12
    v2, R2 = S.compute_jacobian_and_residual(u)
    assert np.array_equal(v2, vals) and np.array_equal(R2, R)
    S.options(M.PREC_MIXED, M.QUAD_SUBDIVISION)
    vm, Rm = S.compute_jacobian_and_residual(u)
    assert np.array_equal(vm.view(np.uint64), vals.view(np.uint64)) and np.array_equal(Rm.view(np.uint64), R.view(np.uint64))


@pytest.mark.parametrize("quad", [M.QUAD_SUBDIVISION, M.QUAD_MOMENT_FIT])
def test_hex27_scatter_mode_graph_replays(monkeypatch, quad):
    """Graph replays of scatter-mode sets zero the values themselves (a fill kernel, no memset
    node) and are bit-identical to eager calls, whatever the buffers held before; with the
    subdivision and with the moment-fitted rule."""
    monkeypatch.setenv("MGPU_GENERIC_SCATTER", "1")
    sets, bufs, eager = [], [], []
    for k, n in enumerate((5, 6)):
        spec, keep = M.make_spec(3, (n, n, n), iwg=M.IWG_STRUC_LINEAR_BULK, ls_kind=M.LS_GYROID,
                                 gyroid_scale=2 * np.pi * n / 4.0, bspline_order=2, lagrange_order=2,
                                 refine_levels=k)
        P = M.Problem(spec, keep)
        S = M.Set(P.desc, keepalive=P)
        S.options(M.PREC_FP64, quad)
        u = np.random.default_rng(k).uniform(-1.0, 1.0, S.n_rows)
        ub, vb, rb = M.DeviceBuffer.from_array(u), M.DeviceBuffer(8 * S.nnz), M.DeviceBuffer(8 * S.n_rows)
        S.assemble_device(ub, vb, rb)
        M.synchronize()
        eager.append((vb.to_array(np.float64, S.nnz), rb.to_array(np.float64, S.n_rows)))
        sets.append(S)
        bufs.append((ub, vb, rb))
    monkeypatch.delenv("MGPU_GENERIC_SCATTER")
    B = M.Batch(sets, [b[0] for b in bufs], [b[1] for b in bufs], [b[2] for b in bufs], n_branches=2)
    for _ in range(3):
        for S, (_, vb, rb) in zip(sets, bufs):
            z = np.full(S.nnz, 7.0)
            M.load_library().mgpu_memcpy_htod(vb.ptr, z.ctypes.data, z.nbytes)
        M.synchronize()
        B.launch()
        B.synchronize()
        for S, (_, vb, rb), (ve, re) in zip(sets, bufs, eager):
            assert np.array_equal(vb.to_array(np.float64, S.nnz), ve)
            assert np.array_equal(rb.to_array(np.float64, S.n_rows), re)
    B.close()


def _device_free():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert M.load_library().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0   # (of its HIP runtime)
    return free.value


def test_thb_scatter_mode_chosen_by_size_properties():
    """A THB set (20^3 base, one level, about 3.3e8 element-matrix entries) that takes the scatter mode without
    being forced, its pool being more than an eighth of the memory left: symmetric K, rigid translations in
    its null space, u^T K u >= 0, R = K u, the mixed option bit for bit."""
    n = 20
    spec, keep = M.make_spec(3, (n, n, n), iwg=M.IWG_STRUC_LINEAR_BULK, ls_kind=M.LS_GYROID,
                             gyroid_scale=2 * np.pi * n / 4.0, bspline_order=2, lagrange_order=2, refine_levels=1)
    P = M.Problem(spec, keep)
    taken = M.DeviceBuffer(_device_free() - (12 << 30))
    S = M.Set(P.desc, keepalive=P)
    taken.free()
    entries = int(np.sum(np.diff(S.topology_offsets()).astype(np.int64) ** 2))
    print("elements", P.n_elements, "rows", S.n_rows, "nnz", S.nnz, "K_e entries", entries, flush=True)
    assert entries > 2 ** 28 and S.statistics()[7] == 3
    rp, ci = S.pattern()
    N = S.n_rows // 3
    u = np.random.default_rng(SEED + 43).uniform(-1.0, 1.0, S.n_rows)
    vals, R = S.compute_jacobian_and_residual(u)
    import scipy.sparse as sp
    K = sp.csr_matrix((vals, ci, rp), shape=(S.n_rows, S.n_rows))
    kmax = np.abs(vals).max()
    assert abs(K - K.T).max() <= 1e-13 * kmax
    for f in range(3):
        t = np.zeros(S.n_rows)
        t[f * N:(f + 1) * N] = 1.0
        assert np.abs(K @ t).max() <= 1e-12 * kmax * np.sqrt(S.n_rows)
    assert u @ (K @ u) >= -1e-12 * kmax * S.n_rows
    assert rel(R, K @ u) <= 1e-12
    S.options(M.PREC_MIXED, M.QUAD_SUBDIVISION)
    vm, Rm = S.compute_jacobian_and_residual(u)
    assert np.array_equal(vm.view(np.uint64), vals.view(np.uint64)) and np.array_equal(Rm.view(np.uint64), R.view(np.uint64))


@pytest.mark.parametrize("left_gib", [3, 12])
def test_large_hex27_set_where_memory_is_short(left_gib):
    """A HEX27 set of 3.7e8 element-matrix entries (a pool of 2.7 GiB) with most of the device's memory
    taken: it assembles without the pool, whether that would not fit (3 GiB left) or would take more
    than an eighth of what is left (12 GiB); with the memory free it keeps the pool.  Both sum the same element
    matrices, up to 27 a value, in another order: 27 x 1.1e-16; R rows of 375 such values."""
    n = 40
    spec, keep = M.make_spec(3, (n, n, n), iwg=M.IWG_STRUC_LINEAR_BULK, ls_kind=M.LS_GYROID,
                             gyroid_scale=2 * np.pi * n / 4.0, bspline_order=2, lagrange_order=2)
    P = M.Problem(spec, keep)
    u = np.random.default_rng(SEED + 54).uniform(-1.0, 1.0, 3 * P.n_adofs_per_type)
    S = M.Set(P.desc, keepalive=P)
    assert S.statistics()[7] == 1
    v1, R1 = S.compute_jacobian_and_residual(u)
    S.close()
    taken = M.DeviceBuffer(_device_free() - (left_gib << 30))
    try:
        S = M.Set(P.desc, keepalive=P)
        assert S.statistics()[7] == 3
        v2, R2 = S.compute_jacobian_and_residual(u)
        S.close()
    finally:
        taken.free()
    assert rel(v2, v1) <= 1e-14 and rel(R2, R1) <= 1e-13


@pytest.mark.parametrize("scatter", ["", "0", "1"])
@pytest.mark.parametrize("order", [1, 2])
def test_hex27_tensor_and_general_rows(order, scatter, monkeypatch):
    """HEX27 elements whose T is a tensor product (nodal rows, p = 2 B-splines) take K_e straight from
    the element's moments, any other T takes K_e = T^T K_p T; both in one set, adofs numbered at random
    (every tensor order among the elements' sorted adofs), against the oracle: FP64 sums in another
    order, K within 1e-13 (5e-16 measured; 27 x 27 products of unit-sized terms).  Summed row by row (the default), by gather
    lists or in scatter mode."""
    spec, keep = M.make_spec(3, (4, 3, 5), iwg=M.IWG_STRUC_LINEAR_BULK, spheres=[[0.45, 0.5, 0.55, 0.34]],
                             bspline_order=order, lagrange_order=2)
    P = M.Problem(spec, keep)
    a = P.arrays()
    rng = np.random.default_rng(SEED + 51)
    adof = np.ascontiguousarray(rng.permutation(P.n_adofs_per_type)[a["t_adof"]].astype(np.int32))
    weight = np.array(a["t_weight"], np.float64)
    t_ptr = a["t_ptr"].astype(np.int64)
    other = rng.choice(P.n_elements, P.n_elements // 3, replace=False)   # T rows that are no tensor product
    for e in other:
        weight[t_ptr[27 * e + 5]:t_ptr[27 * e + 6]] *= 1.25
    d = M.SetDesc()
    ctypes.memmove(ctypes.byref(d), ctypes.byref(P.desc), ctypes.sizeof(M.SetDesc))
    d.t_adof = adof.ctypes.data_as(ctypes.POINTER(ctypes.c_int32))
    d.t_weight = weight.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    if scatter:
        monkeypatch.setenv("MGPU_GENERIC_SCATTER", scatter)
    S = M.Set(d, keepalive=(P, adof, weight))
    monkeypatch.delenv("MGPU_GENERIC_SCATTER", raising=False)
    rp, ci = S.pattern()
    u = rng.uniform(-1.0, 1.0, S.n_rows)
    vo, Ro, _ = O.assemble_desc(d, rp, ci, u)
    for quad in (M.QUAD_SUBDIVISION, M.QUAD_MOMENT_FIT):
        for prec in (M.PREC_FP64, M.PREC_MIXED):
            S.options(prec, quad)
            vals, R = S.compute_jacobian_and_residual(u)
            assert rel(vals, vo) <= 1e-13 and rel(R, Ro) <= 1e-13, (quad, prec, rel(vals, vo), rel(R, Ro))


@pytest.mark.parametrize("case", ["p2_circle_16x12_plane_stress", "thb_sphere_4_hex27_diffusion", "thb_plane_5_hex27_elasticity",
                                  "enriched_gyroid_6_p2_hex27_elasticity"])
def test_rows_mode_sums_in_element_order(case, monkeypatch):
    """Rows mode adds the element matrices into a row in ascending element order, as the gather lists
    do: bit-identical K (HEX27 sets can be forced onto the lists), R the row times u to rounding."""
    spec, keep = CASES[case]()
    P = M.Problem(spec, keep)
    S = M.Set(P.desc, keepalive=P)
    monkeypatch.setenv("MGPU_GENERIC_SCATTER", "0")
    S_lists = M.Set(P.desc, keepalive=P)
    monkeypatch.delenv("MGPU_GENERIC_SCATTER")
    u = np.random.default_rng(SEED + 52).uniform(-1.0, 1.0, S.n_rows)
    v1, R1 = S.compute_jacobian_and_residual(u)
    v2, R2 = S_lists.compute_jacobian_and_residual(u)
    assert np.array_equal(v1.view(np.uint64), v2.view(np.uint64)) and rel(R1, R2) <= 1e-14


# HEX27 node order: half steps along each axis (corners, edges, centre, faces)
HEX27_HALF = ("000 200 220 020 002 202 222 022 100 210 120 010 001 201 221 021 102 212 122 012 "
              "111 110 112 011 211 101 121")


def _slivers():
    """Sub-tets of [-1, 1]^3 that leave a basis function almost untouched: at corners, along edges and
    faces, around the cell's centre, and inside, of extent d."""
    def tet(p, e):
        X = np.array([p, p, p, p], float)
        X[0, 0] += e[0]
        X[1, 1] += e[1]
        X[3, 2] += e[2]
        return X if e[0] * e[1] * e[2] > 0 else X[[1, 0, 2, 3]]
    out = []
    for d in (1e-1, 1e-3, 1e-5):
        out += [("corner", d, [tet((-1, -1, -1), (d, d, d))]), ("corner", d, [tet((1, 1, -1), (-d, -d, d))]),
                ("edge", d, [tet((-1, 1, -1), (d, -d, 2))]), ("face", d, [tet((-1, -1, 1), (2, 2, -d))]),
                ("centre", d, [tet((0, 0, 0), (a * d, b * d, c * d)) for a in (1, -1) for b in (1, -1) for c in (1, -1)]),
                ("axis", d, [tet((0, 0, -1), (d, d, 2))]), ("mid slab", d, [tet((0, -1, -1), (d, 2, 2))]),
                ("inside", d, [tet((0.5, 0.5, 0.5), (d, d, d))])]
    return out


@pytest.mark.parametrize("iwg", [M.IWG_SPATIALDIFF_BULK, M.IWG_STRUC_LINEAR_BULK])
@pytest.mark.parametrize("order", [1, 2])
def test_hex27_small_diagonal_entries_on_slivers(order, iwg):
    """Every diagonal entry of a HEX27 element matrix to its own relative error, however small the
    entry: a diagonal is a sum of w |grad N|^2 over the TET_35 points, all terms of one sign, so the
    error of a correct sum is that of grad N.  The coordinates' rounding, 1e-16 of the cell, is 1e-16 / d of a
    distance d to a corner where grad N vanishes with d^2 (nodal rows) or N and grad N with d^6 (B-spline
    rows, squared): 12 x 1e-16 / d; 200 points' roundings add 1e-14.  Each sliver is an element of its
    own, without shared adofs, against sums in extended precision."""
    spec, keep = M.make_spec(3, (3, 3, 3), iwg=iwg, bspline_order=order, lagrange_order=2)
    P = M.Problem(spec, keep)
    a = P.arrays()
    nf = 3 if iwg == M.IWG_STRUC_LINEAR_BULK else 1
    cases = _slivers()
    # the T rows and box of the middle element, adofs of its own for every sliver, in a random order
    e0 = 13
    tp = a["t_ptr"].astype(np.int64)
    r0, r1 = tp[27 * e0], tp[27 * e0 + 27]
    ids = np.unique(a["t_adof"][r0:r1])
    rng = np.random.default_rng(SEED + 53)
    n = len(cases)
    order_of = [rng.permutation(27) for _ in range(n)]
    col = np.searchsorted(ids, a["t_adof"][r0:r1])
    ig = [np.array(c[2]).reshape(-1) for c in cases]
    nm = 2 if nf == 3 else 1
    box = a["ip_box"].reshape(-1, 6)[e0]
    arrays = {"t_ptr": np.concatenate([[0]] + [tp[27 * e0 + 1:27 * e0 + 28] - r0 + i * (r1 - r0) for i in range(n)]),
              "t_adof": np.concatenate([27 * i + order_of[i][col] for i in range(n)]),
              "t_weight": np.tile(a["t_weight"][r0:r1], n),
              "ig_ptr": np.concatenate([[0], np.cumsum([len(c[2]) for c in cases])]), "ig_xi": np.concatenate(ig),
              "material": np.tile(a["material"].reshape(-1, nm)[e0], n), "ip_box": np.tile(box, n),
              "elem_cell": np.zeros(n, np.int32), "vertex_phi": np.zeros(0)}
    d, keep_arrays = M.desc_from_arrays(P.desc, arrays)
    d.n_elements = n
    d.n_adofs_per_type = 27 * n
    d.elem_cell = None
    d.lattice = M.Lattice()
    S = M.Set(d, keepalive=(P, keep_arrays))
    rp, ci = S.pattern()
    vals, _ = S.compute_jacobian_and_residual(np.zeros(S.n_rows))
    import scipy.sparse as sp
    diag = sp.csr_matrix((vals, ci, rp), shape=(S.n_rows, S.n_rows)).diagonal()
    # reference: the rows' functions at the points, in extended precision
    ld = np.longdouble
    xi, w = (v.astype(ld) for v in O.rule("TET_35"))
    bary = np.stack([xi[:, 0], xi[:, 1], 1 - xi[:, 0] - xi[:, 1] - xi[:, 2], xi[:, 2]], 1)
    h = box[3:].astype(ld)
    # 1D functions of an adof per axis: Lagrange, or uniform quadratic B-splines; which, from T
    T = np.zeros((27, 27))
    for b in range(27):
        for q in range(tp[27 * e0 + b], tp[27 * e0 + b + 1]):
            T[b, col[q - r0]] += a["t_weight"][q]
    half = np.array([[int(c) for c in t] for t in HEX27_HALF.split()])
    T1 = np.array([[0.5, 0.5, 0], [0.125, 0.75, 0.125], [0, 0.5, 0.5]]) if order == 2 else np.eye(3)
    tensor = {tuple(T1[half[:, 0], i] * T1[half[:, 1], j] * T1[half[:, 2], k]): (i, j, k)
              for i in range(3) for j in range(3) for k in range(3)}
    worst = {}
    for i, (kind, size, tets) in enumerate(cases):
        X = np.array(tets).astype(ld)
        x = np.einsum("qv,tvd->tqd", bary, X).reshape(-1, 3)
        J = np.stack([(X[:, r] - X[:, 2]) * (h / 2) for r in (0, 1, 3)], 1)
        det = (J[:, 0, 0] * (J[:, 1, 1] * J[:, 2, 2] - J[:, 2, 1] * J[:, 1, 2]) -
               J[:, 0, 1] * (J[:, 1, 0] * J[:, 2, 2] - J[:, 1, 2] * J[:, 2, 0]) +
               J[:, 0, 2] * (J[:, 1, 0] * J[:, 2, 1] - J[:, 1, 1] * J[:, 2, 0])) / 6
        ws = (det[:, None] * w[None]).reshape(-1)
        u, v = (1 + x) / 2, (1 - x) / 2
        if order == 2:
            f, df = [v * v / 2, (1 + 2 * u * v) / 2, u * u / 2], [-v / 2, -x / 2, u / 2]
        else:
            f, df = [-x * v, 4 * u * v, x * u], [x - ld(0.5), -2 * x, x + ld(0.5)]
        for c in range(27):
            t = tensor[tuple(T[:, c])]
            g2 = [ws @ (np.prod([(df if k == ax else f)[t[k]][:, k] for k in range(3)], axis=0) * 2 / h[ax]) ** 2
                  for ax in range(3)]
            for fld in range(nf):
                if nf == 1:
                    want = ld(arrays["material"][0]) * sum(g2)
                else:
                    E, nu = (ld(m) for m in arrays["material"][:2])
                    lam, mu = E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))
                    want = lam * g2[fld] + mu * (sum(g2) + g2[fld])
                got = diag[fld * 27 * n + 27 * i + order_of[i][c]]
                err = float(abs(got - want) / want)
                worst[kind, size] = max(worst.get((kind, size), 0.0), err)
    for k, e in sorted(worst.items()):
        print(k, "%.1e" % e, flush=True)
    assert all(e <= 1e-14 + 12e-16 / k[1] for k, e in worst.items()), worst
