"""Rows of the reduced matrix with more entries than 13 bits count: sets of bricks, each a fan around one
node that all sets share."""
import ctypes as C

import numpy as np
import pytest


def _fans(sets, elems, seed):
    """(coords, [connectivity]): per element an own cube, turned about node 0."""
    rng = np.random.default_rng(seed)
    corners = np.array([[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0], [0, 0, 1], [1, 0, 1], [1, 1, 1], [0, 1, 1]], float)
    coords, conns, at = [np.zeros((1, 3))], [], 1
    for _ in range(sets):
        conn = np.zeros((elems, 8), np.int64)
        for e in range(elems):
            q = np.linalg.qr(rng.standard_normal((3, 3)))[0]
            q *= np.sign(np.linalg.det(q))
            coords.append(rng.uniform(0.5, 1.5) * corners[1:] @ q.T)
            conn[e, 1:] = np.arange(at, at + 7)
            at += 7
        conns.append(conn)
    return np.concatenate(coords), conns


@pytest.mark.parametrize("sets,widest", [(6, 3 * (1 + 6 * 60 * 7)), (7, 3 * (1 + 7 * 60 * 7))])
def test_plans_take_rows_of_any_length(sets, widest):
    """7,563 and 8,823 entries."""
    from autopdex_amd import _native as N
    coords, conns = _fans(sets, 60, 0)
    mask, plan, params = np.zeros((len(coords), 3), np.uint8), C.c_void_p(), np.zeros(2)
    N.call("apx_plan_create", C.byref(plan), 3, len(coords), coords.ctypes.data, 3, mask.ctypes.data)
    for c in conns:
        N.call("apx_plan_add_set", plan, c.ctypes.data, len(c), 8, N.MODEL_NEO_HOOKE, params.ctypes.data, 2, None)
    N.call("apx_plan_build_pattern", plan)
    info = N.PlanInfo()
    N.call("apx_plan_get_info", plan, C.byref(info))
    ptr, idx = np.empty(info.n_free + 1, np.int32), np.empty(info.nnz, np.int32)
    N.call("apx_plan_csr_pattern", plan, ptr.ctypes.data, idx.ctypes.data)
    N.call("apx_plan_destroy", plan)
    assert np.diff(ptr).max() == widest


@pytest.mark.gpu
@pytest.mark.parametrize("sets", [6, 7])
def test_tangent_with_wide_rows(torch_gpu, sets):
    from autopdex_amd import assembler, models, seeder, spaces
    from oracle import assembly as OA
    from oracle import elements as OE
    from tests import problems as P
    coords, conns = _fans(sets, 60, 1)
    rng = np.random.default_rng(2)
    shape = coords.shape
    mask = rng.random(shape) < 0.02
    mask[0] = False
    pot = models.mixed_reference_domain_potential(models.hyperelastic_integrand(models.neo_hooke, 1.7, 0.6),
                                                  {"u": spaces.fem_iso_line_quad_brick}, *seeder.gauss_legendre_nd(3, 2),
                                                  "u")
    settings = {"connectivity": tuple(conns), "dirichlet dofs": mask, "node coordinates": coords,
                "dirichlet conditions": np.zeros(shape)}
    static = P.static([pot] * sets)
    u = 0.01 * rng.standard_normal(shape)
    print(f"[case] wide rows, {sets} sets", flush=True)
    free = ~mask.ravel()
    want = assembler.assemble_tangent(u, settings, static, form="bcoo").tocsr()[:, free][free]
    want.sort_indices()
    assert (np.diff(want.indptr).max() > 8192) == (sets == 7)
    got = assembler.assemble_tangent(u, settings, static)
    assert np.array_equal(got.indptr, want.indptr) and np.array_equal(got.indices, want.indices)
    scale = np.abs(want.data).max()
    assert np.abs(got.data - want.data).max() <= 1e-12 * scale  # sums of up to 420 elements
    f32 = assembler.assemble_tangent(u, settings, static, precision="fp32")
    assert np.abs(f32.data - want.data).max() <= 1e-4 * scale
    r = assembler.assemble_residual(u, settings, static)
    ro = OA.residual([(OE.NeoHooke(1.7, 0.6), c, None) for c in conns], coords, u.ravel(), 3)
    assert np.abs(r.ravel() - ro).max() <= 1e-11 * np.abs(ro).max()
