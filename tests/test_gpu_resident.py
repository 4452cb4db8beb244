"""Jacobi-PCG in one launch (vectors resident on the compute units) against SuperLU and against the
launch-per-kernel path, at the sizes where the rows are dealt out differently: one workgroup, one
row per thread with 256 or 1024 threads, two and four rows per thread, partly filled last chunks and
workgroups, rows of 9, 18, 50 and 81 entries."""
import ctypes as C

import numpy as np
import pytest

from tests import problems as P

pytestmark = pytest.mark.gpu


def _case(name):
    kind, *n = name.split("-")
    n = [int(v) for v in n]
    if kind == "poisson":
        return P.poisson_rect(*n)
    if kind == "panel":
        return P.tapered_panel(n[0], lam=1.0, mu=0.4, multiplier=0.1)
    if kind == "cube":
        return P.neo_hooke_cube(n[0], disp=0.01)
    return P.cook_membrane_q2(0.1)


def _pcg(prob, vals, b, precision, tol, wait):
    import torch
    from autopdex_amd import _native as N
    from autopdex_amd.backend import current_stream
    N.call("apx_plan_set_resident_wait", prob.plan, wait)
    x = torch.full_like(b, float("nan"))
    ks = N.KrylovStats()
    N.call("apx_pcg", prob.plan, C.c_void_p(vals.data_ptr()), C.c_void_p(b.data_ptr()), C.c_void_p(x.data_ptr()),
           precision, N.APX_PRECOND_JACOBI, tol, 0.0, 0, C.byref(ks), current_stream())
    N.call("apx_plan_set_resident_wait", prob.plan, 2.0)
    return x.cpu().numpy(), ks


# 1/nothing free apart from a few rows, one workgroup (K = 1, 2), 256 threads, 1024 threads with K = 1, 2, 4
@pytest.mark.parametrize("name", ["poisson-2-2", "poisson-9-8", "poisson-33-30", "poisson-46-45", "poisson-61-200",
                                  "poisson-255-257", "poisson-300-299", "poisson-601-603", "poisson-801-1001",
                                  "panel-12", "panel-60", "q2", "cube-4", "cube-13"])
def test_resident_pcg_matches_direct_and_streaming(torch_gpu, name):
    torch = torch_gpu
    import scipy.sparse as sp
    import scipy.sparse.linalg as spla
    from autopdex_amd import _native as N
    from autopdex_amd import backend, learned
    dofs, settings, static, o = _case(name)
    prob = backend.get_problem(dofs, settings, static)
    print(f"[case] resident pcg {name}: {prob.n_free} rows", flush=True)
    vals = learned.tangent(prob)
    indptr, indices = prob.csr_pattern()
    A = sp.csr_matrix((vals.cpu().numpy(), indices, indptr))
    rhs = np.random.default_rng(prob.n_free).standard_normal(prob.n_free)
    b = torch.from_numpy(rhs).cuda()
    x, ks = _pcg(prob, vals, b, N.APX_FP64, 1e-12, 2.0)
    assert ks.converged == 1
    assert np.linalg.norm(A @ x - rhs) <= 1e-9 * np.linalg.norm(rhs)
    if prob.n_free < 100000:
        lu = spla.spsolve(A.tocsc(), rhs)
        assert np.linalg.norm(x - lu) <= 1e-8 * np.linalg.norm(lu)
    xs, kss = _pcg(prob, vals, b, N.APX_FP64, 1e-12, -1.0)  # launch per kernel
    assert kss.converged == 1 and abs(ks.iterations - kss.iterations) <= 2 + kss.iterations // 20
    assert np.linalg.norm(x - xs) <= 1e-8 * np.linalg.norm(xs)
    again, ka = _pcg(prob, vals, b, N.APX_FP64, 1e-12, 2.0)
    assert ka.iterations == ks.iterations and np.array_equal(x, again)
    # no patience at all: the launch may be given up anywhere, the solve is completed all the same
    xz, kz = _pcg(prob, vals, b, N.APX_FP64, 1e-12, 0.0)
    assert kz.converged == 1 and np.linalg.norm(xz - xs) <= 1e-8 * np.linalg.norm(xs)


@pytest.mark.parametrize("name", ["poisson-33-30", "poisson-130-140", "poisson-601-603", "cube-6"])
def test_resident_pcg_fp32(torch_gpu, name):
    torch = torch_gpu
    from autopdex_amd import _native as N
    from autopdex_amd import backend, learned
    dofs, settings, static, o = _case(name)
    prob = backend.get_problem(dofs, settings, static)
    print(f"[case] resident pcg fp32 {name}: {prob.n_free} rows", flush=True)
    vals = learned.tangent(prob).float()
    b = torch.from_numpy(np.random.default_rng(1).standard_normal(prob.n_free)).float().cuda()
    x, ks = _pcg(prob, vals, b, N.APX_FP32, 1e-3, 2.0)
    xs, kss = _pcg(prob, vals, b, N.APX_FP32, 1e-3, -1.0)
    assert ks.converged == 1 and kss.converged == 1
    # both residuals are recursive FP32 ones of at most 1e-3 |b|; the true ones are held to twice that
    for v in (x, xs):
        r = b.double() - learned.spmv(prob, vals.double(), torch.from_numpy(v).double().cuda())
        assert float(r.norm()) <= 2e-3 * float(b.double().norm())


@pytest.mark.parametrize("maxiter", [1, 2, 7])
def test_resident_pcg_stops_at_maxiter(torch_gpu, maxiter):
    torch = torch_gpu
    from autopdex_amd import backend, learned
    dofs, settings, static, o = P.poisson_rect(120, 90)
    prob = backend.get_problem(dofs, settings, static)
    vals = learned.tangent(prob)
    b = torch.from_numpy(np.random.default_rng(3).standard_normal(prob.n_free)).cuda()
    print(f"[case] resident pcg maxiter {maxiter}", flush=True)
    from autopdex_amd import _native as N
    out = []
    for wait in (2.0, -1.0):
        N.call("apx_plan_set_resident_wait", prob.plan, wait)
        x, ks = learned.pcg(prob, vals, b, tol=1e-12, maxiter=maxiter)
        assert ks.iterations == maxiter and ks.converged == 0
        out.append(x.cpu().numpy())
    N.call("apx_plan_set_resident_wait", prob.plan, 2.0)
    # a few iterations of the same recurrence: equal up to the rounding of the sums
    assert np.linalg.norm(out[0] - out[1]) <= 1e-12 * np.linalg.norm(out[1])
