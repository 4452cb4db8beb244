"""Streaming Jacobi-PCG on 9-point matrices read as their upper diagonals, against the same iterations
in scipy: lines shorter, equal and longer than a wavefront's rows, two lines, columns beyond int16,
grid corners off the diagonals, Dirichlet sides, ragged ends, and a matrix that is not symmetric."""
import ctypes as C

import numpy as np
import pytest

from tests import problems as P

pytestmark = pytest.mark.gpu


def _problem(kind, size):
    from autopdex_amd import backend, geometry, mesher, models, seeder, spaces
    coords, elems = mesher.structured_mesh(size, P.UNIT_SQUARE, "quad")
    if kind == "corners":  # free corners: entries off the lines
        mask = geometry.in_sdfs(coords, lambda x: geometry.psdf_polygon(x, P.UNIT_SQUARE))
    elif kind == "side":   # lines of size[1] rows
        mask = np.abs(coords[:, 1]) < 1e-12
    else:                  # "few": all sides and some nodes inside; lines change where they lie
        mask = (np.abs(coords - 0.5) > 0.5 - 1e-12).any(axis=1)
        mask[np.random.default_rng(0).integers(0, mask.size, 5)] = True
    pot = models.mixed_reference_domain_potential(models.poisson_source_integrand(),
                                                  {"phi": spaces.fem_iso_line_quad_brick},
                                                  *seeder.gauss_legendre_nd(dimension=2, order=2), "phi")
    settings = {"connectivity": (elems,), "dirichlet dofs": mask, "node coordinates": coords,
                "dirichlet conditions": np.zeros(mask.shape)}
    return backend.get_problem(np.zeros(mask.shape), settings, P.static([pot]))


def _reference(A, b, its):
    inv = 1.0 / A.diagonal()
    x, r = np.zeros_like(b), b.copy()
    z = inv * r
    p, g = z.copy(), r @ z
    for _ in range(its):
        q = A @ p
        a = g / (p @ q)
        x += a * p
        r -= a * q
        z = inv * r
        g, g0 = r @ z, g
        p = z + (g / g0) * p
    return x


# Each FP64 (FP32) iteration rounds about 4 vectors of sums of up to 12 terms: 7 iterations err by about
# 7 x 4 x 12 half ulps = 3.7e-14 (2e-5) of the largest value; five times that for the recurrence.
@pytest.mark.parametrize("kind,size,precision", [
    ("side", (8500, 31), "fp64"), ("side", (8300, 32), "fp64"), ("side", (4400, 62), "fp64"),
    ("side", (4300, 63), "fp64"), ("side", (2200, 125), "fp64"), ("side", (2, 100000), "fp64"),
    ("corners", (601, 449), "fp64"), ("corners", (263, 1000), "fp64"), ("few", (520, 530), "fp64"),
    ("side", (1, 140000), "fp64"), ("corners", (733, 719), "fp32"), ("side", (5000, 107), "fp32")])
def test_pcg_by_lines_matches_scipy(torch_gpu, kind, size, precision):
    torch = torch_gpu
    import scipy.sparse as sp
    from autopdex_amd import _native as N
    from autopdex_amd import learned
    from autopdex_amd.backend import current_stream
    prob = _problem(kind, size)
    print(f"[case] pcg by lines {kind} {size} {precision}: {prob.n_free} rows", flush=True)
    prec, dt = (N.APX_FP64, torch.float64) if precision == "fp64" else (N.APX_FP32, torch.float32)
    tol = 5 * 3.7e-14 if precision == "fp64" else 5 * 2e-5
    N.call("apx_plan_set_resident_wait", prob.plan, -1.0)  # launch per kernel
    vals = learned.tangent(prob).to(dt)
    indptr, indices = prob.csr_pattern()
    rows = np.repeat(np.arange(prob.n_free), np.diff(indptr))
    rng = np.random.default_rng(prob.n_free)
    b = torch.from_numpy(rng.standard_normal(prob.n_free)).to(dt).cuda()
    # entries below the diagonal away from their mirror images: the whole matrix has to be read
    skew = vals.clone()
    below = np.flatnonzero(np.asarray(indices) < rows)
    skew[torch.from_numpy(rng.choice(below, 50)).cuda()] *= 1.25
    for v, its in ((vals, 1), (vals, 7), (skew, 7), (vals, 7)):
        x = torch.full_like(b, float("nan"))
        ks = N.KrylovStats()
        N.call("apx_pcg", prob.plan, C.c_void_p(v.data_ptr()), C.c_void_p(b.data_ptr()), C.c_void_p(x.data_ptr()), prec,
               N.APX_PRECOND_JACOBI, 1e-14, 0.0, its, C.byref(ks), current_stream())
        A = sp.csr_matrix((v.double().cpu().numpy(), indices, indptr), shape=(prob.n_free,) * 2)
        ref = _reference(A, b.double().cpu().numpy(), its)
        assert ks.iterations == its
        assert np.abs(x.double().cpu().numpy() - ref).max() <= tol * np.abs(ref).max()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_newton_by_lines(torch_gpu, precision):
    """The Newton drivers' matrices (FP64, FP32 rounded) by lines: a converged residual."""
    from autopdex_amd import _native as N
    from autopdex_amd import backend, solver
    from oracle import assembly as OA
    dofs, settings, static, o = P.poisson_rect(301, 1783)
    static = dict(static, **{"hip precision": precision, "linear tolerance": 1e-10 if precision == "fp64" else 1e-6})
    prob = backend.get_problem(dofs, settings, static)
    N.call("apx_plan_set_resident_wait", prob.plan, -1.0)
    print(f"[case] newton by lines {precision}", flush=True)
    sol, infos = solver.solver(dofs, settings, static, newton_tol=1e-9)
    assert not infos[2]
    r = OA.residual(o["sets"], o["coords"], np.asarray(sol).ravel(), 1)
    assert np.linalg.norm(r[~o["mask"]]) <= 1.1e-9


# A network of zero weights with its Jacobi part is the preconditioner D^-1, and flexible CG with it the
# iterations of _reference; tolerance as above times five for its own recurrence of beta.
@pytest.mark.parametrize("kind,size,precision", [("side", (521, 530), "fp64"), ("corners", (600, 470), "fp64"),
                                                 ("corners", (520, 533), "fp32"), ("side", (8500, 31), "fp32")])
def test_flexible_cg_by_lines(torch_gpu, kind, size, precision):
    torch = torch_gpu
    import scipy.sparse as sp
    from autopdex_amd import learned
    prob = _problem(kind, size)
    print(f"[case] flexible cg by lines {kind} {size} {precision}: {prob.n_free} rows", flush=True)
    net = learned.UNetPreconditioner(size[0] + 1, size[1] + 1, 2, (16, 16), 1, 1, relu=False, batch=1, jacobi_skip=True)
    net.set_params(np.zeros(net.n_params))
    net.attach(prob)
    dt = torch.float64 if precision == "fp64" else torch.float32
    vals = learned.tangent(prob).to(dt)
    indptr, indices = prob.csr_pattern()
    rng = np.random.default_rng(prob.n_free)
    b = torch.from_numpy(rng.standard_normal(prob.n_free)).cuda()
    rows = np.repeat(np.arange(prob.n_free), np.diff(indptr))
    skew = vals.clone()
    below = np.flatnonzero(np.asarray(indices) < rows)
    skew[torch.from_numpy(rng.choice(below, 50)).cuda()] *= 1 + 1e-12 if precision == "fp64" else 1 + 1e-6
    for v in (vals, skew):
        x, ks = learned.fcg(prob, v, b, tol=0.0, maxiter=7, precision=precision)
        A = sp.csr_matrix((v.double().cpu().numpy(), indices, indptr), shape=(prob.n_free,) * 2)
        ref = _reference(A, b.cpu().numpy(), 7)
        assert ks.iterations == 7
        assert np.abs(x.cpu().numpy() - ref).max() <= 25 * 3.7e-14 * np.abs(ref).max() + 1e-5 * (v is skew and precision == "fp32")
