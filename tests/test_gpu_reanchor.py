"""Mixed-precision Newton on a linear problem, one PCG run re-anchored to the FP64 residual: the FP32
recursion stops at its own tolerance while the FP64 residual is still above the Newton threshold, so
the next run goes on from a run that ended by itself.  Resident runs count and go on as the
launch-per-kernel ones do, and 'linear maxiter' bounds the total."""
import ctypes as C

import pytest

from tests import problems as P

pytestmark = pytest.mark.gpu


def _newton(torch, prob, wait, vectors64, delta, tol, maxiter=0):
    from autopdex_amd import _native as N
    from autopdex_amd.backend import current_stream
    o = N.NewtonOptions(newton_tol=tol, relative=1, maxiter=30, damping=1.0, precision=N.APX_FP32,
                        precond=N.APX_PRECOND_JACOBI, lin_tol=1e-3, lin_atol=0.0, lin_maxiter=maxiter, reuse_tangent=1,
                        forcing=0, reliable_delta=delta, fp32_element_arith=0, krylov_fp64_vectors=vectors64)
    s = N.NewtonStats()
    u = torch.zeros(prob.n_dofs, dtype=torch.float64, device="cuda")
    zero = torch.zeros_like(u)
    N.call("apx_plan_set_resident_wait", prob.plan, wait)
    N.call("apx_newton", prob.plan, C.c_void_p(u.data_ptr()), C.c_void_p(zero.data_ptr()), C.byref(o), C.byref(s),
           current_stream())
    N.call("apx_plan_set_resident_wait", prob.plan, 2.0)
    return u.cpu().numpy(), s


# Grids of one workgroup, of one with two rows a thread and of several.  delta 1e-30: no reliable updates,
# the first run ends by itself with the FP64 residual above the threshold; 1e-2: with them.
CASES = [((17, 16), 0, 3e-7, 1e-30), ((17, 16), 1, 1e-7, 1e-30), ((44, 43), 0, 3e-6, 1e-30),
         ((44, 43), 1, 1e-6, 1e-30), ((121, 90), 0, 1e-5, 1e-30), ((121, 90), 1, 3e-6, 1e-30),
         ((17, 16), 0, 1e-11, 1e-2), ((44, 43), 1, 1e-11, 1e-2), ((121, 90), 0, 1e-11, 1e-2), ((121, 90), 1, 1e-11, 1e-2)]


@pytest.mark.parametrize("size,vectors64,tol,delta", CASES)
def test_runs_after_a_finished_run(torch_gpu, size, vectors64, tol, delta):
    torch = torch_gpu
    from autopdex_amd import backend
    dofs, settings, static, o = P.poisson_rect(*size)
    prob = backend.get_problem(dofs, settings, static)
    print(f"[case] reanchor {size} vectors64 {vectors64} tol {tol} delta {delta}", flush=True)
    us, ss = _newton(torch, prob, -1.0, vectors64, delta, tol)  # one launch per kernel
    ur, sr = _newton(torch, prob, 2.0, vectors64, delta, tol)
    print(f"  streaming {ss.iterations} anchors {ss.krylov_iterations} its, resident {sr.iterations} anchors "
          f"{sr.krylov_iterations} its", flush=True)
    assert not ss.diverged and not sr.diverged and ss.iterations >= 2
    assert ss.residual_norm <= tol * ss.initial_residual and sr.residual_norm <= tol * sr.initial_residual
    assert sr.iterations == ss.iterations
    # one recurrence whose sums are rounded in another order
    assert abs(sr.krylov_iterations - ss.krylov_iterations) <= 2 + ss.krylov_iterations // 10
    uz, sz = _newton(torch, prob, 0.0, vectors64, delta, tol)  # runs may be given up anywhere
    assert not sz.diverged and sz.iterations == ss.iterations
    assert abs(sz.krylov_iterations - ss.krylov_iterations) <= 2 + ss.krylov_iterations // 10
    bound = min(ss.krylov_iterations, sr.krylov_iterations) * 3 // 4
    for wait in (-1.0, 2.0):
        _, s = _newton(torch, prob, wait, vectors64, delta, tol, maxiter=bound)
        # stopped by the bound: given up, or (the recursion aims at half of the threshold) just converged
        assert s.krylov_iterations == bound and (s.diverged or s.residual_norm <= tol * s.initial_residual)
