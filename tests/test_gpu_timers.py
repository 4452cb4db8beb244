"""The bytes that the assembly timers state: inputs once and outputs once, in the type that is stored."""
import ctypes as C

import pytest

from tests import problems as P

pytestmark = pytest.mark.gpu


def _bytes(prob, name):
    from autopdex_amd import _native as N
    ms, count, nbytes = C.c_double(), C.c_int64(), C.c_int64()
    N.call("apx_get_timing", prob.plan, name, C.byref(ms), C.byref(count), C.byref(nbytes))
    assert count.value > 0
    return nbytes.value


def test_rounded_tangent_of_row_owners_counts_its_fp32_values(torch_gpu):
    from autopdex_amd import _native as N
    from autopdex_amd import backend, solver
    dofs, settings, static, o = P.neo_hooke_cube(4, disp=0.01)
    static = dict(static, **{"hip precision": "mixed", "linear tolerance": 1e-5})
    prob = backend.get_problem(dofs, settings, static)
    print("[case] timers of the row owners", flush=True)
    N.call("apx_set_timing", prob.plan, 1)
    solver.solver(dofs, settings, static, newton_tol=1e-9)
    elements = settings["connectivity"][0].size * 4
    got = _bytes(prob, b"tangent_f64_to_f32"), _bytes(prob, b"residual")
    N.call("apx_set_timing", prob.plan, 0)
    assert got[0] == prob.n_nodes * 3 * 8 + prob.n_dofs * 8 + elements + prob.nnz * 4
    assert got[1] == prob.n_nodes * 3 * 8 + prob.n_dofs * 8 * 2 + elements
