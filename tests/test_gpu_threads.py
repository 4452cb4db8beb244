"""One plan, or one device, used from several threads and streams at once."""
import threading

import numpy as np
import pytest

from tests.test_gpu_captured import _residual, _tangent
from tests.test_gpu_rows import _problem

pytestmark = pytest.mark.gpu


def _in_threads(torch, n, work):
    """work(i) on n threads, each on a stream of its own; exceptions are raised here."""
    errors, start = [], threading.Barrier(n)
    device = torch.cuda.current_device()

    def run(i):
        try:
            torch.cuda.set_device(device)
            with torch.cuda.stream(torch.cuda.Stream()):
                start.wait()
                work(i)
                torch.cuda.current_stream().synchronize()
        except BaseException as e:  # noqa: B902
            errors.append(e)

    threads = [threading.Thread(target=run, args=(i,)) for i in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    if errors:
        raise errors[0]


@pytest.mark.parametrize("kind,size", [("hex", (9, 8, 10)), ("panel", (50, 41)), ("q2", (12, 13))])
def test_assembly_of_one_plan_from_three_threads(torch_gpu, kind, size):
    torch = torch_gpu
    from autopdex_amd import _native as N
    from autopdex_amd import backend
    u, settings, static, _, _ = _problem(kind, size, 1, seed=8)
    prob = backend.get_problem(u, settings, static)
    print(f"[case] assembly from threads {kind} {size}", flush=True)
    rng = np.random.default_rng(9)
    h = np.ptp(settings["node coordinates"], axis=0).max() / max(size) / 50
    us = [torch.from_numpy(h * rng.standard_normal(prob.n_dofs)).cuda() for _ in range(3)]
    rs, ts = [], []
    for v in us:
        rs.append(torch.empty_like(v))
        ts.append(torch.empty(prob.nnz, dtype=torch.float64, device="cuda"))
        _residual(prob, v, rs[-1], torch.cuda.current_stream())
        _tangent(prob, v, ts[-1], N.APX_FP64, torch.cuda.current_stream())
    torch.cuda.synchronize()
    got = [[(torch.empty_like(r), torch.empty_like(t)) for _ in range(30)] for r, t in zip(rs, ts)]
    torch.cuda.synchronize()

    def work(i):
        for r, t in got[i]:
            _residual(prob, us[i], r, torch.cuda.current_stream())
            _tangent(prob, us[i], t, N.APX_FP64, torch.cuda.current_stream())

    _in_threads(torch, 3, work)
    for i in range(3):
        assert all(torch.equal(r, rs[i]) and torch.equal(t, ts[i]) for r, t in got[i])
