"""One plan, or one device, used from several threads and streams at once."""
import ctypes as C
import threading

import numpy as np
import pytest

from tests.test_gpu_captured import _residual, _tangent
from tests.test_gpu_resident_layout import System
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


def _solve(torch, s):
    from autopdex_amd import _native as N
    x, its, completed, given_up = s.run(torch, N.APX_FP64, 1e-12)
    assert completed == 1 and given_up == 0
    assert np.linalg.norm(s.A @ x - s.b) <= 1.1e-12 * np.linalg.norm(s.b)
    return x


def test_resident_solves_on_three_threads(torch_gpu):
    """Systems that together have more workgroups than the device has compute units take turns: every run
    is completed, with the bits that it has alone."""
    torch = torch_gpu
    systems = [System("quad", (900, 901, 1), 0), System("quad", (800, 799, 1), 0), System("brick", (10, 11, 12), 0),
               System("quad", (20, 21, 1), 0)]
    print("[case] resident solves on threads", flush=True)
    alone = [_solve(torch, s) for s in systems]

    def work(i):
        for _ in range(6):
            assert np.array_equal(_solve(torch, systems[i]), alone[i])

    _in_threads(torch, len(systems), work)


def test_a_solve_does_not_wait_for_another_threads_stream(torch_gpu):
    """A solve whose stream still has half a second of other work to do holds no compute units meanwhile: a
    solve on another thread (allocation-free, since freeing memory waits for the whole device) ends before."""
    torch = torch_gpu
    from autopdex_amd import _native as N
    first, second = System("quad", (885, 886, 1), 0), System("quad", (300, 301, 1), 0)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert first.layout(0, cus).workgroups + second.layout(0, cus).workgroups > cus  # not both at once
    data = [tuple(torch.from_numpy(v).cuda() for v in (s.A.data, s.b, np.zeros(s.n))) for s in (first, second)]

    def solve(i):  # no copies from or to the host, which would wait for the stream
        s, entry = ((first, "apx_pcg"), (second, "apx_pcg_noalloc"))[i]
        ks = N.KrylovStats()
        N.call(entry, s.plan, *(C.c_void_p(t.data_ptr()) for t in data[i]), N.APX_FP64, N.APX_PRECOND_JACOBI, 1e-12,
               0.0, 0, C.byref(ks), C.c_void_p(torch.cuda.current_stream().cuda_stream))
        return ks.converged

    assert solve(0) == 1 and solve(1) == 1
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    start.record()
    torch.cuda._sleep(10_000_000)
    end.record()
    end.synchronize()
    cycles = int(10_000_000 * 500 / start.elapsed_time(end))
    print(f"[case] two threads, one with a busy stream: {cycles} cycles", flush=True)
    torch.cuda.synchronize()
    queued, busy, seen = threading.Event(), torch.cuda.Event(), []

    def work(i):
        if i == 0:
            torch.cuda._sleep(cycles)
            busy.record()
            queued.set()
            assert solve(0) == 1
        else:
            assert queued.wait(10)
            threading.Event().wait(0.1)  # the first solve has come to its run
            seen.append((solve(1), busy.query()))

    _in_threads(torch, 2, work)
    assert seen == [(1, False)]
    for s, (_, _, x) in zip((first, second), data):
        assert np.linalg.norm(s.A @ x.cpu().numpy() - s.b) <= 1.1e-12 * np.linalg.norm(s.b)
