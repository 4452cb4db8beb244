"""Captured assembly: replays of a graph may overlap with other calls of the same plan on other
streams, and with each other; every residual keeps the bits that a call alone gives."""
import ctypes as C

import numpy as np
import pytest

from tests import problems as P
from tests.test_gpu_rows import CASES, _problem

pytestmark = pytest.mark.gpu


def _residual(prob, u, r, stream):
    from autopdex_amd import _native as N
    N.call("apx_assemble_residual", prob.plan, C.c_void_p(u.data_ptr()), C.c_void_p(r.data_ptr()),
           C.c_void_p(stream.cuda_stream))


def _capture(torch, call):
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        call(torch.cuda.current_stream())
    return graph


@pytest.mark.parametrize("kind,size,shuffle", CASES + [("traction", (9,), 0)])
def test_captured_residual_has_the_same_bits(torch_gpu, kind, size, shuffle):
    """Every element type, nodes without elements and a second set (the traction's boundary lines)."""
    torch = torch_gpu
    from autopdex_amd import backend
    if kind == "traction":
        u, settings, static, o = P.tapered_panel(*size)
    else:
        u, settings, static, _, _ = _problem(kind, size, shuffle, seed=len(kind) + sum(size))
    prob = backend.get_problem(u, settings, static)
    print(f"[case] captured residual {kind} {size} shuffle {shuffle}", flush=True)
    rng = np.random.default_rng(2)
    h = np.ptp(settings["node coordinates"], axis=0).max() / max(size) / 50
    us = [torch.from_numpy(h * rng.standard_normal(prob.n_dofs)).cuda() for _ in range(3)]
    v, r, alone = us[0].clone(), torch.empty_like(us[0]), []
    graph = _capture(torch, lambda st: _residual(prob, v, r, st))
    many = [_capture(torch, lambda st: _residual(prob, v, r, st)) for _ in range(17)]  # the last ones without scratch
    for w in us:
        want = torch.full_like(w, float("nan"))
        _residual(prob, w, want, torch.cuda.current_stream())
        torch.cuda.synchronize()
        alone.append(want)
    for i, g in ((1, graph), (2, many[0]), (2, many[-1]), (0, graph), (0, many[-1]), (1, many[-2])):
        v.copy_(us[i])
        r.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(r, alone[i])


@pytest.mark.parametrize("kind,size", [("hex", (20, 21, 22)), ("panel", (90, 101)), ("q2", (30, 31))])
def test_replays_overlap_with_other_residuals(torch_gpu, kind, size):
    """Two graphs, replayed on two streams while a third computes residuals of other vectors eagerly."""
    torch = torch_gpu
    from autopdex_amd import backend
    u, settings, static, _, _ = _problem(kind, size, 1, seed=3)
    prob = backend.get_problem(u, settings, static)
    print(f"[case] overlapping residuals {kind} {size}", flush=True)
    rng = np.random.default_rng(4)
    h = np.ptp(settings["node coordinates"], axis=0).max() / max(size) / 50
    us = [torch.from_numpy(h * rng.standard_normal(prob.n_dofs)).cuda() for _ in range(3)]
    alone = [torch.empty_like(v) for v in us]
    for v, r in zip(us, alone):
        _residual(prob, v, r, torch.cuda.current_stream())
    out = [[torch.empty_like(us[0]) for _ in range(8)] for _ in us]

    def eight(i, st):
        for r in out[i]:
            _residual(prob, us[i], r, st)

    graphs = [_capture(torch, lambda st, i=i: eight(i, st)) for i in range(2)]
    streams = [torch.cuda.Stream() for _ in us]
    for _ in range(5):
        for rs in out:
            for r in rs:
                r.fill_(float("nan"))
        torch.cuda.synchronize()
        for i in range(2):
            with torch.cuda.stream(streams[i]):
                graphs[i].replay()
        eight(2, streams[2])
        torch.cuda.synchronize()
        for i, rs in enumerate(out):
            for r in rs:
                assert torch.equal(r, alone[i])
