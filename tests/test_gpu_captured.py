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


def _tangent(prob, u, vals, precision, stream):
    from autopdex_amd import _native as N
    N.call("apx_assemble_tangent", prob.plan, C.c_void_p(u.data_ptr()), C.c_void_p(vals.data_ptr()), precision,
           C.c_void_p(stream.cuda_stream))


@pytest.mark.parametrize("kind,size,sets", [("hex", (12, 13, 14), 1), ("panel", (60, 61), 2), ("q2", (14, 15), 2)])
@pytest.mark.parametrize("captured", ["fp32", "fp64"])
def test_captured_tangent_beside_the_other_precision(torch_gpu, kind, size, sets, captured):
    """A captured tangent keeps its scratch when the other precision comes later and when it runs beside it;
    with two sets, the second is the larger one."""
    torch = torch_gpu
    from autopdex_amd import _native as N
    from autopdex_amd import backend
    u, settings, static, _, _ = _problem(kind, size, 1, seed=6)
    if sets == 2:
        elems = settings["connectivity"][0]
        k = len(elems) // 4
        settings["connectivity"] = (np.ascontiguousarray(elems[:k]), np.ascontiguousarray(elems[k:]))
        static["model"], static["assembling mode"] = static["model"] * 2, static["assembling mode"] * 2
    prob = backend.get_problem(u, settings, static)
    print(f"[case] captured tangent {kind} {size} {captured}", flush=True)
    ud = prob.to_device(u.ravel())
    types = {"fp32": (N.APX_FP32, torch.float32), "fp64": (N.APX_FP64, torch.float64)}
    (mine, dt), (other, odt) = types[captured], types["fp64" if captured == "fp32" else "fp32"]
    vals = torch.empty(prob.nnz, dtype=dt, device="cuda")
    _tangent(prob, ud, vals, mine, torch.cuda.current_stream())
    torch.cuda.synchronize()
    want = vals.clone()
    graph = _capture(torch, lambda st: _tangent(prob, ud, vals, mine, st))
    beside = [torch.empty(prob.nnz, dtype=odt, device="cuda") for _ in range(9)]
    _tangent(prob, ud, beside[0], other, torch.cuda.current_stream())
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for _ in range(4):
        vals.fill_(float("nan"))
        torch.cuda.synchronize()
        with torch.cuda.stream(streams[0]):
            graph.replay()
        for b in beside[1:]:
            _tangent(prob, ud, b, other, streams[1])
        torch.cuda.synchronize()
        assert torch.equal(vals, want)
        assert all(torch.equal(b, beside[0]) for b in beside)
