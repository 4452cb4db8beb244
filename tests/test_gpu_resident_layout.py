"""Resident Jacobi-PCG for each way of dealing out the rows, on matrices whose solution is checked by
the true residual: SPD values on the pattern of a mesh (weighted graph Laplacian plus a shift, condition
number at most 8), with node numberings of small bandwidth and random ones, whose halo is the rest of
the system.  Every case names the layout that it expects, and that the resident launch ran."""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_rows import _book, _q2_grid

pytestmark = pytest.mark.gpu


def _grid(kind, size):
    """(coords, elements, DOFs per node, Dirichlet DOFs)"""
    from autopdex_amd import mesher
    if kind == "quad" or kind == "clamped":
        coords, elems = mesher.structured_mesh(size[:2], ((0, 0), (1, 0), (1, 1), (0, 1)), "quad")
    elif kind == "q2":
        coords, elems = _q2_grid(*size[:2])
    elif kind == "brick":
        coords, elems = mesher.structured_mesh(
            size, ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)), "brick")
    else:
        coords, elems = _book(*size[:2])
    d = {"quad": size[-1], "clamped": 2, "q2": 2}.get(kind, 3)
    mask = np.zeros((len(coords), d), bool)
    if kind == "clamped":
        mask[:size[1] + 1] = True
    return coords, elems, d, mask


class System:
    def __init__(self, kind, size, shuffle):
        import scipy.sparse as sp
        from autopdex_amd import _native as N
        coords, elems, d, mask = _grid(kind, size)
        rng = np.random.default_rng(len(coords))
        if shuffle:
            perm = rng.permutation(len(coords))
            elems, new = perm[elems], np.empty_like(coords)
            new[perm] = coords
            coords = new
        coords, elems = np.ascontiguousarray(coords, np.float64), np.ascontiguousarray(elems, np.int64)
        mask = np.ascontiguousarray(mask, np.uint8)
        self.plan = C.c_void_p()
        N.call("apx_plan_create", C.byref(self.plan), coords.shape[1], len(coords), coords.ctypes.data, d,
               mask.ctypes.data)
        model = N.MODEL_POISSON_SOURCE if d == 1 else N.MODEL_NEO_HOOKE
        params = np.zeros(4)
        N.call("apx_plan_add_set", self.plan, elems.ctypes.data, len(elems), elems.shape[1], model,
               params.ctypes.data, 4, None)
        N.call("apx_plan_finalize", self.plan)
        info = N.PlanInfo()
        N.call("apx_plan_get_info", self.plan, C.byref(info))
        self.n = info.n_free
        ptr, idx = np.empty(self.n + 1, np.int32), np.empty(info.nnz, np.int32)
        N.call("apx_plan_csr_pattern", self.plan, ptr.ctypes.data, idx.ctypes.data)
        rows = np.repeat(np.arange(self.n), np.diff(ptr))
        self.bw, self.row = int(np.abs(idx - rows).max()), int(np.diff(ptr).max())
        # weights in [0.5, 1.5], the same for (i, j) and (j, i)
        low, high = np.minimum(rows, idx).astype(np.int64), np.maximum(rows, idx).astype(np.int64)
        w = -(0.5 + ((low * 7919 + high * 104729) % 1009) / 1009.0)
        w[rows == idx] = 0.0
        w[rows == idx] = 1.3 * np.bincount(rows, -w, self.n)
        self.A = sp.csr_matrix((w, idx, ptr), shape=(self.n, self.n))
        self.b = rng.standard_normal(self.n)

    def __del__(self):
        from autopdex_amd import _native as N
        N.lib().apx_plan_destroy(self.plan)

    def layout(self, precision, cus):
        from autopdex_amd import _native as N
        out = N.ResidentLayout()
        N.call("apx_resident_shape", self.n, self.bw, self.row, precision, cus, C.byref(out))
        return out

    def solve(self, torch, precision, tol, wait=2.0):
        """(x, iterations, resident launches)"""
        from autopdex_amd import _native as N
        N.call("apx_plan_set_resident_wait", self.plan, wait)
        x, its, completed, given_up = self.run(torch, precision, tol)
        assert given_up == 0
        return x, its, completed

    def run(self, torch, precision, tol):
        """(x, iterations, completed resident launches, given up ones)"""
        from autopdex_amd import _native as N
        from autopdex_amd.backend import current_stream
        dt = torch.float64 if precision == N.APX_FP64 else torch.float32
        vals, b = torch.from_numpy(self.A.data).to("cuda", dt), torch.from_numpy(self.b).to("cuda", dt)
        x = torch.full_like(b, float("nan"))
        ks, ms, nbytes = N.KrylovStats(), C.c_double(), C.c_int64()
        N.call("apx_set_timing", self.plan, 1)
        N.call("apx_pcg", self.plan, C.c_void_p(vals.data_ptr()), C.c_void_p(b.data_ptr()), C.c_void_p(x.data_ptr()),
               precision, N.APX_PRECOND_JACOBI, tol, 0.0, 0, C.byref(ks), current_stream())
        counts = []
        for name in (b"pcg_resident_f64" if precision == N.APX_FP64 else b"pcg_resident_f32", b"pcg_resident_given_up"):
            count = C.c_int64()
            N.call("apx_get_timing", self.plan, name, C.byref(ms), C.byref(count), C.byref(nbytes))
            counts.append(count.value)
        N.call("apx_set_timing", self.plan, 0)
        assert ks.converged == 1
        return x.double().cpu().numpy(), ks.iterations, *counts


# (mesh, size, random numbering, expected threads, rows per thread, entries in registers)
WIDE = [("clamped", (2, 256), 0, (1024, 1, 18)),     # a last workgroup of 4 rows, 517 before it
        ("quad", (45, 46, 1), 1, (1024, 1, 9)), ("quad", (64, 64, 1), 1, (1024, 2, 9)),
        ("quad", (70, 70, 1), 1, (1024, 2, 9)), ("quad", (22, 23, 2), 1, (1024, 1, 18)),
        ("quad", (31, 40, 2), 1, (1024, 1, 18)), ("q2", (4, 8), 1, (256, 1, 54)), ("q2", (15, 17), 1, (512, 1, 54)),
        ("brick", (4, 4, 4), 1, (256, 1, 81)), ("brick", (10, 11, 12), 1, (512, 1, 81)),
        ("book", (30, 6), 1, (1024, 1, 0)), ("book", (30, 12), 1, (1024, 1, 0))]
# the mesher's numberings: every layout with one or several workgroups, up to the largest sizes
MESHED = [("quad", (20, 21, 1), 0, (1024, 1, 9)), ("quad", (44, 43, 1), 0, (1024, 2, 9)),
          ("quad", (47, 46, 1), 0, (1024, 1, 9)), ("quad", (120, 121, 1), 0, (1024, 2, 9)),
          ("quad", (800, 801, 1), 0, (512, 6, 9)), ("quad", (900, 901, 1), 0, (512, 8, 9)),
          ("quad", (22, 20, 2), 0, (1024, 1, 18)), ("quad", (60, 61, 2), 0, (1024, 1, 18)),
          ("quad", (362, 362, 2), 0, (512, 3, 18)), ("quad", (450, 449, 2), 0, (512, 4, 18)),
          ("q2", (10, 11), 0, (256, 1, 54)), ("q2", (30, 31), 0, (512, 1, 54)),
          ("brick", (8, 9, 7), 0, (256, 1, 81)), ("brick", (15, 14, 16), 0, (512, 1, 81)),
          ("book", (30, 20), 0, (1024, 1, 0)), ("q2", (130, 131), 0, (1024, 1, 0)), ("q2", (185, 186), 0, (1024, 2, 0)),
          ("quad", (520, 521, 2), 0, (1024, 4, 0))]


@pytest.mark.parametrize("kind,size,shuffle,shape", WIDE + MESHED)
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_resident_pcg_by_layout(torch_gpu, kind, size, shuffle, shape, precision):
    torch = torch_gpu
    from autopdex_amd import _native as N
    s = System(kind, size, shuffle)
    prec = N.APX_FP64 if precision == "fp64" else N.APX_FP32
    lay = s.layout(prec, torch.cuda.get_device_properties(0).multi_processor_count)
    print(f"[case] layout {kind} {size} shuffle {shuffle} {precision}: {s.n} rows of {s.row}, bandwidth {s.bw}, "
          f"{lay.workgroups} workgroups, {lay.lds_bytes} bytes of LDS", flush=True)
    assert (lay.threads, lay.rows_per_thread, lay.row_entries) == shape
    # the recursive residual is at most tol |b|; the true one differs from it by the rounding of at most
    # 60 iterations, 60 * 8 * 1.2e-7 = 6e-5 in FP32 and 1e-13 in FP64
    tol, most = (1e-12, 1.1e-12) if precision == "fp64" else (1e-3, 1.1e-3)
    x, its, resident = s.solve(torch, prec, tol)
    assert resident == 1 and its <= 60
    norm = np.linalg.norm(s.b)
    assert np.linalg.norm(s.A @ x - s.b) <= most * norm
    xs, its_s, resident = s.solve(torch, prec, tol, wait=-1.0)  # one launch per kernel
    assert resident == 0 and abs(its - its_s) <= 1
    assert np.linalg.norm(s.A @ xs - s.b) <= most * norm


def test_a_given_up_launch_is_remembered(torch_gpu):
    """Without patience the launches of a large grid are given up: the solve is completed all the same, the
    plan's next 16 solves do without, a further give-up counts for 64, and setting the wait starts anew."""
    torch = torch_gpu
    from autopdex_amd import _native as N
    s = System("quad", (900, 901, 1), 0)
    norm = np.linalg.norm(s.b)
    N.call("apx_plan_set_resident_wait", s.plan, 0.0)
    tried = []
    for i in range(24):
        x, its, completed, given_up = s.run(torch, N.APX_FP64, 1e-12)
        assert np.linalg.norm(s.A @ x - s.b) <= 1.1e-12 * norm
        if completed or given_up:
            tried.append((i, given_up))
    print(f"[case] resident launches without patience (solve, given up): {tried}", flush=True)
    assert tried[0] == (0, 1)
    assert [i for i, _ in tried] == [0, 17]
    x, its, completed = s.solve(torch, N.APX_FP64, 1e-12)
    assert completed == 1 and np.linalg.norm(s.A @ x - s.b) <= 1.1e-12 * norm
