"""The layout of resident PCG runs, on the CPU: every workgroup's p window, halo and vectors lie within
the LDS that the launch asks for, every row has an owner, and every window position fits its 16 bits."""
import ctypes as C

import pytest

LDS = 160 * 1024  # of a compute unit


def layout(n, bw, row, precision, cus=256):
    from autopdex_amd import _native as N
    out = N.ResidentLayout()
    N.call("apx_resident_shape", n, bw, row, precision, cus, C.byref(out))
    return out


def check(n, bw, row, precision):
    """The workgroups' needs as k_pcg_resident reads and writes them; False: the system does not fit."""
    s = layout(n, bw, row, precision)
    if s.threads == 0:
        return False
    size = 8 if precision == 0 else 4
    own = 64 * s.chunks
    assert 1 <= s.workgroups <= 256 and s.workgroups == -(-n // own)
    assert s.rows_per_thread * s.threads >= min(own, -(-n // 64) * 64)
    assert row <= s.row_entries or s.row_entries == 0
    for g in range(s.workgroups):
        row0, row1 = g * own, min((g + 1) * own, n)
        w0, w1 = max(0, row0 - bw), min(n, row1 + bw)
        halo = (row0 - w0) + (w1 - row1)
        need = (w1 - w0) + halo + (2 * (row1 - row0) if s.vectors_in_lds else 0)
        assert need * size <= s.lds_bytes, (n, bw, row, precision, g, need * size, s.lds_bytes)
        assert w1 - w0 <= 65536
    assert s.lds_bytes <= LDS - 1024  # static words of the reductions beside it
    return True


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("row", [1, 9, 18, 50, 54, 81, 82, 500])
def test_every_workgroup_fits_its_lds(row, precision):
    sizes = {1, 2, 63, 64, 65, 255, 256, 257, 300, 511, 512, 513, 700, 1023, 1024, 1025, 1028, 1100, 1500, 2047, 2048, 2049,
             2100, 3000, 4096, 4097, 5000, 8192, 8200, 10000, 16384, 20000, 65536, 98305, 131000, 262145, 524288, 786500,
             1048576, 3000000}
    fits = 0
    for n in sorted(sizes):
        for bw in sorted({0, 1, 17, 63, 64, 100, 131, 517, 1000, 2000, 4990, 9000, 32767, n // 3, n // 2, n - 2, n - 1}):
            if 0 <= bw < n:
                fits += check(n, bw, row, precision)
    assert fits > 50


@pytest.mark.parametrize("n,bw,row", [(1028, 517, 18), (1100, 1099, 18), (5000, 4990, 9), (300, 299, 54), (384, 221, 81)])
def test_partly_filled_last_workgroup_with_a_wide_halo(n, bw, row):
    assert check(n, bw, row, 0) and check(n, bw, row, 1)


def test_what_does_not_fit():
    assert layout(1 << 22, 2049, 9, 0).threads == 0      # too many rows
    assert layout(100000, 32768, 9, 0).threads == 0      # offsets beyond 16 bits
    assert layout(100000, 30000, 9, 0).threads == 0      # a window beyond the LDS
    assert layout(0, 0, 9, 0).threads == 0
    assert layout(100, 10, 9, 0, cus=0).threads == 0
