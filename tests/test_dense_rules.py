"""Which kernels the dense operators take, asked on the host (smx_measure_dense_backward_form, smx_measure_dense_forward_form)."""
import ctypes

import pytest

from smore_amd import _lib

GENERAL, PER_QUERY, SHARED, REVERSE = range(4)


def form(kind, bsize, num, dim, be=None, ne=None, bc=None, nc=1, low=0):
    """(path, floats per column, wavefronts, reads ahead); entity [B,N,.] against query [B,1,.] unless told otherwise."""
    path, vec, waves, ahead = (ctypes.c_int() for _ in range(4))
    lib = _lib.load()
    rc = lib.smx_measure_dense_backward_form(lib.smx_kind_from_name(kind.encode()), bsize, num, be or bsize, ne or num,
                                             bc or bsize, nc, dim, low, *(ctypes.byref(x) for x in (path, vec, waves, ahead)))
    assert rc == 0, lib.smx_last_error()
    return path.value, vec.value, waves.value, ahead.value


@pytest.mark.parametrize("kind", ["l1", "box_out", "rotate", "beta_kl"])
@pytest.mark.parametrize("dim,low", [(32, 0), (128, 0), (400, 0), (1024, 0), (33, 0), (34, 0), (32, 8), (512, 4)])
@pytest.mark.parametrize("layout", ["per query", "shared"])
def test_every_launch_is_one_that_hip_takes(kind, dim, low, layout):
    """HIP takes launches of fewer than 2^32 threads, and a batch brings a workgroup per query: at the batches around which
    workgroups of sixteen, eight and two wavefronts reach that limit, the kernels taken are below it, or the general ones."""
    for bsize in (1 << 8, (1 << 22) - 1, 1 << 22, 5_000_000, (1 << 23) - 1, 1 << 23, (1 << 25) - 1):
        for num in (1, 2, 8, 32):
            path, vec, waves, _ = form(kind, bsize, num, dim, low=low, **(dict(be=1) if layout == "shared" else {}))
            assert path in ((GENERAL, PER_QUERY) if layout == "per query" else (GENERAL, SHARED))
            few = num if kind != "beta_kl" else (num + 1) // 2
            least = 8 if layout == "shared" else min(few, 8)
            assert (path == GENERAL) == (bsize * least * 64 >= 1 << 32)
            assert path == GENERAL or bsize * waves * 64 < 1 << 32
            assert layout == "shared" or waves <= few, "a wavefront without a row"
    if layout == "shared":      # a workgroup per shared row, too
        for num in ((1 << 23) - 1, 1 << 23):
            path, _, _, _ = form(kind, 2, num, dim, be=1, low=low)
            assert path == (SHARED if num * 512 < 1 << 32 else GENERAL)


@pytest.mark.parametrize("dim", [4, 3])
def test_row_counts_that_an_int_cannot_be_stepped_through(dim):
    """A wavefront's row number goes up to 2 x 16 beyond the last row before it is compared: not beyond 2^31 - 1."""
    top = (1 << 31) - 1
    for num, special in ((top, False), (top - 31, False), (top - 32, True)):
        assert (form("l1", 1, num, dim)[0] == PER_QUERY) == special
        assert (form("l1", 1, num, dim, ne=1, nc=num)[0] == REVERSE) == (special and dim == 4)
    assert form("l1", 1, 1 << 31, dim, ne=1, nc=1)[0] == GENERAL


def test_columns_by_row_length_and_alignment():
    for dim, low, want in ((400, 0, 4), (1024, 0, 4), (1024, 16, 4), (400, 8, 2), (402, 8, 2), (400, 4, 1), (401, 0, 1),
                           (512, 4, 1), (513, 0, 0), (514, 0, 0), (1020, 4, 0), (1028, 0, 0)):
        path, vec, _, _ = form("box_out", 64, 40, dim, low=low)
        assert vec == want and path == (PER_QUERY if want else GENERAL)
        path, vec, _, _ = form("box_out", 64, 40, dim, be=1, low=low)
        assert vec == want and path == (SHARED if want else GENERAL)
    assert form("box_out", 64, 40, 400, ne=1, nc=40)[0] == REVERSE
    assert form("box_out", 64, 40, 401, ne=1, nc=40)[0] == GENERAL
    assert form("box_out", 64, 40, 400, ne=40, nc=40)[0] == GENERAL


def forward_form(bsize, num, dim, be=None, ne=None, nc=1, low=0):
    path, rows = ctypes.c_int(), ctypes.c_int()
    lib = _lib.load()
    rc = lib.smx_measure_dense_forward_form(bsize, num, be or bsize, ne or num, bsize, nc, dim, low, ctypes.byref(path),
                                            ctypes.byref(rows))
    assert rc == 0, lib.smx_last_error()
    return path.value, rows.value


def test_forward_row_numbers_and_launches_stay_in_range():
    """A tile's end and a row number stepped beyond it fit an int, and a launch has fewer than 2^32 threads; the general kernel,
    whose grid is bounded and whose numbers are 64 bits wide, takes the rest."""
    top = (1 << 31) - 1
    for bsize in (1, 2, 3):
        for num in (1, 9, 100_000, top // bsize - 300_000, top // bsize - 100_000, top // bsize - 8, top // bsize):
            for layout, extra in ((PER_QUERY, {}), (SHARED, dict(be=1)), (REVERSE, dict(ne=1, nc=num))):
                path, rows = forward_form(bsize, num, 4, **extra)
                tiles = -(-num // rows) if rows else 0
                if path == GENERAL:
                    assert num > top - 300_000
                else:
                    assert path == layout or num == 1 or bsize == 1 and layout == SHARED
                    assert tiles * rows + 8 <= top and bsize * tiles * 256 < 1 << 32
    assert forward_form(1, top - 8, 4)[0] == forward_form(1, top - 100_000, 4)[0] == GENERAL
    for bsize in ((1 << 24) - 1, 1 << 24):      # a workgroup of 256 threads per query
        assert forward_form(bsize, 1, 4)[0] == (PER_QUERY if bsize < 1 << 24 else GENERAL)
    assert forward_form(64, 40, 400, low=8)[0] == forward_form(64, 40, 401)[0] == GENERAL
