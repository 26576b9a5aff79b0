"""The kernels' dispatch rules on the host, asked of the library's own rule functions.  Nothing is
launched."""

import ctypes

import pytest

import internal_shim


def rows_tile(m, n, k, count):
    out = (ctypes.c_int * 3)()
    internal_shim.load().shim_rows_tile(m, n, k, count, out)
    return list(out)


@pytest.mark.parametrize("count", [1, 2, 64])
@pytest.mark.parametrize("k", [1024, 2048, 3072])
def test_rows_tile_has_no_tile_of_padding_rows(k, count):
    """Two row tiles a block only where there are two, whatever the matrix's width; a group keeps the
    waves that one matrix's launch has."""
    for m in (4, 16, 17, 32, 33, 500):
        for n in (2, 130, 3072, 12224, 12290, 40000, 151936):
            mt, nt, k12 = rows_tile(m, n, k, count)
            single = rows_tile(m, n, k, 1)
            assert (mt, nt) in ((1, 1), (1, 2), (1, 4), (2, 4)) and 16 * (mt - 1) < m, (m, n)
            assert k12 == single[2] == (k == 3072 and single[:2] == [1, 1]), (m, n)
            if count > 1:
                assert mt == 1 or not k12
                assert nt in (1, 4), (m, n)   # the tiles that the grouped kernel has


def test_chain_resid_needs_a_split():
    """The short prefill's output projections write raw partial tiles, which a reduction adds: without a
    split there is none, so y would never be written."""
    for m in (1, 75, 512):
        for k in (512, 1024, 1536, 2048, 3072):
            for ksplit in (0, 1, 2):
                applies = internal_shim.load().shim_chain_resid(m, 1024, k, ksplit)
                assert applies == (ksplit == 2 and k // 2 in (512, 1024, 1536)), (m, k, ksplit)


# (rows, N, K, ep): the rows kernel is the faster one / the tiled kernels are, measured next to the lines
ROWS = [(1, 128, 1024, "F16"), (569, 3072, 1024, "F16"), (1700, 1024, 1024, "F32"), (12288, 128, 1024, "F16"),
        (1536, 1024, 2048, "F16"), (768, 2048, 2048, "F32"), (8000, 128, 2048, "F16"), (1700, 1024, 2048, "RESID"),
        (3400, 512, 2048, "RESID"), (13000, 128, 3072, "F32"), (1700, 1024, 3072, "F16"), (64, 128, 1152, "F16")]
TILED = [(13000, 128, 1024, "F16"), (6800, 256, 1024, "F32"), (1540, 1024, 2048, "F16"), (850, 2048, 2048, "F32"),
         (425, 4096, 2048, "F16"), (10000, 128, 2048, "F16"), (4500, 256, 2048, "F16"), (2800, 512, 2048, "F32"),
         (1800, 1024, 1024, "RESID"), (1800, 1024, 3072, "F16"), (65, 128, 1152, "F16"), (4, 128, 1088, "F16")]


@pytest.mark.parametrize("calls,rows", [(ROWS, 1), (TILED, 0)], ids=["rows", "tiled"])
def test_gemm_takes_the_faster_kernel(calls, rows):
    for m, n, k, ep in calls:
        assert internal_shim.load().shim_rows_apply(m, n, k, getattr(internal_shim, f"EP_{ep}")) == rows, (m, n, k, ep)


def test_linear_takes_the_faster_kernel():
    """A GEMV per row up to 3 rows and for few outputs, the rows kernel past that."""
    gemv = [(3, 3072, 1024, 1), (4, 64, 3072, 1), (100, 2, 2048, 1), (4, 1024, 1024, 1), (4, 1024, 1024, 0),
            (5, 1024, 1024, 0), (33, 64, 2048, 1), (6, 512, 3072, 0), (3, 151936, 1024, 0)]
    rows = [(5, 1024, 1024, 1), (6, 1024, 1024, 0), (4, 2048, 1024, 1), (4, 1024, 2048, 0), (4, 1024, 3072, 0), (4, 1024, 3072, 1),
            (33, 130, 3072, 1), (65535, 2, 1024, 1), (4, 151936, 1024, 1)]
    for calls, want in ((gemv, 0), (rows, 1)):
        for c in calls:
            assert internal_shim.load().shim_rows_linear(*c) == want, c
