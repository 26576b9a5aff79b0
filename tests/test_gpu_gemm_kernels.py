"""The skinny and the 64-row tiled MFMA GEMM, each by itself, on the GPU.

q4d_gemm and q4d_gemm_splitk take the rows kernel for few outputs, so the shapes that pin the other
kernels' operand layout, splits, epilogues and int4 conversion are chosen (tiled: a number of columns
that is no multiple of 128) or called (skinny: the launcher of the batched decode step) past that rule.
Integer-exact inputs: x of small integers and weights that are exact in fp16 after their one rounding,
every partial sum a multiple of 2^-14 below 2^10, so each output equals the float64 product of the same
operands bit for bit.  Scale codes lie on both sides of the one-fma conversion's limit (4094), with and
without a wide code in the matrix."""

import ctypes

import numpy as np
import pytest
import torch

import internal_shim as shim
import oracle as o
from gpu_helpers import q4
from llm_accelerator_amd import _lib
from llm_accelerator_amd._lib import Q4D_F16, Q4D_F32, check
from llm_accelerator_amd.model import current_stream

pytestmark = pytest.mark.gpu

WIDE = np.array([4094, 4095, 4096, 8192, 12288])


def case(rng, n, k, wide, top=128):
    """(packed codes, scale codes, the fp16 weights as float64)."""
    q = rng.integers(-8, 8, size=(n, k))
    scale = rng.integers(1, top, size=(n, k // 64)).astype(np.uint16)
    if wide:  # one group of every third row
        rows = np.arange(0, n, 3)
        scale[rows, rng.integers(0, k // 64, len(rows))] = rng.choice(WIDE, len(rows))
    s16 = (scale.astype(np.float64) / 16384.0).astype(np.float16)
    w16 = (q.astype(np.float16) * np.repeat(s16, 64, axis=1)).astype(np.float64)
    return o.pack_signed_int4(q), scale, w16


def product(x, w16):
    assert (np.abs(x) @ np.abs(w16).T).max() < 1024 and np.array_equal(w16 * 2 ** 14, np.rint(w16 * 2 ** 14))
    return x @ w16.T


def tiled(x, rows=64):
    """[m, k] fp16 in 32-column chunks of 64 rows."""
    m, k = x.shape
    t = torch.full((k // 32, rows, 32), float("nan"), dtype=torch.float16, device=x.device)
    t[:, :m] = x.view(m, k // 32, 32).transpose(0, 1)
    return t


def skinny(mats, x, y, ep, resid=None, part=None, y_tiled=False):
    """launch_gemm as a batched decode step calls it; returns the split that ran."""
    m, k = x.shape
    xt = 2 <= m
    xd = tiled(x) if xt else x
    desc = (_lib.Q4dMatrix * len(mats))(*[w.descriptor() for w in mats])
    used = ctypes.c_int(-1)
    check(shim.load().shim_skinny_gemm(desc, len(mats), xd.data_ptr(), m, y.data_ptr(), ep,
                                       resid.data_ptr() if resid is not None else None,
                                       part.data_ptr() if part is not None else None,
                                       part.numel() if part is not None else 0, int(xt), int(y_tiled),
                                       ctypes.byref(used), current_stream()), "launch_gemm")
    torch.cuda.synchronize()
    return used.value


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("m,segs,k,split", [
    (1, (128,), 1024, False), (5, (2048, 1024, 1024), 1024, False), (64, (256, 128, 128), 1024, False),
    (16, (1024,), 2048, True), (33, (1024,), 3072, True), (64, (1024,), 2048, True), (17, (128,), 1024, True),
])
def test_skinny_integer_exact(dev, m, segs, k, split, wide):
    """The q|k|v shape (three segments, fp32 out) and the output projections (with a partial buffer: K
    split over blocks, then the reduction), fp32, fp16 and in-place residual; the partials start as NaN."""
    rng = np.random.default_rng(m + sum(segs) + k + wide)
    parts = [case(rng, n, k, wide) for n in segs]
    mats = [q4(p, s, dev) for p, s, _ in parts]
    x = rng.integers(-4, 5, size=(m, k)).astype(np.float64)
    ref = product(x, np.concatenate([w for _, _, w in parts]))
    xd = torch.from_numpy(x).to(dev).half()
    n = sum(segs)
    print(f"[skinny exact] M={m} N={n} K={k} split={split} wide={wide}", flush=True)

    def part():
        return torch.full((16 * m * n,), float("nan"), device=dev) if split else None

    y = torch.full((m, n), float("nan"), device=dev)
    used = skinny(mats, xd, y, shim.EP_F32, part=part())
    assert (used > 1) == split
    np.testing.assert_array_equal(y.cpu().numpy(), ref.astype(np.float32))
    y16 = torch.full((m, n), float("nan"), dtype=torch.float16, device=dev)
    skinny(mats, xd, y16, shim.EP_F16, part=part())
    np.testing.assert_array_equal(y16.cpu().numpy(), ref.astype(np.float32).astype(np.float16))
    resid = rng.normal(size=(m, n)).astype(np.float32)
    r = torch.from_numpy(resid).to(dev)
    skinny(mats, xd, r, shim.EP_RESID, resid=r, part=part())
    np.testing.assert_array_equal(r.cpu().numpy(), resid + ref.astype(np.float32))


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("m,n", [(1, 128), (2, 3072), (31, 192), (64, 3072)])
def test_skinny_swiglu(dev, m, n, wide):
    """The gate / up pair with the SwiGLU epilogue, written tiled as the decode step does from two rows
    on: the exact sums g and u, then silu(g) u in fp32 (2^-20 of it: an exponential, a division and two
    products of 2^-23 each) rounded once or twice to fp16 (2^-11, denormals 2^-24)."""
    rng = np.random.default_rng(m + n + wide)
    (pg, sg, wg), (pu, su, wu) = case(rng, n, 1024, wide, 512), case(rng, n, 1024, wide, 512)
    x = rng.integers(-1, 2, size=(m, 1024)).astype(np.float64)
    g, u = product(x, wg), product(x, wu)
    ref = g / (1.0 + np.exp(-g)) * u
    assert np.abs(ref).max() < 60000
    print(f"[skinny swiglu] M={m} N={n} wide={wide}", flush=True)
    yt = m >= 2
    y = torch.full((n // 32, 64, 32) if yt else (m, n), float("nan"), dtype=torch.float16, device=dev)
    assert skinny([q4(pg, sg, dev), q4(pu, su, dev)], torch.from_numpy(x).to(dev).half(), y, shim.EP_SWIGLU,
                  y_tiled=yt) == 1
    out = y[:, :m].transpose(0, 1).reshape(m, n) if yt else y
    if yt:
        assert bool(torch.isnan(y[:, m:]).all())  # rows past M are not written
    out = out.double().cpu().numpy()
    assert np.all(np.abs(out - ref) <= np.abs(ref) * (2.0 ** -11 + 2.0 ** -20) + 2.0 ** -24)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("m,n,k", [(1, 256, 1088), (7, 128, 192), (64, 384, 1984), (65, 256, 1088), (130, 128, 64),
                                   (300, 512, 960)])
def test_tiled_64_rows_integer_exact(dev, m, n, k, wide):
    """The unsplit 64-row tiles through q4d_gemm: fp32, fp16 and in-place residual, partial row tiles, one
    and many K steps."""
    assert k % 128 and n // 128 * ((m + 127) // 128) < 256
    rng = np.random.default_rng(m + n + k + wide)
    packed, scale, w16 = case(rng, n, k, wide)
    w = q4(packed, scale, dev)
    x = rng.integers(-4, 5, size=(m, k)).astype(np.float64)
    ref = product(x, w16)
    xd = torch.from_numpy(x).to(dev).half()
    print(f"[tiled exact] M={m} N={n} K={k} wide={wide}", flush=True)

    def gemm(y, dtype, resid=None):
        desc = w.descriptor()
        check(_lib.load().q4d_gemm(ctypes.byref(desc), xd.data_ptr(), m, y.data_ptr(), dtype,
                                   resid.data_ptr() if resid is not None else None, current_stream()), "q4d_gemm")
        torch.cuda.synchronize()
        return y.cpu().numpy()

    y = gemm(torch.full((m, n), float("nan"), device=dev), Q4D_F32)
    np.testing.assert_array_equal(y, ref.astype(np.float32))
    y16 = gemm(torch.full((m, n), float("nan"), dtype=torch.float16, device=dev), Q4D_F16)
    np.testing.assert_array_equal(y16, ref.astype(np.float32).astype(np.float16))
    resid = rng.normal(size=(m, n)).astype(np.float32)
    r = torch.from_numpy(resid).to(dev)
    np.testing.assert_array_equal(gemm(r, Q4D_F32, r), resid + ref.astype(np.float32))
