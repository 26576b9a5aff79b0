"""q4d_linear over several activation rows (the MFMA kernel, from 4 rows and some 4000 outputs on) on the GPU
vs the oracle: tile edges in both directions, every matrix width, every input and output type."""

import ctypes

import numpy as np
import pytest
import torch

import oracle as o
from gpu_helpers import linear, q4
from llm_accelerator_amd import _lib
from llm_accelerator_amd._lib import Q4D_F16, Q4D_F32
from llm_accelerator_amd.model import Q4Tensor

pytestmark = pytest.mark.gpu

ACC = 4e-6  # fp32 accumulation error relative to sum |w x|, the bar of the one-row GEMV


@pytest.mark.parametrize("m,n,k,xdtype,ydtype,precision", [
    (4, 2, 1024, torch.float32, Q4D_F32, 2),         # few outputs: a GEMV per row
    (4, 1026, 1024, torch.float32, Q4D_F32, 2),      # the first past the GEMVs: one row tile, nearly empty
    (4, 1024, 1024, torch.float32, Q4D_F32, 2),      # ... and the last of them
    (6, 1024, 1024, torch.float16, Q4D_F32, 1),
    (16, 1024, 2048, torch.float32, Q4D_F32, 2),     # one row tile, one weight tile per block
    (17, 1030, 1024, torch.float16, Q4D_F16, 1),     # ragged both ways, fp16 in and out
    (33, 3072, 3072, torch.float32, Q4D_F32, 2),     # two weight tiles per block
    (211, 1024, 3072, torch.float32, Q4D_F16, 2),    # four weight tiles per block
    (300, 2050, 2048, torch.float16, Q4D_F32, 1),
    (50, 96, 1024, torch.float32, Q4D_F32, 1),       # fp32 activations rounded to fp16
])
def test_linear_rows_vs_oracle(dev, m, n, k, xdtype, ydtype, precision):
    rng = np.random.default_rng(m + n + k)
    packed = rng.integers(0, 256, size=(n, k // 2), dtype=np.uint8)
    scale = rng.integers(1, 3000, size=(n, k // 64)).astype(np.uint16)
    x = rng.normal(size=(m, k)) * 10.0 ** rng.integers(-3, 3, size=(m, 1))  # small rows: denormal lo halves
    xt = torch.from_numpy(x.astype(np.float32)).to(dev).to(xdtype)
    lib = _lib.load()
    _lib.check(lib.q4d_set_activation_precision(precision), "q4d_set_activation_precision")
    try:
        y = linear(q4(packed, scale, dev), xt, ydtype).double().cpu().numpy()
    finally:
        _lib.check(lib.q4d_set_activation_precision(2), "q4d_set_activation_precision")
    W = o.dequantize_q4(packed, scale, dtype=np.float64)
    x64 = xt.double().cpu().numpy()
    ref, size = x64 @ W.T, np.abs(x64) @ np.abs(W).T
    # hi + lo halves: 2^-22 of a value, and no finer than the fp16 denormal step 2^-25 of the
    # lo half; one fp16 value: 2^-11, and no finer than 2^-25
    lone = np.abs(W).sum(axis=1)[None, :] * 2.0 ** -25
    xerr = 0.0 if xdtype == torch.float16 else size * (2.0 ** -22 if precision == 2 else 2.0 ** -11) + lone
    out = np.abs(ref) * 2.0 ** -11 + 2.0 ** -25 if ydtype == Q4D_F16 else 0.0
    finite = np.abs(ref) < 65000 if ydtype == Q4D_F16 else np.ones_like(ref, dtype=bool)
    assert finite.mean() > 0.5
    assert np.all((np.abs(y - ref) <= ACC * size + xerr + out)[finite])


@pytest.mark.parametrize("m,n,k", [(20, 256, 3072), (60, 3072, 3072), (211, 1024, 3072), (600, 3072, 2048), (50, 1024, 2048)])
def test_linear_rows_integer_exact(dev, m, n, k):
    """Several 128-column units per wave through the same LDS rows (two and three per wave, and the
    general loop of the largest tile), integers small enough that every sum is exact: equal bits, so a
    row read before the wave's other lanes have stored it, or after the next unit's, shows."""
    rng = np.random.default_rng(m + n + k)
    packed = o.pack_signed_int4(rng.integers(-8, 8, size=(n, k)))
    scale = rng.integers(1, 32, size=(n, k // 64)).astype(np.uint16)
    x = rng.integers(-4, 5, size=(m, k)).astype(np.float32)
    W = o.dequantize_q4(packed, scale, dtype=np.float64)
    assert (np.abs(x).astype(np.float64) @ np.abs(W).T).max() < 1024  # multiples of 2^-14: exact in fp32
    print(f"[linear rows exact] {m} x {n} x {k}", flush=True)
    y = linear(q4(packed, scale, dev), torch.from_numpy(x).to(dev)).cpu().numpy()
    np.testing.assert_array_equal(y, (x.astype(np.float64) @ W.T).astype(np.float32))


def test_linear_rows_one_bad_row_stays_alone(dev):
    """A row holding an infinity or a NaN does not reach the other rows of its tile."""
    rng = np.random.default_rng(3)
    w = q4(rng.integers(0, 256, size=(256, 512), dtype=np.uint8), np.full((256, 16), 100, dtype=np.uint16), dev)
    x = torch.randn(20, 1024, device=dev)
    clean = linear(w, x)
    x[5, 17], x[9, 1000] = float("inf"), float("nan")
    y = linear(w, x)
    keep = [i for i in range(20) if i not in (5, 9)]
    assert torch.equal(y[keep], clean[keep])
    assert not torch.isfinite(y[5]).any() and not torch.isfinite(y[9]).any()


def test_linear_group_rows_equal_single_calls(dev):
    """q4d_linear_group at 4 rows and more: each output equals its own q4d_linear call."""
    from llm_accelerator_amd.model import current_stream
    rng = np.random.default_rng(4)
    ws = [q4(rng.integers(0, 256, size=(130, 512), dtype=np.uint8),
             rng.integers(1, 3000, size=(130, 16)).astype(np.uint16), dev) for _ in range(3)]
    xs = [torch.randn(18, 1024, device=dev) for _ in ws]
    ys = [torch.full((18, 130), float("nan"), device=dev) for _ in ws]
    descs = (_lib.Q4dMatrix * 3)(*[w.descriptor() for w in ws])
    xp, yp = ((ctypes.c_void_p * 3)(*[t.data_ptr() for t in ts]) for ts in (xs, ys))
    _lib.check(_lib.load().q4d_linear_group(descs, xp, Q4D_F32, yp, Q4D_F32, 18, 3, current_stream()),
               "q4d_linear_group")
    for w, x, y in zip(ws, xs, ys):
        assert torch.equal(y, linear(w, x))


@pytest.mark.parametrize("m,n,k,count,xdtype,ydtype,precision", [
    (16, 258, 1024, 70, torch.float32, Q4D_F32, 2),     # 64 + 6: four weight tiles per block, then one
    (4, 130, 1024, 70, torch.float32, Q4D_F32, 2),      # few outputs: the grouped GEMV
    (5, 1026, 3072, 64, torch.float32, Q4D_F16, 2),     # four weight tiles per block, the waves of one
    (20, 258, 3072, 2, torch.float32, Q4D_F32, 2),      # one tile, 12 waves
    (33, 3072, 3072, 3, torch.float32, Q4D_F32, 2),     # two weight tiles alone, two row tiles together
    (40, 512, 2048, 65, torch.float16, Q4D_F16, 1),     # 64 + 1: the last a launch of its own
    (17, 512, 3072, 66, torch.float32, Q4D_F32, 1),
    (64, 258, 1024, 30, torch.float16, Q4D_F32, 1),
    (70, 130, 2048, 64, torch.float32, Q4D_F32, 2),     # two row tiles, the general loop
])
def test_linear_group_rows_one_launch_and_bits(dev, m, n, k, count, xdtype, ydtype, precision):
    """q4d_linear_group over several rows: one launch per 64 matrices (the kernels a captured call
    records), and each output equals its own q4d_linear call bit for bit whatever tile the group takes."""
    from llm_accelerator_amd.model import current_stream
    lib = _lib.load()
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    mats = [Q4Tensor(torch.randint(0, 256, (n, k // 2), generator=g, device=dev, dtype=torch.uint8),
                     torch.randint(1, 3000, (n, k // 64), generator=g, device=dev).to(torch.int16).view(torch.uint16))
            for _ in range(count)]
    xs = [torch.randn(m, k, generator=g, device=dev).to(xdtype) for _ in range(count)]
    ydt = torch.float16 if ydtype == Q4D_F16 else torch.float32
    ys = [torch.full((m, n), float("nan"), device=dev, dtype=ydt) for _ in range(count)]
    descs = (_lib.Q4dMatrix * count)(*[w.descriptor() for w in mats])
    xp, yp = ((ctypes.c_void_p * count)(*[t.data_ptr() for t in ts]) for ts in (xs, ys))
    xcode = Q4D_F16 if xdtype == torch.float16 else Q4D_F32
    print(f"[linear group rows] {count} x {m} x {n} x {k}", flush=True)

    def call():
        _lib.check(lib.q4d_linear_group(descs, xp, xcode, yp, ydtype, m, count, current_stream()), "q4d_linear_group")

    _lib.check(lib.q4d_set_activation_precision(precision), "q4d_set_activation_precision")
    try:
        call()
        for w, x, y in zip(mats, xs, ys):
            assert torch.equal(y, linear(w, x, ydtype))
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph):
            call()
    finally:
        _lib.check(lib.q4d_set_activation_precision(2), "q4d_set_activation_precision")
    nodes = ctypes.c_size_t(0)
    lib.hipGraphGetNodes.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.POINTER(ctypes.c_size_t)]
    assert lib.hipGraphGetNodes(graph.raw_cuda_graph(), None, ctypes.byref(nodes)) == 0
    assert nodes.value == (count + 63) // 64


@pytest.mark.parametrize("m,n,k,top", [(1, 128, 1024, 1500), (33, 1024, 3072, 1500), (64, 384, 2048, 9000),
                                       (100, 3072, 1024, 4095), (500, 3072, 1024, 1500), (401, 1024, 3072, 1500),
                                       (64, 128, 1152, 65535), (700, 4096, 1024, 9000), (2000, 1024, 2048, 9000),
                                       (2000, 4096, 1024, 9000)])
def test_gemm_vs_fp16_operands(dev, m, n, k, top):
    """q4d_gemm against the product of the same fp16 operands (weights rounded once): the rows
    kernel's tile sizes and general K loop (1152 columns), the pipelined kernel (700 x 4096, 2000 x
    1024) and the 128-row tiles (2000 x 4096), with scale codes on both sides of the fast
    conversion's limit (4094)."""
    from llm_accelerator_amd.model import current_stream
    rng = np.random.default_rng(m + n + k)
    packed = rng.integers(0, 256, size=(n, k // 2), dtype=np.uint8)
    scale = rng.integers(1, top + 1, size=(n, k // 64)).astype(np.uint16)
    scale[0, :2] = min(top, 4094), top
    w = q4(packed, scale, dev)
    x = torch.from_numpy(rng.normal(size=(m, k)).astype(np.float16)).to(dev)
    resid = torch.from_numpy(rng.normal(size=(m, n)).astype(np.float32)).to(dev)
    y = torch.full((m, n), float("nan"), device=dev)
    desc = w.descriptor()
    _lib.check(_lib.load().q4d_gemm(ctypes.byref(desc), x.data_ptr(), m, y.data_ptr(), Q4D_F32, resid.data_ptr(),
                                    current_stream()), "q4d_gemm")
    q = o.unpack_signed_int4(packed, k).astype(np.float16)
    w16 = (q * np.repeat((scale / 16384.0).astype(np.float16), 64, axis=1)).astype(np.float64)
    x64 = x.double().cpu().numpy()
    assert np.isfinite(w16).all()
    bound = 2.0 ** -16 * (np.abs(x64) @ np.abs(w16).T) + 2.0 ** -22
    assert np.all(np.abs(y.double().cpu().numpy() - resid.double().cpu().numpy() - x64 @ w16.T) <= bound)
