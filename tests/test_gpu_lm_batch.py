"""The resident batched LM head (at most 64 rows) on the GPU: every activation-tile count, table
sizes that leave waves without work, wide scale codes, ties, with and without logits."""

import ctypes

import numpy as np
import pytest
import torch

import oracle as o
from gpu_helpers import head_model, q4
from llm_accelerator_amd import _lib
from llm_accelerator_amd._lib import check
from llm_accelerator_amd.model import Q4Tensor, current_stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,vocab,top,logits", [(1, 128, 1500, True), (16, 4224, 1500, True), (17, 40064, 9000, True),
                                                    (33, 1024, 1500, False), (64, 33024, 4095, True), (65, 1024, 1500, True)])
def test_lm_head_batch_vs_fp16_operands(dev, batch, vocab, top, logits):
    """Logits against the product of the same fp16 operands, the argmax against the returned
    logits (two planted copies of a winning row: the lower index wins); 65 rows take the tiled
    kernel."""
    rng = np.random.default_rng(batch + vocab)
    packed = rng.integers(0, 256, size=(vocab, 512), dtype=np.uint8)
    scale = rng.integers(1, top + 1, size=(vocab, 16)).astype(np.uint16)
    packed[vocab - 1] = packed[vocab // 2]
    scale[vocab - 1] = scale[vocab // 2]
    table = q4(packed, scale, dev)
    hidden = torch.from_numpy((rng.normal(size=(batch, 1024)) * 3).astype(np.float32)).to(dev)
    gamma = torch.from_numpy((1 + 0.1 * rng.normal(size=1024)).astype(np.float32)).to(dev)
    m = head_model(table, gamma)
    lib = _lib.load()
    nbytes = int(lib.q4d_workspace_bytes(ctypes.byref(m), batch))
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    tok = torch.full((batch,), -1, dtype=torch.int32, device=dev)
    score = torch.zeros(batch, device=dev)
    out = torch.full((batch, vocab), float("nan"), device=dev)
    check(lib.q4d_lm_head_argmax_batch(ctypes.byref(m), hidden.data_ptr(), batch, tok.data_ptr(), score.data_ptr(),
                                       out.data_ptr() if logits else None, ws.data_ptr(), nbytes, current_stream()),
          "q4d_lm_head_argmax_batch")
    h = hidden.double().cpu().numpy()
    xn = h / np.sqrt((h * h).mean(axis=1, keepdims=True) + 1e-6) * gamma.double().cpu().numpy()
    w16 = (o.unpack_signed_int4(packed, 1024).astype(np.float16) *
           np.repeat((scale / 16384.0).astype(np.float16), 64, axis=1)).astype(np.float64)
    ref, size = xn @ w16.T, np.abs(xn) @ np.abs(w16).T
    tok, score = tok.cpu().numpy(), score.double().cpu().numpy()
    # activations rounded to fp16 once (2^-11 each), fp32 sums (2^-16 of the absolute sum)
    bound = (2.0 ** -11 + 2.0 ** -16) * size + 1e-6
    if logits:
        y = out.double().cpu().numpy()
        assert np.all(np.abs(y - ref) <= bound)
        assert np.array_equal(tok, y.argmax(axis=1)) and np.array_equal(score, y.max(axis=1))
    rows = np.arange(batch)
    assert np.all(tok < vocab - 1) and np.all(np.abs(score - ref[rows, tok]) <= bound[rows, tok])
    assert np.all(score >= ref.max(axis=1) - bound.max(axis=1))


@pytest.mark.parametrize("batch", [1, 16, 24, 48, 64])
def test_lm_head_batch_every_wave_loops(dev, batch):
    """The real vocabulary, where every wave of each instance takes several table tiles: scale codes past
    the fast conversion's limit (4094) only from a wave's second tile on, and for each row a winner with an
    equal copy in its wave's next tile, in its last one, in a neighbouring wave's or anywhere after it."""
    vocab, tiles = 151936, 151936 // 16
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    stride = cus * {1: 8, 2: 16, 3: 12, 4: 8}[(batch + 15) // 16]  # tiles from one of a wave's to its next
    assert tiles > 2 * stride
    rng = np.random.default_rng(batch)
    g = torch.Generator(device=dev).manual_seed(batch)
    packed = torch.randint(0, 256, (vocab, 512), generator=g, device=dev, dtype=torch.uint8)
    scale = torch.randint(1, 1501, (vocab, 16), generator=g, device=dev)
    late = 16 * stride + torch.randperm(vocab - 16 * stride, generator=g, device=dev)[:2000]
    scale[late, torch.randint(0, 16, (2000,), generator=g, device=dev)] = 9000
    hidden = 3 * torch.randn(batch, 1024, generator=g, device=dev)
    gamma = 1 + 0.1 * torch.randn(1024, generator=g, device=dev)
    h = hidden.double()
    xn = h / torch.sqrt((h * h).mean(-1, keepdim=True) + 1e-6) * gamma.double()
    winners, taken = [], set()
    for b in range(batch):
        while True:
            first = int(rng.integers(0, vocab))
            last = first + 16 * stride * ((vocab - 1 - first) // (16 * stride))
            copy = (first + 16 * stride, last, first + 16, int(rng.integers(first, vocab)))[b % 4]
            if first < copy < vocab and not {first, copy} & taken:
                break
        taken |= {first, copy}
        winners.append(first)
        code = 9000 if first >= 16 * stride else 4000
        q = np.where(xn[b].cpu().numpy() >= 0, 7, -8)
        for r in (first, copy):
            packed[r] = torch.from_numpy(o.pack_signed_int4(q[None])[0]).to(dev)
            scale[r] = code
    table = Q4Tensor(packed, scale.to(torch.int16).view(torch.uint16))
    m = head_model(table, gamma)
    lib = _lib.load()
    nbytes = int(lib.q4d_workspace_bytes(ctypes.byref(m), batch))
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    tok = torch.full((batch,), -1, dtype=torch.int32, device=dev)
    score = torch.zeros(batch, device=dev)
    out = torch.full((batch, vocab), float("nan"), device=dev)
    print(f"[lm head loops] {batch} rows, {tiles} tiles, {stride} waves", flush=True)
    check(lib.q4d_lm_head_argmax_batch(ctypes.byref(m), hidden.data_ptr(), batch, tok.data_ptr(), score.data_ptr(),
                                       out.data_ptr(), ws.data_ptr(), nbytes, current_stream()), "q4d_lm_head_argmax_batch")
    assert tok.tolist() == winners
    assert torch.equal(score, out[torch.arange(batch, device=dev), tok.long()])
    for r0 in range(0, vocab, 16384):  # the same bound as above, against the fp16 weights
        p, s = packed[r0:r0 + 16384], scale[r0:r0 + 16384]
        q = torch.stack([p & 15, p >> 4], -1).reshape(len(p), -1).to(torch.int16)
        w16 = (torch.where(q >= 8, q - 16, q).half() * (s / 16384).half().repeat_interleave(64, 1)).double()
        ref = xn @ w16.t().contiguous()
        bound = (2.0 ** -11 + 2.0 ** -16) * (xn.abs() @ w16.abs().t().contiguous()) + 1e-6
        assert bool(((out[:, r0:r0 + 16384].double() - ref).abs() <= bound).all()), r0
