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
from llm_accelerator_amd.model import current_stream

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
