"""Cached attention past 512 positions: a batch's sequences cut into parts from their own positions
(parts of one sub-chunk, the largest number of parts, more sequences than lanes, positions out of
range), with and without a merge."""

import ctypes

import numpy as np
import pytest
import torch

from llm_accelerator_amd import _lib
from llm_accelerator_amd._lib import Q4dModel, check
from llm_accelerator_amd.model import KVCache, Qwen3Config, current_stream

pytestmark = pytest.mark.gpu

CASES = [  # lengths, capacity, kv heads
    ([1], 576, 8), ([576], 576, 8), ([1025], 2048, 8), ([8192], 8192, 8), ([64, 8191], 8192, 8),
    ([1, 65, 640, 641, 1500, 0, 2048, 4000], 2048, 8),          # two positions out of range
    ([700 - 11 * (i % 63) for i in range(63)], 704, 8),         # all lanes but one a sequence
    ([1 + (53 * i) % 704 for i in range(64)], 704, 4),          # every lane a sequence
    ([1 + (37 * i) % 640 for i in range(100)], 640, 4),         # two groups of lanes
    ([576 - 8 * (i % 72) for i in range(64)] + [-3], 576, 8),   # one part each, a position out of range
    ([101] * 24, 640, 8), ([191, 192, 193, 256, 320, 321, 384, 385], 1024, 8),  # too short to cut, and just not
    ([1024] * 12, 1024, 8), ([700] * 16, 1024, 8), ([513] * 17, 576, 8),  # equal batches, two parts and one
    ([4000] + [200 + i for i in range(31)], 4096, 8),           # one long sequence beside short ones
    ([2624 - i for i in range(36)], 2624, 8),                   # past one block per CU, long enough for two parts
    ([2600 - 40 * i for i in range(63)], 2624, 8),              # the same, ragged
    ([640 - 5 * i for i in range(126)] + [641], 640, 4),        # two groups of lanes with extra parts
]


@pytest.mark.parametrize("lengths,cap,kvh", CASES, ids=lambda v: f"{len(v)}" if isinstance(v, list) else str(v))
def test_span_attention_vs_fp64(dev, lengths, cap, kvh):
    lib = _lib.load()
    B = len(lengths)
    g = torch.Generator(device=dev).manual_seed(sum(lengths) + cap)
    kv = KVCache(Qwen3Config(num_attention_heads=2 * kvh, num_key_value_heads=kvh), 1, B, cap, dev)
    kv.data.normal_(generator=g)
    q = torch.randn(B, 2 * kvh, 128, generator=g, device=dev)
    m = Q4dModel(hidden_size=1024, intermediate_size=3072, num_layers=1, num_q_heads=2 * kvh, num_kv_heads=kvh,
                 head_dim=128, vocab_size=2, max_ctx=cap, rms_norm_eps=1e-6, attn_scaling=128 ** -0.5)
    nbytes = int(lib.q4d_workspace_bytes(ctypes.byref(m), B))
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    pos = torch.tensor([n - 1 for n in lengths], dtype=torch.int32, device=dev)
    out = torch.full((B, 2 * kvh, 128), 7.0, device=dev)
    kvd = kv.descriptor()
    first = None
    for _ in range(2):  # the second call finds the counters as the first left them
        check(lib.q4d_cached_attention(ctypes.byref(m), ctypes.byref(kvd), 0, q.data_ptr(), pos.data_ptr(),
                                       out.data_ptr(), _lib.Q4D_F32, ws.data_ptr(), nbytes, current_stream()),
              "q4d_cached_attention")
        first = out.clone() if first is None else first
    assert torch.equal(first, out)
    for b, n in enumerate(lengths):
        if not 0 < n <= cap:
            assert bool((out[b] == 7.0).all())
            continue
        k, v = (kv.data[0, i, b, :, :n].double().repeat_interleave(2, 0) for i in range(2))
        p = torch.softmax((k * q[b].double()[:, None]).sum(-1) * 128 ** -0.5, -1)
        ref, size = (p[..., None] * v).sum(1), (p[..., None] * v.abs()).sum(1)
        # fp32 dots of 128, exponents and sums over the positions, relative to the absolute sum
        np.testing.assert_array_less((out[b].double() - ref).abs().cpu().numpy(), (2.0 ** -16 * size + 1e-7).cpu().numpy())
    status = ws[:4].view(torch.int32).item()
    assert status == (_lib.STATUS_BAD_POSITION if any(not 0 < n <= cap for n in lengths) else 0)


@pytest.mark.parametrize("lengths,cap,whole", [
    ([101] * 24, 640, True), ([150] * 8, 8192, True), ([192, 64, 1], 1024, True),  # a split would save too little
    ([1024] * 24, 1024, True), ([700] * 20, 2048, True), ([600] * 63, 1024, True),  # about one block per CU already
    ([1024] * 8, 1024, False), ([8192], 8192, False), ([4000] + [200] * 15, 4096, False), ([640] * 4, 640, False),
])
def test_span_attention_splits_where_it_pays(dev, lengths, cap, whole):
    """Whether any sequence is cut into parts, read from the workspace: a cut leaves its partials there,
    whole sequences write nothing but their output."""
    lib = _lib.load()
    B = len(lengths)
    kv = KVCache(Qwen3Config(), 1, B, cap, dev)
    kv.data.normal_()
    q = torch.randn(B, 16, 128, device=dev)
    m = Q4dModel(hidden_size=1024, intermediate_size=3072, num_layers=1, num_q_heads=16, num_kv_heads=8,
                 head_dim=128, vocab_size=2, max_ctx=cap, rms_norm_eps=1e-6, attn_scaling=128 ** -0.5)
    nbytes = int(lib.q4d_workspace_bytes(ctypes.byref(m), B))
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    pos = torch.tensor([n - 1 for n in lengths], dtype=torch.int32, device=dev)
    out = torch.empty(B, 16, 128, device=dev)
    kvd = kv.descriptor()
    check(lib.q4d_cached_attention(ctypes.byref(m), ctypes.byref(kvd), 0, q.data_ptr(), pos.data_ptr(), out.data_ptr(),
                                   _lib.Q4D_F32, ws.data_ptr(), nbytes, current_stream()), "q4d_cached_attention")
    assert bool((ws != 0).any()) == (not whole)
