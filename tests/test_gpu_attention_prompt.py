"""Causal attention over prompts on the GPU: several sequences per call, partial query and key
tiles, head counts that do and do not split over the XCDs, and extreme scores."""

import numpy as np
import pytest
import torch

from llm_accelerator_amd import _lib, common
from llm_accelerator_amd.model import current_stream

pytestmark = pytest.mark.gpu


def reference(q, k, v, repeat, scaling):
    """float64 on the fp16-rounded operands the kernel uses (q with scaling * log2 e folded in)."""
    b, h, s, d = q.shape
    qh = (q * np.float32(scaling * 1.4426950408889634)).half().double()
    kh, vh = k.half().double(), v.half().double()
    out, size = torch.empty_like(qh), torch.empty_like(qh)
    mask = torch.triu(torch.ones(s, s, dtype=torch.bool, device=q.device), 1)
    for i in range(b):
        for j in range(h):
            t = (qh[i, j] @ kh[i, j // repeat].t().contiguous()).masked_fill(mask, float("-inf"))
            p = torch.softmax(t * np.log(2.0), dim=-1)
            out[i, j], size[i, j] = p @ vh[i, j // repeat], p @ vh[i, j // repeat].abs()
    return out, size


@pytest.mark.parametrize("b,h,kvh,s", [(1, 16, 8, 1), (3, 16, 8, 31), (2, 16, 8, 33), (1, 16, 8, 64), (5, 4, 1, 65),
                                       (2, 16, 8, 97), (1, 3, 3, 200), (2, 8, 8, 640), (1, 32, 8, 1025)])
def test_prompt_attention_vs_fp64(dev, b, h, kvh, s):
    g = torch.Generator(dev).manual_seed(b * 1000 + s)
    q, k, v = (torch.randn(b, n, s, 128, device=dev, generator=g) for n in (h, kvh, kvh))
    q[:, 0] *= 30        # a head with one-hot rows: the running maximum moves by hundreds
    k[:, :, 0] *= 8      # key 0, the only one every query sees
    scaling = 128 ** -0.5
    print(f"[prompt attention] {b} x {h}/{kvh} heads x {s}", flush=True)
    out, _ = common.manual_causal_attention(q, common.manual_repeat_kv(k, h // kvh),
                                            common.manual_repeat_kv(v, h // kvh), scaling)
    ref, size = reference(q, k, v, h // kvh, scaling)
    # probabilities rounded to fp16 against a maximum up to 2^8 below theirs (2^-11 each),
    # fp32 scores (exponent error 2^-22 of |score| <= 2^12, times ln 2)
    assert torch.all((out.double() - ref).abs() <= 2.0 ** -9 * size + 1e-6)


@pytest.mark.parametrize("b,h,kvh,s", [(1, 16, 8, 1), (3, 16, 8, 67), (2, 5, 1, 130)])
def test_prompt_attention_stays_in_its_workspace(dev, b, h, kvh, s):
    """A workspace of exactly the stated bytes between two guards: the guards stay, and the output is
    that of a call with room to spare."""
    lib = _lib.load()
    q, k, v = (torch.randn(b, n, s, 128, device=dev) for n in (h, kvh, kvh))
    need = int(lib.q4d_causal_attention_workspace_bytes(b, h, kvh, s))
    outs = []
    for nbytes in (need, 4 * need + 4096):
        ws = torch.full((256 + nbytes + 4096,), 0x5A, dtype=torch.uint8, device=dev)
        out = torch.full_like(q, float("nan"))
        _lib.check(lib.q4d_causal_attention(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), b, h, kvh, s, 128,
                                            0.09, ws.data_ptr() + 256, nbytes, current_stream()), "q4d_causal_attention")
        outs.append(out)
        assert bool((ws[:256] == 0x5A).all()) and bool((ws[256 + need:] == 0x5A).all())
    assert torch.equal(*outs) and bool(torch.isfinite(outs[0]).all())


def test_prompt_attention_sequences_are_independent(dev):
    q, k, v = (torch.randn(4, n, 130, 128, device=dev) for n in (16, 8, 8))
    both = common.manual_causal_attention(q, common.manual_repeat_kv(k, 2), common.manual_repeat_kv(v, 2), 0.09)[0]
    for i in range(4):
        one = common.manual_causal_attention(q[i:i + 1], common.manual_repeat_kv(k[i:i + 1], 2),
                                             common.manual_repeat_kv(v[i:i + 1], 2), 0.09)[0]
        assert torch.equal(both[i:i + 1], one)
