"""Short prefills (the GEMMs of q4d_chain.hip) on the GPU: the same bits as the tiled kernels
of longer ones, at the edges of the token tiles and of the switch between the two."""

import numpy as np
import pytest
import torch

from llm_accelerator_amd.decode import Prefill
from llm_accelerator_amd.model import KVCache, Qwen3Config, build_model, random_host_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["usual scales", "wide scales"])
def model(dev, request):
    cfg = Qwen3Config(num_hidden_layers=2, vocab_size=4096)
    host = random_host_weights(cfg, seed=21)
    if request.param == "wide scales":  # codes past the fast conversion's limit in some groups
        for L in host["layers"]:
            for name in ("q_proj", "o_proj", "up_proj", "down_proj"):
                L[name][1][5::64, 3::7] = 4095 + L[name][1][5::64, 3::7]
    return build_model(cfg, host, 1024, dev)


@pytest.fixture(scope="module")
def whole(model, dev):
    """One call over 800 tokens (tiled kernels throughout)."""
    tokens = torch.randint(0, 4096, (800,), dtype=torch.int32, device=dev, generator=torch.Generator(dev).manual_seed(3))
    kv = KVCache(model.config, 2, 1, 1024, dev)
    Prefill(model, kv, 800).run(tokens)
    return tokens, kv.data[:, :, 0, :, :800].clone()


@pytest.mark.parametrize("cuts", [[1, 16, 17, 33], [64, 65], [250, 257], [500, 513], [3, 515, 600]])
def test_short_chunks_equal_one_call(model, whole, dev, cuts):
    """Chunk lengths 1 .. 512: one, two and four 16-token tiles per block, partial tiles, and
    both sides of each kernel's limit; every K/V row equals the one call's bit for bit."""
    tokens, ref = whole
    kv = KVCache(model.config, 2, 1, 1024, dev)
    run = Prefill(model, kv, 800)
    bounds = [0] + cuts + [800]
    for a, b in zip(bounds, bounds[1:]):
        print(f"[prefill short] tokens {a}..{b}", flush=True)
        run.run(tokens[a:b].contiguous(), start_pos=a)
    assert torch.equal(kv.data[:, :, 0, :, :800].view(torch.int16), ref.view(torch.int16))
    assert not np.any(kv.data[:, :, 0, :, 800:].cpu().numpy())
