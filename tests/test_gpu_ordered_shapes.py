"""ORDERED layers at the token counts where its projection kernels change form: chains of a few tokens,
matrix-core products at 1, 2, 4 and (gate/up) 8 tokens per wave, with remainders; key counts around the
attention's 64-key tiles; and row scales outside the range in which a weight is formed with one multiplication.
All bit for bit against the oracle (verification/real_host_top_backend.py runs the same layers on the host);
the forms of 8 and 16 tokens per wave, which long prompts take, against chunks of the same prompt."""

from __future__ import annotations

import numpy as np
import pytest

from _cases import (LayerCase, bits_equal, decode_layer, first_mismatch, quantized_kv_history, random_hidden,
                    random_layer)
from _oracle import oracle
from work_llm_accelerator_amd.layout import HIDDEN, KV_WIDTH

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def layer():
    """A random layer whose q, up and down rows include a negative, a zero, a denormal and a huge scale."""
    case = random_layer(seed=77)
    for name, row, value in (("q_s", 3, -0.01), ("q_s", 700, 0.0), ("up_s", 40, np.float32(1e-41)),
                             ("down_s", 9, np.float32(2.0 ** 122)), ("down_s", 1500, np.float32(-1e-41))):
        case.v[name][row] = value
    case.v["down_w"][9 * 4480:10 * 4480] = 0  # the huge row: three weights, so that its sum stays finite
    case.v["down_w"][9 * 4480 + 7] = 0x1F
    case.v["down_w"][9 * 4480 + 4001] = 0x01
    return case


def model_of(case: LayerCase):
    from work_llm_accelerator_amd.model import DeviceModel

    return DeviceModel(1, case.weight_ddr, case.scale_ddr)


@pytest.mark.parametrize("tokens", [1, 2, 5, 6, 9, 17, 33, 63, 65, 129, 260])
def test_prefill_tokens(layer, tokens):
    import torch

    from work_llm_accelerator_amd.model import FLAG_NO_BF16_ROUND, MODE_ORDERED, KvCache

    print(f"ordered prefill of {tokens} tokens", flush=True)
    x = random_hidden(900 + tokens, tokens)
    kc, vc = np.zeros(tokens * KV_WIDTH, np.float32), np.zeros(tokens * KV_WIDTH, np.float32)
    out = np.zeros(tokens * HIDDEN, np.float32)
    assert oracle().oracle_prefill_layer_uncapped(x, tokens, layer.weight_ddr, layer.scale_ddr, kc, vc, out) == 0
    model = model_of(layer)
    cache = KvCache.allocate(1, 1, tokens)
    hidden = torch.from_numpy(x.reshape(1, tokens, HIDDEN)).cuda()
    model.prefill(MODE_ORDERED | FLAG_NO_BF16_ROUND, hidden, cache)
    model.synchronize()
    for got, ref in ((hidden, out), (cache.k, kc), (cache.v, vc)):
        got = got.cpu().numpy().reshape(-1)
        assert bits_equal(got, ref), first_mismatch(got, ref)
    model.close()


@pytest.mark.parametrize("tokens", [715, 2003])
def test_prefill_in_chunks(layer, tokens):
    """715 tokens: 8 a wave for q/k/v, 16 for gate/up; 2003: 16 for every projection.  In chunks of 128 all
    run at 4 (each chunk's last tokens at fewer), which the oracle is compared with above."""
    import torch

    from work_llm_accelerator_amd.model import FLAG_NO_BF16_ROUND, MODE_ORDERED, KvCache

    print(f"ordered prefill of {tokens} tokens, whole and in chunks", flush=True)
    x = torch.from_numpy(random_hidden(920 + tokens, tokens).reshape(1, tokens, HIDDEN)).cuda()
    model = model_of(layer)
    whole, parts = KvCache.allocate(1, 1, tokens), KvCache.allocate(1, 1, tokens)
    out = x.clone()
    model.prefill(MODE_ORDERED | FLAG_NO_BF16_ROUND, out, whole)
    model.synchronize()
    for past in range(0, tokens, 128):
        chunk = x[:, past:past + 128].clone()
        model.prefill(MODE_ORDERED | FLAG_NO_BF16_ROUND, chunk, parts, past=past)
        model.synchronize()
        got, ref = out[0, past:past + 128].cpu().numpy().reshape(-1), chunk.cpu().numpy().reshape(-1)
        assert bits_equal(got, ref), (past, first_mismatch(got, ref))
    for got, ref in ((whole.k, parts.k), (whole.v, parts.v)):
        got, ref = got.cpu().numpy().reshape(-1), ref.cpu().numpy().reshape(-1)
        assert bits_equal(got, ref), first_mismatch(got, ref)
    model.close()


@pytest.mark.parametrize("batch,longest", [(1, 62), (1, 63), (1, 64), (1, 300), (2, 65), (4, 130), (5, 64), (6, 20),
                                           (9, 70), (33, 12), (65, 5)])
def test_decode_batch(layer, batch, longest):
    import torch

    from work_llm_accelerator_amd.model import FLAG_NO_BF16_ROUND, MODE_ORDERED, KvCache

    print(f"ordered decode of {batch} sequences, up to {longest} keys", flush=True)
    past = [longest - (i * 7) % (longest // 2 + 1) for i in range(batch)]
    rows = longest + 3
    x = random_hidden(950 + batch, batch)
    k, v = quantized_kv_history(960 + batch, batch * rows)
    model = model_of(layer)
    cache = KvCache.allocate(1, batch, rows)
    cache.k.copy_(torch.from_numpy(k.reshape(1, batch, rows, KV_WIDTH)))
    cache.v.copy_(torch.from_numpy(v.reshape(1, batch, rows, KV_WIDTH)))
    hidden = torch.from_numpy(x.reshape(batch, HIDDEN)).cuda()
    pos = torch.tensor(past, dtype=torch.int32, device="cuda")
    model.decode(MODE_ORDERED | FLAG_NO_BF16_ROUND, hidden, pos, longest + 1, cache)
    model.synchronize()
    got, gk, gv = hidden.cpu().numpy(), cache.k.cpu().numpy()[0], cache.v.cpu().numpy()[0]
    for b, p in enumerate(past):
        kc, vc = k.reshape(batch, -1)[b].copy(), v.reshape(batch, -1)[b].copy()
        st, out = decode_layer(oracle().oracle_decode_layer_smoke_forward, layer, x[b * HIDDEN:(b + 1) * HIDDEN].copy(),
                               p, kc, vc)
        assert st == 0
        for g, r in ((got[b], out), (gk[b].reshape(-1), kc), (gv[b].reshape(-1), vc)):
            assert bits_equal(g, r), (b, p, first_mismatch(g, r))
    model.close()
