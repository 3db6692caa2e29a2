"""FAST prefill at the token counts where its launches change form: the K splits of the O and down projections,
one or two heads per Q/K/V block, the skinny kernels' 64 tokens with several sequences in a tile, and the attention's key splits (a query tile's keys over several blocks,
splits past a query's last key, a single query tile behind a long history).  Every size against ORDERED on the
same input, per tensor within 1e-3 of its maximum (the FAST contract of the layer)."""

from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-3


@pytest.fixture(scope="module")
def model():
    from work_llm_accelerator_amd.model import DeviceModel

    m = DeviceModel(2, synthetic_seed=31)
    yield m
    m.close()


def run(model, mode, x, batch, seq, past, seed, layers):
    import torch

    from work_llm_accelerator_amd.model import FLAG_NO_BF16_ROUND, KvCache, fill_kv_synthetic

    cache = KvCache.allocate(layers[1], batch, past + seq)
    fill_kv_synthetic(cache, seed)
    hidden = x.clone()
    torch.cuda.synchronize()
    model.prefill(mode | FLAG_NO_BF16_ROUND, hidden, cache, past=past, layers=layers)
    model.synchronize()
    return hidden, cache.k, cache.v


@pytest.mark.parametrize("batch,seq,past", [(1, 65, 0), (1, 130, 0), (3, 90, 0), (1, 257, 0), (1, 400, 0), (2, 400, 33),
                                            (1, 1025, 0), (1, 5, 3000), (1, 16, 700), (1, 33, 2047), (2, 70, 1500),
                                            (1, 1, 0), (1, 17, 0), (3, 21, 5), (64, 1, 7), (1, 64, 0),
                                            (1, 2100, 0), (2, 1500, 0), (3, 1661, 0)])
def test_layer_against_ordered(model, batch, seq, past):
    import torch

    from work_llm_accelerator_amd.model import MODE_FAST, MODE_ORDERED

    print(f"prefill {batch} x {seq} after {past}", flush=True)
    x = torch.randn(batch, seq, 1536, generator=torch.Generator(device="cuda").manual_seed(seq), device="cuda")
    got = run(model, MODE_FAST, x, batch, seq, past, 7, (0, 1))
    ref = run(model, MODE_ORDERED, x, batch, seq, past, 7, (0, 1))
    for g, r in zip(got, ref):
        assert float((g - r).abs().max() / r.abs().max()) <= TOL


@pytest.mark.parametrize("seq", [100, 513])
def test_two_layers_as_one_call(model, seq):
    """The layer boundary inside the down projection's reduce step against two one-layer calls, whose boundary is
    a launch of its own: the sum of squares of the RMSNorm is taken in another fp32 order, so the next layer's
    15-bit codes may differ by a step here and there."""
    import torch

    from work_llm_accelerator_amd.model import MODE_FAST

    x = torch.randn(1, seq, 1536, generator=torch.Generator(device="cuda").manual_seed(seq), device="cuda")
    both, k, v = run(model, MODE_FAST, x, 1, seq, 0, 9, (0, 2))
    first, k0, v0 = run(model, MODE_FAST, x, 1, seq, 0, 9, (0, 1))
    assert torch.equal(k[0], k0[0]) and torch.equal(v[0], v0[0])
    second, k1, v1 = run(model, MODE_FAST, first, 1, seq, 0, 9, (1, 1))
    for g, r in ((both, second), (k[1], k1[0]), (v[1], v1[0])):
        assert float((g - r).abs().max() / r.abs().max()) <= TOL
