"""FAST decode at the batch sizes and history lengths where its launches change form: the attention's splits by the
batch's own lengths (65 to 1024 sequences: equal, ragged, one long sequence among short ones, fresh sequences), the
plain grid above that, up to 48 splits of one or two long sequences, and the projections of 65 to 256 and more
tokens with the RoPE epilogue.  Against ORDERED on the same input, per tensor within 1e-3 of its maximum (the FAST
contract of the layer)."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-3


@pytest.fixture(scope="module")
def model():
    from work_llm_accelerator_amd.model import DeviceModel

    m = DeviceModel(1, synthetic_seed=41)
    yield m
    m.close()


def positions(kind: str, batch: int, longest: int) -> np.ndarray:
    rng = np.random.default_rng(batch)
    if kind == "equal":
        return np.full(batch, longest - 1)
    if kind == "one long":
        p = rng.integers(0, 12, batch)
        p[batch // 3] = longest - 1
        return p
    p = rng.integers(0, longest, batch)
    p[0], p[-1] = 0, longest - 1
    return p


@pytest.mark.parametrize("batch,longest,kind", [(65, 300, "equal"), (65, 1, "equal"), (66, 700, "ragged"),
                                                (150, 200, "ragged"), (150, 2000, "one long"), (257, 70, "ragged"),
                                                (700, 40, "ragged"), (1025, 20, "ragged"), (1, 3000, "equal"),
                                                (1, 1537, "equal"), (2, 5000, "ragged")])
def test_layer_against_ordered(model, batch, longest, kind):
    import torch

    from work_llm_accelerator_amd.model import FLAG_NO_BF16_ROUND, MODE_FAST, MODE_ORDERED, KvCache, fill_kv_synthetic

    print(f"decode {batch} sequences, {kind}, up to {longest} keys", flush=True)
    pos = torch.tensor(positions(kind, batch, longest), dtype=torch.int32, device="cuda")
    x = torch.randn(batch, 1536, generator=torch.Generator(device="cuda").manual_seed(batch), device="cuda")
    out = []
    for mode in (MODE_FAST, MODE_ORDERED):
        cache = KvCache.allocate(1, batch, longest + 1)
        fill_kv_synthetic(cache, 5)
        hidden = x.clone()
        torch.cuda.synchronize()
        model.decode(mode | FLAG_NO_BF16_ROUND, hidden, pos, longest, cache)
        model.synchronize()
        out.append((hidden, cache.k, cache.v))
    for g, r in zip(*out):
        assert float((g - r).abs().max() / r.abs().max()) <= TOL


def test_positions_outside_the_cache(model):
    """More than 64 sequences, some positions past max_keys or negative: those rows stay unwritten and attend over
    what the cache holds, as in ORDERED."""
    import torch

    from work_llm_accelerator_amd.model import FLAG_NO_BF16_ROUND, MODE_FAST, MODE_ORDERED, KvCache, fill_kv_synthetic

    batch, rows = 70, 40
    p = np.arange(batch) % rows
    p[3], p[40], p[69] = rows + 5, -2, rows
    pos = torch.tensor(p, dtype=torch.int32, device="cuda")
    x = torch.randn(batch, 1536, generator=torch.Generator(device="cuda").manual_seed(3), device="cuda")
    out = []
    for mode in (MODE_FAST, MODE_ORDERED):
        cache = KvCache.allocate(1, batch, rows)
        fill_kv_synthetic(cache, 6)
        hidden = x.clone()
        torch.cuda.synchronize()
        model.decode(mode | FLAG_NO_BF16_ROUND, hidden, pos, rows, cache)
        model.synchronize()
        out.append((hidden, cache.k, cache.v))
    for g, r in zip(*out):
        assert float((g - r).abs().max() / r.abs().max()) <= TOL
