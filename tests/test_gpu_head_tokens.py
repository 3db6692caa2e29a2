"""The multi-token lm_head at its token tiles' edges (one, two and three tiles per pass, several passes) and at
vocabularies of fewer rows than the launch has waves, against the oracle as tests/test_gpu_head.py does."""

from __future__ import annotations

import numpy as np
import pytest

from test_gpu_head import bf16_bits_np, check_head, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [16, 17, 32, 48, 49, 97])
@pytest.mark.parametrize("vocab", [128, 4224])
def test_head_tokens(torch, count, vocab):  # noqa: F811
    from work_llm_accelerator_amd.model import DeviceModel

    rng = np.random.default_rng(vocab + count)
    table = bf16_bits_np(rng.standard_normal((vocab, 1536)).astype(np.float32) * 0.02)
    norm = bf16_bits_np(1.0 + 0.1 * rng.standard_normal(1536).astype(np.float32))
    m = DeviceModel(1, synthetic_seed=2)
    m.set_head(table, norm)
    check_head(torch, m, vocab, table, norm, count, 50 + count)
    m.close()
