"""The K splits of the pipelined FAST projections add up exactly, on rows far from zero mean.

A split's partial used to be an fp32 value that still held the zero point 8 sum(X) of the stored weights
u = q + 8, so its rounding was relative to that term, not to the result; rows of one sign make the term up to
thousands of times the result.  Here every activation is positive (20000 .. 32512, the largest 32512, so the
token scale is 1 and the code is the input itself) and the row scales are powers of two, so an output is the
integer sum_k q X rounded to fp32 once, and is compared bit for bit with numpy's.

* the projection by itself, for the shapes whose K is split over blocks and for some whose K is not;
* the O projection inside the layer, whose reduce step is fused with the RMSNorm and the quantization (one
  token per sequence at position 0: the context row is the V row, the bias alone with zero weights);
* the down projection inside the layer: a constant normalized row makes the SiLU.up row a multiple of chosen
  integers, and the outputs are those integers' sums times one unknown token scale.
"""

from __future__ import annotations

import numpy as np
import pytest

from _fastcode import QMAX, unpack_int4

pytestmark = pytest.mark.gpu


def pack(q: np.ndarray) -> np.ndarray:
    nib = (q.reshape(-1, 2) & 0xF).astype(np.uint8)
    return nib[:, 0] | (nib[:, 1] << 4)


def one_sign(rng, shape) -> np.ndarray:
    x = rng.integers(20000, QMAX + 1, shape).astype(np.float64)
    x[..., 7] = QMAX
    return x


SHAPES = [(40, 1536, 1040), (65, 1536, 1536), (150, 1536, 2048), (150, 8960, 1536), (300, 8960, 1536),
          (600, 8960, 1536), (700, 1536, 1536), (1030, 1536, 1536), (1030, 8960, 1536), (1200, 8960, 1536),
          (1700, 8960, 1536), (2050, 8960, 1536)]


@pytest.mark.parametrize("tokens,in_dim,out_dim", SHAPES)
def test_projection(tokens, in_dim, out_dim):
    import ctypes

    import torch

    from work_llm_accelerator_amd import abi

    print(f"projection of rows of one sign: {tokens} x {in_dim} -> {out_dim}", flush=True)
    rng = np.random.default_rng(tokens + in_dim)
    packed = rng.integers(0, 256, out_dim * in_dim // 2, dtype=np.uint8)
    packed[:in_dim // 2], packed[in_dim // 2:in_dim] = 0x77, 0x88  # rows of the largest and smallest weights
    q = unpack_int4(packed, out_dim, in_dim).astype(np.float64)
    x = one_sign(rng, (tokens, in_dim))
    x[0], x[1] = QMAX, -QMAX  # with those rows the largest sums there are
    want = (x @ q.T).astype(np.float32)  # exact in float64, one rounding
    dev = [torch.from_numpy(a).cuda() for a in (packed, np.ones(out_dim, np.float32), x.astype(np.float32))]
    y = torch.empty((tokens, out_dim), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    w, sw, xd, yd = (ctypes.c_void_p(t.data_ptr()) for t in (*dev, y))
    lib = abi.load()
    assert lib.qwen_hip_fast_project(w, sw, None, out_dim, in_dim, xd, tokens, 0, yd, None) == 0, abi.last_error(lib)
    assert np.array_equal(y.cpu().numpy().view(np.uint32), want.view(np.uint32))


def layer_output(case, kind: str, tokens: int) -> np.ndarray:
    """Hidden rows of `tokens` sequences whose only token is at position 0, through one layer."""
    import torch

    from work_llm_accelerator_amd.model import FLAG_NO_BF16_ROUND, MODE_FAST, DeviceModel, KvCache

    print(f"{kind}: {tokens} sequences of one token", flush=True)
    model = DeviceModel(1, case.weight_ddr, case.scale_ddr)
    cache = KvCache.allocate(1, tokens, 1)
    hidden = torch.ones(tokens, 1, 1536, device="cuda")
    if kind == "prefill":
        model.prefill(MODE_FAST | FLAG_NO_BF16_ROUND, hidden, cache)
    else:
        hidden = hidden[:, 0]
        pos = torch.zeros(tokens, dtype=torch.int32, device="cuda")
        model.decode(MODE_FAST | FLAG_NO_BF16_ROUND, hidden, pos, 1, cache)
    model.synchronize()
    out = hidden.reshape(tokens, 1536).cpu().numpy()
    model.close()
    return out


LAYERS = [("prefill", 47), ("prefill", 65), ("prefill", 200), ("prefill", 257), ("prefill", 512), ("prefill", 600),
          ("prefill", 1000), ("prefill", 1030), ("prefill", 1200), ("prefill", 1700), ("decode", 65),
          ("decode", 150), ("decode", 300)]


@pytest.mark.parametrize("kind,tokens", [("prefill", 1), ("prefill", 16), *LAYERS])
def test_o_projection(kind, tokens):
    from _cases import empty_layer

    rng = np.random.default_rng(tokens)
    case = empty_layer()
    case.v["v_bias"][:] = one_sign(rng, 256)
    case.v["o_w"][:] = rng.integers(0, 256, 1536 * 1536 // 2, dtype=np.uint8)
    context = np.repeat(case.v["v_bias"].reshape(2, 128), 6, axis=0).reshape(-1).astype(np.float64)
    want = (unpack_int4(case.v["o_w"], 1536, 1536).astype(np.float64) @ context).astype(np.float32)
    got = layer_output(case, kind, tokens)
    assert np.array_equal(got.view(np.uint32), np.broadcast_to(want.view(np.uint32), got.shape))


@pytest.mark.parametrize("kind,tokens", LAYERS[1:])
def test_down_projection(kind, tokens):
    from _cases import empty_layer

    rng = np.random.default_rng(tokens)
    case = empty_layer()
    # attention output 1 in every column: V's column 0 of each head, one weight a row
    case.v["v_bias"][0] = 1.0
    o = np.zeros((1536, 1536), np.int64)
    o[:, 0] = 1
    case.v["o_w"][:] = pack(o)
    # gate 48 in every row (its SiLU is the row itself); up in proportion to n, whose code is 4 n exactly
    case.v["gate_w"][:] = pack(np.ones((8960, 1536), np.int64))
    case.v["gate_s"][:] = 1.0 / 32.0
    n = rng.integers(4064, 8129, 8960)
    n[5] = QMAX // 4
    up = n[:, None] // 1536 + (np.arange(1536)[None, :] < (n % 1536)[:, None])
    case.v["up_w"][:] = pack(up)
    case.v["up_s"][:] = 2.0**-10
    q = rng.integers(-7, 8, (1536, 8960))
    q[0] = 1  # the row that tells the token scale
    case.v["down_w"][:] = pack(q)
    sums = q.astype(np.float64) @ (4.0 * n)
    got = layer_output(case, kind, tokens).astype(np.float64)
    scale = (got[:, :1] - 1.0) / sums[0]
    want = 1.0 + sums[None, :] * scale
    # the sum's rounding, the scale's product and the residual's addition, of the row itself and of row 0
    bound = 2.0**-24 * (6.0 * np.abs(sums[None, :] * scale) + 2.0)
    assert np.all(np.abs(got - want) <= bound), float((np.abs(got - want) / bound).max())
