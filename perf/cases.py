"""The work that a user of this library has it do, as cases that a timing program can run.

listed() names the cases, draw() makes more of the same ranges.  A case is one call sequence of the
public Python / C entry points: a decode or prefill step of a DeviceModel (either mode), a whole
generation step (embedding, layers, head), or a call of the drop-in C ABI on host buffers.

Sizes are those of the repository's benchmark and tests (64 x 4096 decode, 8 x 2048 prefill, a
512-token prompt and batch-1 generation after it, the 128-token prefill and one-layer decode of the
drop-in ABI) and of what lies between and around them (ragged batches, a short odd prompt, a chunk of a
long prompt, a long history).  Layer stacks are cut to a few layers: the random-weight model amplifies
rounding from layer to layer, so a result after many layers says nothing about a kernel.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from work_llm_accelerator_amd import abi
from work_llm_accelerator_amd.layout import LAYOUT
from work_llm_accelerator_amd.model import FLAG_NO_BF16_ROUND, MODE_FAST, MODE_ORDERED, DeviceModel, KvCache

HIDDEN, INTERMEDIATE, KV_WIDTH, HEAD_DIM, Q_HEADS, VOCAB = 1536, 8960, 256, 128, 12, 151936
LAYER_BYTES = 23_508_992
LAYER_MACS = 46_792_704
MATRICES = (("q", HIDDEN, HIDDEN), ("k", KV_WIDTH, HIDDEN), ("v", KV_WIDTH, HIDDEN), ("o", HIDDEN, HIDDEN),
            ("gate", INTERMEDIATE, HIDDEN), ("up", INTERMEDIATE, HIDDEN), ("down", HIDDEN, INTERMEDIATE))


# ---- the cases ------------------------------------------------------------------------------
def _decode(kind: str, layers: int, batch: int, lo: int, hi: int, mode: str = "fast", **more) -> dict:
    """One new token for each of `batch` sequences whose histories hold lo..hi tokens."""
    return {**more, "kind": kind, "mode": mode, "layers": layers, "batch": batch, "lo": lo, "hi": hi}


def _prefill(layers: int, batch: int, seq: int, past: int = 0, mode: str = "fast", **more) -> dict:
    """`seq` new tokens for each of `batch` sequences that hold `past` tokens already."""
    return {**more, "kind": "prefill", "mode": mode, "layers": layers, "batch": batch, "seq": seq, "past": past}


def listed() -> list:
    return [
        # interactive generation: the whole step of one sequence, token id to logits, after a 512-token prompt
        _decode("generate", 8, 1, 577, 577, name="generate_b1"),
        # a small serving batch: the whole step of 24 conversations of different lengths
        _decode("generate", 8, 24, 150, 1100, name="generate_b24"),
        # one user deep in a long document
        _decode("decode", 4, 1, 9001, 9001, name="decode_b1_long"),
        # the benchmark's decode: bound by the key/value stream
        _decode("decode", 4, 64, 4096, 4096, name="decode_b64_kv4096"),
        # throughput serving: many conversations of different lengths, an odd count above one token tile of 64
        _decode("decode", 4, 150, 100, 900, name="decode_b150"),
        # a short chat turn
        _prefill(4, 1, 47, name="prefill_1x47"),
        # the benchmark's prompt for generation
        _prefill(4, 1, 512, name="prefill_1x512"),
        # the benchmark's prefill: bound by the matrix cores
        _prefill(1, 8, 2048, name="prefill_8x2048"),
        # a later chunk of a long prompt
        _prefill(4, 1, 385, past=3000, name="prefill_chunk_385_at_3000"),
        # the reference's arithmetic bit for bit, resident on the GPU: a decode step and a prefill of 128 tokens
        _decode("decode", 4, 1, 577, 577, mode="ordered", name="ordered_decode_b1"),
        _prefill(2, 1, 128, mode="ordered", name="ordered_prefill_1x128"),
        # a caller of the reference's host library that switched to this one: one layer on host buffers
        {"name": "dropin_decode_layer", "kind": "dropin_decode", "past": 576},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["generate", "decode", "decode", "one", "prefill", "prefill", "prompt", "chunk", "ordered_decode",
                       "ordered_prefill", "dropin"])
    if kind == "generate":
        batch, hi = _log_int(rng, 1, 24), _log_int(rng, 16, 1100)
        return _decode("generate", 8, batch, max(1, hi // rng.randint(1, 8)), hi)
    if kind == "decode":
        batch = _log_int(rng, 2, 150)
        hi = _log_int(rng, 16, min(9000, 262144 // batch))
        return _decode("decode", 4, batch, max(1, hi // rng.randint(1, 8)), hi)
    if kind == "one":
        keys = _log_int(rng, 16, 9001)
        return _decode("decode", 4, 1, keys, keys)
    if kind == "prompt":
        return _prefill(4, 1, _log_int(rng, 16, 1024))
    if kind == "prefill":
        batch = _log_int(rng, 1, 8)
        return _prefill(1, batch, _log_int(rng, 64, min(4096, 16384 // batch)))
    if kind == "chunk":
        return _prefill(4, 1, _log_int(rng, 16, 512), past=_log_int(rng, 16, 4000))
    if kind == "ordered_decode":
        batch, hi = _log_int(rng, 1, 8), _log_int(rng, 16, 577)
        return _decode("decode", 4, batch, max(1, hi // 2), hi, mode="ordered")
    if kind == "ordered_prefill":
        return _prefill(2, 1, _log_int(rng, 8, 128), mode="ordered")
    return {"kind": "dropin_decode", "past": _log_int(rng, 1, 576)}


def _positions(case: dict) -> np.ndarray:
    """History lengths of the batch, spread evenly over lo..hi in a scattered order."""
    if case["kind"] == "dropin_decode":
        return np.array([case["past"]])
    batch, lo, hi = case["batch"], case["lo"], case["hi"]
    even = lo + (np.arange(batch) * (hi - lo)) // max(1, batch - 1)
    return even[np.argsort((np.arange(batch) * 7919) % 104729, kind="stable")]


def _layers(case: dict) -> int:
    return case.get("layers", 1)


def work(case: dict) -> dict:
    if case["kind"] == "prefill":
        tokens = case["batch"] * case["seq"]
        attended = case["batch"] * sum(case["past"] + i + 1 for i in range(case["seq"]))
        history = case["batch"] * case["past"]
    else:
        pos = _positions(case)
        tokens, attended, history = len(pos), int(pos.sum()) + len(pos), int(pos.sum())
    layers = _layers(case)
    nbytes = layers * (LAYER_BYTES + 2048 * (history + tokens)) + 2 * tokens * HIDDEN * 4
    flops = layers * (2.0 * LAYER_MACS * tokens + 4.0 * HIDDEN * attended)
    if case["kind"] == "generate":
        nbytes += VOCAB * HIDDEN * 2 + tokens * VOCAB * 4
        flops += 2.0 * tokens * VOCAB * HIDDEN
    return {"bytes": float(nbytes), "flops": flops}


def tolerance(case: dict):
    if case.get("mode", "ordered") == "ordered":
        return "exact"  # this mode's results are defined to the bit
    # about four times the measured distance from exact(): 2.2e-4 to 5.4e-4 after one to four layers (the
    # 15-bit activation code); 2.3e-3 for logits, which are rounded to bf16, after eight
    return {"rel": 1e-2} if case["kind"] == "generate" else {"rel": 2e-3}


# ---- inputs ---------------------------------------------------------------------------------
def _generator(seed: int, part: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1_000_003 + part) & 0x7FFFFFFFFFFFFFFF)


def _normal(gen, *shape, sigma: float = 1.0) -> torch.Tensor:
    return torch.randn(*shape, generator=gen, device="cuda") * sigma


def _bf16(x: torch.Tensor) -> torch.Tensor:
    return x.to(torch.float32).to(torch.bfloat16).to(x.dtype)


def _layer(seed: int, layer: int) -> dict:
    """One layer's parameters: N(0, 0.02) bf16 weights quantized per row to INT4 (scale max|w| / 7), bf16
    biases and norm weights around 1."""
    gen = _generator(seed, 1000 + layer)
    p = {}
    for name, out_dim, in_dim in MATRICES:
        w = _bf16(_normal(gen, out_dim, in_dim, sigma=0.02))
        scale = w.abs().amax(dim=1) / 7.0
        p[name] = torch.clamp(torch.round(w / scale[:, None]), -8, 7).to(torch.int8)
        p[name + "_scale"] = scale
    for name, n in (("q_bias", HIDDEN), ("k_bias", KV_WIDTH), ("v_bias", KV_WIDTH)):
        p[name] = _bf16(_normal(gen, n, sigma=0.02))
    for name in ("input_layernorm", "post_attention_layernorm"):
        p[name] = _bf16(1.0 + _normal(gen, HIDDEN, sigma=0.1))
    return p


def _images(seed: int, layers: int) -> tuple:
    """The per-layer weight and scale images of the stack, in host memory."""
    weight = torch.zeros(layers, LAYER_BYTES, dtype=torch.uint8, device="cuda")
    scale = torch.zeros(layers, LAYER_BYTES // 4, dtype=torch.float32, device="cuda")
    for i in range(layers):
        p = _layer(seed, i)
        for name, out_dim, in_dim in MATRICES:
            nibble = (p[name].reshape(-1, 2) & 0xF).to(torch.uint8)
            at = getattr(LAYOUT, name + "_weight_offset_bytes")
            weight[i, at:at + out_dim * in_dim // 2] = nibble[:, 0] | (nibble[:, 1] << 4)
            at = getattr(LAYOUT, name + "_scale_offset_bytes") // 4
            scale[i, at:at + out_dim] = p[name + "_scale"]
        for name, attr in (("q_bias", "q_bias_offset_bytes"), ("k_bias", "k_bias_offset_bytes"),
                           ("v_bias", "v_bias_offset_bytes"),
                           ("input_layernorm", "input_layernorm_weight_offset_bytes"),
                           ("post_attention_layernorm", "post_attention_layernorm_weight_offset_bytes")):
            at = getattr(LAYOUT, attr) // 4
            scale[i, at:at + p[name].numel()] = p[name]
    return weight.cpu().numpy().reshape(-1), scale.cpu().numpy().reshape(-1)


def _head(seed: int) -> tuple:
    gen = _generator(seed, 3)
    table = (torch.randn(VOCAB, HIDDEN, generator=gen, device="cuda", dtype=torch.float32) * 0.02).to(torch.bfloat16)
    return table, (1.0 + _normal(gen, HIDDEN, sigma=0.1)).to(torch.bfloat16)


def _tokens(seed: int, count: int) -> torch.Tensor:
    return torch.randint(0, VOCAB, (count,), generator=_generator(seed, 4), device="cuda", dtype=torch.int32)


def _hidden(case: dict, seed: int) -> torch.Tensor:
    shape = (case["batch"], case["seq"], HIDDEN) if case["kind"] == "prefill" else (len(_positions(case)), HIDDEN)
    return _normal(_generator(seed, 5), *shape)


def _cache_rows(case: dict) -> int:
    """Rows of each sequence's cache: the tokens so far, and room for the next ones of a generation."""
    return case["past"] + case["seq"] if case["kind"] == "prefill" else int(_positions(case).max()) + 16


def _history(case: dict, seed: int, layer: int) -> tuple:
    """K and V rows of one layer's cache, [sequences][rows][256]."""
    gen = _generator(seed, 2000 + layer)
    rows = _cache_rows(case)
    batch = len(_positions(case)) if case["kind"] != "prefill" else case["batch"]
    return _normal(gen, batch, rows, KV_WIDTH), _normal(gen, batch, rows, KV_WIDTH)


def prepare(case: dict, seed: int) -> dict:
    layers = _layers(case)
    weight, scale = _images(seed, layers)
    state = {"case": case}
    if case["kind"] == "dropin_decode":
        at = {f: getattr(LAYOUT, f) for f in LAYOUT.__dataclass_fields__}
        sizes = {name: (out_dim, in_dim) for name, out_dim, in_dim in MATRICES}

        def packed(name):
            first = at[name + "_weight_offset_bytes"]
            return weight[first:first + sizes[name][0] * sizes[name][1] // 2]

        def words(attr, n):
            return scale[at[attr] // 4:at[attr] // 4 + n]

        k, v = _history(case, seed, 0)
        state["k"] = k[0, :case["past"] + 1].reshape(-1).cpu().numpy()
        state["v"] = v[0, :case["past"] + 1].reshape(-1).cpu().numpy()
        state["x"] = _hidden(case, seed).reshape(-1).cpu().numpy()
        state["out"] = np.zeros(HIDDEN, np.float32)
        state["lib"] = abi.load()
        state["weights"] = [
            words("input_layernorm_weight_offset_bytes", HIDDEN),
            words("post_attention_layernorm_weight_offset_bytes", HIDDEN),
            *(packed(name) for name in ("q", "k", "v", "o", "gate", "up", "down")),
            *(words(name + "_bias_offset_bytes", sizes[name][0]) for name in ("q", "k", "v")),
            *(words(name + "_scale_offset_bytes", sizes[name][0]) for name in ("q", "k", "v", "o", "gate", "up", "down")),
        ]
        return state
    model = DeviceModel(layers, weight, scale)
    sequences = case["batch"]
    cache = KvCache.allocate(layers, sequences, _cache_rows(case))
    for i in range(layers):
        k, v = _history(case, seed, i)
        cache.k[i], cache.v[i] = k, v
    state.update(model=model, cache=cache, mode=MODE_FAST if case["mode"] == "fast" else MODE_ORDERED)
    if case["kind"] == "prefill":
        state["x"] = _hidden(case, seed)
    else:
        pos = _positions(case)
        state["positions"] = torch.tensor(pos, dtype=torch.int32, device="cuda")
        state["max_keys"] = int(pos.max()) + 1
        if case["kind"] == "generate":
            table, norm = _head(seed)
            model.set_head(table.view(torch.int16).cpu().numpy().view(np.uint16),
                           norm.view(torch.int16).cpu().numpy().view(np.uint16))
            state["ids"] = _tokens(seed, sequences)
            state["logits"] = torch.empty(sequences, VOCAB, dtype=torch.float32, device="cuda")
            state["hidden"] = torch.empty(sequences, HIDDEN, dtype=torch.float32, device="cuda")
        else:
            state["x"] = _hidden(case, seed)
    if "x" in state:
        state["hidden"] = torch.empty_like(state["x"])
    torch.cuda.synchronize()
    return state


# ---- one pass -------------------------------------------------------------------------------
def run(state: dict):
    case = state["case"]
    if case["kind"] == "dropin_decode":
        status = state["lib"].qwen_decode_layer_smoke_forward(state["x"], case["past"], *state["weights"], state["k"],
                                                              state["v"], state["out"])
        if status != 0:
            raise RuntimeError(f"qwen_decode_layer_smoke_forward: status {status}")
        return {"out": state["out"], "k": state["k"], "v": state["v"]}
    model, cache, hidden = state["model"], state["cache"], state["hidden"]
    # no bf16 rounding between layers: a tie that falls the other way is 30 times the kernels' own rounding
    mode = state["mode"] | FLAG_NO_BF16_ROUND
    if case["kind"] == "generate":
        model.embed(state["ids"], hidden)
        model.decode(mode, hidden, state["positions"], state["max_keys"], cache, order=False)
        model.logits(hidden, state["logits"], order=False)
        torch.cuda.current_stream().wait_stream(model.stream)
        return {"logits": state["logits"], "k": cache.k, "v": cache.v}
    hidden.copy_(state["x"])  # the layers work in place
    if case["kind"] == "decode":
        model.decode(mode, hidden, state["positions"], state["max_keys"], cache)
    else:
        model.prefill(mode, hidden, cache, past=case["past"])
    torch.cuda.current_stream().wait_stream(model.stream)
    return {"hidden": hidden, "k": cache.k, "v": cache.v}


# ---- the same in 64 bits, in plain torch ----------------------------------------------------
def _rms(x, w, prefill: bool):
    mean = (x * x).mean(dim=-1, keepdim=True) + 1e-6
    root = mean.sqrt()
    if prefill:  # six Newton steps from max(1, mean), as the prefill layer defines its root
        root = mean.clamp(min=1.0)
        for _ in range(6):
            root = 0.5 * (root + mean / root)
    return x / root * w


def _exp(v, prefill: bool):
    """exp, or the prefill layer's: 0 from -16 down, halved into [-1, ...), six terms, squared back."""
    if not prefill:
        return v.exp()
    s, halves = v.clone(), torch.zeros_like(v, dtype=torch.int8)
    for _ in range(4):
        low = s < -1.0
        s = torch.where(low, s * 0.5, s)
        halves += low
    term, series = torch.ones_like(s), torch.ones_like(s)
    for degree in range(1, 7):
        term = term * s / degree
        series = series + term
    for i in range(4):
        series = torch.where(halves > i, series * series, series)
    return torch.where(v <= -16.0, torch.zeros_like(v), series.clamp(min=0.0))


def _rope_rows(pos, prefill: bool) -> tuple:
    """(cos, sin) [n, 64] of positions [n]: the decode layer's are libm's in double, the prefill layer's
    its own fp32 angles, folded by repeated subtraction, and short series."""
    if not prefill:
        p = torch.arange(64, device="cuda", dtype=torch.float64)
        angle = pos.to(torch.float64)[:, None] * torch.pow(torch.tensor(1e6, dtype=torch.float64, device="cuda"),
                                                          -2.0 * p / HEAD_DIM)
        return angle.cos().float().double(), angle.sin().float().double()
    freq, f = [], np.float32(1.0)
    for _ in range(64):
        freq.append(f)
        f = np.float32(f * np.float32(0.8058421877614801))
    angle = pos.to(torch.float32)[:, None] * torch.tensor(np.array(freq), device="cuda")
    pi, two_pi = float(np.float32(math.pi)), torch.tensor(np.float32(2 * math.pi), device="cuda")
    while bool((angle > pi).any()):
        angle = torch.where(angle > pi, angle - two_pi, angle)
    r = angle.double()
    fold = torch.where(r > math.pi / 2, pi - r, torch.where(r < -math.pi / 2, -pi - r, r))
    sign = torch.where(fold == r, 1.0, -1.0)
    x2 = fold * fold
    sin = fold * (1.0 + x2 * (-1.0 / 6.0 + x2 * (1.0 / 120.0 - x2 / 5040.0)))
    cos = sign * (1.0 + x2 * (-0.5 + x2 * (1.0 / 24.0 - x2 / 720.0)))
    return cos, sin


def _rotate(x, rope, heads: int):
    cos, sin = rope[0][:, None], rope[1][:, None]
    h = x.reshape(-1, heads, HEAD_DIM)
    even, odd = h[..., :64], h[..., 64:]
    return torch.cat([even * cos - odd * sin, odd * cos + even * sin], dim=-1).reshape(x.shape)


def _attend(q, k, v, first: int, prefill: bool):
    """q [n, 1536] at positions first.. over rows k, v [rows, 256]: causal, query head h on KV head h // 6."""
    n, rows = q.shape[0], first + q.shape[0]
    out = torch.empty(n, Q_HEADS, HEAD_DIM, dtype=torch.float64, device="cuda")
    masked = torch.arange(rows, device="cuda")[None, :] > first + torch.arange(n, device="cuda")[:, None]
    for h in range(Q_HEADS):
        kv = slice((h // 6) * HEAD_DIM, (h // 6 + 1) * HEAD_DIM)
        score = q[:, h * HEAD_DIM:(h + 1) * HEAD_DIM] @ k[:rows, kv].T.contiguous() / math.sqrt(HEAD_DIM)
        score = score.masked_fill(masked, -1e30)
        e = _exp(score - score.amax(dim=1, keepdim=True), prefill)
        e = e.masked_fill(masked, 0.0)
        out[:, h] = (e @ v[:rows, kv].contiguous()) / e.sum(dim=1, keepdim=True)
    return out.reshape(n, HIDDEN)


def _layer64(p: dict, x, k, v, starts, prefill: bool):
    """One layer of x [sequences, n, 1536]; sequence b's tokens take positions starts[b].. and rows of k, v."""
    def weight(name):
        return (p[name].double() * p[name + "_scale"].double()[:, None]).T.contiguous()

    sequences, n, _ = x.shape
    flat = _rms(x, p["input_layernorm"].double(), prefill).reshape(-1, HIDDEN)
    pos = (torch.tensor(np.array(starts), device="cuda")[:, None] + torch.arange(n, device="cuda")).reshape(-1)
    rope = _rope_rows(pos, prefill)
    q = _rotate(flat @ weight("q") + p["q_bias"].double(), rope, Q_HEADS).reshape(sequences, n, HIDDEN)
    new_k = _rotate(flat @ weight("k") + p["k_bias"].double(), rope, 2).reshape(sequences, n, KV_WIDTH)
    new_v = (flat @ weight("v") + p["v_bias"].double()).reshape(sequences, n, KV_WIDTH)
    context = torch.empty(sequences, n, HIDDEN, dtype=torch.float64, device="cuda")
    for b in range(sequences):
        first = int(starts[b])
        k[b, first:first + n], v[b, first:first + n] = new_k[b], new_v[b]
        context[b] = _attend(q[b], k[b], v[b], first, prefill)
    a = context.reshape(-1, HIDDEN) @ weight("o")
    post = _rms(a, p["post_attention_layernorm"].double(), prefill)
    gate = post @ weight("gate")
    s = gate / (1.0 + _exp(-gate, prefill)) * (post @ weight("up"))
    return (a + s @ weight("down")).reshape(x.shape)


def exact(case: dict, seed: int):
    prefill = case["kind"] == "prefill"
    starts = [case["past"]] * case["batch"] if prefill else _positions(case)
    if case["kind"] == "generate":
        table, norm = _head(seed)
        x = table[_tokens(seed, len(starts)).long()].double()[:, None]
    else:
        x = _hidden(case, seed).double().reshape(len(starts), -1, HIDDEN)
    ks, vs = [], []
    for i in range(_layers(case)):
        k, v = (r.double() for r in _history(case, seed, i))
        x = _layer64(_layer(seed, i), x, k, v, starts, prefill)
        ks.append(k)
        vs.append(v)
    if case["kind"] == "dropin_decode":
        rows = case["past"] + 1
        return {"out": x.reshape(-1), "k": ks[0][0, :rows].reshape(-1), "v": vs[0][0, :rows].reshape(-1)}
    k, v = torch.stack(ks), torch.stack(vs)
    if case["kind"] == "generate":
        h = _bf16(x[:, 0])
        n = _bf16(_bf16(h / ((h * h).mean(dim=-1, keepdim=True) + 1e-6).sqrt()) * norm.double())
        logits = torch.cat([n @ part.double().T.contiguous() for part in table.split(16384)], dim=1)
        return {"logits": logits, "k": k, "v": v}
    return {"hidden": x.reshape(len(starts), -1, HIDDEN) if prefill else x[:, 0], "k": k, "v": v}
