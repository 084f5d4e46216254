"""The work that a serving program has this framework do, as cases that can be timed and compared.

A case is one pass of the attention part of a model step through the public operators: the KV append (or the fused
q/k norm, rotary embedding and append) followed by the attention call over every row's populated prefix, in the
adapters' order; or the singleton projections of one decoder layer.  The shapes are those of xinfer_amd/workloads.py
and of the tests: 16 query / 8 KV heads of 128 features, 16 / 4 of 256, 8 / 8 of 64, 32 / 8 of 128; batches from one
row to a few tens; 1 to 512 new tokens a row; prefixes up to 16384 keys.

`counts` and `lengths` are comma-separated texts, one number per row: the new tokens and the populated keys after
the append.  Inputs are N(0, 1) bf16, as in xinfer_amd/workloads.py.
"""

import math

import torch

from xinfer_amd.attention import batched_attention_metadata, cache_extent, load_attention_ops
from xinfer_amd.kv_cache import append_kv_batched
from xinfer_amd.norm_rope import qk_norm_rope_append
from xinfer_amd.projection_gemv import projection_gemv

SHAPES = {  # (query heads, KV heads, features)
    "16x8x128": (16, 8, 128),
    "16x4x256": (16, 4, 256),
    "8x8x64": (8, 8, 64),
    "32x8x128": (32, 8, 128),
}
EPS = 1e-6
LAYER_PROJECTIONS = "8224x1024,7168x1024,5120x1024,1024x3584,1024x2048"


def _numbers(text):
    return [int(x) for x in str(text).split(",")]


def _case(name, kind, shape, capacity, counts, lengths, layers=1):
    return {"name": name, "kind": kind, "shape": shape, "capacity": capacity, "layers": layers,
            "counts": ",".join(map(str, counts)), "lengths": ",".join(map(str, lengths))}


def listed():
    return [
        # One request, one new token, a short context: the smallest decode call (latency).
        _case("decode_b1_l1024", "flash", "16x8x128", 4096, [1], [1024]),
        # A ragged decode batch of eight requests, log-uniform contexts up to 16384 keys.
        _case("decode_b8_ragged", "step", "16x8x128", 16384, [1] * 8, [13312, 2162, 386, 9459, 1399, 3852, 55, 182]),
        # Decode with 256 features per head and four query heads per KV head.
        _case("decode_b4_d256", "step", "16x4x256", 16384, [1] * 4, [1024, 4096, 8192, 16384]),
        # A full server: 32 requests decode together, most contexts short, some long.
        _case("decode_b32_ragged", "step", "16x8x128", 8192, [1] * 32,
              [4021, 33, 517, 1260, 95, 7710, 208, 2475, 61, 1033, 345, 5822, 18, 764, 150, 3001,
               49, 6345, 411, 27, 1888, 90, 640, 4490, 121, 2210, 303, 77, 985, 1501, 8190, 242]),
        # Six new tokens a row over long contexts: checking drafted tokens, or short follow-up turns.
        _case("chunk_b8_t6", "step", "16x8x128", 16384, [6, 6, 5, 6, 2, 6, 6, 4],
              [9010, 1203, 4777, 305, 15021, 2650, 640, 6111]),
        # One 512-token chunk of a prompt at offset 1536: chunked prefill.
        _case("prefill_b1_n512", "step", "16x8x128", 4096, [512], [2048]),
        # Short prompts of odd lengths from an empty cache, small heads.
        _case("prompts_b3_d64", "step", "8x8x64", 1024, [77, 201, 13], [77, 201, 13]),
        # Four chunks of long prompts, 32 query heads.
        _case("prefill_b4_long", "step", "32x8x128", 16384, [512, 512, 389, 512], [8704, 5120, 12001, 2560]),
        # A ragged prefill batch, 256 features: the largest call.
        _case("prefill_b8_d256", "step", "16x4x256", 16384, [356, 138, 422, 459, 325, 298, 113, 124],
              [14244, 13896, 2059, 4214, 12262, 14086, 12837, 9315]),
        # Continuous batching: seven requests decode while one prompt chunk is read; the fused entry points.
        _case("mixed_b8_fused", "fused", "16x8x128", 8192, [1, 1, 384, 1, 1, 1, 1, 1],
              [2047, 611, 1409, 5003, 96, 1233, 3170, 402]),
        # A decode step captured once and replayed as lengths change: the attention parts of eight layers.
        _case("captured_b8_8layers", "captured", "16x8x128", 4096, [1] * 8, [4000, 18, 1021, 255, 2077, 640, 97, 3333],
              layers=8),
        # The singleton projections of one decoder layer at one new token.
        {"name": "projections_bf16", "kind": "gemv", "dtype": "bf16", "shapes": LAYER_PROJECTIONS},
    ]


def _log_uniform(rng, low, high):
    return min(high, int(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))


def _draw_once(rng):
    kind = rng.choice(["flash", "step", "step", "step", "step", "fused", "captured", "gemv"])
    if kind == "gemv":
        shapes = rng.sample(LAYER_PROJECTIONS.split(","), 2) + [
            "%dx%d" % (_log_uniform(rng, 512, 8224), 8 * _log_uniform(rng, 64, 512)) for _ in range(2)]
        return {"kind": "gemv", "dtype": rng.choice(["bf16", "bf16", "fp32"]), "shapes": ",".join(shapes)}
    shape = rng.choice(["16x8x128", "16x8x128", "16x4x256", "8x8x64", "32x8x128"])
    what = rng.choice(["decode", "decode", "chunk", "prefill", "mixed"])
    if kind == "flash":
        rows, what = 1, rng.choice(["decode", "prefill"])
    elif what == "prefill":
        rows = rng.randint(1, 8)
    else:
        rows = _log_uniform(rng, 1, 32)
    capacity = rng.choice([4096, 16384] if rows <= 8 else [4096, 8192])
    layers = 1
    if kind == "captured":
        capacity, layers = 4096, rng.randint(2, 8)
        rows = min(rows, 16)
    if what == "decode":
        counts = [1] * rows
    elif what == "chunk":
        t = rng.randint(2, 16)
        counts = [rng.randint(1, t) for _ in range(rows)]
    elif what == "prefill":
        counts = [_log_uniform(rng, 17, 512) for _ in range(rows)]
    else:
        counts = [1] * rows
        counts[rng.randrange(rows)] = _log_uniform(rng, 17, 512)
    lengths = [n + (0 if rng.random() < 0.15 else _log_uniform(rng, 16, capacity - n)) for n in counts]
    return {k: v for k, v in _case("", kind, shape, capacity, counts, lengths, layers).items() if k != "name"}


def draw(rng):
    largest = next(_cost(c) for c in listed() if c["name"] == "prefill_b8_d256")
    while True:
        case = _draw_once(rng)
        if _cost(case) <= largest:
            return case


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 4e12, w["flops"] / 5e14)


def work(case):
    if case["kind"] == "gemv":
        size = 4 if case["dtype"] == "fp32" else 2
        shapes = [[int(x) for x in s.split("x")] for s in case["shapes"].split(",")]
        return {"bytes": sum((n * k + n + k) * size for n, k in shapes), "flops": sum(2 * n * k for n, k in shapes)}
    hq, hkv, d = SHAPES[case["shape"]]
    counts, lengths = _numbers(case["counts"]), _numbers(case["lengths"])
    tokens, padded = sum(counts), len(counts) * max(counts)
    keys = 2 * 2 * hkv * d  # bytes of one token's K and V
    # Every populated key and every query is read once, every output (padded tokens are zeros) is written once.
    moved = sum(lengths) * keys + tokens * hq * d * 2 + padded * hq * d * 2
    if case["kind"] != "flash":
        moved += 2 * tokens * keys  # the new tokens' K and V, read and appended
    if case["kind"] in ("fused", "captured"):
        moved += 2 * padded * hq * d * 2 + padded * 2 * d * 2  # projected queries in and out, rotary tables
    flops = 4 * hq * d * sum(n * (length - n) + n * (n + 1) // 2 for n, length in zip(counts, lengths))
    return {"bytes": moved * case["layers"], "flops": flops * case["layers"]}


def tolerance(case):
    if case["kind"] == "gemv":
        # fp32 sums in another order; or one rounding of such a sum to bf16.
        return {"rel": 1e-5} if case["dtype"] == "fp32" else {"rel": 4e-3}
    # Outputs rounded to bf16 (2^-9 at most, 1.7e-3 rms), softmax weights of prefill rounded to bf16.
    return {"rel": 1e-2}


def _layer_inputs(case, generator):
    """One layer's tensors: caches as populated before the step, and the step's projections."""
    hq, hkv, d = SHAPES[case["shape"]]
    counts, lengths = _numbers(case["counts"]), _numbers(case["lengths"])
    b, t, c = len(counts), max(counts), case["capacity"]

    def normal(*shape):
        return torch.randn(*shape, generator=generator, device="cuda", dtype=torch.float32).to(torch.bfloat16)

    layer = {"k": normal(b, hkv, c, d), "v": normal(b, hkv, c, d), "q": normal(b, t, hq, d),
             "new_k": normal(b, t, hkv, d), "new_v": normal(b, t, hkv, d)}
    if case["kind"] in ("fused", "captured"):
        layer["q_weight"] = (1 + 0.1 * normal(d).float()).to(torch.bfloat16)
        layer["k_weight"] = (1 + 0.1 * normal(d).float()).to(torch.bfloat16)
    return layer


def _positions(case):
    counts, lengths = _numbers(case["counts"]), _numbers(case["lengths"])
    positions = torch.zeros(len(counts), max(counts), dtype=torch.int64)
    for r, (n, length) in enumerate(zip(counts, lengths)):
        positions[r, :n] = torch.arange(length - n, length)
    return positions.cuda()


def _rotary(case, positions):
    d = SHAPES[case["shape"]][2]
    inverse = 1e6 ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d)
    angles = positions[..., None].double() * inverse
    angles = torch.cat((angles, angles), dim=-1)
    return angles.cos().to(torch.bfloat16), angles.sin().to(torch.bfloat16)


def _inputs(case, seed):
    generator = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] == "gemv":
        dtype = torch.float32 if case["dtype"] == "fp32" else torch.bfloat16
        pairs = []
        for shape in case["shapes"].split(","):
            n, k = (int(x) for x in shape.split("x"))
            x = torch.randn(1, 1, k, generator=generator, device="cuda").to(dtype)
            pairs.append((x, (torch.randn(n, k, generator=generator, device="cuda") * k ** -0.5).to(dtype)))
        return {"pairs": pairs}
    state = {"positions": _positions(case), "layers": [_layer_inputs(case, generator) for _ in range(case["layers"])]}
    if case["kind"] in ("fused", "captured"):
        state["cos"], state["sin"] = _rotary(case, state["positions"])
    return state


def prepare(case, seed):
    load_attention_ops(model="qwen3")
    state = _inputs(case, seed)
    state["kind"] = case["kind"]
    if case["kind"] == "gemv":
        return state
    counts = torch.tensor(_numbers(case["counts"]), dtype=torch.int32)
    lengths = torch.tensor(_numbers(case["lengths"]), dtype=torch.int32)
    state["offsets"], state["device_offsets"], state["blocks"] = batched_attention_metadata(lengths, counts, "cuda")
    state["scale"] = SHAPES[case["shape"]][2] ** -0.5
    state["cu_query"] = state["device_offsets"][0]
    if case["kind"] == "flash":
        state["extent"] = cache_extent(int(lengths[0]))
    if case["kind"] in ("flash", "step"):
        # A model step's projections transposed to heads, as the adapters hand them over.
        for layer in state["layers"]:
            for name in ("q", "new_k", "new_v"):
                layer[name] = layer[name].transpose(1, 2)
    if case["kind"] == "captured":
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream), torch.inference_mode():
            _step(state)
        torch.cuda.current_stream().wait_stream(stream)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]), torch.inference_mode():
            state["outputs"] = _step(state)
    return state


def _step(state):
    """The attention part of every layer of a model step; returns each layer's output and caches."""
    outputs = []
    for layer in state["layers"]:
        k, v = layer["k"], layer["v"]
        if state["kind"] == "step":
            append_kv_batched(layer["new_k"], layer["new_v"], state["positions"], state["cu_query"], k, v)
            out = torch.ops.xinfer.batched_flash_attention(layer["q"], k, v, state["offsets"], state["device_offsets"],
                                                           state["blocks"], state["scale"])
        else:
            q = qk_norm_rope_append(layer["q"], layer["new_k"], layer["new_v"], layer["q_weight"], layer["k_weight"],
                                    EPS, state["cos"], state["sin"], state["positions"], state["cu_query"], k, v)
            attention = (torch.ops.xinfer.batched_flash_attention_bthd if state["kind"] == "fused"
                         else torch.ops.xinfer.batched_flash_attention_graph)
            out = attention(q, k, v, state["offsets"], state["device_offsets"], state["blocks"], state["scale"])
        outputs.append({"out": out, "k": k, "v": v})
    return outputs


def run(state):
    with torch.inference_mode():
        if state["kind"] == "gemv":
            return [projection_gemv(x, weight) for x, weight in state["pairs"]]
        if state["kind"] == "flash":
            layer = state["layers"][0]
            return torch.ops.xinfer.flash_attention(layer["q"], layer["k"], layer["v"], state["extent"],
                                                    state["scale"])
        if state["kind"] == "captured":
            state["graph"].replay()
            return state["outputs"]
        return _step(state)


def _norm_rope(x, weight, cos, sin):
    x = x.double()
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()
    half = x.shape[-1] // 2
    rotated = torch.cat((-x[..., half:], x[..., :half]), dim=-1)
    return x * cos.double()[:, :, None] + rotated * sin.double()[:, :, None]


def _attention(q, k, v, counts, lengths, scale):
    """softmax(scale * q k^T) v in 64 bits, lower-right causal; q [B, T, Hq, D], caches [B, Hkv, C, D] -> [B, Hq, T, D]."""
    b, t, hq, d = q.shape
    hkv = k.shape[1]
    out = torch.zeros(b, hq, t, d, dtype=torch.float64, device=q.device)
    for r, (n, length) in enumerate(zip(counts, lengths)):
        hidden = torch.arange(length, device=q.device)[None] > (length - n + torch.arange(n, device=q.device))[:, None]
        for h in range(hkv):
            group = hq // hkv
            rows = q[r, :n, h * group:(h + 1) * group].double().transpose(0, 1).reshape(group * n, d)
            keys, values = k[r, h, :length].double(), v[r, h, :length].double()
            scores = (rows @ keys.t().contiguous() * scale).reshape(group, n, length)
            scores.masked_fill_(hidden, -math.inf)
            out[r, h * group:(h + 1) * group, :n] = (scores.softmax(-1).reshape(group * n, length) @ values).reshape(
                group, n, d)
    return out


def exact(case, seed):
    state = _inputs(case, seed)
    if case["kind"] == "gemv":
        return [(x.double().reshape(1, -1) @ weight.double().t().contiguous()).reshape(1, 1, -1)
                for x, weight in state["pairs"]]
    counts, lengths = _numbers(case["counts"]), _numbers(case["lengths"])
    scale = SHAPES[case["shape"]][2] ** -0.5
    outputs = []
    for layer in state["layers"]:
        q, new_k, k, v = layer["q"], layer["new_k"], layer["k"], layer["v"]
        if case["kind"] in ("fused", "captured"):
            q = _norm_rope(q, layer["q_weight"], state["cos"], state["sin"])
            new_k = _norm_rope(new_k, layer["k_weight"], state["cos"], state["sin"])
        if case["kind"] != "flash":
            k, v = k.double(), v.double()
            for r, (n, length) in enumerate(zip(counts, lengths)):
                k[r, :, length - n:length] = new_k[r, :n].transpose(0, 1).double()
                v[r, :, length - n:length] = layer["new_v"][r, :n].transpose(0, 1).double()
        out = _attention(q, k, v, counts, lengths, scale)
        if case["kind"] == "flash":
            return out
        outputs.append({"out": out.transpose(1, 2).contiguous() if case["kind"] == "fused" else out, "k": k, "v": v})
    return outputs
