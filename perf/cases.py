"""The work a user of this framework has it do, as cases that can be timed and compared: paged
attention steps, dense attention and a decoder layer on device "HIP".

Every case goes through the public entry points (the C ABI's bindings `capi`, and `plugin_capi`'s
InferRequest for the decoder layer) with all tensors resident on the GPU.  The listed cases are the
benchmark configurations of this repository and ordinary sizes between and beside them; `draw` gives
more of the same ranges.  Torch allocates and fills the memory; the bindings take any object with
`ptr` and `nbytes`.
"""
import ctypes
import math
import random

import numpy as np
import torch

from openvino_contrib_amd import capi
from openvino_contrib_amd import plugin_capi as P
from openvino_contrib_amd import workloads as W

DTYPES = {"f32": (W.F32, torch.float32), "f16": (W.F16, torch.float16), "bf16": (W.BF16, torch.bfloat16),
          "u8": (W.U8, torch.uint8)}

# ----------------------------------------------------------------------------------- the cases
# A paged step: `prompts` sequences of chunk_lo..chunk_hi new tokens behind past_lo..past_hi cached ones, then
# `decodes` sequences of one new token whose contexts are uniform in ctx_lo..ctx_hi.  The lengths are part of
# the case (drawn from `lengths`), everything else comes from prepare()'s seed.
PAGED = dict(path="paged", q="f16", cache="f16", heads=32, kv_heads=8, size=128, block=32, window=0, lengths=1,
             prompts=0, chunk_lo=0, chunk_hi=0, past_lo=0, past_hi=0, decodes=0, ctx_lo=0, ctx_hi=0)
# v13::ScaledDotProductAttention; mask: "none", "causal", "padding" (boolean, one row of keys per batch entry)
# or "bias" (additive, of the operands' type, one [queries, keys] matrix for all)
SDPA = dict(path="sdpa", dtype="bf16", batch=1, heads=32, kv_heads=8, queries=128, keys=128, size=128, mask="causal", std=1.0)
# One decoder layer (norm, projections, rotary embedding, paged attention, gated MLP, residuals) compiled for
# device "HIP": bf16 weights and activations, fp16 cache, the batch as in a paged step
LAYER = dict(PAGED, path="layer", q="bf16", hidden=4096, ffn=14336)


def listed():
    return [
        # the next token of a single conversation: one launch or two, all latency
        dict(PAGED, name="decode_one", decodes=1, ctx_lo=778, ctx_hi=778),
        # a decode step of a serving batch
        dict(PAGED, name="decode_f16", decodes=64, ctx_lo=512, ctx_hi=8192, lengths=1003),
        # the same on a quantised cache, twice the batch and the context
        dict(PAGED, name="decode_u8", cache="u8", heads=64, decodes=128, ctx_lo=1024, ctx_hi=16384, lengths=1004),
        # continuous batching: chunks of prompts beside decoding sequences, with a sliding window
        dict(PAGED, name="mixed_bf16", q="bf16", heads=64, window=4096, prompts=8, chunk_lo=512, chunk_hi=512, past_hi=4096,
             decodes=120, ctx_lo=256, ctx_hi=8192, lengths=1005),
        # new prompts of uneven length into a quantised cache
        dict(PAGED, name="prompt_u8", q="bf16", cache="u8", prompts=6, chunk_lo=100, chunk_hi=3000, lengths=6),
        # one attention operator of a small fp32 model
        dict(SDPA, name="sdpa_f32_small", dtype="f32", heads=8, kv_heads=8, queries=128, keys=128, size=64),
        # an fp32 text encoder: padded sentences in a batch
        dict(SDPA, name="sdpa_f32_encoder", dtype="f32", batch=8, heads=12, kv_heads=12, queries=384, keys=384, size=64, mask="padding"),
        # an image encoder: every patch and one token more attend each other
        dict(SDPA, name="sdpa_f16_encoder", dtype="f16", batch=16, heads=16, kv_heads=16, queries=577, keys=577, size=64, mask="none"),
        # prompt attention of a decoder in a stateful (contiguous cache) model
        dict(SDPA, name="sdpa_bf16_causal", batch=4, queries=2048, keys=2048, std=0.5),
        # a decoder layer with a handful of conversations, with a serving batch, and over new prompts
        dict(LAYER, name="layer_decode_few", decodes=4, ctx_lo=256, ctx_hi=4096, lengths=4),
        dict(LAYER, name="layer_decode", decodes=64, ctx_lo=512, ctx_hi=8192, lengths=1003),
        dict(LAYER, name="layer_prompt", prompts=3, chunk_lo=200, chunk_hi=1200, lengths=3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    """Seconds, roughly, at rates well below the card's: what keeps a drawn case below the largest listed one."""
    w = work(case)
    rate = 3e13 if case.get("dtype") == "f32" else 4e14
    return w["bytes"] / 4e12 + w["flops"] / rate


def draw(rng):
    kind = rng.choices(("decode", "chunks", "sdpa", "layer"), (3, 2, 4, 3))[0]
    largest = max(_cost(c) for c in listed() if c["path"] == ("layer" if kind == "layer" else "sdpa" if kind == "sdpa" else "paged"))
    while True:
        if kind == "sdpa":
            f32 = rng.random() < 0.5
            size = rng.choice((64, 64, 128) if f32 else (64, 64, 80, 96, 128, 128))
            mask = rng.choice(("none", "causal", "padding", "bias"))
            kv = rng.choice((8, 12, 16) if mask != "causal" else (4, 8, 8, 12))
            heads = kv * (rng.choice((1, 1, 4)) if mask == "causal" else 1)
            n = _log_int(rng, 48, 2048 if f32 else 4096)
            keys = n if mask == "causal" or rng.random() < 0.8 else _log_int(rng, 48, 2048)
            case = dict(SDPA, dtype="f32" if f32 else rng.choice(("f16", "bf16")), batch=_log_int(rng, 1, 16), heads=heads,
                        kv_heads=kv, queries=n, keys=keys, size=size, mask=mask)
        else:
            case = dict(LAYER if kind == "layer" else PAGED, lengths=rng.randrange(1 << 30))
            if kind == "layer":
                kv = rng.choice((4, 8, 8))
                heads = rng.choice((4, 4, 8) if kv == 4 else (3, 4)) * kv
                hidden = heads * 128
                case.update(heads=heads, kv_heads=kv, hidden=hidden, ffn=rng.choice((hidden * 7 // 2, hidden * 8 // 3 // 256 * 256)))
            else:
                heads, kv = rng.choice(((32, 8), (32, 8), (64, 8), (16, 4), (16, 16)))
                case.update(q=rng.choice(("f16", "bf16")), cache=rng.choice(("f16", "bf16", "u8", "u8")), heads=heads, kv_heads=kv,
                            size=rng.choice((64, 128, 128, 128)), block=rng.choice((16, 32)), window=rng.choice((0, 0, 0, 4096)))
                if case["cache"] != "u8" and rng.random() < 0.7:
                    case["cache"] = case["q"]  # a 16-bit cache mostly has the activations' type
            chunks = kind == "chunks" or (kind == "layer" and rng.random() < 0.33)
            if chunks:
                case["prompts"] = _log_int(rng, 1, 8)
                case["chunk_hi"] = _log_int(rng, 64, 3000)
                case["chunk_lo"] = max(2, int(case["chunk_hi"] * rng.uniform(0.1, 1.0)))
                case["past_hi"] = rng.choice((0, 0, _log_int(rng, 64, 4096)))
            if not chunks or rng.random() < 0.4:
                case["decodes"] = _log_int(rng, 1, 128 if kind != "layer" else 64)
                case["ctx_hi"] = _log_int(rng, 64, 16384 if kind != "layer" else 8192)
                case["ctx_lo"] = max(1, int(case["ctx_hi"] * rng.uniform(0.05, 1.0)))
        if _cost(case) <= largest:
            return case


def _sequences(case):
    """[(cached tokens, new tokens)] of a paged step."""
    r = random.Random(case["lengths"])
    seqs = [(r.randint(case["past_lo"], case["past_hi"]), r.randint(case["chunk_lo"], case["chunk_hi"])) for _ in range(case["prompts"])]
    return seqs + [(r.randint(case["ctx_lo"], case["ctx_hi"]) - 1, 1) for _ in range(case["decodes"])]


# --------------------------------------------------------------------------------------- work
def work(case):
    """What a pass cannot do without: every input once, every output once, two operations per multiply-add."""
    if case["path"] == "sdpa":
        e = DTYPES[case["dtype"]][1].itemsize
        B, Hq, Hkv, Lq, Lk, D = (case[k] for k in ("batch", "heads", "kv_heads", "queries", "keys", "size"))
        mask = B * Lk if case["mask"] == "padding" else Lq * Lk * e if case["mask"] == "bias" else 0
        return {"bytes": e * B * D * (2 * Hq * Lq + 2 * Hkv * Lk) + mask, "flops": W.sdpa_flops(B, Hq, Lq, Lk, D, case["mask"] == "causal")}
    Hq, Hkv, D, window = case["heads"], case["kv_heads"], case["size"], case["window"]
    row = W.cache_row_bytes(DTYPES[case["cache"]][0], D)
    tokens = keys = pairs = 0
    for past, new in _sequences(case):
        tokens += new
        # cached rows some new token attends (those of the step's own tokens are written, counted below)
        keys += min(past, window - 1) if window else past
        seen = np.arange(past + 1, past + new + 1)
        pairs += int(np.minimum(seen, window).sum() if window else seen.sum())
    e = DTYPES[case["q"]][1].itemsize
    nbytes = 2 * Hkv * row * (keys + tokens) + e * tokens * D * (2 * Hq + 2 * Hkv)
    flops = 4 * D * Hq * pairs
    if case["path"] == "layer":  # the activations between the operators are not counted
        hidden, ffn = case["hidden"], case["ffn"]
        weights = hidden * (2 * Hq + 2 * Hkv) * D + 3 * hidden * ffn
        nbytes = 2 * Hkv * row * (keys + tokens) + 2 * weights + 2 * 2 * tokens * hidden
        flops += 2 * tokens * weights
    return {"bytes": int(nbytes), "flops": int(flops)}


def tolerance(case):
    """About four times the distance of this framework's outputs from the same path in fp64 on these inputs: rel / max of
    5e-7 / 6e-6 with fp32 operands, 4e-4 / 6e-3 with fp16 ones, 2.7e-3 / 5e-2 where queries or cache are bf16, and
    3.8e-3 / 2e-2 for the layer, whose activations are bf16.  Cache bytes of a u8 cache are exact."""
    if case["path"] == "layer":
        return {"rel": 1.4e-2, "max": 0.1}
    types = (case["dtype"],) if case["path"] == "sdpa" else (case["q"], case["cache"])
    if "f32" in types:
        return {"rel": 2e-6, "max": 3e-5}
    return {"rel": 1e-2, "max": 0.2} if "bf16" in types else {"rel": 1.6e-3, "max": 0.025}


# ------------------------------------------------------------------------------------ prepare
class Buffer:
    """A torch tensor as the bindings take device memory."""

    def __init__(self, tensor):
        self.tensor, self.ptr, self.nbytes = tensor, ctypes.c_void_p(tensor.data_ptr()), tensor.numel() * tensor.element_size()


def _normal(gen, shape, dtype, std=1.0):
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    return (x * std).to(dtype)


def _quantised(x):
    """fp32 [..., size] -> bytes [..., size + 8]: [scale f32][zero-point f32][bytes], the u8 cache's rows."""
    lo, hi = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
    scale = (hi - lo) / 255.0
    zero = -lo / scale
    q = torch.clamp(torch.round(x / scale + zero), 0, 255).to(torch.uint8)
    return torch.cat([scale.view(torch.uint8), zero.view(torch.uint8), q], -1)


def _cache(gen, blocks, case):
    shape = (blocks, case["kv_heads"], case["block"], case["size"])
    if case["cache"] != "u8":
        out = torch.empty(shape, device="cuda", dtype=DTYPES[case["cache"]][1])
        for b in range(0, blocks, 4096):
            out[b:b + 4096] = _normal(gen, (min(4096, blocks - b),) + shape[1:], out.dtype)
        return out
    out = torch.empty(shape[:3] + (case["size"] + 8,), device="cuda", dtype=torch.uint8)
    for b in range(0, blocks, 4096):
        out[b:b + 4096] = _quantised(_normal(gen, (min(4096, blocks - b),) + shape[1:], torch.float32))
    return out


def _paged_inputs(case, gen):
    """Device tensors of a batch: the caches, a block table that scatters every sequence over the pool, lengths."""
    seqs = _sequences(case)
    past = np.array([p for p, _ in seqs], np.int32)
    new = np.array([n for _, n in seqs], np.int32)
    begins = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
    table = np.concatenate([[0], np.cumsum((past.astype(np.int64) + new + case["block"] - 1) // case["block"])]).astype(np.int32)
    blocks = int(table[-1]) + 3
    i32 = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
    positions = np.concatenate([np.arange(p, p + n) for p, n in seqs])
    return dict(tokens=int(begins[-1]), seqs=len(seqs), blocks=blocks, longest=int((past + new).max()), past=i32(past), begins=i32(begins),
                table=torch.randperm(blocks, generator=gen, device="cuda")[:int(table[-1])].to(torch.int32), table_begins=i32(table),
                positions=i32(positions), last_position=int(positions.max()), keys=_cache(gen, blocks, case), values=_cache(gen, blocks, case))


def _prepare_paged(case, gen):
    s = _paged_inputs(case, gen)
    q_code, q_type = DTYPES[case["q"]]
    Hq, Hkv, D, T = case["heads"], case["kv_heads"], case["size"], s["tokens"]
    s["desc"] = capi.PaDesc(q_code, q_code, DTYPES[case["cache"]][0], q_code, Hq, Hkv, D, case["block"], s["blocks"], T, s["seqs"],
                            s["longest"], case["window"], 0.0, 0, 0, None, None)
    s["workspace"] = torch.empty(max(16, capi.paged_attention_workspace_size(s["desc"])), device="cuda", dtype=torch.uint8)
    s["q"], s["k"], s["v"] = (_normal(gen, (T, h * D), q_type) for h in (Hq, Hkv, Hkv))
    s["out"] = torch.empty_like(s["q"])
    order = ("q", "k", "v", "keys", "values", "past", "begins", "table", "table_begins", "out", "workspace")
    s["args"] = [Buffer(s[n]) for n in order]
    return s


def _prepare_sdpa(case, gen):
    code, dtype = DTYPES[case["dtype"]]
    B, Hq, Hkv, Lq, Lk, D = (case[k] for k in ("batch", "heads", "kv_heads", "queries", "keys", "size"))
    s = {"desc": capi.SdpaDesc(code, B, Hq, Hkv, Lq, Lk, D, int(case["mask"] == "causal"), 0.0)}
    s["q"], s["k"], s["v"] = (_normal(gen, (B, h, n, D), dtype, case["std"]) for h, n in ((Hq, Lq), (Hkv, Lk), (Hkv, Lk)))
    s["out"] = torch.empty_like(s["q"])
    s["args"] = [Buffer(s[n]) for n in ("q", "k", "v")]
    s["result"] = Buffer(s["out"])
    if case["mask"] == "padding":  # sentences of a quarter of the length to all of it
        lengths = torch.randint(max(1, Lk // 4), Lk + 1, (B, 1), generator=gen, device="cuda")
        s["mask"] = (torch.arange(Lk, device="cuda")[None, :] < lengths).to(torch.uint8)
        s["mask_args"] = (W.U8, (Lk, 0, 0, 1), Buffer(s["mask"]))
    elif case["mask"] == "bias":
        s["mask"] = _normal(gen, (Lq, Lk), dtype)
        s["mask_args"] = (code, (0, 0, Lk, 1), Buffer(s["mask"]))
    return s


def _prepare_layer(case, gen):
    s = _paged_inputs(case, gen)
    hidden, ffn, Hq, Hkv, D, T = case["hidden"], case["ffn"], case["heads"], case["kv_heads"], case["size"], s["tokens"]
    g = P.GraphText("decoder_layer")
    bound = {}

    def device(name, code, tensor):
        bound[name] = (tensor, code)
        return g.parameter(name, code, list(tensor.shape))

    def weight(name, rows, cols):
        return device(name, W.BF16, _normal(gen, (rows, cols), torch.bfloat16, cols ** -0.5))

    def gamma(name):
        x = 1.0 + 0.1 * torch.randn(hidden, generator=gen, device="cuda")
        return g.constant(name, x.to(torch.bfloat16).view(torch.int16).cpu().numpy(), "bf16")

    def matmul(name, x, w):
        return g.add("MatMul", name, [x, w], transpose_a=False, transpose_b=True)

    x = device("hidden", W.BF16, _normal(gen, (T, hidden), torch.bfloat16))
    angle = torch.arange(s["last_position"] + 1, device="cuda", dtype=torch.float64)[:, None] * (
        10000.0 ** (-torch.arange(0, D, 2, device="cuda", dtype=torch.float64) / D))[None, :]
    cos = device("cos", W.F32, torch.cat([angle.cos(), angle.cos()], 1).float())
    sin = device("sin", W.F32, torch.cat([angle.sin(), angle.sin()], 1).float())
    positions = device("positions", P.I32, s["positions"])
    index = [device(n, P.I32, s[n]) for n in ("past", "begins", "table", "table_begins")]
    host = {"scale": (np.zeros((0,), np.float32), W.F32), "sliding_window": (np.array([case["window"]], np.int32), P.I32),
            "alibi_slopes": (np.zeros((0,), np.float32), W.F32), "max_context_len": (np.array([s["longest"]], np.int32), P.I32)}
    scalars = [g.parameter(n, code, [0] if n == "alibi_slopes" else [-1]) for n, (_, code) in host.items()]
    caches = [device(n, DTYPES[case["cache"]][0], s[n]) for n in ("keys", "values")]
    n1 = g.add("RMS", "norm1", [x, gamma("gamma1")], epsilon=1e-5, output_type="dynamic")
    q, k, v = (matmul(n, n1, weight("w" + n, h * D, hidden)) for n, h in (("q", Hq), ("k", Hkv), ("v", Hkv)))
    rope = dict(head_size=D, rotary_ndims=D, gather_position_arg_id=3)
    q = g.add("RoPE", "rope_q", [q, cos, sin, positions], head_cnt=Hq, **rope)
    k = g.add("RoPE", "rope_k", [k, cos, sin, positions], head_cnt=Hkv, **rope)
    a = g.add("PagedAttentionExtension", "attention", [q, k, v] + caches + index + scalars)
    h1 = g.add("Add", "residual1", [matmul("o", a, weight("wo", hidden, Hq * D)), x])
    n2 = g.add("RMS", "norm2", [h1, gamma("gamma2")], epsilon=1e-5, output_type="dynamic")
    act = g.add("GLU", "glu", [matmul("gate_up", n2, weight("wgu", 2 * ffn, hidden))], axis=-1, split_lengths=ffn, glu_type=0,
                split_to_glu_idx=0, output_type="dynamic")
    g.result("out", g.add("Add", "residual2", [matmul("down", act, weight("wd", hidden, ffn)), h1]))
    plugin = P.Plugin()
    compiled = plugin.compile_model(g.model())
    request = compiled.create_infer_request()
    for i, name in enumerate(compiled.input_names()):
        if name in host:
            request.set_input(i, *host[name])
        else:
            tensor, code = bound[name]
            request.set_device_input(i, tensor.data_ptr(), code, list(tensor.shape))
    s["out"] = torch.empty((T, hidden), device="cuda", dtype=torch.bfloat16)
    request.set_device_output(0, s["out"].data_ptr(), W.BF16, [T, hidden])
    return dict(s, request=request, compiled=compiled, plugin=plugin, bound=bound)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = {"paged": _prepare_paged, "sdpa": _prepare_sdpa, "layer": _prepare_layer}[case["path"]](case, gen)
    return dict(s, path=case["path"])


# ---------------------------------------------------------------------------------------- run
def run(state):
    if state["path"] == "sdpa":
        if "mask" in state:
            capi.sdpa_masked(state["desc"], *state["args"], *state["mask_args"], state["result"])
        else:
            capi.sdpa(state["desc"], *state["args"], state["result"])
        return state["out"]
    if state["path"] == "layer":
        state["request"].infer()
    else:
        capi.paged_attention(state["desc"], *state["args"])
    return state["out"], state["keys"], state["values"]
