"""What the framework is used for, as cases that can be timed.

Five kinds of work, each through the public calls of aq_mi355.Context as a serving program makes them:

  layer  the quantised projections of one decoder layer (q|k|v, o, gate|up with the gated activation, down) for `rows`
         rows of activations: one row is a decode step, 2..64 rows are batched or speculative decoding, more are prefill
  moe    a routed expert block: router, gathered gate|up with the activation, gathered down projection, combine
  head   the lm_head of a decode step: scores, the best 40, temperature / top-p sampling; or greedy tokens of a batch
  load   GGUF blocks turned into affine tensors on the device when a checkpoint is loaded
  host   the plug-in surface that takes host slices (QuantMatVec.MatVec, ProjQuantMatMulInto): weights come from host
         memory at every call

Widths are 4 and 8 bits; groups of 64 are the MLX default, groups of 32 what GGUF checkpoints (Q4_0, Q4_K, Q8_0) become,
groups of 128 the coarser MLX form.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "go-inference_amd"))
import aq_mi355  # noqa: E402

_context = None


def context():
    """One device context for the program, as a server holds it."""
    global _context
    if _context is None:
        _context = aq_mi355.Context(0)
    return _context


def listed():
    return [
        # one token through a narrow layer, call by call: a few MB per projection, so launches and latency are what counts
        dict(name="token_narrow", kind="layer", rows=1, hidden=1536, q=2048, kv=256, ffn=6144, bits=4, group=64, layers=1,
             tiled=False),
        # one token through four layers of the benchmark's size, weights in the layout made at load, the step recorded
        # once and replayed: how a decode loop runs
        dict(name="token_step", kind="layer", rows=1, hidden=4096, q=4096, kv=1024, ffn=14336, bits=4, group=64, layers=4,
             tiled=True),
        # one token through the same layer with 8-bit codes, call by call
        dict(name="token_8bit", kind="layer", rows=1, hidden=4096, q=4096, kv=1024, ffn=14336, bits=8, group=64, layers=1,
             tiled=False),
        # a batch of 21 sequences decoding together on a GGUF-derived layer (groups of 32)
        dict(name="batch_21_group32", kind="layer", rows=21, hidden=3840, q=4096, kv=2048, ffn=15360, bits=4, group=32,
             layers=1, tiled=False),
        # prefill of a long prompt: the benchmark's matmul size
        dict(name="prefill_2048", kind="layer", rows=2048, hidden=4096, q=4096, kv=1024, ffn=14336, bits=4, group=64,
             layers=1, tiled=False),
        # a prompt of 509 tokens on the GGUF-derived layer
        dict(name="prefill_509_group32", kind="layer", rows=509, hidden=3840, q=4096, kv=2048, ffn=15360, bits=4, group=32,
             layers=1, tiled=False),
        # a prompt of 777 tokens on a smaller layer with 8-bit codes
        dict(name="prefill_777_8bit", kind="layer", rows=777, hidden=2560, q=2048, kv=512, ffn=10240, bits=8, group=64,
             layers=1, tiled=False),
        # eight sequences decoding through a block of 128 experts, eight per token
        dict(name="moe_decode", kind="moe", tokens=8, experts=128, top_k=8, hidden=2816, ffn=1408, bits=4, group=64),
        # a prompt of 512 tokens through a block of 128 narrower experts
        dict(name="moe_prefill", kind="moe", tokens=512, experts=128, top_k=8, hidden=2816, ffn=704, bits=4, group=64),
        # the next token of one sequence, sampled from the 40 best of a 262144-word vocabulary
        dict(name="head_sample", kind="head", mode="sample", rows=1, vocab=262144, hidden=1536, bits=4, group=32),
        # a Q4_K tensor of an MLP projection becoming an affine tensor at load
        dict(name="load_q4_k", kind="load", format="Q4_K", rows=15360, cols=3840),
        # one projection over host slices, the contract of QuantMatVec.MatVec
        dict(name="host_matvec", kind="host", rows=1, hidden=2048, out=8192, bits=4, group=64),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], evenly spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(max(round(v / step) * step, math.ceil(lo / step) * step), hi // step * step))


def draw(rng):
    kind = rng.choices(["layer", "moe", "head", "load", "host"], [9, 4, 2, 2, 2])[0]
    bits = rng.choice([4, 4, 4, 8])
    if kind == "layer":
        group = rng.choice([64, 64, 64, 32, 32, 128])
        step = 128 if group == 128 else 64
        hidden = _log(rng, 768, 4096, step)
        c = dict(kind=kind, hidden=hidden, q=_log(rng, 1024, 4096, step), kv=_log(rng, 256, 2048, step),
                 ffn=_log(rng, 1.5 * hidden, min(4 * hidden, 15360), step), bits=bits, group=group)
        # every third is a single token (in half of those cases a recorded step of some layers), the others spread from
        # a pair of rows to a long prompt, at most the work of the listed prompts
        weights = hidden * (2 * c["q"] + 2 * c["kv"] + 3 * c["ffn"])
        most = 509 * 224_000_000 if group == 32 else 2048 * 218_000_000
        c["rows"] = 1 if rng.random() < 0.34 else _log(rng, 2, min(509 if group == 32 else 2048, most // weights))
        c["layers"] = rng.randint(2, 4) if c["rows"] == 1 and rng.random() < 0.5 else 1
        c["tiled"] = bool(c["layers"] > 1 and bits == 4 and group == 64 and not any(c[k] % 128 for k in ("hidden", "q", "ffn")))
        return c
    if kind == "moe":
        group = rng.choice([64, 64, 64, 32])
        # decode batches and prompts; expert sizes from narrow to the benchmark's
        c = dict(kind=kind, tokens=_log(rng, 1, 512), experts=rng.choice([16, 32, 64, 128]), top_k=rng.choice([2, 4, 8]),
                 hidden=_log(rng, 1024, 2816, 64), bits=bits, group=group)
        c["ffn"] = _log(rng, 512, 1408 if c["tokens"] < 128 else 704, 64)
        return c
    if kind == "head":
        mode = rng.choice(["sample", "greedy"])
        return dict(kind=kind, mode=mode, rows=1 if mode == "sample" else _log(rng, 1, 16), vocab=_log(rng, 32000, 262144),
                    hidden=_log(rng, 1024, 2560, 128), bits=bits, group=rng.choice([32, 64]))
    if kind == "load":
        return dict(kind=kind, format=rng.choice(["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"]), rows=_log(rng, 1024, 65536),
                    cols=_log(rng, 1024, 8192, 256))
    return dict(kind=kind, rows=rng.choice([1, _log(rng, 2, 256)]), hidden=_log(rng, 512, 4096, 64),
                out=_log(rng, 512, 14336, 8), bits=bits, group=rng.choice([32, 64]))


# ---- inputs ---------------------------------------------------------------------------------------------------------

class _Maker:
    """Seeded tensors of the distributions the benchmark states."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, dtype=torch.bfloat16, scale=1.0):
        return (torch.randn(*shape, generator=self.g, device="cuda") * scale).to(dtype)

    def words(self, n, k, bits):
        return torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k * bits // 32), generator=self.g, device="cuda", dtype=torch.int32)

    def affine(self, n, k, bits, group):
        """Packed codes, scales and biases of an [n, k] affine tensor: uniform codes, small scales, centred weights."""
        spread = 1.0 if bits == 4 else 1.0 / 16
        s = (torch.randn(n, k // group, generator=self.g, device="cuda").abs() * 0.02 + 1e-3) * spread
        s = s.to(torch.bfloat16)
        b = (s.float() * -(1 << (bits - 1)) + torch.randn(n, k // group, generator=self.g, device="cuda") * 1e-3)
        return self.words(n, k, bits), s, b.to(torch.bfloat16)


def _p(t):
    return t.data_ptr() if isinstance(t, torch.Tensor) else t


class _Graph:
    def __init__(self, ctx, handle):
        self.ctx, self.handle = ctx, handle

    def __del__(self):
        self.ctx.graph_destroy(self.handle)


_GGUF = {  # tensor type, bytes per block, columns per block, byte offsets of the block's half-precision factors
    "Q4_0": (aq_mi355.GGUF_Q4_0, 18, 32, (0,)),
    "Q8_0": (aq_mi355.GGUF_Q8_0, 34, 32, (0,)),
    "Q4_K": (aq_mi355.GGUF_Q4_K, 144, 256, (0, 2)),
    "Q5_K": (aq_mi355.GGUF_Q5_K, 176, 256, (0, 2)),
    "Q6_K": (aq_mi355.GGUF_Q6_K, 210, 256, (208,)),
}


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, _Maker(seed), seed)


def _prepare_layer(c, make, seed):
    ctx, M, H, F = context(), c["rows"], c["hidden"], c["ffn"]
    bits, group = c["bits"], c["group"]
    shapes = {"q": (c["q"], H), "k": (c["kv"], H), "v": (c["kv"], H), "o": (H, c["q"]), "gate": (F, H), "up": (F, H),
              "down": (H, F)}
    layers = []
    for _ in range(c["layers"]):
        w = {name: make.affine(n, k, bits, group) for name, (n, k) in shapes.items()}
        torch.cuda.synchronize()
        if c["tiled"]:
            flat = {name: tuple(t.data_ptr() for t in w[name]) for name in w}
            tiled = {name: ctx.tile_weights(*flat[name], *shapes[name], group, bits) for name in w}
            ctx.sync()
            w = {name: (tiled[name], None, None) for name in w}
        layers.append(w)
    s = dict(kind="layer", case=c, layers=layers, flags=aq_mi355.AQ_W_TILED if c["tiled"] else 0, graph=None)
    # the activations that the rest of the model hands to each projection
    s["x"], s["attn"], s["h"] = make.normal(M, H), make.normal(M, c["q"]), make.normal(M, H)
    out = {name: torch.empty(M, n, device="cuda", dtype=torch.bfloat16) for name, (n, _) in shapes.items() if name != "up"}
    s["outs"] = [out] + [{name: torch.empty_like(t) for name, t in out.items()} for _ in layers[1:]]
    if c["layers"] > 1:
        # a decode loop records its step once and replays it
        torch.cuda.synchronize()
        _run_layers(ctx, s)
        ctx.sync()
        ctx.capture_begin()
        _run_layers(ctx, s)
        s["graph"] = _Graph(ctx, ctx.capture_end())
    return s


def _run_layers(ctx, s):
    c = s["case"]
    M, H, Q, KV, F, bits, group, flags = (c["rows"], c["hidden"], c["q"], c["kv"], c["ffn"], c["bits"], c["group"], s["flags"])
    x, attn, h = s["x"].data_ptr(), s["attn"].data_ptr(), s["h"].data_ptr()
    # up to 64 rows are decoding (matvec calls), more are prefill (matmul calls)
    few = M <= 64
    multi, one = (ctx.qmv_multi, ctx.qmv) if few else (ctx.qmm_multi, ctx.qmm)
    for w, y in zip(s["layers"], s["outs"]):
        y = {name: t.data_ptr() for name, t in y.items()}
        w = {name: tuple(_p(t) for t in arrays) for name, arrays in w.items()}
        qkv = (w["q"], w["k"], w["v"])
        multi(x, [t[0] for t in qkv], [t[1] for t in qkv], [t[2] for t in qkv], [y["q"], y["k"], y["v"]], [Q, KV, KV], M, H,
              group, bits, flags)
        one(attn, *w["o"], y["o"], M, Q, H, group, bits, flags)
        ctx.qmv_gate_up(h, w["gate"], w["up"], y["gate"], M, H, F, group, bits, aq_mi355.AQ_ACT_GELU_TANH, flags)
        one(y["gate"], *w["down"], y["down"], M, F, H, group, bits, flags)


def _prepare_moe(c, make, seed):
    T, E, k, H, F = c["tokens"], c["experts"], c["top_k"], c["hidden"], c["ffn"]
    routes = T * k
    s = dict(kind="moe", case=c, gate_up=make.affine(E * 2 * F, H, c["bits"], c["group"]),
             down=make.affine(E * H, F, c["bits"], c["group"]), x=make.normal(T, H),
             logits=make.normal(T, E, dtype=torch.float32, scale=1.5), iota=torch.arange(routes, device="cuda", dtype=torch.int32))
    for name, shape, dtype in (("ids", (T, k), torch.int32), ("token", (T, k), torch.int32), ("weights", (T, k), torch.float32),
                               ("gated", (routes, F), torch.bfloat16), ("rows", (routes, H), torch.bfloat16),
                               ("out", (T, H), torch.bfloat16)):
        s[name] = torch.empty(*shape, device="cuda", dtype=dtype)
    return s


def _prepare_head(c, make, seed):
    M = c["rows"]
    s = dict(kind="head", case=c, w=make.affine(c["vocab"], c["hidden"], c["bits"], c["group"]), x=make.normal(M, c["hidden"]),
             draw=float(np.random.default_rng(seed).random()))
    s["scores"] = torch.empty(c["vocab"] if c["mode"] == "sample" else 1, device="cuda", dtype=torch.int64)
    s["top"] = torch.empty(40, device="cuda", dtype=torch.int64)
    s["best"] = torch.empty(M, device="cuda", dtype=torch.int64)
    return s


def _prepare_load(c, make, seed):
    kind, nbytes, ncols, factors = _GGUF[c["format"]]
    blocks = c["rows"] * c["cols"] // ncols
    src = torch.randint(0, 256, (blocks, nbytes), generator=make.g, device="cuda", dtype=torch.uint8)
    for at in factors:  # the blocks' scales: small positive halves
        d = (torch.rand(blocks, 1, generator=make.g, device="cuda") * 0.01 + 1e-4).to(torch.float16)
        src[:, at:at + 2] = d.view(torch.uint8)
    lay = aq_mi355.gguf_affine_layout(kind, c["rows"], c["cols"])
    empty = lambda n: torch.empty(n, device="cuda", dtype=torch.int16)  # noqa: E731
    return dict(kind="load", case=c, type=kind, src=src, packed=empty(lay.packed_bytes // 2), scales=empty(lay.scales_bytes // 2),
                biases=empty(lay.scales_bytes // 2))


def _prepare_host(c, make, seed):
    M, K, N = c["rows"], c["hidden"], c["out"]
    w, sc, bi = make.affine(N, K, c["bits"], c["group"])
    bits16 = lambda t: t.view(torch.int16).cpu().numpy().view(np.uint16)  # noqa: E731
    s = dict(kind="host", case=c, w=w.cpu().numpy(), scales=bits16(sc), biases=bits16(bi))
    x = make.normal(M, K, dtype=torch.float32)
    s["x"] = bits16(x.to(torch.bfloat16)) if M == 1 else x.cpu().numpy()
    return s


# ---- one pass -------------------------------------------------------------------------------------------------------

def run(state):
    return globals()["_run_" + state["kind"]](context(), state)


def _run_layer(ctx, s):
    if s["graph"] is not None:
        ctx.graph_launch(s["graph"].handle)
    else:
        _run_layers(ctx, s)
    return s["outs"]


def _run_moe(ctx, s):
    c = s["case"]
    T, E, k, H, F, bits, group = c["tokens"], c["experts"], c["top_k"], c["hidden"], c["ffn"], c["bits"], c["group"]
    routes = T * k
    at = {name: t.data_ptr() for name, t in s.items() if isinstance(t, torch.Tensor)}
    gate_up, down = (tuple(t.data_ptr() for t in s[name]) for name in ("gate_up", "down"))
    ctx.moe_route(at["logits"], T, E, k, at["ids"], at["weights"], at["token"])
    ctx.gather_qmv_gate_up(at["x"], *gate_up, at["token"], at["ids"], at["gated"], routes, T, H, F, E, 2 * F, 0, F, group, bits)
    ctx.gather_qmv(at["gated"], *down, at["iota"], at["ids"], at["rows"], routes, routes, F, H, E, H, 0, group, bits)
    ctx.moe_combine(at["rows"], at["weights"], at["out"], T, k, H)
    return s["out"], s["ids"], s["weights"]


def _run_head(ctx, s):
    c = s["case"]
    w = tuple(t.data_ptr() for t in s["w"])
    x, best = s["x"].data_ptr(), s["best"].data_ptr()
    if c["mode"] == "greedy":
        ctx.qmv_greedy(x, *w, best, c["rows"], c["hidden"], c["vocab"], c["group"], c["bits"])
        packed = (s["best"],)
    else:
        ctx.qmv_scores(x, *w, s["scores"].data_ptr(), 1, c["hidden"], c["vocab"], c["group"], c["bits"])
        ctx.packed_topk(s["scores"].data_ptr(), c["vocab"], 40, s["top"].data_ptr())
        ctx.packed_topk_sample(s["top"].data_ptr(), 40, 0.8, 0.95, 30.0, s["draw"], best)
        packed = (s["top"], s["best"])
    # a packed value holds the token (complemented) in its low word; its high word, the order-preserving key of the score,
    # has the bits of minus the score where the score is positive, as the best ones are
    return [(t.view(torch.int32)[0::2], t.view(torch.float32)[1::2]) for t in packed]


def _run_load(ctx, s):
    c, src = s["case"], s["src"]
    ctx.gguf_to_affine(s["type"], src.data_ptr(), src.numel(), c["rows"], c["cols"], s["packed"].data_ptr(), s["scales"].data_ptr(),
                       s["biases"].data_ptr())
    return s["packed"], s["scales"], s["biases"]


def _run_host(ctx, s):
    c = s["case"]
    if c["rows"] == 1:
        y = ctx.matvec_host(s["x"], s["w"], s["scales"], s["biases"], c["out"], c["hidden"], c["group"], c["bits"])
        return torch.from_numpy(y).view(torch.bfloat16)
    return ctx.proj_quant_matmul_host(s["x"], s["w"], s["scales"], s["biases"], c["rows"], c["hidden"], c["out"], c["group"], c["bits"])


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def _weight_bytes(n, k, bits, group):
    return n * k * bits / 8 + 2 * n * (k // group) * 2


def work(case):
    c, kind = case, case["kind"]
    if kind == "layer":
        M, H, Q, KV, F = c["rows"], c["hidden"], c["q"], c["kv"], c["ffn"]
        shapes = [(Q, H), (KV, H), (KV, H), (H, Q), (F, H), (F, H), (H, F)]
        weights = sum(_weight_bytes(n, k, c["bits"], c["group"]) for n, k in shapes)
        # x, the attention's output and the MLP's input in; q, k, v, o, the gated values (also read again) and down out
        acts = 2 * M * (H + Q + H + Q + 2 * KV + H + 2 * F + H)
        return {"bytes": c["layers"] * (weights + acts), "flops": c["layers"] * 2.0 * M * sum(n * k for n, k in shapes)}
    if kind == "moe":
        T, E, k, H, F = c["tokens"], c["experts"], c["top_k"], c["hidden"], c["ffn"]
        distinct = E * (1 - (1 - k / E) ** T)
        expert = _weight_bytes(2 * F, H, c["bits"], c["group"]) + _weight_bytes(H, F, c["bits"], c["group"])
        acts = 4 * T * E + 2 * T * H + 2 * T * k * (2 * F + 2 * H) + 2 * T * H
        return {"bytes": distinct * expert + acts, "flops": 2.0 * T * k * 3 * H * F}
    if kind == "head":
        M, N, K = c["rows"], c["vocab"], c["hidden"]
        scores = 2 * 8 * N if c["mode"] == "sample" else 8 * M
        return {"bytes": _weight_bytes(N, K, c["bits"], c["group"]) + 2 * M * K + scores, "flops": 2.0 * M * N * K}
    if kind == "load":
        lay = aq_mi355.gguf_affine_layout(_GGUF[c["format"]][0], c["rows"], c["cols"])
        return {"bytes": lay.src_bytes + lay.packed_bytes + 2 * lay.scales_bytes, "flops": 0}
    M, K, N = c["rows"], c["hidden"], c["out"]
    wide = 2 if M == 1 else 4
    return {"bytes": _weight_bytes(N, K, c["bits"], c["group"]) + wide * M * (K + N), "flops": 2.0 * M * N * K}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"
    if case["kind"] == "head":
        return {"rel": 1e-5, "max": 1e-4}  # tokens as they are, scores as fp32 sums in another order
    # bf16 results: another order of the fp32 sums moves some values to the neighbouring bf16, and the down projection
    # reads such values
    return {"rel": 5e-3, "max": 0.03}
