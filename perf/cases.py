"""The workloads by which this library's speed is measured.

Each case is work that a program running a quantized Qwen3-like model has the library do
through ``dyninfer_amd.Context``: single linears, a decode step captured once as a HIP
graph and replayed (the form serving programs run it in), the matmuls of one layer over a
prompt chunk (issued eagerly, as prompts differ in length), and the embedding gather.
Sizes are those of the repository's benchmark (the 0.6B and 8B decode steps, 512-token
prompt chunks) and ragged ones between.  Weights are random blocks in the on-disk layouts
with scales of the size trained weights have; activations are normal with a few large
channels, as a norm's output has.
"""
from __future__ import annotations

import math

import torch

import dyninfer_amd as d

# (weights per block, bytes per block) of the GGUF layouts
BLOCK = {"q4_0": (32, 18), "q4_1": (32, 20), "q8_0": (32, 34), "q6_k": (256, 210), "q4_k": (256, 144),
         "q5_k": (256, 176), "iq4_xs": (256, 136)}
GROUP = 64  # scale group of the MLX weights

SIZE_06B = dict(hidden=1024, q=2048, kv=1024, ffn=3072)
SIZE_8B = dict(hidden=4096, q=4096, kv=1024, ffn=12288)
VOCAB = 151936


def listed():
    return [
        # One small linear called by itself at one row: the latency of a single call.
        dict(name="linear_1row", kind="linear", enc="q4_0", rows=1, n=3072, k=1024, count=1, io="f32"),
        # The token embeddings of a 512-token prompt chunk (a tied 0.6B table).
        dict(name="embed_512", kind="embed", enc="q6_k", ids=512, n=VOCAB, k=1024),
        # Decode steps, all layers and the output head, as a captured graph.  One sequence on the
        # small model in its mixed encoding: over a hundred launches of one to four megabytes.
        dict(name="step_06b_mixed_1", kind="step", mix="mixed", rows=1, layers=28, vocab=VOCAB, io="f32", **SIZE_06B),
        # The small model in MLX form serving eight sequences, bf16 activations.
        dict(name="step_06b_mlx_8", kind="step", mix="mlx", rows=8, layers=28, vocab=VOCAB, io="bf16", **SIZE_06B),
        # One sequence on the 8B model (Q4_0 with Q6_K): the weight stream itself.
        dict(name="step_8b_q4_0_1", kind="step", mix="q4_0", rows=1, layers=36, vocab=VOCAB, io="f32", **SIZE_8B),
        # Four sequences on the 8B model in the common K-quant mix.
        dict(name="step_8b_q4km_4", kind="step", mix="q4_k_m", rows=4, layers=36, vocab=VOCAB, io="f32", **SIZE_8B),
        # Sixteen sequences on the 8B model.
        dict(name="step_8b_q4_0_16", kind="step", mix="q4_0", rows=16, layers=36, vocab=VOCAB, io="f32", **SIZE_8B),
        # A short ragged prompt (45 tokens) through one 8B layer in the five-bit K-quant.
        dict(name="prompt_45_8b_q5k", kind="layer", mix="q5_k", rows=45, io="f32", **SIZE_8B),
        # A ragged prompt (333 tokens) through one layer of the small MLX model.
        dict(name="prompt_333_06b_mlx", kind="layer", mix="mlx", rows=333, io="bf16", **SIZE_06B),
        # A full 512-token chunk through one layer of the small model.
        dict(name="prompt_512_06b_mixed", kind="layer", mix="mixed", rows=512, io="f32", **SIZE_06B),
        # A full chunk through one 8B layer of the K-quant mix, bf16 activations.
        dict(name="prompt_512_8b_q4km", kind="layer", mix="q4_k_m", rows=512, io="bf16", **SIZE_8B),
        # A long prompt in one call per linear through one 8B layer.
        dict(name="prompt_2048_8b_q4_0", kind="layer", mix="q4_0", rows=2048, io="f32", **SIZE_8B),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` in lo..hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "step", "layer", "layer", "embed"])
    if kind == "embed":
        return dict(kind=kind, enc=rng.choice(sorted(BLOCK) + ["mlx_u4"]), ids=_log(rng, 1, 4096),
                    n=_log(rng, 1000, VOCAB), k=_log(rng, 512, 4096, 256))
    io = rng.choice(["f32", "bf16"])
    if kind == "linear":
        enc = rng.choice(sorted(BLOCK) + ["mlx_u4"])
        step = 256 if enc.endswith("_k") or enc == "iq4_xs" else GROUP
        c = dict(kind=kind, enc=enc, rows=_log(rng, 1, 2048), n=_log(rng, 200, 16384), k=_log(rng, 512, 12288, step),
                 count=rng.choice([1, 1, 2, 3]), io=io)
        if rng.random() < 0.4:  # decode rows as often as prompts
            c["rows"] = rng.randint(1, 16)
        c["rows"] = min(c["rows"], int(3e11 / (c["n"] * c["k"])))
        c["count"] = max(1, min(c["count"], int(3e11 / (2.0 * c["rows"] * c["n"] * c["k"]))))
        return c
    size = dict(hidden=_log(rng, 512, 4096, 256), q=_log(rng, 512, 4096, 256), kv=_log(rng, 256, 1024, 128),
                ffn=_log(rng, 1024, 12288, 256))
    mix = rng.choice(["mixed", "mlx", "q4_0", "q4_k_m", "q5_k", "iq4_xs"])
    if kind == "step":
        return dict(kind=kind, mix=mix, rows=_log(rng, 1, 16), layers=rng.randint(2, 12), vocab=_log(rng, 2000, 50000),
                    io=io, **size)
    return dict(kind=kind, mix=mix, rows=_log(rng, 17, 2048), io=io, **size)


# ------------------------------------------------------------------ weights and activations
def _weight(enc, n, k, gen):
    def f16(count, scale, signed=False):
        v = torch.randn(count, device="cuda", generator=gen)
        return ((v if signed else 0.5 + 0.25 * v.abs()) * scale).half().view(torch.uint8).view(count, 2)

    if enc == "mlx_u4":
        g = n * (k // GROUP)
        words = torch.randint(0, 256, (n * k // 2,), dtype=torch.uint8, device="cuda", generator=gen).view(torch.int32)
        scales = ((0.5 + 0.25 * torch.randn(g, device="cuda", generator=gen).abs()) * 0.006).bfloat16()
        biases = (scales.float() * -7.5 * (1 + 0.1 * torch.randn(g, device="cuda", generator=gen))).bfloat16()
        return d.QWeight(d.ENC_MLX_U4, n, k, words, scales, biases, GROUP, d.DTYPE_BF16)
    bw, bb = BLOCK[enc]
    nb = n * (k // bw)
    b = torch.randint(0, 256, (nb, bb), dtype=torch.uint8, device="cuda", generator=gen)
    if enc == "q6_k":
        b[:, 208:210] = f16(nb, 4e-5)
    elif enc in ("q4_k", "q5_k"):
        b[:, 0:2] = f16(nb, 2e-4 if enc == "q4_k" else 1e-4)
        b[:, 2:4] = f16(nb, 1.5e-3)
    elif enc == "iq4_xs":
        b[:, 0:2] = f16(nb, 3e-5)
    elif enc == "q8_0":
        b[:, 0:2] = f16(nb, 4e-4)
    else:
        b[:, 0:2] = f16(nb, 6e-3)
        if enc == "q4_1":
            b[:, 2:4] = f16(nb, 4e-2, signed=True)
    return d.QWeight(getattr(d, "ENC_" + enc.upper()), n, k, b.view(-1))


def _activation(rows, k, io, gen):
    x = torch.randn(rows, k, device="cuda", generator=gen)
    loud = torch.randint(0, k, (max(1, k // 256),), device="cuda", generator=gen)
    x[:, loud] *= 12.0
    return x.bfloat16() if io == "bf16" else x


def _launches(case):
    """(encoding, [(role, N)], K, activation) of each call of the case, in order, with its layer."""
    if case["kind"] == "linear":
        return [(0, case["enc"], [("y%d" % i, case["n"]) for i in range(case["count"])], case["k"], "h")]
    h, q, kv, f = case["hidden"], case["q"], case["kv"], case["ffn"]
    out = []
    for layer in range(case.get("layers", 1)):
        mix = case["mix"]
        main = {"mixed": ("q4_0", "q4_1")[layer % 2], "mlx": "mlx_u4", "q4_k_m": "q4_k"}.get(mix, mix)
        down = {"q4_0": "q6_k", "mixed": "q8_0", "q4_k_m": ("q6_k", "q4_k")[layer % 2]}.get(mix, main)
        down = "q4_0" if down == "q6_k" and f % 256 else down
        if mix == "q4_k_m":
            out.append((layer, main, [("q", q), ("k", kv)], h, "h"))
            out.append((layer, "q6_k", [("v", kv)], h, "h"))
        else:
            out.append((layer, main, [("q", q), ("k", kv), ("v", kv)], h, "h"))
        out.append((layer, main, [("o", h)], q, "attn"))
        out.append((layer, main, [("gate", f), ("up", f)], h, "h"))
        out.append((layer, down, [("down", h)], f, "act"))
    if case.get("vocab"):
        out.append((0, "mlx_u4" if case["mix"] == "mlx" else "q6_k", [("logits", case["vocab"])], h, "h"))
    return out


class _State:
    pass


def _make(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    s = _State()
    s.kind = case["kind"]
    if s.kind == "embed":
        s.w = _weight(case["enc"], case["n"], case["k"], gen)
        s.ids = torch.randint(0, case["n"], (case["ids"],), device="cuda", generator=gen)
        s.out = torch.empty(case["ids"], case["k"], device="cuda")
        return s
    s.x, s.y, s.calls = {}, {}, []
    ydt = torch.bfloat16 if case["io"] == "bf16" else torch.float32
    launches = _launches(case)
    layers = {}
    for layer, _, outs, _, _ in launches:
        for role, n in outs:
            layers[role] = (max(layer + 1, layers.get(role, (0, 0))[0]), n)
    for role, (count, n) in layers.items():  # every layer's outputs, one buffer for each kind of linear
        s.y[role] = torch.empty(count, case["rows"], n, device="cuda", dtype=ydt)
    for layer, enc, outs, k, act in launches:
        if act not in s.x:
            s.x[act] = _activation(case["rows"], k, case["io"], gen)
        ws = [_weight(enc, n, k, gen) for _, n in outs]
        s.calls.append((ws, s.x[act], [s.y[role][layer] for role, _ in outs]))
    return s


def prepare(case, seed):
    s = _make(case, seed)
    s.ctx = d.Context(0)
    if s.kind == "embed":
        return s
    code = d.DTYPE_BF16 if case["io"] == "bf16" else d.DTYPE_F32
    need = max(d.prefill_workspace_bytes(ws, case["rows"], code, code) for ws, _, _ in s.calls)
    s.work = torch.empty(need, dtype=torch.uint8, device="cuda") if need else None
    if s.kind == "step":  # a serving program captures its step once and replays it for every token
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _issue(s)
        side.synchronize()
        s.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s.graph, stream=side):
            _issue(s)
        torch.cuda.synchronize()
        for y in s.y.values():
            y.zero_()
    return s


def _issue(s):
    for ws, x, ys in s.calls:
        if len(ws) == 1:
            s.ctx.qlinear(ws[0], x, ys[0], workspace=s.work)
        else:
            s.ctx.qlinear_multi(ws, x, ys, workspace=s.work)


def run(s):
    if s.kind == "embed":
        return s.ctx.embedding(s.w, s.ids, s.out)
    if s.kind == "step":
        s.graph.replay()
    else:
        _issue(s)
    return s.y


# ------------------------------------------------------------------ what a pass cannot do without
def _bytes(enc, n, k):
    if enc == "mlx_u4":
        return n * k // 2 + 2 * n * (k // GROUP) * 2
    bw, bb = BLOCK[enc]
    return n * (k // bw) * bb


def work(case):
    if case["kind"] == "embed":
        return {"bytes": case["ids"] * (_bytes(case["enc"], 1, case["k"]) + 4 * case["k"] + 8),
                "flops": 2 * case["ids"] * case["k"]}
    es = 2 if case["io"] == "bf16" else 4
    total, flops, acts = 0, 0, {}
    for _, enc, outs, k, act in _launches(case):
        acts[act] = case["rows"] * k * es
        for _, n in outs:
            total += _bytes(enc, n, k) + case["rows"] * n * es
            flops += 2 * case["rows"] * n * k
    return {"bytes": total + sum(acts.values()), "flops": flops}


def tolerance(case):
    if case["kind"] == "embed":
        return "exact"
    # Activations (and from a few rows on, weights) are rounded to f16 once: measured 2e-4 to 4e-4
    # against 64 bits with f32 outputs, 1.7e-3 where the outputs are rounded to bf16.
    return {"rel": 7e-3} if case["io"] == "bf16" else {"rel": 1.5e-3}


# ------------------------------------------------------------------ the results in 64 bits
def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _nibbles(b):
    return torch.cat([b & 15, b >> 4], -1).double()


_IQ4 = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _dense(w, enc, lo, hi):
    """Rows lo..hi of a weight in 64 bits, from its bytes."""
    n, k = hi - lo, w.cols
    if enc == "mlx_u4":
        b = w.data.view(torch.uint8).view(w.rows, k // 2)[lo:hi]
        q = torch.stack([b & 15, b >> 4], -1).reshape(n, k // GROUP, GROUP).double()
        sc = w.scales.view(w.rows, -1)[lo:hi].double()[..., None]
        return (q * sc + w.biases.view(w.rows, -1)[lo:hi].double()[..., None]).reshape(n, k)
    bw, bb = BLOCK[enc]
    b = w.data.view(w.rows, k // bw, bb)[lo:hi].reshape(-1, bb)
    dd = _f16(b[:, 208:210] if enc == "q6_k" else b[:, 0:2])
    if enc == "q4_0":
        v = (_nibbles(b[:, 2:]) - 8) * dd
    elif enc == "q4_1":
        v = _nibbles(b[:, 4:]) * dd + _f16(b[:, 2:4])
    elif enc == "q8_0":
        v = b[:, 2:].contiguous().view(torch.int8).double() * dd
    elif enc == "q6_k":
        ql, qh = b[:, :128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)
        high = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        v = ((low | (high << 4)).double() - 32).view(-1, 16, 16) * (sc * dd)[..., None]
    elif enc == "iq4_xs":
        ib = torch.arange(8, device=b.device)
        high = b[:, 2:3].int() | (b[:, 3:4].int() << 8)
        ls = ((b[:, 4:8].int()[:, ib // 2] >> (4 * (ib % 2))) & 15) | (((high >> (2 * ib)) & 3) << 4)
        qs = b[:, 8:].view(-1, 8, 16)
        v = torch.tensor(_IQ4, device=b.device, dtype=torch.float64)[torch.cat([qs & 15, qs >> 4], -1).long()]
        v = v * ((ls - 32).double() * dd)[..., None]
    else:
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, -128:].view(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32)
        if enc == "q5_k":
            q = q | (torch.stack([(b[:, 16:48] >> i) & 1 for i in range(8)], 1) << 4)
        v = q.double() * (sc * dd)[..., None] - (mn * _f16(b[:, 2:4]))[..., None]
    return v.reshape(n, k)


def exact(case, seed):
    s = _make(case, seed)
    if s.kind == "embed":
        out = torch.empty(case["ids"], case["k"], device="cuda", dtype=torch.float64)
        for i, row in enumerate(s.ids.tolist()):
            out[i] = _dense(s.w, case["enc"], row, row + 1)[0]
        return out
    y = {role: torch.empty(t.shape, dtype=torch.float64, device="cuda") for role, t in s.y.items()}
    for (ws, x, _), (layer, enc, outs, _, _) in zip(s.calls, _launches(case)):
        x64 = x.double()
        for w, (role, n) in zip(ws, outs):
            for lo in range(0, n, 8192):
                hi = min(n, lo + 8192)
                y[role][layer][:, lo:hi] = x64 @ _dense(w, enc, lo, hi).t().contiguous()
    return y
