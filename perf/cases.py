"""The work a program has this framework do, as cases that can be timed and compared: decode steps through stacks and
layers of routed experts, prefill and batched-decode chunks, the drop-in block and dense calls, and the trunk's 4-bit
products. Experts are Gaussian weights quantized to ggml blocks by plain torch, so that `exact` needs nothing of this
package; activations are Gaussian, routing comes from a router weight or from skewed logits.

Kinds (key "kind") and the entry points they pass through:
  stack    layer.DecodeStack, captured once as a program would, one step a pass
  layer    layer.decode of 1-16 tokens through one layer, launched eagerly (a speculative decoder's verify rows)
  prefill  grouped.prefill of a chunk or a batch of tokens through one layer
  block    route.probs -> gguf_experts.experts -> trunk.shared_expert_rows -> route.tail: the drop-in calls of one block
  dense    gguf_experts.dense: rows of one slot each, unweighted, any ggml types
  qmv      trunk.qmv_rows: the trunk's 4-bit affine product
"""
import math

import torch

from larder_amd import gguf_experts, grouped, layer, route, trunk

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
# (weights a block, bytes a block) of the ggml types
BLOCK = {"Q4_0": (32, 18), "Q4_1": (32, 20), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q5_K": (256, 176),
         "Q6_K": (256, 210)}
# layer shapes: hidden, experts, picks, width, shared width (0: none), renormalised
SHAPES = {
    "e60": dict(H=2048, E=60, k=4, I=1408, Is=5632, norm=False),
    "e128": dict(H=2048, E=128, k=8, I=768, Is=0, norm=True),
    "e256": dict(H=2048, E=256, k=8, I=512, Is=512, norm=True),
    "e512": dict(H=4096, E=512, k=10, I=512, Is=512, norm=True),
}


def listed():
    return [
        # one token of a chat through the 48-layer model, everything resident: the headline of a serving process
        dict(name="decode_48_layers", kind="stack", shape="e128", types="Q4_0/Q4_0/Q4_0", layers=48, T=1, dtype="f16"),
        # one token through layers of many small Q4_K experts and a shared one
        dict(name="decode_q4_k_shared", kind="stack", shape="e512", types="Q4_K/Q4_K/Q4_K", layers=4, T=1, dtype="f16"),
        # one token's block by the drop-in calls: the smallest work, launches and latency
        dict(name="block_one_token", kind="block", shape="e256", types="Q4_0/Q4_0/Q4_0", T=1),
        # a speculative decoder's verify rows through a layer with a wide shared expert
        dict(name="verify_5_rows", kind="layer", shape="e60", types="Q4_0/Q4_0/Q4_0", T=5, dtype="f16"),
        # the widest decode pass, of the usual k-quant mix
        dict(name="decode_16_rows_mix", kind="layer", shape="e256", types="Q4_K/Q4_K/Q6_K", T=16, dtype="bf16"),
        # continuous batching: 64 sequences, one token each, experts picked unevenly
        dict(name="batch_64", kind="prefill", shape="e128", types="Q4_0/Q4_0/Q4_0", T=64, dtype="f16", routing="zipf"),
        # a short, odd prompt through a layer with a shared expert, routed by the layer itself
        dict(name="prompt_333", kind="prefill", shape="e60", types="Q4_0/Q4_0/Q4_0", T=333, dtype="bf16",
             routing="router"),
        # a prompt chunk over many experts: few rows each
        dict(name="prompt_2048_q4_k", kind="prefill", shape="e512", types="Q4_K/Q4_K/Q4_K", T=2048, dtype="bf16",
             routing="router"),
        # a full prompt chunk
        dict(name="prompt_8192", kind="prefill", shape="e128", types="Q4_0/Q4_0/Q4_0", T=8192, dtype="bf16",
             routing="skewed"),
        # the drop-in's prompt path (2,048 tokens' picks) on the usual k-quant mix
        dict(name="dense_16384_mix", kind="dense", shape="e128", types="Q4_K/Q4_K/Q6_K", rows=16384, dtype="bf16"),
        # the same on 8-bit experts, fewer and an odd number of rows
        dict(name="dense_3001_q8_0", kind="dense", shape="e60", types="Q8_0/Q8_0/Q8_0", rows=3001, dtype="bf16"),
        # a token's logits over the vocabulary, and the widest trunk product
        dict(name="vocabulary_1_row", kind="qmv", K=2048, N=248320, G=64, T=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["stack", "layer", "prefill", "prefill", "block", "dense", "qmv"])
    if kind == "stack":
        shape = rng.choice(["e60", "e128", "e256", "e512"])
        t = rng.choice(["Q4_0/Q4_0/Q4_0", "Q4_K/Q4_K/Q4_K", "Q4_K/Q4_K/Q6_K"])
        t = "Q4_0/Q4_0/Q4_0" if shape == "e60" else t
        most = 4 if shape == "e512" else 24
        return dict(kind=kind, shape=shape, types=t, layers=rng.randint(most // 4, most), T=rng.choice([1, 1, 1, 2, 3]),
                    dtype=rng.choice(["f16", "bf16"]))
    if kind == "layer":
        shape = rng.choice(["e60", "e128", "e256", "e512"])
        t = rng.choice(["Q4_0/Q4_0/Q4_0", "Q4_K/Q4_K/Q4_K", "Q4_K/Q4_K/Q6_K", "Q4_0/Q4_0/Q8_0", "Q6_K/Q6_K/Q6_K"])
        if shape == "e60":
            t = "Q4_0/Q4_0/Q8_0" if t == "Q4_0/Q4_0/Q8_0" else "Q4_0/Q4_0/Q4_0"
        return dict(kind=kind, shape=shape, types=t, T=rng.randint(1, 16), dtype=rng.choice(["f16", "bf16", "f32"]))
    if kind == "prefill":
        shape = rng.choice(["e60", "e128", "e256", "e512"])
        t = rng.choice(["Q4_0/Q4_0/Q4_0", "Q4_K/Q4_K/Q4_K", "Q4_K/Q4_K/Q6_K"])
        t = "Q4_0/Q4_0/Q4_0" if shape == "e60" else t
        s = SHAPES[shape]
        routing = rng.choice(["zipf", "skewed", "router"]) if not s["Is"] else "router"
        return dict(kind=kind, shape=shape, types=t, T=_log_int(rng, 17, 2048 if shape == "e512" else 4096),
                    dtype=rng.choice(["f16", "bf16"]), routing=routing)
    if kind == "block":
        return dict(kind=kind, shape=rng.choice(["e128", "e256"]), types=rng.choice(["Q4_0/Q4_0/Q4_0", "Q4_K/Q4_K/Q6_K"]),
                    T=rng.randint(1, 8))
    if kind == "dense":
        shape = rng.choice(["e60", "e128", "e256"])
        t = rng.choice(["Q4_0/Q4_0/Q4_0", "Q8_0/Q8_0/Q8_0", "Q4_1/Q4_1/Q4_1"] if shape == "e60" else
                       ["Q4_0/Q4_0/Q4_0", "Q4_K/Q4_K/Q6_K", "Q6_K/Q6_K/Q6_K", "Q5_K/Q5_K/Q5_K", "Q8_0/Q8_0/Q8_0",
                        "Q4_1/Q4_1/Q4_1", "Q4_K/Q4_K/Q4_K"])
        return dict(kind=kind, shape=shape, types=t, rows=_log_int(rng, 64, 16384),
                    dtype=rng.choice(["f16", "bf16", "f32"]))
    K, G = rng.choice([(2048, 64), (4096, 64), (512, 64), (2560, 32), (640, 32)])
    return dict(kind=kind, K=K, N=_log_int(rng, 32, 32768), G=G, T=rng.randint(1, 8))


# ---- inputs ----------------------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _half(v):
    return v.to(torch.float16).view(torch.uint8).reshape(v.shape + (2,))


def _nibbles(lo, hi):
    return lo | (hi << 4)


def _pack(w, t):
    """w [n, block] float32 as blocks of ggml type t, uint8 [n, bytes a block]."""
    n = w.shape[0]
    if t == "Q4_0":
        m = w.gather(1, w.abs().argmax(1, keepdim=True))
        d = (m / -8).to(torch.float16).float()
        q = (w / torch.where(d == 0, 1, d) + 8.5).floor().clamp(0, 15).to(torch.uint8)
        return torch.cat([_half(d[:, 0]), _nibbles(q[:, :16], q[:, 16:])], 1)
    if t == "Q4_1":
        m = w.amin(1, keepdim=True).to(torch.float16).float()
        d = ((w.amax(1, keepdim=True) - m) / 15).to(torch.float16).float()
        q = ((w - m) / d).round().clamp(0, 15).to(torch.uint8)
        return torch.cat([_half(d[:, 0]), _half(m[:, 0]), _nibbles(q[:, :16], q[:, 16:])], 1)
    if t == "Q8_0":
        d = (w.abs().amax(1, keepdim=True) / 127).to(torch.float16).float()
        q = (w / d).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([_half(d[:, 0]), q], 1)
    if t == "Q6_K":
        s = w.view(n, 16, 16)
        a = s.abs().amax(2) / 31
        d = (a.amax(1, keepdim=True) / 127).to(torch.float16).float()
        sc = (a / d).round().clamp(1, 127)
        q = ((s / (d * sc)[:, :, None]).round().clamp(-32, 31) + 32).to(torch.uint8).view(n, 2, 4, 32)
        ql = _nibbles(q[:, :, 0:2] & 15, q[:, :, 2:4] & 15).reshape(n, 128)
        h = q >> 4
        qh = (h[:, :, 0] | (h[:, :, 1] << 2) | (h[:, :, 2] << 4) | (h[:, :, 3] << 6)).reshape(n, 64)
        return torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), _half(d[:, 0])], 1)
    top = 15 if t == "Q4_K" else 31
    s = w.view(n, 8, 32)
    lo = (-s.amin(2)).clamp(min=0)
    step = (s.amax(2) + lo) / top
    d = (step.amax(1, keepdim=True) / 63).to(torch.float16).float()
    dmin = (lo.amax(1, keepdim=True) / 63).to(torch.float16).float()
    sc = (step / d).round().clamp(1, 63)
    m = (lo / torch.where(dmin == 0, 1, dmin)).round().clamp(0, 63)
    q = ((s + (dmin * m)[:, :, None]) / (d * sc)[:, :, None]).round().clamp(0, top).to(torch.uint8)
    sc, m = sc.to(torch.uint8), m.to(torch.uint8)
    head = torch.cat([_half(d[:, 0]), _half(dmin[:, 0]), sc[:, :4] | ((sc[:, 4:] >> 4) << 6),
                      m[:, :4] | ((m[:, 4:] >> 4) << 6), _nibbles(sc[:, 4:] & 15, m[:, 4:] & 15)], 1)
    q = q.view(n, 4, 2, 32)
    qs = _nibbles(q[:, :, 0] & 15, q[:, :, 1] & 15).reshape(n, 128)
    if t == "Q4_K":
        return torch.cat([head, qs], 1)
    hi = (q.view(n, 8, 32) >> 4) << torch.arange(8, dtype=torch.uint8, device=q.device)[None, :, None]
    return torch.cat([head, hi.sum(1).to(torch.uint8), qs], 1)


def _experts(t, n, rows, cols, gen):
    """n experts uint8 [n, rows, row bytes] of ggml type t, quantized from N(0, 0.02^2)."""
    be, bb = BLOCK[t]
    out = torch.empty((n * rows, cols // be * bb), dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 27) // cols)
    for r in range(0, n * rows, step):
        w = torch.randn((min(step, n * rows - r), cols), generator=gen, device="cuda") * 0.02
        out[r:r + step] = _pack(w.view(-1, be), t).view(w.shape[0], -1)
    return out.view(n, rows, -1)


def _raw_layer(case, gen, router):
    """(experts, router weight or None, shared experts or None, shared gate or None) of one layer."""
    s = SHAPES[case["shape"]]
    H, I, Is = s["H"], s["I"], s["Is"]
    t = case["types"].split("/")
    w = tuple(_experts(q, s["E"], r, c, gen) for q, r, c in zip(t, (I, I, H), (H, H, I)))
    if not router:
        return w, None, None, None
    wr = (torch.randn((s["E"], H), generator=gen, device="cuda") * 0.02).to(torch.float16)
    if not Is:
        return w, wr, None, None
    shared = tuple(_experts(q, 1, r, c, gen) for q, r, c in zip(t, (Is, Is, H), (H, H, Is)))
    return w, wr, shared, (torch.randn(H, generator=gen, device="cuda") * 0.02).to(torch.float16)


def _layer(case, raw):
    s = SHAPES[case["shape"]]
    w, wr, shared, wsg = raw
    return layer.MoELayer(*w, case["types"].split("/"), s["k"], s["norm"], wr=wr, shared=shared, wsg=wsg)


def _x(case, gen, rows):
    H = SHAPES[case["shape"]]["H"]
    return torch.randn((rows, H), generator=gen, device="cuda").to(DTYPES[case["dtype"]])


def _logits(case, gen, rows):
    """Router logits that pick experts unevenly: N(0, 1) plus a prior per expert, Gaussian or half a Zipf(1.1)'s."""
    E = SHAPES[case["shape"]]["E"]
    if case.get("routing") == "zipf":
        prior = -0.55 * torch.log(torch.randperm(E, generator=gen, device="cuda").float() + 1)
    else:
        prior = torch.randn(E, generator=gen, device="cuda")
    return torch.randn((rows, E), generator=gen, device="cuda") + prior


def _affine(N, K, G, gen):
    """A 4-bit affine weight (w int32 [N, K / 8], scales and biases bf16 [N, K / G]) of values around N(0, 0.02^2)."""
    w = torch.randint(-2 ** 31, 2 ** 31, (N, K // 8), generator=gen, device="cuda", dtype=torch.int64).to(torch.int32)
    sc = (0.004 + 0.002 * torch.rand((N, K // G), generator=gen, device="cuda")).to(torch.bfloat16)
    return w, sc, (-7.5 * sc.float() * (1 + 0.1 * torch.randn((N, K // G), generator=gen, device="cuda"))).to(
        torch.bfloat16), G


def _inputs(case, seed):
    """What both prepare and exact start from: raw tensors, made from the seed alone."""
    gen = _gen(seed)
    kind = case["kind"]
    if kind == "qmv":
        return dict(w=_affine(case["N"], case["K"], case["G"], gen),
                    x=torch.randn((case["T"], case["K"]), generator=gen, device="cuda").to(torch.bfloat16))
    s = SHAPES[case["shape"]]
    if kind == "stack":
        return dict(x=_x(case, gen, case["T"]), raw=[_raw_layer(case, gen, True) for _ in range(case["layers"])])
    if kind == "layer":
        return dict(x=_x(case, gen, case["T"]), raw=_raw_layer(case, gen, True))
    if kind == "prefill":
        own = case["routing"] == "router"
        return dict(x=_x(case, gen, case["T"]), raw=_raw_layer(case, gen, own),
                    logits=None if own else _logits(case, gen, case["T"]))
    if kind == "dense":
        lg = _logits(case, gen, -(-case["rows"] // s["k"]))
        return dict(x=_x(case, gen, case["rows"]), raw=_raw_layer(case, gen, False),
                    slots=lg.topk(s["k"], 1).indices.reshape(-1)[:case["rows"]].to(torch.int32))
    T, H = case["T"], s["H"]  # block
    Is = s["Is"] or 512
    return dict(x=torch.randn((T, H), generator=gen, device="cuda").to(torch.bfloat16),
                raw=_raw_layer(case, gen, False), logits=_logits(case, gen, T).to(torch.bfloat16),
                shared=(_affine(Is, H, 64, gen), _affine(Is, H, 64, gen), _affine(H, Is, 64, gen)),
                gate=torch.randn((T, 1), generator=gen, device="cuda").to(torch.bfloat16))


def prepare(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    st = dict(kind=kind, case=case, x=d["x"])
    if kind == "qmv":
        return dict(st, w=d["w"])
    if kind == "stack":
        stack = layer.DecodeStack([_layer(case, r) for r in d["raw"]], case["T"], DTYPES[case["dtype"]])
        stack.capture()
        return dict(st, stack=stack)
    if kind == "layer":
        L = _layer(case, d["raw"])
        return dict(st, layer=L, bufs=layer.DecodeBuffers(L, case["T"]), out=torch.empty_like(d["x"]))
    if kind == "prefill":
        L = _layer(case, d["raw"])
        if L.wr is not None:  # the router's own forms, converted once a layer
            L.router_gemm_weight()
            L.router_norms()
        return dict(st, layer=L, bufs=grouped.PrefillBuffers(L, case["T"]), out=torch.empty_like(d["x"]),
                    logits=d["logits"])
    if kind == "dense":
        return dict(st, w=d["raw"][0], slots=d["slots"])
    return dict(st, bufs=tuple((w,) for w in d["raw"][0]), logits=d["logits"], shared=d["shared"], gate=d["gate"])


def run(st):
    kind, case, x = st["kind"], st["case"], st["x"]
    if kind == "qmv":
        return trunk.qmv_rows(x, *st["w"])
    if kind == "stack":
        st["stack"].x_in.copy_(x)
        st["stack"].graph.replay()
        return st["stack"].x_out
    if kind == "layer":
        out = layer.decode(st["layer"], x, st["bufs"], st["out"], residual=x)
        return dict(out=out, ids=st["bufs"].ids)
    if kind == "prefill":
        out = grouped.prefill(st["layer"], x, st["bufs"], st["out"], residual=x, logits=st["logits"])
        return dict(out=out, ids=st["bufs"].ids, scores=st["bufs"].scores)
    if kind == "dense":
        return gguf_experts.dense(x, st["w"], st["slots"], case["types"], x.dtype)
    s = SHAPES[case["shape"]]
    inds, scores = route.probs(st["logits"], s["k"], s["norm"])
    y = gguf_experts.experts(x[:, None, None], st["bufs"], inds, case["types"])
    shared = trunk.shared_expert_rows(x, *st["shared"])
    return dict(out=route.tail(y.squeeze(-2), scores, shared, st["gate"]), inds=inds)


# ---- what a pass cannot do without -----------------------------------------------------------------------------

def _row_bytes(t, n):
    return n // BLOCK[t][0] * BLOCK[t][1]


def work(case):
    if case["kind"] == "qmv":
        K, N, T = case["K"], case["N"], case["T"]
        return {"bytes": N * (K / 2 + 4 * K / case["G"]) + 2 * T * (K + N), "flops": 2 * T * N * K}
    s = SHAPES[case["shape"]]
    H, E, k, I, kind = s["H"], s["E"], s["k"], s["I"], case["kind"]
    tg, tu, td = case["types"].split("/")
    rows = case["rows"] if kind == "dense" else case["T"] * k
    tokens = -(-rows // k)
    expert = I * (_row_bytes(tg, H) + _row_bytes(tu, H)) + H * _row_bytes(td, I)
    used = E * (1 - (1 - k / E) ** tokens)  # experts that get a row, were they picked evenly
    size = 2 if case.get("dtype") != "f32" else 4
    b, f = used * expert, 6 * rows * H * I
    if kind == "dense":
        return {"bytes": b + 2 * rows * H * size, "flops": f}
    T = case["T"]
    b += 2 * T * H * size
    own = kind in ("stack", "layer") or case.get("routing") == "router"
    b += E * H * 2 if own else T * E * 4
    f += 2 * T * E * H if own else 0
    if s["Is"] and own:
        b += expert / I * s["Is"] + 2 * H
        f += 6 * T * H * s["Is"]
    if kind == "block":
        Is = s["Is"] or 512
        b += 3 * H * Is * (0.5 + 4 / 64)
        f += 6 * T * H * Is
    n = case.get("layers", 1)
    return {"bytes": n * b, "flops": n * f}


def tolerance(case):
    kind = case["kind"]
    if kind == "qmv":  # its bf16 steps are fixed one by one
        return "exact"
    if kind == "stack":  # 16-bit residuals, and now and then another pick where two logits nearly tie
        return {"rel": 2e-2, "max": 0.5}
    if case.get("dtype") == "bf16" or kind == "block":  # one bf16 rounding of the output
        return {"rel": 8e-3, "max": 0.1, "differ": 1e-4}
    return {"rel": 1e-3, "max": 0.04, "differ": 1e-4}  # f16 operands, float32 sums


# ---- the same in 64 bits ---------------------------------------------------------------------------------------

def _values(b, t):
    """Blocks uint8 [..., row bytes] of ggml type t as float64 [..., row length]."""
    be, bb = BLOCK[t]
    lead = b.shape[:-1]
    b = b.reshape(-1, bb)
    n = b.shape[0]

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    if t in ("Q4_0", "Q4_1"):
        qs = b[:, bb - 16:]
        q = torch.cat([qs & 15, qs >> 4], 1).double()
        v = (q - 8) * half(0) if t == "Q4_0" else q * half(0) + half(2)
    elif t == "Q8_0":
        v = b[:, 2:].contiguous().view(torch.int8).double() * half(0)
    elif t == "Q6_K":
        ql, qh = b[:, :128].view(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)
        hi = torch.cat([(qh >> (2 * g)) & 3 for g in range(4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        v = ((lo | (hi << 4)).double() - 32).reshape(n, 16, 16) * (half(208) * sc)[:, :, None]
    else:
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        m = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, bb - 128:].reshape(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
        if t == "Q5_K":
            j = torch.arange(8, dtype=torch.uint8, device=b.device)[None, :, None]
            q = q | (((b[:, None, 16:48] >> j) & 1) << 4)
        v = q.double() * (half(0) * sc)[:, :, None] - (half(2) * m)[:, :, None]
    return v.reshape(lead + (-1,))


def _affine_values(w, sc, bi, G):
    j = torch.arange(8, device=w.device) * 4
    q = ((w[:, :, None] >> j) & 15).reshape(w.shape[0], -1).double()
    return q * sc.double().repeat_interleave(G, 1) + bi.double().repeat_interleave(G, 1)


def _mlp(x, w, types):
    """down(silu(gate x) * up x) for x [n, H] through one expert's blocks."""
    g, u = (x @ _values(b, t).T for b, t in zip(w[:2], types))
    return (g * torch.sigmoid(g) * u) @ _values(w[2], types[2]).T


def _expert_rows(x, ids, w, types):
    """Row i of x through expert ids[i]."""
    y = torch.zeros((x.shape[0], w[2].shape[1]), dtype=torch.float64, device=x.device)
    for e in ids.unique().tolist():
        at = (ids == e).nonzero()[:, 0]
        y[at] = _mlp(x[at], [b[e] for b in w], types)
    return y


def _pick(logits, k, norm):
    """The k best (ties to the lower index), best first, and their softmax probabilities."""
    ids = logits.sort(dim=1, descending=True, stable=True).indices[:, :k]
    p = torch.softmax(logits, 1).gather(1, ids)
    return ids, p / p.sum(1, keepdim=True) if norm else p


def _whole_layer(case, raw, x, logits=None):
    s = SHAPES[case["shape"]]
    types = case["types"].split("/")
    w, wr, shared, wsg = raw
    ids, p = _pick(x @ wr.double().T if logits is None else logits.double(), s["k"], s["norm"])
    y = _expert_rows(x.repeat_interleave(s["k"], 0), ids.reshape(-1), w, types)
    out = (y.view(x.shape[0], s["k"], -1) * p[:, :, None]).sum(1)
    if shared is not None:
        out += torch.sigmoid(x @ wsg.double())[:, None] * _mlp(x, [b[0] for b in shared], types)
    return x + out, ids.to(torch.int32), p


def exact(case, seed):
    d = _inputs(case, seed)
    kind, x = case["kind"], d["x"].double()
    if kind == "qmv":
        w, sc, bi, G = d["w"]
        return torch.cat([x @ _affine_values(w[r:r + 16384], sc[r:r + 16384], bi[r:r + 16384], G).T
                          for r in range(0, w.shape[0], 16384)], 1)
    if kind == "stack":
        for raw in d["raw"]:
            x = _whole_layer(case, raw, x)[0]
        return x
    if kind == "layer":
        out, ids, _ = _whole_layer(case, d["raw"], x)
        return dict(out=out, ids=ids)
    if kind == "prefill":
        out, ids, p = _whole_layer(case, d["raw"], x, d["logits"])
        return dict(out=out, ids=ids, scores=p)
    if kind == "dense":
        return _expert_rows(x, d["slots"].long(), d["raw"][0], case["types"].split("/"))
    s = SHAPES[case["shape"]]
    k, T = s["k"], case["T"]
    ids, p = _pick(d["logits"].double(), k, s["norm"])
    y = _expert_rows(x.repeat_interleave(k, 0), ids.reshape(-1), d["raw"][0], case["types"].split("/"))
    g, u, dn = (_affine_values(*a) for a in d["shared"])
    h = x @ g.T
    out = (y.view(T, k, -1) * p[:, :, None]).sum(1) + torch.sigmoid(d["gate"].double()) * (
        (h * torch.sigmoid(h) * (x @ u.T)) @ dn.T)
    return dict(out=out, inds=ids.flip(-1).to(torch.int32))
