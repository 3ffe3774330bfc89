"""The work that is timed on an MI355X: EXL3 linears, MoE layers and quantized-KV attention as a serving engine runs them.

Three kinds of case, each through the entry points that the engine glue calls:

  linear   fused linears (`torch.ops.exl3_mi355x.linear`): q/k/v, o, gate/up, down of dense decoder layers, from one
           token's decode to a prefill chunk.
  moe      routed SiLU-gated expert layers (`ops.moe_forward`).
  kv       decode attention over the paged quantized KV cache (`ops.kv_decode_attention`), batches of ragged lengths.

Engines reserve their workspaces at load and replay decode steps from a HIP graph (`graph`: true, `layers` layers in
one graph, each with its own weights or cache); prefill chunks and single calls run eagerly.
"""
from __future__ import annotations

import math

import torch

from trellis_serve_amd import ops
from trellis_serve_amd.runtime import ops as runtime_ops

# one decoder layer of the dense 27B-class model of the benchmark: q/k/v, o, gate/up, down
DECODER = "5120:6144+1024+1024 6144:5120 5120:17408+17408 17408:5120"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
HEAD_DIM = 128
PAGE = 16


def listed():
    return [
        # one small linear on its own, one token, called eagerly: latency and host path (the benchmark's single linear)
        dict(name="linear_4096_m1_eager", kind="linear", linears="4096:4096", layers=1, rows=1, K=4, codebook=0,
             dtype="fp16", graph=False),
        # one user's decode step: the linears of two decoder layers in the step's graph
        dict(name="decoder_m1", kind="linear", linears=DECODER, layers=2, rows=1, K=3, codebook=1, dtype="fp16",
             graph=True),
        # decode of a full small batch, bf16 activations (the usual model dtype)
        dict(name="decoder_m16_bf16", kind="linear", linears=DECODER, layers=2, rows=16, K=3, codebook=1,
             dtype="bf16", graph=True),
        # decode of a ragged larger batch (or speculative tokens of several users)
        dict(name="decoder_m43", kind="linear", linears=DECODER, layers=1, rows=43, K=4, codebook=1, dtype="fp16",
             graph=True),
        # a short prompt's prefill through the attention-side linears
        dict(name="prefill_attn_m333_bf16", kind="linear", linears="5120:6144+1024+1024 6144:5120", layers=1,
             rows=333, K=5, codebook=2, dtype="bf16", graph=False),
        # a prefill chunk through the largest fused linear
        dict(name="prefill_gate_up_m4096", kind="linear", linears="5120:17408+17408", layers=1, rows=4096, K=3,
             codebook=1, dtype="fp16", graph=False),
        # one user's MoE decode step: two expert layers of 128 experts, top-8
        dict(name="moe_t1", kind="moe", layers=2, tokens=1, experts=128, top_k=8, hidden=2048, inter=768, K_gate_up=3,
             K_down=3, codebook=1, dtype="bf16", graph=True),
        # a decode batch of the same layers, down stored at a higher bitrate
        dict(name="moe_t37", kind="moe", layers=2, tokens=37, experts=128, top_k=8, hidden=2048, inter=768,
             K_gate_up=3, K_down=4, codebook=1, dtype="bf16", graph=True),
        # a large decode batch or a short prompt
        dict(name="moe_t256", kind="moe", layers=1, tokens=256, experts=128, top_k=8, hidden=2048, inter=768,
             K_gate_up=3, K_down=3, codebook=1, dtype="fp16", graph=False),
        # a prefill chunk
        dict(name="moe_t2048", kind="moe", layers=1, tokens=2048, experts=128, top_k=8, hidden=2048, inter=768,
             K_gate_up=3, K_down=3, codebook=1, dtype="bf16", graph=False),
        # chat-length decode: ragged lengths up to 4k, the page table as wide as the engine's 8k context limit
        dict(name="kv8_b16_4k", kind="kv", layers=2, batch=16, q_heads=40, kv_heads=8, longest=4096, table=8192,
             bits=8, graph=True),
        # long-context decode: ragged lengths up to 32k at 4 bits
        dict(name="kv4_b7_32k", kind="kv", layers=2, batch=7, q_heads=40, kv_heads=8, longest=32768, table=32768,
             bits=4, graph=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):  # a multiple of 128, as the format requires
    return 128 * _log_int(rng, lo // 128, hi // 128)


def draw(rng):
    kind = rng.choice(["linear", "linear", "moe", "kv"])
    if kind == "linear":
        while True:
            rows = _log_int(rng, 1, 4096)
            if rng.random() < 0.4:
                linears = rng.choice(DECODER.split())
            else:
                k = _width(rng, 1024, 17408)
                linears = "%d:%s" % (k, "+".join(str(_width(rng, 512, 17408)) for _ in range(rng.randint(1, 3))))
            n = sum(sum(ns) for _, ns in _linears(linears))
            k = _linears(linears)[0][0]
            if n <= 34816 and rows * k * n <= 4096 * 5120 * 34816:
                break
        return dict(kind="linear", linears=linears, layers=1 if rows > 64 else 2, rows=rows,
                    K=rng.choice([2, 3, 3, 4, 4, 5, 6, 8]), codebook=rng.randint(0, 2),
                    dtype=rng.choice(["fp16", "bf16"]), graph=rows <= 64)
    if kind == "moe":
        experts = rng.choice([8, 16, 60, 64, 128])
        tokens = _log_int(rng, 1, 2048)
        hidden, inter = _width(rng, 1024, 4096), _width(rng, 512, 1536)
        top_k = rng.randint(2, 8)
        return dict(kind="moe", layers=2 if tokens <= 64 else 1, tokens=tokens, experts=experts, top_k=top_k,
                    hidden=hidden, inter=inter, K_gate_up=rng.choice([2, 3, 4, 5]), K_down=rng.choice([3, 4, 6]),
                    codebook=rng.randint(0, 2), dtype=rng.choice(["fp16", "bf16"]), graph=tokens <= 64)
    bits = rng.choice([4, 8])
    kv_heads = rng.choice([1, 2, 4, 8])
    while True:
        batch, longest = _log_int(rng, 1, 64), _log_int(rng, 64, 32768)
        if batch * longest * kv_heads * bits <= 16 * 32768 * 8 * 4:
            break
    table = min(32768, max(longest, 256) * rng.choice([1, 1, 2, 4]))
    return dict(kind="kv", layers=2, batch=batch, q_heads=kv_heads * rng.choice([1, 4, 5, 8, 16]), kv_heads=kv_heads,
                longest=longest, table=table, bits=bits, graph=True)


# ---- inputs ----------------------------------------------------------------------------------------------------

def _linears(text):
    """"k:n0+n1 k:n" -> [(k, [n0, n1]), (k, [n])]"""
    return [(int(k), [int(n) for n in ns.split("+")]) for k, ns in (part.split(":") for part in text.split())]


def _signs(g, shape, scale):
    """Sign vector with the magnitudes of a quantized checkpoint: +-scale, spread by 30 %."""
    sign = torch.randint(0, 2, shape, generator=g, device="cuda") * 2 - 1
    return (sign * scale * (0.7 + 0.6 * torch.rand(shape, generator=g, device="cuda"))).half()


def _trellis(g, shape):
    return torch.randint(-32768, 32768, shape, dtype=torch.int16, generator=g, device="cuda")


def _linear_inputs(case, g):
    layers = []
    for _ in range(case["layers"]):
        for k, ns in _linears(case["linears"]):
            x = torch.randn((case["rows"], k), generator=g, device="cuda").to(DTYPES[case["dtype"]])
            layers.append((x, [_trellis(g, (k // 16, n // 16, 16 * case["K"])) for n in ns],
                           [_signs(g, (k,), 1.0) for _ in ns], [_signs(g, (n,), k ** -0.5) for n in ns]))
    return layers


def _moe_inputs(case, g):
    layers = []
    E, H, I, T = case["experts"], case["hidden"], case["inter"], case["tokens"]
    for _ in range(case["layers"]):
        x = torch.randn((T, H), generator=g, device="cuda").to(DTYPES[case["dtype"]])
        # a router's logits: per-token scores over experts of uneven popularity
        logits = torch.randn((T, E), generator=g, device="cuda") \
            + 0.5 * torch.randn((1, E), generator=g, device="cuda")
        w, ids = torch.topk(logits, case["top_k"], dim=1)
        experts = {}
        for name, k, n, K in (("gate", H, I, case["K_gate_up"]), ("up", H, I, case["K_gate_up"]),
                              ("down", I, H, case["K_down"])):
            experts[name + "_trellis"] = _trellis(g, (E, k // 16, n // 16, 16 * K))
            experts[name + "_suh"] = _signs(g, (E, k), 1.0)
            experts[name + "_svh"] = _signs(g, (E, n), k ** -0.5)
        layers.append((x, ids.to(torch.int32), torch.softmax(w, dim=1), experts))
    return layers


def _lengths(case):
    """A batch of users at different points of their sequences: evenly spread lengths up to the longest."""
    B = case["batch"]
    return [max(1, case["longest"] * (i + 1) // B) for i in range(B)]


def _kv_inputs(case, g):
    layers = []
    B, Hkv, bits = case["batch"], case["kv_heads"], case["bits"]
    qmax = 127 if bits == 8 else 7

    def codes(pages):  # normal keys and values on the code grid
        c = torch.empty((pages, Hkv, PAGE, HEAD_DIM), dtype=torch.int8, device="cuda")
        for p in range(0, pages, 1024):
            part = torch.randn(c[p:p + 1024].shape, generator=g, device="cuda") * (qmax / 3.0)
            c[p:p + 1024] = part.round_().clamp_(-qmax, qmax).to(torch.int8)
        if bits == 8:
            return c
        return ((c[..., 0::2] & 15) | (c[..., 1::2] << 4)).view(torch.uint8)

    for _ in range(case["layers"]):
        order = torch.randperm(B, generator=g, device="cuda").tolist()
        lens = [_lengths(case)[i] for i in order]
        need = [-(-n // PAGE) for n in lens]
        pages = sum(need) + B
        perm = torch.randperm(pages, generator=g, device="cuda").to(torch.int32)
        table = torch.zeros((B, -(-case["table"] // PAGE)), dtype=torch.int32, device="cuda")
        at = 0
        for b, n in enumerate(need):
            table[b, :n] = perm[at:at + n]
            at += n
        q = torch.randn((B, case["q_heads"], HEAD_DIM), generator=g, device="cuda").half()
        scale = [((0.5 + torch.rand((pages, Hkv), generator=g, device="cuda")) * 3.0 / qmax).half() for _ in range(2)]
        layers.append((q, codes(pages), codes(pages), scale[0], scale[1], table,
                       torch.tensor(lens, dtype=torch.int32, device="cuda")))
    return layers


_INPUTS = {"linear": _linear_inputs, "moe": _moe_inputs, "kv": _kv_inputs}


def _inputs(case, seed):
    return _INPUTS[case["kind"]](case, torch.Generator(device="cuda").manual_seed(seed))


def _reserve(case):
    """The engine's reservations at load, for the largest layer and batch of every case (made once, kept after)."""
    dev = torch.device("cuda", torch.cuda.current_device())
    if case["kind"] == "linear":
        ops.reserve_linear(dev, runtime_ops.PREFILL_ROWS - 1, 17408, 34816, 3)
        for k, ns in _linears(case["linears"]):
            if case["rows"] < runtime_ops.PREFILL_ROWS:
                ops.reserve_linear(dev, case["rows"], k, sum(ns), case["K"])
            else:
                ops.reserve_prefill(dev, case["rows"], k, sum(ns), len(ns))
    elif case["kind"] == "moe":
        ops.reserve_moe(dev, 2048, 8, 128, 4096, 1536, 3, 3)
        ops.reserve_moe(dev, case["tokens"], case["top_k"], case["experts"], case["hidden"], case["inter"],
                        case["K_gate_up"], case["K_down"])
    else:
        for group in (5, 8, 16):
            ops.reserve_kv(dev, 64, 8 * group, 8, 32768 // PAGE)
        ops.reserve_kv(dev, case["batch"], case["q_heads"], case["kv_heads"], -(-case["table"] // PAGE))


# ---- one pass --------------------------------------------------------------------------------------------------

def _call(case, inputs):
    if case["kind"] == "linear":
        return [runtime_ops.linear(x, trellis, suh, svh, case["codebook"]) for x, trellis, suh, svh in inputs]
    if case["kind"] == "moe":
        return [ops.moe_forward(x, ids, w, experts, case["codebook"]) for x, ids, w, experts in inputs]
    return [ops.kv_decode_attention(q, k, v, ks, vs, table, lens, case["bits"])
            for q, k, v, ks, vs, table, lens in inputs]


def prepare(case, seed):
    state = {"case": case, "inputs": _inputs(case, seed), "graph": None}
    _reserve(case)
    if case["graph"]:  # as an engine captures its decode step: one call outside, then the capture
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _call(case, state["inputs"])
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = _call(case, state["inputs"])
    return state


def run(state):
    if state["graph"] is None:
        return _call(state["case"], state["inputs"])
    state["graph"].replay()
    return state["out"]


# ---- what a pass cannot do without -----------------------------------------------------------------------------

def work(case):
    layers = case["layers"]
    if case["kind"] == "linear":
        M, K = case["rows"], case["K"]
        nbytes = flops = 0
        for k, ns in _linears(case["linears"]):
            n = sum(ns)
            nbytes += k * n * K // 8 + 2 * k * len(ns) + 2 * n + 2 * M * (k + n)
            flops += 2 * M * k * n
    elif case["kind"] == "moe":
        T, E, H, I, top = case["tokens"], case["experts"], case["hidden"], case["inter"], case["top_k"]
        touched = E * (1.0 - (1.0 - top / E) ** T)  # expected over even routing
        per_expert = H * I * (2 * case["K_gate_up"] + case["K_down"]) / 8 + 2 * (2 * (H + I) + I + H)
        nbytes = touched * per_expert + T * (4 * H + 8 * top)
        flops = 2 * T * top * 3 * H * I
    else:
        pages = sum(-(-n // PAGE) for n in _lengths(case))
        tokens = sum(_lengths(case))
        block = PAGE * HEAD_DIM * case["bits"] // 8 + 2
        nbytes = pages * case["kv_heads"] * 2 * block + 4 * pages + 4 * case["batch"] \
            + 4 * case["batch"] * case["q_heads"] * HEAD_DIM
        flops = 4 * tokens * case["q_heads"] * HEAD_DIM
    return {"bytes": layers * nbytes, "flops": layers * flops}


def tolerance(case):
    # Outputs are rounded once to fp16 or bf16, and the rotated activations (and the MoE's g, u, a and d rows) to fp16,
    # from fp32 sums: about four times the error seen against exact() (linears 4.6e-4 in fp16 and 1.8e-3 in bf16, MoE
    # 8.8e-4 and 1.9e-3, attention 2.7e-4).
    if case["kind"] == "moe":
        return {"rel": 8e-3 if case["dtype"] == "bf16" else 4e-3}
    if case["kind"] == "kv":
        return {"rel": 1.2e-3}
    return {"rel": 8e-3 if case["dtype"] == "bf16" else 2e-3}


# ---- the same outputs in 64 bits, in plain torch ---------------------------------------------------------------

def _f16(bits):
    bits = bits - 65536 * (bits >= 32768)
    return bits.to(torch.int16).view(torch.float16).double()


def _codebook(cb):
    """The fp16 value of each of the 65536 states (format definition), as float64."""
    s = torch.arange(65536, dtype=torch.int64, device="cuda")
    if cb == 2:  # MUL1: fp16 fma of 1024 + the byte sum of the hash
        x = (s * 0x83DCD12D) & 0xFFFFFFFF
        total = 1024 + (x & 255) + ((x >> 8) & 255) + ((x >> 16) & 255) + ((x >> 24) & 255)
        one = torch.ones((), dtype=torch.int64, device="cuda")
        return (total.double() * _f16(one * 0x1EEE) + _f16(one * 0xC931)).half().double()
    x = (s * 0xCBAC1FED if cb == 1 else s * 89226354 + 64248484) & 0xFFFFFFFF
    x = (x & 0x8FFF8FFF) ^ 0x3B603B60
    return (_f16(x & 0xFFFF) + _f16(x >> 16)).half().double()


def _decode(trellis, cb, lut):
    """int16 [k/16, n/16, 16K] -> the inner weights, float64 [k, n]."""
    tk, tn, words = trellis.shape
    K = words // 16
    t = torch.arange(256, device="cuda")
    start = (t * K + K - 16) % (256 * K)  # first bit of the 16-bit window that ends at bit (t + 1) K, MSB first
    first, shift = start // 32, 48 - start % 32
    row = 8 * ((t >> 1) & 1) + 2 * ((t >> 3) & 3) + (t & 1)
    place = row * 16 + (t >> 5) + 8 * ((t >> 2) & 1)
    out = torch.empty((tk, 16, tn, 16), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 16) // tn)
    for i in range(0, tk, step):
        h = trellis[i:i + step].long() & 0xFFFF
        w = h[..., 0::2] | (h[..., 1::2] << 16)
        pair = (w[..., first] << 32) | w[..., (first + 1) % (8 * K)]
        tile = torch.empty(pair.shape, dtype=torch.float64, device="cuda")
        tile[..., place] = lut[(pair >> shift) & 0xFFFF]
        out[i:i + step] = tile.view(*tile.shape[:2], 16, 16).permute(0, 2, 1, 3)
    return out.view(tk * 16, tn * 16)


def _rotate(x):
    h = torch.ones((1, 1), dtype=torch.float64, device="cuda")
    while h.shape[0] < 128:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (x.reshape(-1, 128) @ (h / 128 ** 0.5)).view(x.shape)


def _exact_linear(x, trellis, suh, svh, cb, lut):
    return _rotate(_rotate(x * suh.double()) @ _decode(trellis, cb, lut)) * svh.double()


def _exact_moe(case, x, ids, w, experts, lut):
    y = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
    for e in range(case["experts"]):
        tokens, choice = torch.nonzero(ids == e, as_tuple=True)
        if not len(tokens):
            continue

        def part(name, v):
            return _exact_linear(v, *(experts[name + "_" + p][e] for p in ("trellis", "suh", "svh")),
                                 case["codebook"], lut)

        xe = x[tokens].double()
        a = torch.nn.functional.silu(part("gate", xe)) * part("up", xe)
        y.index_add_(0, tokens, part("down", a) * w[tokens, choice].double()[:, None])
    return y


def _exact_kv(case, q, k, v, ks, vs, table, lens):
    def values(codes, scale, pages):  # [tokens, kv heads, head dim]
        c = codes[pages]
        if case["bits"] == 4:
            c = torch.stack([c & 15, c >> 4], -1).view(*c.shape[:-1], HEAD_DIM).to(torch.int8)
            c = c - 16 * (c >= 8)
        d = c.double() * scale[pages].double()[:, :, None, None]
        return d.permute(0, 2, 1, 3).reshape(-1, case["kv_heads"], HEAD_DIM)

    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    group = case["q_heads"] // case["kv_heads"]
    for b, n in enumerate(lens.tolist()):
        pages = table[b, :-(-n // PAGE)].long()
        kk, vv = values(k, ks, pages)[:n], values(v, vs, pages)[:n]
        for h in range(case["kv_heads"]):
            qh = q[b, h * group:(h + 1) * group].double()
            p = torch.softmax(qh @ kk[:, h].t().contiguous() * HEAD_DIM ** -0.5, dim=1)
            out[b, h * group:(h + 1) * group] = p @ vv[:, h].contiguous()
    return out


def exact(case, seed):
    inputs = _inputs(case, seed)
    if case["kind"] == "kv":
        return [_exact_kv(case, *layer) for layer in inputs]
    lut = _codebook(case["codebook"])
    if case["kind"] == "moe":
        return [_exact_moe(case, *layer, lut) for layer in inputs]
    return [torch.cat([_exact_linear(x.double(), t, su, sv, case["codebook"], lut)
                       for t, su, sv in zip(trellis, suh, svh)], dim=1) for x, trellis, suh, svh in inputs]
