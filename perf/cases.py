"""The work that the framework's speed is judged by: routed experts on quantised weights, quantised linears, and latent attention.

A case is one call of a public entry point on one GPU, the way a serving loop makes it for one layer:

  moe          MoEHandle.forward: the routed experts of one layer, by weight format (what KTMoEWrapper and KTransformersExperts call)
  linear       LinearHandle.forward: one projection, by weight format (what KLinearMarlin, KLinearFP8 and KLinearTorch call)
  mla_decode   MLAWrapper.run: one decode step of a batch of requests over a paged latent cache
  mla_prefill  mla_prefill: a prompt chunk's causal attention over expanded keys and values

listed() holds the cases that are always timed; draw() gives more of the same ranges: tokens from one to a prompt chunk, the layer sizes of
this repository's benchmark and generic ones, every weight format of its benchmark's workloads.  exact() states each call in 64-bit arithmetic.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from ktransformers_amd._native import LinearHandle, MLAWrapper, MoEHandle, mla_prefill

CHUNK = 2048          # tokens of the largest prompt chunk: what an engine sizes its expert handles for
GGML_Q4_K = 12        # ggml's type id; a block is 256 weights in 144 bytes
PAGE = 64             # tokens per page of the latent cache
LORA, ROPE = 512, 64  # latent and rotated part of a cached row

#: (experts, experts per token, hidden, intermediate) of the layers that this repository's benchmark runs in each format
MOE_SIZES = {
    "AMXINT4": ((64, 6, 2048, 1408), (256, 8, 7168, 2048)),
    "FP8": ((256, 8, 7168, 2048), (64, 6, 2048, 1408)),
    "RAWINT4": ((384, 8, 7168, 2048), (64, 8, 2048, 1024)),
    "GGUF": ((8, 2, 4096, 14336), (64, 6, 2048, 1536)),
}
#: (in, out) of the projections of its attention and shared-expert operators; 576 and 1000 are ragged ones
LINEAR_SIZES = ((7168, 2112), (1536, 24576), (16384, 7168), (7168, 4096), (2048, 7168), (18432, 7168), (2048, 3072), (2048, 576), (4096, 1000))


def listed():
    return [
        # one token through a small mixture: the shortest call of a chat's decode loop, launches and latency
        {"name": "moe-int4-small-t1", "kind": "moe", "fmt": "AMXINT4", "E": 64, "k": 6, "H": 2048, "I": 1408, "T": 1},
        # a decode step of 32 concurrent requests at DeepSeek-V3's expert sizes: the weights of most experts stream once
        {"name": "moe-int4-v3-t32", "kind": "moe", "fmt": "AMXINT4", "E": 256, "k": 8, "H": 7168, "I": 2048, "T": 32},
        # a full prompt chunk at the same sizes
        {"name": "moe-int4-v3-t2048", "kind": "moe", "fmt": "AMXINT4", "E": 256, "k": 8, "H": 7168, "I": 2048, "T": 2048},
        # a ragged prompt on block-fp8 experts
        {"name": "moe-fp8-v3-t1000", "kind": "moe", "fmt": "FP8", "E": 256, "k": 8, "H": 7168, "I": 2048, "T": 1000},
        # a decode batch and a prompt chunk on Kimi-K2's group-scaled int4 experts
        {"name": "moe-rawint4-k2-t16", "kind": "moe", "fmt": "RAWINT4", "E": 384, "k": 8, "H": 7168, "I": 2048, "T": 16},
        {"name": "moe-rawint4-k2-t2048", "kind": "moe", "fmt": "RAWINT4", "E": 384, "k": 8, "H": 7168, "I": 2048, "T": 2048},
        # a user's prompt of a few hundred tokens on Mixtral-8x7B's Q4_K experts
        {"name": "moe-q4k-mixtral-t500", "kind": "moe", "fmt": "GGUF", "E": 8, "k": 2, "H": 4096, "I": 14336, "T": 500},
        # the attention's output projection for a batch of 48 requests, 4-bit weights
        {"name": "linear-w4-o-t48", "kind": "linear", "fmt": "W4", "K": 16384, "N": 7168, "T": 48},
        # the first projections of a 300-token prompt, block-fp8 weights
        {"name": "linear-fp8-qkv-t300", "kind": "linear", "fmt": "FP8", "K": 7168, "N": 2112, "T": 300},
        # the query up-projection of a 1000-token prompt, bf16 weights
        {"name": "linear-bf16-q-t1000", "kind": "linear", "fmt": "BF16", "K": 1536, "N": 24576, "T": 1000},
        # a decode step of 8 requests of unequal length up to 8192 cached tokens
        {"name": "mla-decode-b8", "kind": "mla_decode", "heads": 128, "B": 8, "ctx": 8192},
        # a 1000-token chunk behind a 3096-token context
        {"name": "mla-prefill-t1000", "kind": "mla_prefill", "heads": 128, "T": 1000, "ctx": 4096},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("moe", "moe", "moe", "moe", "linear", "linear", "mla_decode", "mla_prefill"))
    if kind == "moe":
        fmt = rng.choice(tuple(MOE_SIZES))
        T = _log_int(rng, 1, CHUNK)
        if rng.random() < 0.6:
            E, k, H, I = rng.choice(MOE_SIZES[fmt])
        else:
            E, k = rng.choice((8, 16, 32, 64, 128)), rng.choice((2, 4, 6, 8))
            H, I = 512 * rng.randint(2, 12), 512 * rng.randint(1, 6)
        return {"kind": kind, "fmt": fmt, "E": E, "k": k, "H": H, "I": I, "T": T}
    if kind == "linear":
        K, N = rng.choice(LINEAR_SIZES) if rng.random() < 0.7 else (128 * rng.randint(8, 80), 8 * rng.randint(16, 1500) + rng.choice((0, 0, 1)))
        return {"kind": kind, "fmt": rng.choice(("W4", "FP8", "BF16")), "K": K, "N": N, "T": _log_int(rng, 1, CHUNK)}
    heads = rng.choice((16, 64, 128))
    if kind == "mla_decode":
        B = _log_int(rng, 1, 32)
        return {"kind": kind, "heads": heads, "B": B, "ctx": min(_log_int(rng, 100, 32768), 131072 // B)}
    T = _log_int(rng, 64, CHUNK)
    return {"kind": kind, "heads": heads, "T": T, "ctx": T + rng.choice((0, 0, _log_int(rng, 1, 8192 - CHUNK)))}


# ---- inputs: every tensor comes from the seed and a salt of its own, so that exact() can make the same ones again -------------------------


def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000 + salt)
    return g


def _normal(shape, seed, salt, std=1.0, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=_gen(seed, salt))


def _bytes(shape, seed, salt):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=_gen(seed, salt))


def _routing(case, seed):
    """(ids, weights): the k experts of each token and their softmax weights, under unequal popularity of the experts as routers have it."""
    r = np.random.default_rng(seed)
    E, k, T = case["E"], case["k"], case["T"]
    score = r.standard_normal((T, E)).astype(np.float32) + 0.7 * r.standard_normal(E).astype(np.float32)
    ids = np.argsort(-score, axis=1, kind="stable")[:, :k]
    top = np.exp(np.take_along_axis(score, ids, axis=1))
    return ids.astype(np.int64), (top / top.sum(axis=1, keepdims=True)).astype(np.float32)


def _matrices(case):
    """(rows, columns, standard deviation of the weights) of gate, up and down."""
    H, I = case["H"], case["I"]
    return ((I, H, H ** -0.5), (I, H, H ** -0.5), (H, I, I ** -0.5))


def _moe_weights(case, seed, m):
    """The checkpoint's tensors of matrix m (0 gate, 1 up, 2 down) of all experts: (weights,) or (weights, scales)."""
    n, kk, std = _matrices(case)[m]
    E, fmt = case["E"], case["fmt"]
    if fmt == "AMXINT4":
        return (_normal((E, n, kk), seed, 10 + m, std),)
    if fmt == "FP8":
        w = torch.empty((E, n, kk), dtype=torch.float8_e4m3fn, device="cuda")
        for e in range(0, E, 16):   # a normal weight over its block's scale: codes of magnitude up to 448
            w[e:e + 16] = _normal((min(16, E - e), n, kk), seed, 20 + 3 * e + m, 100.0).clamp_(-448, 448).to(torch.float8_e4m3fn)
        scale = std / 100.0 * (0.5 + torch.rand((E, -(-n // 128), -(-kk // 128)), device="cuda", generator=_gen(seed, 13 + m)))
        return w, scale
    if fmt == "RAWINT4":
        scale = std / 4.6 * (0.5 + torch.rand((E, n, kk // 32), device="cuda", generator=_gen(seed, 13 + m)))
        return _bytes((E, n, kk // 2), seed, 10 + m), scale.to(torch.bfloat16)
    # Q4_K: fp16 d, fp16 dmin, 12 bytes of 6-bit scales and minima, 128 bytes of nibbles; d * 32 * nibble and dmin * 32 around equal means
    b = _bytes((E, n, kk // 256, 144), seed, 10 + m)
    unit = 0.5 + torch.rand((E, n, kk // 256), device="cuda", generator=_gen(seed, 13 + m))
    d = (unit * (std / 160.0)).to(torch.float16)
    b[..., 0:2] = d.view(torch.uint8).view(E, n, kk // 256, 2)
    b[..., 2:4] = (d.float() * 7.5).to(torch.float16).view(torch.uint8).view(E, n, kk // 256, 2)
    return (b,)


def _linear_weights(case, seed):
    K, N, fmt = case["K"], case["N"], case["fmt"]
    if fmt == "FP8":
        w = _normal((N, K), seed, 10, 100.0).clamp_(-448, 448).to(torch.float8_e4m3fn)
        scale = K ** -0.5 / 100.0 * (0.5 + torch.rand((-(-N // 128), K // 128), device="cuda", generator=_gen(seed, 11)))
        return w, scale
    return (_normal((N, K), seed, 10, K ** -0.5),)


def _lengths(case, seed):
    """Cached tokens of each request: the longest as stated, the others between a quarter of it and all of it."""
    r = np.random.default_rng(seed)
    n = r.integers(max(1, case["ctx"] // 4), case["ctx"] + 1, size=case["B"])
    n[0] = case["ctx"]
    return n.astype(np.int32)


def _sm_scale():
    return (128 + ROPE) ** -0.5


def _decode_inputs(case, seed):
    n = _lengths(case, seed)
    pages = -(-n // PAGE)
    first = np.concatenate([[0], np.cumsum(pages)]).astype(np.int32)
    table = np.random.default_rng(seed + 1).permutation(int(first[-1])).astype(np.int32)   # pages are handed out in no order
    q_nope = _normal((case["B"], case["heads"], LORA), seed, 1)
    q_pe = _normal((case["B"], case["heads"], ROPE), seed, 2)
    cache = _normal((int(first[-1]), PAGE, LORA + ROPE), seed, 3)
    return n, first, table, q_nope, q_pe, cache


def _prefill_inputs(case, seed):
    T, kv, H = case["T"], case["ctx"], case["heads"]
    pad = -(-kv // 64) * 64
    q = _normal((T, H, 128 + ROPE), seed, 1)
    k_nope = _normal((H, pad, 128), seed, 2)
    k_nope[:, kv:] = 0
    rows = _normal((kv, LORA + ROPE), seed, 3)     # the latent cache; its rotated part is read in place
    v_t = _normal((H, 128, pad), seed, 4)
    v_t[:, :, kv:] = 0
    return q, k_nope, rows, v_t


# ---- the calls ------------------------------------------------------------------------------------------------------------------------


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    if case["kind"] == "moe":
        fmt = case["fmt"]
        h = MoEHandle(case["E"], case["k"], case["H"], case["I"], max(CHUNK, case["T"]), fmt, dev, group_size={"RAWINT4": 32, "FP8": 128}.get(fmt, 0))
        w = [_moe_weights(case, seed, m) for m in range(3)]
        if fmt == "AMXINT4":
            h.load_bf16(*(t[0] for t in w))
        elif fmt == "GGUF":
            h.load_gguf(*(t[0].view(case["E"], t[0].shape[1], -1) for t in w), GGML_Q4_K, GGML_Q4_K, GGML_Q4_K)
        else:
            (h.load_fp8 if fmt == "FP8" else h.load_rawint4)(*(t[0] for t in w), *(t[1] for t in w))
        ids, weights = (torch.from_numpy(a).to(dev) for a in _routing(case, seed))
        return {"kind": "moe", "h": h, "x": _normal((case["T"], case["H"]), seed, 1), "ids": ids, "w": weights}
    if case["kind"] == "linear":
        h = LinearHandle(case["K"], case["N"], case["fmt"], {"W4": 64, "FP8": 128, "BF16": 0}[case["fmt"]], max(CHUNK, case["T"]), dev)
        (h.load_fp8 if case["fmt"] == "FP8" else h.load_bf16)(*_linear_weights(case, seed))
        return {"kind": "linear", "h": h, "x": _normal((case["T"], case["K"]), seed, 1)}
    if case["kind"] == "mla_decode":
        n, first, table, q_nope, q_pe, cache = _decode_inputs(case, seed)
        B = case["B"]
        first, table, n_dev, one = (torch.from_numpy(a).to(dev) for a in (first, table, n, np.arange(B + 1, dtype=np.int32)))
        wrapper = MLAWrapper(B, int(first[-1]), use_cuda_graph=False, device=dev, max_q_tokens=B)
        live = torch.tensor([B], dtype=torch.int32, device=dev)
        plan = (one, first, table, n_dev, live, case["heads"], LORA, ROPE, PAGE, _sm_scale(), torch.bfloat16, torch.bfloat16, case["ctx"])
        return {"kind": "mla_decode", "wrapper": wrapper, "plan": plan, "q_nope": q_nope, "q_pe": q_pe, "cache": cache}
    q, k_nope, rows, v_t = _prefill_inputs(case, seed)
    return {"kind": "mla_prefill", "q": q, "k_nope": k_nope, "rows": rows, "v_t": v_t, "kv": case["ctx"]}


def run(state):
    if state["kind"] == "moe":
        return state["h"].forward(state["x"], state["ids"], state["w"])
    if state["kind"] == "linear":
        return state["h"].forward(state["x"])
    if state["kind"] == "mla_decode":
        state["wrapper"].plan(*state["plan"])
        cache = state["cache"]
        return state["wrapper"].run(state["q_nope"], state["q_pe"], cache[:, :, :LORA], cache[:, :, LORA:])
    q = state["q"]
    return mla_prefill(q[:, :, :128], q[:, :, 128:], state["k_nope"], state["rows"][:, LORA:], state["v_t"], state["kv"], _sm_scale())


def work(case):
    """Each weight that the routing names, each input and each output once; two operations per multiply-add."""
    if case["kind"] == "moe":
        T, k, H, I = case["T"], case["k"], case["H"], case["I"]
        used = len(np.unique(_routing(case, 0)[0]))
        per_weight = {"AMXINT4": 0.5, "FP8": 1.0 + 4 / 16384, "RAWINT4": 0.5 + 2 / 32, "GGUF": 144 / 256}[case["fmt"]]
        rows = 4 * (2 * I + H) if case["fmt"] == "AMXINT4" else 0
        return {"bytes": used * (3 * H * I * per_weight + rows) + T * (4 * H + 12 * k), "flops": 6 * T * k * H * I}
    if case["kind"] == "linear":
        per_weight = {"W4": 0.5 + 2 / 64, "FP8": 1.0 + 4 / 16384, "BF16": 2.0}[case["fmt"]]
        return {"bytes": case["K"] * case["N"] * per_weight + 2 * case["T"] * (case["K"] + case["N"]), "flops": 2 * case["T"] * case["K"] * case["N"]}
    if case["kind"] == "mla_decode":
        tokens = int(_lengths(case, 0).sum())
        return {"bytes": tokens * (LORA + ROPE) * 2 + case["B"] * case["heads"] * (2 * LORA + ROPE) * 2, "flops": 2 * case["heads"] * tokens * (2 * LORA + ROPE)}
    T, kv, H = case["T"], case["ctx"], case["heads"]
    seen = T * kv - T * (T - 1) // 2
    return {"bytes": 2 * (H * kv * 256 + kv * ROPE + T * H * (192 + 128)), "flops": 2 * H * seen * (192 + 128)}


def tolerance(case):
    """About four times what the paths differ by from the 64-bit statement.  That is the rounding of bf16 results and intermediates (0.002 to
    0.004 over all), and in the formats that quantise activations to 8 bits the codes that these roundings move (0.005 with Q8_K, 0.007 with
    a scale per 32, 0.012 with one scale per row; the FP8 linear 0.0034)."""
    if case["kind"] == "moe":
        return {"AMXINT4": {"rel": 0.03, "max": 0.4}, "RAWINT4": {"rel": 0.025, "max": 0.2}, "GGUF": {"rel": 0.02, "max": 0.15}, "FP8": {"rel": 0.015, "max": 0.1}}[case["fmt"]]
    if case["kind"] == "linear":
        return {"rel": 0.013, "max": 0.1} if case["fmt"] == "FP8" else {"rel": 0.008, "max": 0.04}
    return {"rel": 0.008, "max": 0.1}


# ---- the same calls in 64-bit arithmetic ------------------------------------------------------------------------------------------------


def _int8_rows(x, group):
    """x with each group of a row as int8 codes times its scale (largest magnitude / 127), in 64 bits."""
    g = x.view(x.shape[0], -1, group)
    d = g.abs().amax(-1, keepdim=True) / 127.0
    return (torch.round(g / torch.where(d > 0, d, torch.ones_like(d))).clamp(-128, 127) * d).view(x.shape)


def _q8_k(x):
    """x as ggml's Q8_K: per 256, the element of largest magnitude becomes -127."""
    g = x.view(x.shape[0], -1, 256)
    top = torch.gather(g, 2, g.abs().argmax(-1, keepdim=True))
    inv = torch.where(top != 0, -127.0 / top, torch.zeros_like(top))
    return (torch.round(g * inv).clamp(max=127) * torch.where(top != 0, 1 / inv, torch.zeros_like(top))).view(x.shape)


def _dequantised(case, tensors, e):
    """Expert e's matrix in 64 bits, as its format defines the values."""
    fmt, w = case["fmt"], tensors[0][e]
    if fmt == "AMXINT4":   # per row d = max / 112, codes rounded to int8 and then to a multiple of 16, both as the format's converter does in 32 bits
        f = w.float()
        d = (f.abs().amax(1, keepdim=True).double() / 112.0).float()
        i = torch.round(f * (1.0 / d)).clamp(-128, 127)
        return (torch.sign(i) * torch.floor((i.abs() + 8) / 16) * 16).double() * d.double()
    if fmt == "FP8":
        return _fp8_blocks(w, tensors[1][e])
    if fmt == "RAWINT4":
        q = torch.stack(((w & 15), (w >> 4)), dim=-1).view(w.shape[0], -1).double() - 8.0
        return (q.view(w.shape[0], -1, 32) * tensors[1][e].double().unsqueeze(-1)).view(w.shape[0], -1)
    d, dmin = (w[..., a:a + 2].contiguous().view(torch.float16).double() for a in (0, 2))     # [n, blocks, 1]
    s = w[..., 4:16].int()
    scale = torch.cat((s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)), -1).double()
    low = torch.cat((s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)), -1).double()
    q = w[..., 16:].view(*w.shape[:2], 4, 32)
    q = torch.stack((q & 15, q >> 4), dim=3).view(*w.shape[:2], 8, 32).double()
    return ((d * scale).unsqueeze(-1) * q - (dmin * low).unsqueeze(-1)).view(w.shape[0], -1)


def _fp8_blocks(w, scale):
    s = scale.double().repeat_interleave(128, 0)[:w.shape[0]].repeat_interleave(128, 1)[:, :w.shape[1]]
    return w.to(torch.float32).double() * s


def _moe_exact(case, seed):
    tensors = [_moe_weights(case, seed, m) for m in range(3)]
    ids, weights = (torch.from_numpy(a).cuda() for a in _routing(case, seed))
    x = _normal((case["T"], case["H"]), seed, 1).double()
    seen = {"AMXINT4": lambda v: _int8_rows(v, v.shape[1]), "RAWINT4": lambda v: _int8_rows(v, 32), "GGUF": _q8_k, "FP8": lambda v: v}[case["fmt"]]
    xq, y = seen(x), torch.zeros_like(x)
    for e in range(case["E"]):
        t, j = torch.nonzero(ids == e, as_tuple=True)
        if t.numel():
            g, u = (xq[t] @ _dequantised(case, tensors[m], e).t() for m in (0, 1))
            a = seen(g / (1 + torch.exp(-g)) * u)
            y.index_add_(0, t, (a @ _dequantised(case, tensors[2], e).t()) * weights[t, j].double().unsqueeze(1))
    return y


def _linear_exact(case, seed):
    x, w = _normal((case["T"], case["K"]), seed, 1), _linear_weights(case, seed)
    if case["fmt"] == "BF16":
        return x.double() @ w[0].double().t()
    if case["fmt"] == "FP8":   # activations in e4m3 with one 32-bit scale (largest magnitude / 448) per 128 inputs
        f = x.float().view(case["T"], -1, 128)
        s = f.abs().amax(-1, keepdim=True) / 448.0
        a = (f / s).to(torch.float8_e4m3fn).to(torch.float32).double() * s.double()
        return a.view(x.shape) @ _fp8_blocks(*w).t()
    # 4 bits per weight: scale = max * 2 / 15 per 64 inputs and code = round(w / scale), in the weights' own bf16; the multiplicand is a bf16 too
    g = w[0].view(case["N"], -1, 64)
    s = g.abs().amax(2, keepdim=True) * (2 / 15)
    q = torch.clamp(torch.round(g / s).float() + 8, 0, 15) - 8
    return x.double() @ (q * s.float()).to(torch.bfloat16).double().view(w[0].shape).t()


def _decode_exact(case, seed):
    n, first, table, q_nope, q_pe, cache = _decode_inputs(case, seed)
    out = []
    for b in range(case["B"]):
        rows = cache[torch.from_numpy(table[first[b]:first[b + 1]]).long().cuda()].view(-1, LORA + ROPE)[:int(n[b])].double()
        q = torch.cat((q_nope[b], q_pe[b]), dim=1).double()
        out.append(torch.softmax(q @ rows.t() * _sm_scale(), dim=1) @ rows[:, :LORA])
    return torch.stack(out)


def _prefill_exact(case, seed):
    q, k_nope, rows, v_t = _prefill_inputs(case, seed)
    T, kv = case["T"], case["ctx"]
    hidden = torch.ones((T, kv), dtype=torch.bool, device="cuda").triu(kv - T + 1)
    out = torch.empty((T, case["heads"], 128), dtype=torch.float64, device="cuda")
    for h in range(case["heads"]):
        k = torch.cat((k_nope[h, :kv], rows[:, LORA:]), dim=1).double()
        s = (q[:, h].double() @ k.t() * _sm_scale()).masked_fill_(hidden, -math.inf)
        out[:, h] = torch.softmax(s, dim=1) @ v_t[h, :, :kv].double().t()
    return out


def exact(case, seed):
    return {"moe": _moe_exact, "linear": _linear_exact, "mla_decode": _decode_exact, "mla_prefill": _prefill_exact}[case["kind"]](case, seed)
