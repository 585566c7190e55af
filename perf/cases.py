"""The work a program has this framework do, as measurable cases: the
dequant-fused matvec / matmul, the routed MoE layer, one decode step of a
whole (short) model and the MLA attention, each through its public entry
point on device-resident tensors, from the smallest call to the largest.

Sizes are those of the repository's own configurations and benchmark (the
stories15M and Qwen3-30B-A3B shapes, the DeepSeek-V3-class layer, the matvec
sweep) or generic ragged ones.  Weights are seeded GGML blocks built here in
torch (quants uniform over their range, scales set so the dequantized values
have a standard deviation of about 0.02, as the benchmark's are) and
converted once to the device layout, as a program does at load.
"""
import math

import numpy as np
import torch

import loom_amd
from loom_amd import COMBINE_EXPERT_ASC, COMBINE_SELECTION, GATING_SIGMOID, GATING_SOFTMAX
from loom_amd import NUMERICS_FAST, NUMERICS_PARITY, Q4_0, Q4_K, Q6_K, Q8_0
from loom_amd import backend as be
from loom_amd.frame import Decoder, DeviceModel, qwen3_30b_a3b, stories15m

TYPES = {"q4_0": Q4_0, "q8_0": Q8_0, "q4_k": Q4_K, "q6_k": Q6_K}
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210)}  # (values, GGML bytes)
STD = 0.02


def listed():
    return [
        # one small projection at one token: the latency of a call
        {"name": "matvec_small", "kind": "matmul", "t": "q4_0", "n": 1, "rows": 768, "cols": 2048},
        # a square projection for a handful of concurrent sequences
        {"name": "matmul_lanes", "kind": "matmul", "t": "q8_0", "n": 6, "rows": 4096, "cols": 4096},
        # a short prompt through a matrix whose sizes fit no tile
        {"name": "matmul_ragged", "kind": "matmul", "t": "q6_k", "n": 77, "rows": 1003, "cols": 2816},
        # prefill: 512 prompt tokens through the query projection
        {"name": "matmul_prefill", "kind": "matmul", "t": "q4_k", "n": 512, "rows": 4096, "cols": 2048},
        # the routed layer in single-sequence decode
        {"name": "moe_token", "kind": "moe", "n": 1, "dim": 2048, "ffn": 768, "experts": 128, "used": 8,
         "gate": "q4_k", "down": "q6_k", "sigmoid": False, "shared": 0},
        # a Q4_0 model's routed layer for an odd number of sequences
        {"name": "moe_lanes", "kind": "moe", "n": 13, "dim": 2048, "ffn": 768, "experts": 128, "used": 8,
         "gate": "q4_0", "down": "q4_0", "sigmoid": False, "shared": 0},
        # the routed layer in a large decode batch or a prefill chunk
        {"name": "moe_batch", "kind": "moe", "n": 128, "dim": 2048, "ffn": 768, "experts": 128, "used": 8,
         "gate": "q4_k", "down": "q6_k", "sigmoid": False, "shared": 0},
        # a DeepSeek-class layer (sigmoid gating, shared expert) in batched decode
        {"name": "moe_shared", "kind": "moe", "n": 24, "dim": 7168, "ffn": 2048, "experts": 64, "used": 8,
         "gate": "q4_k", "down": "q4_k", "sigmoid": True, "shared": 2048},
        # one token of one sequence at a long context, whole call to logits
        {"name": "decode_token", "kind": "decode", "model": "qwen3", "layers": 2, "n": 1, "ctx": 4096, "fast": False},
        # one step of 32 sequences of different lengths, whole call to logits
        {"name": "decode_lanes", "kind": "decode", "model": "qwen3", "layers": 2, "n": 32, "ctx": 4096,
         "fast": False},
        # a small dense model's token: launch-bound
        {"name": "decode_dense", "kind": "decode", "model": "stories", "layers": 6, "n": 1, "ctx": 200, "fast": False},
        # latent attention of one layer at a long context
        {"name": "mla_attn", "kind": "mla", "t": "q4_k", "heads": 128, "seq": 4096},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("matmul", "matmul", "matmul", "moe", "moe", "decode", "decode", "mla"))
    if kind == "matmul":
        t = rng.choice(sorted(TYPES))
        bv = BLOCK[t][0]
        while True:
            n, rows = _log_int(rng, 1, 512), _log_int(rng, 256, 16384)
            cols = bv * _log_int(rng, 256 // bv, 8192 // bv)
            if n * rows * cols <= 512 * 4096 * 2048 and rows * cols <= 4096 * 8192:
                return {"kind": kind, "t": t, "n": n, "rows": rows, "cols": cols}
    if kind == "moe":
        dim, ffn, experts, used = rng.choice(((2048, 768, 128, 8), (1024, 512, 32, 4), (1536, 1280, 60, 6),
                                              (7168, 2048, 16, 4)))
        gate, down = rng.choice((("q4_k", "q6_k"), ("q4_k", "q4_k"), ("q8_0", "q8_0"), ("q4_0", "q4_0")))
        n = _log_int(rng, 1, 128 if dim <= 2048 else 32)
        return {"kind": kind, "n": n, "dim": dim, "ffn": ffn, "experts": experts, "used": used, "gate": gate,
                "down": down, "sigmoid": rng.random() < 0.5, "shared": rng.choice((0, 0, ffn))}
    if kind == "decode":
        if rng.random() < 0.6:
            return {"kind": kind, "model": "qwen3", "layers": 2, "n": _log_int(rng, 1, 32),
                    "ctx": _log_int(rng, 16, 4096), "fast": rng.random() < 0.4}
        return {"kind": kind, "model": "stories", "layers": 6, "n": _log_int(rng, 1, 32), "ctx": _log_int(rng, 8, 250),
                "fast": rng.random() < 0.4}
    return {"kind": kind, "t": rng.choice(("q4_k", "q6_k", "q8_0")), "heads": rng.choice((16, 64, 128)),
            "seq": _log_int(rng, 16, 4096)}


# ---- seeded inputs -----------------------------------------------------------------


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed((seed * 1000003 + salt) % (1 << 62))


def _blocks(g, t, rows, cols, planes=1):
    """Random GGML blocks [planes * rows * cols / block values][block bytes]."""
    bv, bb = BLOCK[t]
    u = planes * rows * cols // bv
    words = torch.randint(-(1 << 63), (1 << 63) - 1, ((u * bb + 7) // 8,), generator=g, device="cuda")
    raw = words.view(torch.uint8)[:u * bb].view(u, bb)
    spread = 0.75 + 0.5 * torch.rand(u, generator=g, device="cuda")  # block scales differ

    def put(off, scale):
        raw[:, off:off + 2] = scale.to(torch.float16).view(torch.uint8).view(u, 2)

    if t == "q4_k":
        raw[:, 4:16] = (raw[:, 4:16] & 0xD7) | 0x28  # scales and mins in their upper range
        put(0, spread * (STD / (4.6 * 52.0)))
        put(2, spread * (7.5 * STD / (4.6 * 52.0)))
    elif t == "q6_k":
        s = raw[:, 192:208]
        m = 64 + (s & 63).to(torch.int16)  # |scale| in 64..127
        raw[:, 192:208] = torch.where(s >= 128, -m, m).to(torch.int8).view(torch.uint8)
        put(208, spread * (STD / (18.5 * 96.0)))
    elif t == "q8_0":
        q = raw[:, 2:34]
        raw[:, 2:34] = torch.where(q == 128, torch.full_like(q, 129), q)  # -128 is not a Q8_0 quant
        put(0, spread * (STD / 73.0))
    else:
        put(0, spread * (STD / 4.6))
    return raw.reshape(-1)


def _device(t, raw, rows, cols, planes=1):
    return be.repack_dev(TYPES[t], raw, rows, cols, planes)


def _randn(g, *shape, scale=1.0):
    return torch.randn(shape, generator=g, device="cuda") * scale


def _router(g, experts, dim):
    """A router with Zipf(1.1)-skewed logits, as the benchmark's."""
    w = _randn(g, experts, dim, scale=1.0 / math.sqrt(dim)).contiguous()
    z = -1.1 * torch.log(torch.randperm(experts, generator=g, device="cuda").float() + 1)
    return w, (z - z.mean()).contiguous()


def _moe_tensors(case):
    """(name, type, rows, cols, planes) of a MoE case's matrices."""
    d, f, e, s = case["dim"], case["ffn"], case["experts"], case["shared"]
    out = [("gate", case["gate"], f, d, e), ("up", case["gate"], f, d, e), ("down", case["down"], d, f, e)]
    if s:
        out += [("sgate", case["gate"], s, d, 1), ("sup", case["gate"], s, d, 1), ("sdown", case["down"], d, s, 1)]
    return out


def _spec(case):
    """The model of a decode case; the cache holds the context and a margin."""
    if case["model"] == "qwen3":
        return qwen3_30b_a3b(ctx_len=(case["ctx"] + 64 + 63) // 64 * 64, n_layers=case["layers"])
    return stories15m(ctx_len=256)


def _spec_tensors(s):
    """(name, type, rows, cols, planes) of a decode model's matrices."""
    name = {v: k for k, v in TYPES.items()}
    out = [("embed", s.embed_t, s.vocab, s.dim, 1), ("output", s.output_t, s.vocab, s.dim, 1)]
    for li in range(s.n_layers):
        p = f"l{li}."
        out += [(p + "wq", s.wq_t, s.qd, s.dim, 1), (p + "wk", s.wk_t, s.kvd, s.dim, 1),
                (p + "wv", s.wv_t, s.kvd, s.dim, 1), (p + "wo", s.wo_t, s.dim, s.qd, 1)]
        if s.n_expert:
            out += [(p + "gate", s.moe_gate_t, s.moe_ffn, s.dim, s.n_expert),
                    (p + "up", s.moe_gate_t, s.moe_ffn, s.dim, s.n_expert),
                    (p + "down", s.moe_down_t, s.dim, s.moe_ffn, s.n_expert)]
        else:
            out += [(p + "ffn_gate", s.ffn_gate_t, s.ffn, s.dim, 1), (p + "ffn_up", s.ffn_gate_t, s.ffn, s.dim, 1),
                    (p + "ffn_down", s.ffn_down_t, s.dim, s.ffn, 1)]
    return [(n, name[t], r, c, pl) for n, t, r, c, pl in out]


def _positions(case, seed):
    """Sequence lengths of a decode case: one lane at the context, more lanes
    spread over the upper half of it, up to 16 lengths (neighbouring lanes of a
    wide batch share one: samples of one prompt)."""
    n, ctx = case["n"], case["ctx"]
    if n == 1:
        return [ctx]
    r = np.random.default_rng(seed)
    share = -(-n // 16)
    lens = [int(v) for v in r.integers((ctx + 1) // 2, ctx + 1, -(-n // share))]
    return [lens[lane // share] for lane in range(n)]


def _runs(pos):
    """(first lane, end lane, position) of neighbouring lanes that share one."""
    out = []
    for lane, p in enumerate(pos):
        if out and out[-1][2] == p:
            out[-1][1] = lane + 1
        else:
            out.append([lane, lane + 1, p])
    return out


def _kv_rows(seed, lane, which, layers, pos, kvd):
    """The cached fp16 rows of one lane: [layers][pos][kvd]."""
    return _randn(_gen(seed, 7000 + 2 * lane + which), layers, pos, kvd, scale=0.5).to(torch.float16)


def prepare(case, seed):
    loom_amd.init(0)
    kind = case["kind"]
    g = _gen(seed, 1)
    if kind == "matmul":
        t, n, rows, cols = case["t"], case["n"], case["rows"], case["cols"]
        return {"kind": kind, "t": TYPES[t], "n": n, "rows": rows, "cols": cols,
                "w": _device(t, _blocks(g, t, rows, cols), rows, cols), "x": _randn(g, n, cols),
                "out": torch.empty(n, rows, device="cuda")}
    if kind == "moe":
        n, dim = case["n"], case["dim"]
        router, bias = _router(g, case["experts"], dim)
        w = {nm: _device(t, _blocks(_gen(seed, 10 + i), t, r, c, p), r, c, p)
             for i, (nm, t, r, c, p) in enumerate(_moe_tensors(case))}
        gt, dt = TYPES[case["gate"]], TYPES[case["down"]]
        sh = (w["sgate"], w["sup"], w["sdown"], gt, gt, dt, case["shared"]) if case["shared"] else None
        layer = be.MoeLayer(dim, case["ffn"], case["experts"], case["used"], router, w["gate"], w["up"], w["down"],
                            gt, gt, dt, router_bias=bias,
                            gating=GATING_SIGMOID if case["sigmoid"] else GATING_SOFTMAX, weights_norm=True,
                            weights_scale=2.5 if case["sigmoid"] else 1.0, shexp=sh)
        return {"kind": kind, "layer": layer, "x": _randn(g, n, dim), "out": torch.empty(n, dim, device="cuda"),
                "ids": torch.empty(n, case["used"], dtype=torch.int32, device="cuda"),
                "gates": torch.empty(n, case["used"], device="cuda"),
                "combine": COMBINE_SELECTION if n == 1 else COMBINE_EXPERT_ASC}
    if kind == "decode":
        s = _spec(case)
        m = DeviceModel.synth(s, seed=seed % 100000 + 1)
        for i, (nm, t, r, c, p) in enumerate(_spec_tensors(s)):
            m.tensors[nm].dev.copy_(_device(t, _blocks(_gen(seed, 100 + i), t, r, c, p), r, c, p))
        for li in range(s.n_layers if s.n_expert else 0):
            router, bias = _router(_gen(seed, 5000 + li), s.n_expert, s.dim)
            m.f32[f"l{li}.router"].copy_(router)
            m.f32[f"l{li}.router_bias"].copy_(bias)
        m.set_numerics(NUMERICS_FAST if case["fast"] else NUMERICS_PARITY)
        dec = Decoder(m, case["n"])
        pos = _positions(case, seed)
        for lane, p in enumerate(pos):
            dec.k_cache[lane, :, :p] = _kv_rows(seed, lane, 0, s.n_layers, p, s.kvd).view(torch.int16)
            dec.v_cache[lane, :, :p] = _kv_rows(seed, lane, 1, s.n_layers, p, s.kvd).view(torch.int16)
        tok = torch.randint(0, s.vocab, (case["n"],), generator=g, device="cuda").to(torch.int32)
        # the appended cache rows, seen in place
        rows = [c.view(torch.float16)[a:b, :, p] for a, b, p in _runs(pos) for c in (dec.k_cache, dec.v_cache)]
        return {"kind": kind, "dec": dec, "tok": tok, "pos": torch.tensor(pos, dtype=torch.int32, device="cuda"),
                "rows": rows}
    t, h, seq = case["t"], case["heads"], case["seq"]
    nope, rope, kvr, vd = 128, 64, 512, 128
    kv_b = _blocks(g, t, h * (nope + vd), kvr)
    attn = be.MlaAttn(TYPES[t], kv_b, h, nope, vd, kvr, rope, 1.0 / math.sqrt(nope + rope))
    return {"kind": kind, "attn": attn, "seq": seq, "c": _randn(g, seq, kvr), "r": _randn(g, seq, rope),
            "qn": _randn(g, h, nope), "qr": _randn(g, h, rope), "out": torch.empty(h, vd, device="cuda")}


def run(st):
    kind = st["kind"]
    if kind == "matmul":
        be.matvec_dev(st["t"], st["out"], st["w"], st["x"], st["n"], st["rows"], st["cols"])
        return st["out"]
    if kind == "moe":
        if st["combine"] == COMBINE_EXPERT_ASC:  # the batched form adds to its accumulator
            st["out"].zero_()
        st["layer"](st["x"], st["out"], st["combine"], ids=st["ids"], gates=st["gates"])
        return st["out"], st["ids"], st["gates"]
    if kind == "decode":
        # the step advances the positions; a repeated pass starts from the same ones
        st["dec"].pos.copy_(st["pos"])
        st["dec"].step(tokens=st["tok"])
        return [st["dec"].logits] + st["rows"]
    st["attn"](st["c"], st["r"], st["seq"], st["qn"], st["qr"], st["out"])
    return st["out"]


# ---- what a pass cannot do without ---------------------------------------------------


def _bytes(t, rows, cols):
    return rows * cols // BLOCK[t][0] * BLOCK[t][1]


def _distinct(n, experts, used):
    """Experts that n tokens reach under the Zipf-skewed router (simulated)."""
    r = np.random.default_rng(0)
    z = -1.1 * np.log(np.arange(1, experts + 1))
    tops = [len(np.unique(np.argsort(-(r.standard_normal((n, experts)) + z), axis=1)[:, :used])) for _ in range(4)]
    return float(np.mean(tops))


def _moe_work(n, dim, ffn, experts, used, gate, down, shared):
    e = _distinct(n, experts, used)
    b = e * (2 * _bytes(gate, ffn, dim) + _bytes(down, dim, ffn)) + experts * dim * 4 + 2 * n * dim * 4
    f = 2 * n * experts * dim + 6 * n * used * dim * ffn
    if shared:
        b += 2 * _bytes(gate, shared, dim) + _bytes(down, dim, shared)
        f += 6 * n * dim * shared
    return b, f


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        n, rows, cols = case["n"], case["rows"], case["cols"]
        return {"bytes": _bytes(case["t"], rows, cols) + 4 * n * (rows + cols), "flops": 2 * n * rows * cols}
    if kind == "moe":
        b, f = _moe_work(case["n"], case["dim"], case["ffn"], case["experts"], case["used"], case["gate"],
                         case["down"], case["shared"])
        return {"bytes": int(b), "flops": int(f)}
    if kind == "decode":
        s, n = _spec(case), case["n"]
        b = f = 0
        for nm, t, r, c, p in _spec_tensors(s):
            if nm == "embed":
                b += n * _bytes(t, 1, c)
            elif p == 1:
                b += _bytes(t, r, c)
                f += 2 * n * r * c
        if s.n_expert:
            mb, mf = _moe_work(n, s.dim, s.moe_ffn, s.n_expert, s.n_used, "q4_k", "q6_k", 0)
            b, f = b + s.n_layers * mb, f + s.n_layers * mf
        pos = sum(_positions(case, 0))
        b += s.n_layers * pos * s.kvd * 4 + n * s.vocab * 4
        f += s.n_layers * pos * s.qd * 4
        return {"bytes": int(b), "flops": int(f)}
    h, seq = case["heads"], case["seq"]
    return {"bytes": _bytes(case["t"], h * 256, 512) + seq * 576 * 4 + h * (192 + 128) * 4,
            "flops": 2 * h * (256 * 512 + seq * (576 + 512))}


def tolerance(case):
    """About four times the largest distance the path shows from the 64-bit
    result over the listed and some thirty drawn cases: 8.2e-7 for a matmul
    (f32 sums of exact integer dots, up to 256 of them); 1.1e-4 where an activation is rounded to
    int8 twice and a last-bit difference can move a rounding (the MoE layer,
    the latent attention 0.8e-4); 1.5e-2 for the two-layer and 2.5e-2 for the
    six-layer decode, where such steps travel through every later layer."""
    if case["kind"] == "matmul":
        return {"rel": 3e-6}
    if case["kind"] == "moe":
        return {"rel": 5e-4, "differ": 1e-3}
    if case["kind"] == "mla":
        return {"rel": 3e-4}
    return {"rel": 6e-2 if case["model"] == "qwen3" else 1e-1}


# ---- the same in 64 bits ---------------------------------------------------------------


def _f16(raw, off):
    return raw[:, off:off + 2].contiguous().view(torch.float16).double()


def _dequant(t, raw, rows, cols):
    """GGML blocks -> f64 [rows][cols]."""
    raw = raw.view(-1, BLOCK[t][1])
    u = raw.shape[0]
    if t == "q4_k":
        a, b, c = (raw[:, k:k + 4].int() for k in (4, 8, 12))
        sc = torch.cat([a & 63, (c & 15) | ((a >> 6) << 4)], 1).double()
        mn = torch.cat([b & 63, (c >> 4) | ((b >> 6) << 4)], 1).double()
        q = raw[:, 16:].view(u, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).view(u, 8, 32).double()
        v = (_f16(raw, 0) * sc)[..., None] * q - (_f16(raw, 2) * mn)[..., None]
    elif t == "q6_k":
        ql, qh = raw[:, :128].view(u, 2, 64).int(), raw[:, 128:192].view(u, 2, 32).int()
        lo, hi = ql[..., :32], ql[..., 32:]
        q = torch.stack([(lo & 15) | ((qh & 3) << 4), (hi & 15) | (((qh >> 2) & 3) << 4),
                         (lo >> 4) | (((qh >> 4) & 3) << 4), (hi >> 4) | (((qh >> 6) & 3) << 4)], 2) - 32
        sc = raw[:, 192:208].contiguous().view(torch.int8).double()
        v = (_f16(raw, 208) * sc)[..., None] * q.view(u, 16, 16).double()
    elif t == "q8_0":
        v = _f16(raw, 0) * raw[:, 2:].contiguous().view(torch.int8).double()
    else:
        q = raw[:, 2:].int()
        v = _f16(raw, 0) * (torch.cat([q & 15, q >> 4], 1) - 8).double()
    return v.reshape(rows, cols)


def _plane(t, raw, rows, cols, p):
    nb = _bytes(t, rows, cols)
    return _dequant(t, raw[p * nb:(p + 1) * nb], rows, cols)


def _act(t, x):
    """Activations as the int8 formats hold them: one scale per 256 (K
    quants) or 32 values, rounded to nearest in f32 -- the format's own
    definition -- and widened."""
    bv = BLOCK[t][0]
    v = x.float().reshape(-1, bv)
    d = v.abs().amax(1, keepdim=True) / 127.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    y = v * inv
    q = torch.where(y >= 0, (y + 0.5).floor(), (y - 0.5).ceil()).clamp(-127, 127)
    return (q.double() * d.double()).reshape(x.shape)


def _linear(t, w, x):
    return _act(t, x) @ w.t()


def _silu(x):
    return x / (1.0 + torch.exp(-x))


def _moe_exact(x, router, bias, used, sigmoid, wscale, gate_t, down_t, plane, shared):
    """x f64 [n][dim]; plane(name, e) the f64 matrix of expert e."""
    logits = x @ router.double().t() + bias.double()
    p = torch.sigmoid(logits) if sigmoid else torch.softmax(logits, 1)
    ids = torch.sort(p, dim=1, descending=True, stable=True).indices[:, :used]
    gates = torch.gather(p, 1, ids)
    gates = gates / gates.sum(1, keepdim=True) * wscale
    out = torch.zeros_like(x)
    for e in ids.unique().tolist():
        t, s = (ids == e).nonzero(as_tuple=True)
        h = _silu(_linear(gate_t, plane("gate", e), x[t])) * _linear(gate_t, plane("up", e), x[t])
        out.index_add_(0, t, gates[t, s][:, None] * _linear(down_t, plane("down", e), h))
    if shared:
        h = _silu(_linear(gate_t, plane("sgate", 0), x)) * _linear(gate_t, plane("sup", 0), x)
        out += _linear(down_t, plane("sdown", 0), h)
    return out, ids, gates


def _rope(x, pos, base, dim, neox):
    """x [..., head_dim] rotated at pos."""
    i = torch.arange(dim // 2, device="cuda", dtype=torch.float64)
    a = pos * base ** (-2.0 * i / dim)
    c, s = torch.cos(a), torch.sin(a)
    y = x.clone()
    if neox:
        u, v = x[..., :dim // 2], x[..., dim // 2:dim]
        y[..., :dim // 2], y[..., dim // 2:dim] = u * c - v * s, u * s + v * c
    else:
        u, v = x[..., 0:dim:2], x[..., 1:dim:2]
        y[..., 0:dim:2], y[..., 1:dim:2] = u * c - v * s, u * s + v * c
    return y


def _decode_exact(case, seed):
    s, n = _spec(case), case["n"]
    mats = {nm: (t, _blocks(_gen(seed, 100 + i), t, r, c, p), r, c)
            for i, (nm, t, r, c, p) in enumerate(_spec_tensors(s))}
    g = _gen(seed, 1)
    tok = torch.randint(0, s.vocab, (n,), generator=g, device="cuda")
    pos = _positions(case, seed)

    def lin(nm, x):
        t, raw, r, c = mats[nm]
        return _linear(t, _plane(t, raw, r, c, 0), x)

    def norm(x):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + s.eps)

    t, raw, r, c = mats["embed"]
    x = torch.cat([_plane(t, raw, 1, c, int(k)) for k in tok.tolist()])
    heads, group = s.n_heads, s.n_heads // s.n_kv_heads
    krows, vrows = [[] for _ in pos], [[] for _ in pos]
    for li in range(s.n_layers):
        p = f"l{li}."
        y = norm(x)
        q = lin(p + "wq", y).view(n, heads, s.head_dim)
        k = lin(p + "wk", y).view(n, s.n_kv_heads, s.head_dim)
        v = lin(p + "wv", y)
        if s.qk_norm:
            q, k = norm(q), norm(k)
        att = torch.empty(n, heads, s.head_dim, dtype=torch.float64, device="cuda")
        for lane, ps in enumerate(pos):
            kr = _rope(k[lane], ps, s.rope_base, s.rope_dim, s.rope_neox).reshape(-1).to(torch.float16)
            vr = v[lane].to(torch.float16)
            krows[lane].append(kr)
            vrows[lane].append(vr)
            ks = torch.cat([_kv_rows(seed, lane, 0, s.n_layers, ps, s.kvd)[li], kr[None]]).double()
            vs = torch.cat([_kv_rows(seed, lane, 1, s.n_layers, ps, s.kvd)[li], vr[None]]).double()
            qr = _rope(q[lane], ps, s.rope_base, s.rope_dim, s.rope_neox)
            for h in range(s.n_kv_heads):
                sl, hd = slice(h * group, (h + 1) * group), slice(h * s.head_dim, (h + 1) * s.head_dim)
                w = torch.softmax(qr[sl] @ ks[:, hd].t() / math.sqrt(s.head_dim), 1)
                att[lane, sl] = w @ vs[:, hd]
        x = x + lin(p + "wo", att.view(n, -1))
        y = norm(x)
        if s.n_expert:
            router, bias = _router(_gen(seed, 5000 + li), s.n_expert, s.dim)

            def plane(nm, e, p=p):
                t, raw, r, c = mats[p + nm]
                return _plane(t, raw, r, c, e)

            x = x + _moe_exact(y, router, bias, s.n_used, False, 1.0, "q4_k", "q6_k", plane, 0)[0]
        else:
            x = x + lin(p + "ffn_down", _silu(lin(p + "ffn_gate", y)) * lin(p + "ffn_up", y))
    rows = [torch.stack([torch.stack(r) for r in c[a:b]]) for a, b, _ in _runs(pos) for c in (krows, vrows)]
    return [lin("output", norm(x))] + rows


def exact(case, seed):
    kind = case["kind"]
    g = _gen(seed, 1)
    if kind == "matmul":
        t, n, rows, cols = case["t"], case["n"], case["rows"], case["cols"]
        w = _dequant(t, _blocks(g, t, rows, cols), rows, cols)
        return _linear(t, w, _randn(g, n, cols))
    if kind == "moe":
        router, bias = _router(g, case["experts"], case["dim"])
        mats = {nm: (t, _blocks(_gen(seed, 10 + i), t, r, c, p), r, c)
                for i, (nm, t, r, c, p) in enumerate(_moe_tensors(case))}

        def plane(nm, e):
            t, raw, r, c = mats[nm]
            return _plane(t, raw, r, c, e)

        x = _randn(g, case["n"], case["dim"]).double()
        out, ids, gates = _moe_exact(x, router, bias, case["used"], case["sigmoid"],
                                     2.5 if case["sigmoid"] else 1.0, case["gate"], case["down"], plane,
                                     case["shared"])
        return out, ids.int(), gates
    if kind == "decode":
        return _decode_exact(case, seed)
    t, h, seq = case["t"], case["heads"], case["seq"]
    nope, rope, kvr, vd = 128, 64, 512, 128
    w = _dequant(t, _blocks(g, t, h * (nope + vd), kvr), h * (nope + vd), kvr).view(h, nope + vd, kvr)
    c, r = _randn(g, seq, kvr).double(), _randn(g, seq, rope).double()
    qn, qr = _randn(g, h, nope).double(), _randn(g, h, rope).double()
    qa = (qn[:, :, None] * w[:, :nope]).sum(1)
    p = torch.softmax((qa @ c.t() + qr @ r.t()) / math.sqrt(nope + rope), 1)
    o = _act(t, p @ c)
    return (w[:, nope:] * o[:, None, :]).sum(2)
