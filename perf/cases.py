"""What a program of this framework has it do, as timed cases.

Each case is one call (or, for a whole token, one stack call) of the public
entry points on device data.  Weights and inputs are synthetic: weights come
from the framework's counter-based generator (every weight is a function of
the case, the seed and its index, packed on the device as the loaders'
organs are), hidden states and inputs are N(0, 1) draws.  `exact` redraws
the same weights with plain torch and evaluates the path in 64 bits.
"""
from __future__ import annotations

import ctypes as C
import math
from types import SimpleNamespace

import torch

from hawking_amd import moe, organs, runtime
from hawking_amd._lib import HK_BIN, HK_BIN_RICE, HK_MIXED, HK_Q4, HK_Q8, HK_U3

KINDS = {"q4": HK_Q4, "bin": HK_BIN, "mixed": HK_MIXED, "q8": HK_Q8, "u3": HK_U3, "rice": HK_BIN_RICE}
SIGMA = 0.02


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # the smallest call: one residual-coded matrix (an expert's up
        # projection) times one vector, where launches and latency count
        dict(name="organ_rice_512x2048", op="gemv", kind="rice", group=128, rows=512, cols=2048, n=1),
        # one projection of a wide model at batch 1 (4-bit, 7168 columns)
        dict(name="organ_q4_2048x7168", op="gemv", kind="q4", group=32, rows=2048, cols=7168, n=1),
        # a routed wave: the gate and up matrices of ten experts in one call
        dict(name="wave_mixed_20x512x2048", op="gemv", kind="mixed", group=128, rows=512, cols=2048, n=20),
        # many matrices streamed from HBM in one call, one bit a weight ...
        dict(name="stream_bin_8192x512x2048", op="gemv", kind="bin", group=128, rows=512, cols=2048, n=8192),
        # ... and in the mixed format of 1.45 bits a weight
        dict(name="stream_mixed_4096x512x2048", op="gemv", kind="mixed", group=128, rows=512, cols=2048, n=4096),
        # the low-rank down projections (3-bit factors) of many experts
        dict(name="stream_lowrank_2048x2048x160x768", op="lowrank", rows=2048, rank=160, cols=768, n=2048),
        # the end of every token: final norm, 8-bit lm_head, greedy pick
        dict(name="head_q8_151936x2048", op="head", kind="q8", group=64, rows=151936, cols=2048, n_valid=151669),
        # one MoE layer of a token, 4-bit experts
        dict(name="layer_q4_2048x512", op="stack", kind="q4", group=32, n_layers=1, hidden=2048, inter=512,
             shared_inter=512, n_experts=512, top_k=10),
        # the whole token of the 48-layer mixed model
        dict(name="token_mixed_48", op="stack", kind="mixed", group=128, n_layers=48, hidden=2048, inter=512,
             shared_inter=512, n_experts=512, top_k=10),
        # two layers of the model whose experts mix three codecs (binary
        # gate, binary + residual up, low-rank down, 8-bit router and shared)
        dict(name="layers_mixed15_2", op="mixed15", n_layers=2, hidden=2048, inter=512, shared_inter=512,
             n_experts=512, top_k=10, rank=160),
        # 32 tokens through a 256-expert block (batched decode, prefill)
        dict(name="batch_q4_32x7168", op="batch", tokens=32, hidden=7168, inter=2048, shared_inter=2048,
             n_experts=256, top_k=8, n_group=1, topk_group=1, group=32),
        # the encode direction: a matrix of f32 weights packed to 4 bits
        dict(name="pack_q4_2048x7168", op="pack", kind="q4", group=32, rows=2048, cols=7168),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _organ_shape(rng, kind):
    group = {"q4": rng.choice((32, 64, 128)), "q8": 64, "u3": 64}.get(kind, 128)
    unit = 32 if kind == "u3" else group
    cols = unit * max(1, _log(rng, 256, 7168) // unit)
    return group, _log(rng, 16, 8192), cols


def draw(rng):
    """One more case over the ranges the listed ones stand for."""
    op = rng.choice(("one", "one", "wave", "wave", "stream", "lowrank", "head", "layer", "token", "mixed15", "batch",
                     "batch", "pack"))
    if op in ("one", "wave", "stream"):
        kind = rng.choice(tuple(KINDS))
        group, rows, cols = _organ_shape(rng, kind)
        if op != "one":
            rows, cols = min(rows, 2304), max(cols, 512)
        most = (1 << 30) if kind == "rice" else (3 << 29)  # weights of one call
        n = 1 if op == "one" else _log(rng, 2, 64) if op == "wave" else _log(rng, 64, 2048)
        return dict(op="gemv", kind=kind, group=group, rows=rows, cols=cols, n=max(1, min(n, most // (rows * cols))))
    if op == "lowrank":
        return dict(op="lowrank", rows=_log(rng, 256, 4096), rank=32 * rng.randint(1, 12),
                    cols=32 * rng.randint(8, 64), n=_log(rng, 1, 1024))
    if op == "head":
        rows = _log(rng, 4096, 160000)
        return dict(op="head", kind=rng.choice(("q8", "q8", "q4", "bin")), group=0, rows=rows,
                    cols=128 * rng.randint(4, 32), n_valid=max(1, rows - rng.randint(0, 300)))
    if op in ("layer", "token"):
        kind = rng.choice(("q4", "mixed"))
        top_k = rng.randint(2, 10)
        return dict(op="stack", kind=kind, group=32 if kind == "q4" else 128,
                    n_layers=1 if op == "layer" else rng.randint(4, 24), hidden=128 * rng.randint(4, 32),
                    inter=128 * rng.randint(1, 4), shared_inter=rng.choice((0, 128, 256, 512)),
                    n_experts=_log(rng, 16, 384), top_k=top_k)
    if op == "mixed15":
        return dict(op="mixed15", n_layers=1, hidden=128 * rng.randint(4, 20), inter=128 * rng.randint(1, 5),
                    shared_inter=64 * rng.randint(1, 8), n_experts=_log(rng, 16, 256), top_k=rng.randint(2, 10),
                    rank=32 * rng.randint(1, 6))
    if op == "batch":
        n_group = rng.choice((1, 4, 8))
        n_experts = 8 * rng.randint(4, 24)
        return dict(op="batch", tokens=_log(rng, 1, 64), hidden=128 * rng.randint(6, 48),
                    inter=128 * rng.randint(2, 14), shared_inter=128 * rng.randint(2, 14), n_experts=n_experts,
                    top_k=rng.randint(2, 8), n_group=n_group, topk_group=max(1, n_group // 2), group=32)
    kind = rng.choice(("q4", "bin", "q8", "u3"))
    group, rows, cols = _organ_shape(rng, kind)
    return dict(op="pack", kind=kind, group=group, rows=max(rows, 256), cols=max(cols, 512))


# ---------------------------------------------------------------- preparation

_CTX = None


def _ctx():
    global _CTX
    if _CTX is None:
        _CTX = runtime.Context(0)
    return _CTX


def _gen(seed, tag):
    return torch.Generator("cuda").manual_seed((seed * 1000003 + tag) & 0x7FFFFFFFFFFF)


def _randn(seed, tag, *shape):
    return torch.randn(*shape, generator=_gen(seed, tag), device="cuda", dtype=torch.float32)


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _vec(t):
    """A device vector for the calls that take an object with a .ptr."""
    return SimpleNamespace(ptr=_ptr(t), t=t)


def _pad4(n):
    return (n + 3) // 4 * 4


def _key(seed, tag):
    """Generator key of one tensor of a case."""
    return _stream_key(seed, (0xCA5E << 44) | tag)


def _head_case(case):
    group = {"q8": 64, "q4": 32}.get(case["kind"], 128)
    return dict(case, group=group, cols=case["cols"] // group * group)


def _organ(case, seed, tag, rows=None, cols=None, kind=None, sigma=SIGMA):
    return organs.SyntheticOrgan(_ctx(), KINDS[kind or case["kind"]], rows or case["rows"], cols or case["cols"],
                                 _key(seed, 2 * tag), _key(seed, 2 * tag + 1), group=case.get("group", 64),
                                 sigma=sigma)


def _moe_shape(case):
    if case["op"] == "batch":
        return moe.MoeShape(n_layers=1, hidden=case["hidden"], inter=case["inter"],
                            shared_inter=case["shared_inter"], n_experts=case["n_experts"], top_k=case["top_k"],
                            expert_kind=HK_Q4, expert_group=case["group"], shared_gate=False, router=1,
                            n_group=case["n_group"], topk_group=case["topk_group"], norm_topk_prob=True,
                            routed_scaling_factor=2.5)
    return moe.MoeShape(n_layers=case["n_layers"], hidden=case["hidden"], inter=case["inter"],
                        shared_inter=case["shared_inter"], n_experts=case["n_experts"], top_k=case["top_k"],
                        expert_kind=KINDS[case["kind"]], expert_group=case["group"])


def _mixed15_dims(case):
    return moe.Mixed15Dims(case["hidden"], case["inter"], case["shared_inter"], case["n_experts"], case["top_k"],
                           case["rank"])


def prepare(case, seed):
    ctx, op = _ctx(), case["op"]
    s = SimpleNamespace(case=case, ctx=ctx)
    if op == "gemv":
        n, rows, cols = case["n"], case["rows"], case["cols"]
        s.organs = [_organ(case, seed, i) for i in range(n)]
        s.set = organs.OrganSet(ctx, s.organs) if n > 1 else None
        s.x = _vec(_randn(seed, 1, n, cols))
        s.y = _vec(torch.zeros(n, _pad4(rows), device="cuda"))
        s.out = [s.y.t[:, :rows]]
    elif op == "lowrank":
        n, rows, rank, cols = case["n"], case["rows"], case["rank"], case["cols"]
        s.left = organs.OrganSet(ctx, [_organ(case, seed, 2 * i, rows, rank, "u3", 0.05) for i in range(n)])
        s.right = organs.OrganSet(ctx, [_organ(case, seed, 2 * i + 1, rank, cols, "u3") for i in range(n)])
        s.x = _vec(_randn(seed, 1, n, cols))
        s.y = _vec(torch.zeros(n, _pad4(rows), device="cuda"))
        s.mid = _vec(torch.zeros(n, rank, device="cuda"))
        s.out = [s.y.t[:, :rows]]
    elif op == "head":
        c = _head_case(case)
        s.organ = _organ(c, seed, 0)
        s.h = _randn(seed, 1, c["cols"])
        s.w = _randn(seed, 2, c["cols"]) * 0.02
        s.xn = torch.zeros(c["cols"], device="cuda")
        s.logits = torch.zeros(_pad4(c["rows"]), device="cuda")
        s.pick = torch.zeros(2, dtype=torch.int64, device="cuda")
        s.token = torch.zeros(1, dtype=torch.int32, device="cuda")
        s.out = [s.logits[:c["rows"]], s.token]
    elif op == "stack":
        s.model = moe.MoeModel(ctx, _moe_shape(case))
        s.model.fill_synthetic(seed)
        s.h = _randn(seed, 1, case["hidden"])
        s.y = torch.zeros(case["hidden"], device="cuda")
        s.ids = torch.zeros(case["n_layers"], case["top_k"], dtype=torch.int32, device="cuda")
        s.w = torch.zeros(case["n_layers"], case["top_k"], device="cuda")
        s.out = [s.y, s.ids, s.w]
    elif op == "mixed15":
        s.layers, _, _ = moe.synthetic_mixed15_layers(ctx, seed, case["n_layers"], _mixed15_dims(case))
        s.h = _randn(seed, 1, case["hidden"])
        s.y = torch.zeros(case["hidden"], device="cuda")
        s.ids = torch.zeros(case["n_layers"], case["top_k"], dtype=torch.int32, device="cuda")
        s.w = torch.zeros(case["n_layers"], case["top_k"], device="cuda")
        s.out = [s.y, s.ids, s.w]
    elif op == "batch":
        s.model = moe.MoeModel(ctx, _moe_shape(case))
        s.model.fill_synthetic(seed)
        s.x = _randn(seed, 1, case["tokens"], case["hidden"]).bfloat16()
        s.y = torch.zeros(case["tokens"], case["hidden"], device="cuda")
        s.ids = torch.zeros(case["tokens"], case["top_k"], dtype=torch.int32, device="cuda")
        s.w = torch.zeros(case["tokens"], case["top_k"], device="cuda")
        s.out = [s.y, s.ids, s.w]
    else:
        rows, cols, n = case["rows"], case["cols"], case["rows"] * case["cols"]
        g, per = {"q4": (case["group"], case["group"] // 2), "bin": (128, 16), "q8": (64, 64), "u3": (64, 24)}[case["kind"]]
        groups = (n + g - 1) // g
        s.weights = _randn(seed, 1, rows, cols) * SIGMA
        s.scales = torch.zeros(groups, dtype=torch.int16, device="cuda")
        s.codes = torch.zeros(groups * per, dtype=torch.uint8, device="cuda")
        s.out = [s.scales, s.codes]
    torch.cuda.synchronize()
    return s


def run(s):
    case, ctx, op = s.case, s.ctx, s.case["op"]
    if op == "gemv":
        if s.set is None:
            s.organs[0].matvec_device(s.x.ptr, s.y.ptr)
        else:
            s.set.gemv(s.x, case["cols"], s.y, s.y.t.shape[1])
    elif op == "lowrank":
        organs.gemv_lowrank_set(ctx, s.left, s.right, s.x, case["cols"], s.y, s.y.t.shape[1], mid=s.mid,
                                mid_stride=case["rank"])
    elif op == "head":
        ctx.call("hk_terminal_greedy", _ptr(s.h), _ptr(s.w), 1e-6, s.organ.h, case["n_valid"], _ptr(s.xn),
                 _ptr(s.logits), _ptr(s.pick), _ptr(s.token), ctx.stream)
    elif op == "stack":
        if case["n_layers"] == 1:
            s.model.decode_layer_device(0, _ptr(s.h), _ptr(s.y), _ptr(s.ids), _ptr(s.w))
        else:
            s.model.decode_stack_device(_ptr(s.h), _ptr(s.y), _ptr(s.ids), _ptr(s.w))
    elif op == "mixed15":
        moe.mixed15_decode_stack(ctx, s.layers, _ptr(s.h), _ptr(s.y), _ptr(s.ids), _ptr(s.w))
    elif op == "batch":
        s.model.forward_batch_device(0, _ptr(s.x), case["tokens"], _ptr(s.y), _ptr(s.ids), _ptr(s.w))
    elif case["kind"] == "q4":
        ctx.call("hk_pack_q4", _ptr(s.weights), case["rows"], case["cols"], case["group"], _ptr(s.scales),
                 _ptr(s.codes), ctx.stream)
    elif case["kind"] == "u3":
        ctx.call("hk_pack_u3", _ptr(s.weights), case["rows"] * case["cols"], _ptr(s.scales), _ptr(s.codes), ctx.stream)
    else:
        ctx.call("hk_pack_bin" if case["kind"] == "bin" else "hk_pack_q8", _ptr(s.weights), case["rows"],
                 case["cols"], _ptr(s.scales), _ptr(s.codes), ctx.stream)
    return s.out


# ---------------------------------------------------------------- work and tolerance

def _packed_bytes(kind, group, rows, cols):
    n = rows * cols
    return {"q4": n / 2 + 2 * n / group, "bin": n / 8 + n / 64, "q8": n + n / 32, "u3": n * 3 / 8 + n / 32,
            "mixed": 0.7 * (n / 8 + n / 64) + 0.3 * (n / 4 + n / 32) + n / 1024,
            "rice": n / 8 + n / 64 + 0.02 * n * 9.4 / 8}[kind]


def work(case):
    op = case["op"]
    if op == "gemv":
        n, r, c = case["n"], case["rows"], case["cols"]
        return {"bytes": n * (_packed_bytes(case["kind"], case["group"], r, c) + 4 * (r + c)), "flops": 2 * n * r * c}
    if op == "lowrank":
        n, r, k, c = case["n"], case["rows"], case["rank"], case["cols"]
        b = _packed_bytes("u3", 64, r, k) + _packed_bytes("u3", 64, k, c) + 4 * (r + k + c)
        return {"bytes": n * b, "flops": 2 * n * k * (r + c)}
    if op == "head":
        c = _head_case(case)
        return {"bytes": _packed_bytes(c["kind"], c["group"], c["rows"], c["cols"]) + 4 * (c["rows"] + 3 * c["cols"]),
                "flops": 2 * c["rows"] * c["cols"]}
    if op == "pack":
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * n + _packed_bytes(case["kind"], case["group"], case["rows"], case["cols"]), "flops": 4 * n}
    H, I, SI, E, K = (case[k] for k in ("hidden", "inter", "shared_inter", "n_experts", "top_k"))
    if op == "stack":
        L, kind, g = case["n_layers"], case["kind"], case["group"]
        per = 4 * H * (E + 4) + K * 3 * _packed_bytes(kind, g, I, H) + 3 * _packed_bytes(kind, g, SI, H)
        return {"bytes": L * per, "flops": 2 * L * H * (E + 3 * K * I + 3 * SI)}
    if op == "mixed15":
        L, r = case["n_layers"], case["rank"]
        per = (4 * 3 * H + _packed_bytes("q8", 64, E + 1, H) + 3 * _packed_bytes("q8", 64, SI, H) +
               K * (_packed_bytes("bin", 128, I, H) + _packed_bytes("rice", 128, I, H) +
                    _packed_bytes("u3", 64, H, r) + _packed_bytes("u3", 64, r, I)))
        return {"bytes": L * per, "flops": 2 * L * (H * (E + 3 * SI) + K * (2 * I * H + r * (H + I)))}
    T = case["tokens"]
    active = E * (1 - (1 - K / E) ** T)
    b = 4 * E * (H + 1) + 3 * active * _packed_bytes("q4", case["group"], I, H) + 3 * _packed_bytes(
        "q4", case["group"], SI, H) + T * H * 6
    return {"bytes": b, "flops": 2 * T * H * (E + 3 * K * I + 3 * SI)}


def tolerance(case):
    op = case["op"]
    if op == "pack":
        return "exact"
    # f32 results of exact integer dot products: 2e-7 from the 64-bit result
    if op in ("gemv", "lowrank"):
        return {"rel": 1e-6, "max": 1e-5}
    if op == "head":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    if op == "stack" and case["n_layers"] > 1:
        # a layer's rounding feeds every later one (4e-7 after 48), and a
        # near-tie in a router may order two of the experts either way
        return {"rel": 2e-6, "max": 2e-5, "differ": 0.01}
    return {"rel": 1.5e-6, "max": 1.5e-5, "differ": 0.01}


# ---------------------------------------------------------------- the path in 64 bits

_M = (1 << 64) - 1


def _i64(v):
    v &= _M
    return v - (1 << 64) if v >> 63 else v


def _mix_int(z):
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _M
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _M
    return z ^ (z >> 31)


def _stream_key(seed, stream):
    return _mix_int(_mix_int((seed ^ 0x6A09E667F3BCC909) & _M) ^ (stream & _M))


def _xor_shift(z, k):
    t = z >> k
    t &= (1 << (64 - k)) - 1
    return z.bitwise_xor_(t)


def _words(key, ctr):
    """SplitMix64 words of a key at counters ctr (int64 tensor, overwritten)."""
    z = ctr.add_(1).mul_(_i64(0x9E3779B97F4A7C15)).add_(_i64(key))
    z = _xor_shift(z, 30).mul_(_i64(0xBF58476D1CE4E5B9))
    z = _xor_shift(z, 27).mul_(_i64(0x94D049BB133111EB))
    return _xor_shift(z, 31)


def _normal(key, n, sigma):
    """n draws of the weight generator (Irwin-Hall of twelve 16-bit uniforms), f32."""
    base = torch.arange(n, device="cuda", dtype=torch.int64) * 3
    s = torch.zeros(n, device="cuda", dtype=torch.int64)
    for w in range(3):
        v = _words(key, base + w)
        for j in range(4):
            s += (v >> (16 * j)) & 0xFFFF
    return (2 * s + (12 - 786432)).float() * (1.0 / 131072.0) * torch.tensor(sigma, dtype=torch.float32).item()


def _round_away(v):
    return torch.sign(v) * torch.floor(v.abs() + 0.5)


def _max_over(g, by):
    """max |g| of each group / by, correctly rounded (a division by a Python
    number would multiply by its reciprocal)."""
    m = g.abs().amax(1, keepdim=True)
    return m / torch.full_like(m, by)


def _q4(w, group):
    g = w.view(-1, group)
    s = _max_over(g, 7.0).half().float()
    q = torch.where(s != 0, torch.clamp(torch.round(g / s), -8, 7), torch.zeros_like(g))
    return s, q


def _binary(w):
    g = w.view(-1, 128)
    s = g.abs().double().mean(1, keepdim=True).float().half().float()
    return s, torch.where(g >= 0, s, -s)


def _uniform(w, bound):
    n = w.numel()
    g = torch.nn.functional.pad(w, (0, -n % 64)).view(-1, 64)
    s = _max_over(g, float(bound))
    q = torch.clamp(_round_away((g / torch.where(s > 0, s, torch.ones_like(s))).double()), -bound, bound)
    return s.half(), q


def _weights(kind, group, rows, cols, key, coin_key, sigma):
    """The decoded matrix of a synthetic organ, float64."""
    n = rows * cols
    w = _normal(key, n, sigma)
    if kind == "q4":
        s, q = _q4(w, group)
        d = s.double() * q.double()
    elif kind in ("q8", "u3"):
        s, q = _uniform(w, 127 if kind == "q8" else 3)
        d = (s.double() * q).view(-1)[:n]
    elif kind == "mixed":
        _, b = _binary(w)
        g = w.view(-1, 64)
        s = _max_over(g, 1.5).half().float()
        c = torch.clamp(torch.round(g / torch.where(s > 0, s, torch.ones_like(s)) + 1.5), 0, 3)
        q2 = ((c - 1.5) * s).view(-1, 128)
        coin = _words(coin_key, torch.arange(n // 128, device="cuda", dtype=torch.int64))
        pick = ((coin >> 32) & 0xFFFFFFFF) < 3006477107
        d = torch.where(pick[:, None], b, q2).double()
    else:
        _, b = _binary(w)
        d = b.double().view(-1)
        if kind == "rice":
            res = w - b.view(-1)
            top = torch.sort(res.abs(), descending=True, stable=True).indices[:max(1, math.ceil(n * 0.02))]
            v = res[top].double()
            scale = float((v * v).mean().sqrt().float().half())
            d[top] += torch.where(v >= 0, scale, -scale)
    return d.view(rows, cols)


def _case_weights(case, seed, tag, rows=None, cols=None, kind=None, sigma=SIGMA):
    return _weights(kind or case["kind"], case.get("group", 64), rows or case["rows"], cols or case["cols"],
                    _key(seed, 2 * tag), _key(seed, 2 * tag + 1), sigma)


def _silu(v):
    return v / (1 + torch.exp(-v))


def _moe_weights(case, seed, layer, expert, proj):
    """A projection (0 gate, 1 up, 2 down) of a model's expert, or a dense tensor."""
    rows, cols = case["inter"] if expert < case["n_experts"] else case["shared_inter"], case["hidden"]
    if proj == 2:
        rows, cols = cols, rows
    sid = moe.moe_stream_id(layer, expert, proj)
    return _weights(case.get("kind", "q4"), case["group"], rows, cols, _stream_key(seed, sid),
                    _stream_key(seed, sid + moe.PROJ_COIN), SIGMA)


def _moe_dense(seed, layer, proj, n, sigma):
    return _normal(_stream_key(seed, moe.moe_stream_id(layer, 0, proj)), n, sigma).double()


def _rmsnorm(h, w):
    return h / torch.sqrt((h * h).mean() + 1e-6) * (1 + w)


def _topk(score, k):
    ids = torch.sort(score, descending=True, stable=True).indices[..., :k]
    return ids, torch.gather(score, -1, ids)


def _exact_stack(case, seed):
    H, E, K = case["hidden"], case["n_experts"], case["top_k"]
    h = _randn(seed, 1, H).double()
    all_ids, all_w = [], []
    for layer in range(case["n_layers"]):
        xn = _rmsnorm(h, _moe_dense(seed, layer, moe.PROJ_NORM, H, 0.02))
        ids, w = _topk(torch.softmax(_moe_dense(seed, layer, moe.PROJ_ROUTER, E * H, SIGMA).view(E, H) @ xn, 0), K)
        w = w / w.sum()
        out = h.clone()
        jobs = list(zip(ids.tolist(), w.tolist()))
        if case["shared_inter"]:
            gate = _moe_dense(seed, layer, moe.PROJ_SHARED_GATE, H, SIGMA) @ xn
            jobs.append((E, float(torch.sigmoid(gate))))
        for e, we in jobs:
            g, u, d = (_moe_weights(case, seed, layer, e, p) for p in range(3))
            out += we * (d @ (_silu(g @ xn) * (u @ xn)))
        h = out
        all_ids.append(ids.int())
        all_w.append(w)
    return [h, torch.stack(all_ids), torch.stack(all_w)]


def _exact_mixed15(case, seed):
    d = _mixed15_dims(case)
    names = {v: k for k, v in KINDS.items()}

    def tensor(layer, expert, proj):
        kind, rows, cols, group, sigma = moe.mixed15_tensor(d, expert, proj)
        return _weights(names[kind], group, rows, cols,
                        _stream_key(seed, moe.mixed15_stream_id(layer, expert, proj)), 0, sigma)

    h, E = _randn(seed, 1, d.hidden).double(), d.n_experts
    all_ids, all_w = [], []
    for layer in range(case["n_layers"]):
        nw = _normal(_stream_key(seed, moe.mixed15_stream_id(layer, E, moe.MIXED15_NORM)), d.hidden, 0.02).double()
        xn = _rmsnorm(h, nw)
        ids, w = _topk(torch.softmax(tensor(layer, E, moe.MIXED15_ROUTER) @ xn, 0), d.top_k)
        w = w / w.sum()
        out = h.clone()
        for e, we in zip(ids.tolist(), w.tolist()):
            act = _silu(tensor(layer, e, moe.MIXED15_GATE) @ xn) * (tensor(layer, e, moe.MIXED15_UP) @ xn)
            out += we * (tensor(layer, e, moe.MIXED15_DOWN_LEFT) @ (tensor(layer, e, moe.MIXED15_DOWN_RIGHT) @ act))
        act = (_silu(tensor(layer, E, moe.MIXED15_SHARED_GATE_PROJ) @ xn) *
               (tensor(layer, E, moe.MIXED15_SHARED_UP) @ xn))
        gate = torch.sigmoid(tensor(layer, E, moe.MIXED15_SHARED_GATE) @ xn)
        out += gate * (tensor(layer, E, moe.MIXED15_SHARED_DOWN) @ act)
        h = out
        all_ids.append(ids.int())
        all_w.append(w)
    return [h, torch.stack(all_ids), torch.stack(all_w)]


def _exact_batch(case, seed):
    T, H, E, K, G = (case[k] for k in ("tokens", "hidden", "n_experts", "top_k", "n_group"))
    x = _randn(seed, 1, T, H).bfloat16().double()
    score = torch.sigmoid(x @ _moe_dense(seed, 0, moe.PROJ_ROUTER, E * H, SIGMA).view(E, H).T)
    biased = score + _moe_dense(seed, 0, 19, E, 0.01)  # 19: the router bias
    if case["topk_group"] < G:
        strength = torch.topk(biased.view(T, G, E // G), min(2, E // G), dim=2).values.sum(2)
        keep = torch.zeros(T, G, dtype=torch.bool, device="cuda")
        keep.scatter_(1, _topk(strength, case["topk_group"])[0], True)
        biased = biased.masked_fill(~keep.repeat_interleave(E // G, 1), -math.inf)
    ids, _ = _topk(biased, K)
    w = torch.gather(score, 1, ids)
    w = w / (w.sum(1, keepdim=True) + 1e-20) * 2.5
    y = torch.zeros(T, H, dtype=torch.float64, device="cuda")
    for e in sorted(set(ids.flatten().tolist())) + [E]:
        g, u, d = (_moe_weights(case, seed, 0, e, p) for p in range(3))
        if e < E:
            t, slot = torch.nonzero(ids == e, as_tuple=True)
            y[t] += w[t, slot][:, None] * ((_silu(x[t] @ g.T) * (x[t] @ u.T)) @ d.T)
        else:
            y += (_silu(x @ g.T) * (x @ u.T)) @ d.T
    return [y, ids.int(), w]


def exact(case, seed):
    op = case["op"]
    if op == "gemv":
        x = _randn(seed, 1, case["n"], case["cols"]).double()
        return [torch.stack([_case_weights(case, seed, i) @ x[i] for i in range(case["n"])])]
    if op == "lowrank":
        n, rows, rank, cols = case["n"], case["rows"], case["rank"], case["cols"]
        x = _randn(seed, 1, n, cols).double()
        return [torch.stack([_case_weights(case, seed, 2 * i, rows, rank, "u3", 0.05) @
                             (_case_weights(case, seed, 2 * i + 1, rank, cols, "u3") @ x[i]) for i in range(n)])]
    if op == "head":
        c = _head_case(case)
        h, w = _randn(seed, 1, c["cols"]).double(), (_randn(seed, 2, c["cols"]) * 0.02).double()
        logits = _case_weights(c, seed, 0) @ _rmsnorm(h, w)
        return [logits, logits[:c["n_valid"]].argmax().int().view(1)]
    if op == "stack":
        return _exact_stack(case, seed)
    if op == "mixed15":
        return _exact_mixed15(case, seed)
    if op == "batch":
        return _exact_batch(case, seed)
    w = (_randn(seed, 1, case["rows"], case["cols"]) * SIGMA).view(-1)
    if case["kind"] == "q4":
        s, q = _q4(w, case["group"])
        q = (q + 8).to(torch.uint8).view(-1, 2)
        codes = q[:, 0] | (q[:, 1] << 4)
    elif case["kind"] == "bin":
        s, d = _binary(w)
        bit = 1 << torch.arange(8, device="cuda")
        codes = ((w.view(-1, 8) >= 0).long() * bit).sum(1).to(torch.uint8)
    elif case["kind"] == "q8":
        s, q = _uniform(w, 127)
        codes = (q + 127).to(torch.uint8).view(-1)
    else:
        s, q = _uniform(w, 3)
        bits = (((q + 3).long().view(-1, 8, 1) >> torch.arange(3, device="cuda")) & 1).view(-1, 8)
        codes = (bits << torch.arange(8, device="cuda")).sum(1).to(torch.uint8)
    return [s.half().view(-1).view(torch.int16), codes]
