"""What the speed of this library is measured on: the calls a program that
runs MLA attention makes through the public entry points, over the sizes it
makes them with.

    listed()            the cases looked at one by one
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what the program holds before the call (on the GPU)
    run(state)          one pass; returns its outputs whole
    work(case)          the bytes and flops a pass cannot do without
    tolerance(case)     how far another correct implementation may be off
    exact(case, seed)   the outputs in 64 bits, plain torch

Kinds ("op"):
    decode         absorbed MLA decode over a latent cache, a plan per cache
    sparse         the same over top-k index lists, checked on the device
    prefill        causal prefill (up-projection + attention), with a prefix
    linear         dense projection of T tokens
    affine         4-bit affine projection of T tokens
    moe            routed 4-bit experts of T tokens
    decode_block   one token through the whole attention block
    prefill_block  a prompt chunk through the whole attention block
    index          lightning-index scores of S query tokens and the top-k of
                   each row: a whole prompt (4 tokens to a key), or the one
                   token of a decode step
"""
from __future__ import annotations

import ctypes as C
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "minirun-app_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import minirun_hip as M  # noqa: E402

R, DR, NOPE, V = 512, 64, 128, 128  # latent, rotary key, nope and value widths
SCALE = (NOPE + DR) ** -0.5
HIDDEN, Q_LORA = 7168, 1536
# projections of the attention layer, [out, in] (128 heads, and the gated form with 96)
SHAPES = {"q_a": (1536, 7168), "q_b": (24576, 1536), "kv_a": (576, 7168), "o_proj": (7168, 16384),
          "q_b_96": (18432, 1536), "g_proj_96": (12288, 7168), "o_proj_96": (7168, 12288)}
_DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest decode layer: one token of a short chat on a small model
        # (16 heads, 512 rows); launches and latency are all of it
        {"name": "decode_h16_n512", "op": "decode", "batch": 1, "heads": 16, "ctx": 512, "out": "bf16"},
        # the headline: one token, 128 heads over a 32K-row latent cache
        {"name": "decode_h128_n32768", "op": "decode", "batch": 1, "heads": 128, "ctx": 32768, "out": "bf16"},
        # a serving batch in mid-conversation, an odd row count, 96 heads
        {"name": "decode_b6_h96_n3001", "op": "decode", "batch": 6, "heads": 96, "ctx": 3001, "out": "bf16"},
        # sparse decode: top-2048 rows of 128K-row caches, four tokens, the
        # index lists checked on the device
        {"name": "sparse_b4_h128_k2048", "op": "sparse", "batch": 4, "heads": 128, "ctx": 131072, "topk": 2048,
         "sinks": False, "padded": False},
        # prefill of a 4096-token prompt, 128 heads
        {"name": "prefill_t4096_h128", "op": "prefill", "tokens": 4096, "prefix": 0, "heads": 128},
        # a dense projection of a small batch (speculative tokens or a batch of
        # decodes): the gate projection of 24 tokens
        {"name": "linear_t24_g_proj", "op": "linear", "tokens": 24, "out_features": 12288, "in_features": 7168,
         "y": "bf16"},
        # the 4-bit output projection of a small batch
        {"name": "affine_t13_o_proj", "op": "affine", "tokens": 13, "out_features": 7168, "in_features": 16384,
         "group": 64, "scales": "bf16", "y": "bf16"},
        # the 4-bit output projection over an odd-sized prompt
        {"name": "affine_t1111_o_proj", "op": "affine", "tokens": 1111, "out_features": 7168, "in_features": 16384,
         "group": 64, "scales": "bf16", "y": "bf16"},
        # routed experts of a prompt chunk: 200 tokens, 8 of 128 experts each
        {"name": "moe_t200_e128_k8", "op": "moe", "tokens": 200, "experts": 128, "per_token": 8,
         "out_features": 768, "in_features": 2048},
        # one token through the whole attention block, 4-bit weights, rotary, 32K rows
        {"name": "decode_block_affine_n32768", "op": "decode_block", "weights": "affine", "heads": 128,
         "ctx": 32768, "rotary": True, "gate": False},
        # a prompt chunk behind a cached prefix through the whole block: dense
        # bf16 weights, 96 heads, output gate, no rotation
        {"name": "prefill_block_t2000_p1000", "op": "prefill_block", "weights": "dense", "heads": 96,
         "tokens": 2000, "position": 1000, "rotary": False, "gate": True},
        # lightning indexer of an odd-sized prompt compressed 4:1, top 512 of
        # each row
        {"name": "index_s4001_n1000", "op": "index", "rows": 4001, "keys": 1000, "heads": 64, "topk": 512},
    ]


def _log(rng, lo, hi):
    import math

    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes over the whole range (over their logarithm), any
    parity; never dearer than the dearest listed one."""
    op = rng.choice(["decode", "decode", "sparse", "prefill", "linear", "affine", "affine", "moe", "decode_block",
                     "prefill_block", "index"])
    if op == "decode":
        batch = _log(rng, 1, 16)
        return {"op": op, "batch": batch, "heads": rng.choice([16, 32, 64, 96, 128]),
                "ctx": _log(rng, 64, min(65536, 131072 // batch)), "out": rng.choice(["bf16", "bf16", "bf16", "f32"])}
    if op == "sparse":
        return {"op": op, "batch": _log(rng, 1, 8), "heads": rng.choice([64, 96, 128]),
                "ctx": _log(rng, 8192, 131072), "topk": _log(rng, 256, 4096), "sinks": rng.random() < 0.5,
                "padded": rng.random() < 0.5}
    if op == "prefill":
        return {"op": op, "tokens": _log(rng, 8, 2048), "prefix": rng.choice([0, _log(rng, 16, 2048)]),
                "heads": rng.choice([16, 64, 96, 128])}
    if op in ("linear", "affine"):
        if rng.random() < 0.6:
            o, i = rng.choice(sorted(SHAPES.values()))
        else:
            o, i = 8 * _log(rng, 64, 2048), 64 * _log(rng, 8, 256)
        c = {"op": op, "tokens": _log(rng, 1, 2048), "out_features": o, "in_features": i,
             "y": rng.choice(["bf16", "bf16", "f32"])}
        if op == "affine":
            c.update(group=64, scales=rng.choice(["bf16", "bf16", "f16", "f32"]))
        return c
    if op == "moe":
        o, i = rng.choice([(768, 2048), (2048, 768), (1408, 2048), (512, 1024)])
        return {"op": op, "tokens": _log(rng, 1, 512), "experts": rng.choice([64, 128]),
                "per_token": rng.choice([4, 6, 8]), "out_features": o, "in_features": i}
    if op == "decode_block":
        affine = rng.random() < 0.5
        return {"op": op, "weights": "affine" if affine else "dense", "heads": 128 if affine else 96,
                "ctx": _log(rng, 256, 32768), "rotary": affine, "gate": not affine}
    if op == "prefill_block":
        affine = rng.random() < 0.5
        return {"op": op, "weights": "affine" if affine else "dense", "heads": 128 if affine else 96,
                "tokens": _log(rng, 16, 1200), "position": rng.choice([0, _log(rng, 16, 1200)]),
                "rotary": affine, "gate": not affine}
    rows = rng.choice([1, _log(rng, 64, 4096)])
    return {"op": op, "rows": rows, "keys": _log(rng, 512, 65536) if rows == 1 else rows // 4, "heads": 64,
            "topk": rng.choice([512, 1024, 2048])}


# ---------------------------------------------------------------- inputs
class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)

    def normal(self, *shape, std=1.0, dtype=torch.bfloat16):
        return (std * torch.randn(*shape, generator=self.g, device="cuda")).to(dtype)

    def norm_weight(self, n):
        return (1 + 0.02 * torch.randn(n, generator=self.g, device="cuda")).to(torch.bfloat16)

    def affine(self, out, inp, group=64, scales=torch.bfloat16, experts=0):
        """4-bit rows as a quantizer lays out zero-mean weights of standard
        deviation about in^-1/2: scales of a narrow spread, biases about 7.5
        scales below zero."""
        lead = (experts, out) if experts else (out,)
        packed = torch.randint(-2 ** 31, 2 ** 31, (*lead, inp // 8), generator=self.g, device="cuda",
                               dtype=torch.int64).to(torch.int32)
        s = (0.217 * inp ** -0.5) * (1 + 0.2 * torch.randn(*lead, inp // group, generator=self.g, device="cuda")).abs()
        s = s.to(scales)
        b = (s.float() * (-7.5 + 0.2 * torch.randn(*lead, inp // group, generator=self.g, device="cuda"))).to(scales)
        return M.AffineWeights(packed, s, b, group_size=group)

    def dense(self, out, inp):
        return M.DenseWeights(self.normal(out, inp, std=inp ** -0.5))

    def indices(self, batch, ctx, k, padded):
        window = min(128, k)
        rows = []
        for _ in range(batch):
            far = torch.randperm(ctx - window, generator=self.g, device="cuda")[: k - window]
            row = torch.cat([far, torch.arange(ctx - window, ctx, device="cuda")]).sort().values
            if padded:  # a short list, filled up with -1
                row[k - k // 7:] = -1
            rows.append(row)
        return torch.stack(rows).to(torch.int32).contiguous()


def _block_inputs(case, r):
    H = case["heads"]
    mk = (lambda o, i: r.affine(o, i)) if case["weights"] == "affine" else r.dense
    w = {"input_norm": r.norm_weight(HIDDEN) if case["weights"] == "affine" else None,
         "q_a_norm": r.norm_weight(Q_LORA), "kv_a_norm": r.norm_weight(R),
         "q_a": mk(Q_LORA, HIDDEN), "q_b": mk(H * (NOPE + DR), Q_LORA), "kv_a": mk(R + DR, HIDDEN),
         "kv_b": mk(H * (NOPE + V), R), "o_proj": mk(HIDDEN, H * V)}
    if case["gate"]:
        w["g_proj"] = mk(H * V, HIDDEN)
    return w


def _rope(positions):
    c, s = M.rope_table(positions, M.rope_frequencies(DR))
    return torch.from_numpy(c).cuda(), torch.from_numpy(s).cuda()


def prepare(case, seed):
    op = case["op"]
    r = _Rand(seed)
    st = {"op": op}
    if op in ("decode", "sparse"):
        B, H, N = case["batch"], case["heads"], case["ctx"]
        q_lat, q_rope = r.normal(B, H, R), r.normal(B, H, DR)
        cache = r.normal(B, N, R + DR, std=0.5)
        kw = {}
        if op == "sparse":
            kw["indices"] = r.indices(B, N, case["topk"], case["padded"])
            kw["index_status"] = torch.zeros(B, 3, dtype=torch.int32, device="cuda")
            if case["sinks"]:
                kw["sinks"] = r.normal(H, dtype=torch.float32)
        out = torch.empty(B, H, R, dtype=_DT[case.get("out", "bf16")], device="cuda")
        plan, out, ws = M.decode_args(q_lat, q_rope, cache[..., :R], cache[..., R:], scale=SCALE, out=out, **kw)
        st.update(plan=plan, out=out, keep=(q_lat, q_rope, cache, ws, kw), status=kw.get("index_status"))
    elif op == "prefill":
        T, P, H = case["tokens"], case["tokens"] + case["prefix"], case["heads"]
        q = r.normal(T, H, NOPE + DR)
        cache = r.normal(P, R + DR, std=0.5)
        kv_b = r.normal(H * (NOPE + V), R, std=R ** -0.5)
        plan, out, ws = M.prefill_args(q, cache[:, :R], cache[:, R:], kv_b)
        st.update(plan=plan, out=out, keep=(q, cache, kv_b, ws))
    elif op == "linear":
        st.update(x=r.normal(case["tokens"], case["in_features"]), y=_DT[case["y"]],
                  w=r.dense(case["out_features"], case["in_features"]))
    elif op == "affine":
        st.update(x=r.normal(case["tokens"], case["in_features"]), y=_DT[case["y"]],
                  w=r.affine(case["out_features"], case["in_features"], case["group"], _DT[case["scales"]]))
    elif op == "moe":
        T, E, K = case["tokens"], case["experts"], case["per_token"]
        st.update(x=r.normal(T, case["in_features"]),
                  w=r.affine(case["out_features"], case["in_features"], experts=E),
                  ids=torch.rand(T, E, generator=r.g, device="cuda").topk(K, dim=1).indices.to(torch.int32).contiguous())
    elif op == "decode_block":
        w = _block_inputs(case, r)
        N = case["ctx"]
        cache = r.normal(N, R + DR, std=0.5)
        x = r.normal(HIDDEN)
        cos, sin = _rope([N - 1]) if case["rotary"] else (None, None)
        out = torch.empty(HIDDEN, dtype=torch.bfloat16, device="cuda")
        plan, ws = M.block_args(x, w, cache, N - 1, cos, sin, out, heads=case["heads"])
        st.update(plan=plan, out=out, cache=cache, first=N - 1, keep=(w, x, cos, sin, ws))
    elif op == "prefill_block":
        w = _block_inputs(case, r)
        T, p0 = case["tokens"], case["position"]
        cache = r.normal(p0 + T, R + DR, std=0.5)
        x = r.normal(T, HIDDEN)
        cos, sin = _rope(list(range(p0, p0 + T))) if case["rotary"] else (None, None)
        out = torch.empty(T, HIDDEN, dtype=torch.bfloat16, device="cuda")
        plan, ws = M.prefill_block_args(x, w, cache, p0, cos, sin, out, heads=case["heads"])
        st.update(plan=plan, out=out, cache=cache, first=p0, keep=(w, x, cos, sin, ws))
    elif op == "index":
        S, T, H = case["rows"], case["keys"], case["heads"]
        st.update(q=r.normal(S, H, 128), k=r.normal(T, 128),
                  w=r.normal(S, H, std=(128 * H) ** -0.5, dtype=torch.float32), topk=case["topk"],
                  start=4 * T - 1 if S == 1 else 0, status=torch.zeros(1, dtype=torch.int32, device="cuda"))
    else:
        raise ValueError(op)
    return st


# ---------------------------------------------------------------- one pass
def run(st):
    op = st["op"]
    if op in ("decode", "sparse", "prefill", "decode_block", "prefill_block"):
        entry = {"decode": "mr_mla_decode", "sparse": "mr_mla_decode", "prefill": "mr_mla_prefill",
                 "decode_block": "mr_mla_decode_block", "prefill_block": "mr_mla_prefill_block"}[op]
        lib = M.load()
        if getattr(lib, entry)(C.byref(st["plan"]), torch.cuda.current_stream().cuda_stream) != M.OK:
            raise M.MRError(1, M.last_error())
        if op == "sparse":
            return {"out": st["out"], "status": st["status"]}
        if op.endswith("block"):  # the rows the call appended, and the cache they are part of
            return {"out": st["out"], "rows": st["cache"][st["first"]:], "cache": st["cache"]}
        return st["out"]
    if op == "linear":
        return M.linear(st["x"], st["w"], out_dtype=st["y"])
    if op == "affine":
        return M.affine_mm(st["x"], st["w"], out_dtype=st["y"])
    if op == "moe":
        return M.affine_gather_mm(st["x"], st["w"], st["ids"])
    scores = M.lightning_index_scores(st["q"], st["k"], st["w"])
    ids = M.lightning_select(scores, st["topk"], 4, st["start"], 0, check=False, status=st["status"])
    return {"scores": scores, "ids": ids, "status": st["status"]}


# ---------------------------------------------------------------- what a pass cannot do without
def _weight_bytes(case, o, i, group=64, sbytes=2):
    if case.get("weights") == "affine" or case["op"] in ("affine", "moe"):
        return o * i // 2 + 2 * sbytes * o * (i // group)
    return 2 * o * i


def _pairs(T, prefix):
    return T * prefix + T * (T + 1) // 2


def work(case):
    op = case["op"]
    if op == "decode":
        B, H, N = case["batch"], case["heads"], case["ctx"]
        ob = 4 if case["out"] == "f32" else 2
        return {"bytes": B * (N * 2 * (R + DR) + H * (2 * (R + DR) + ob * R)), "flops": 2 * B * H * N * (2 * R + DR)}
    if op == "sparse":
        B, H, K = case["batch"], case["heads"], case["topk"]
        return {"bytes": B * (K * (2 * (R + DR) + 4) + H * 2 * (2 * R + DR)), "flops": 2 * B * H * K * (2 * R + DR)}
    if op == "prefill":
        T, P, H = case["tokens"], case["tokens"] + case["prefix"], case["heads"]
        return {"bytes": 2 * (T * H * (NOPE + DR + V) + P * (R + DR) + H * (NOPE + V) * R),
                "flops": 2 * H * (P * R * (NOPE + V) + _pairs(T, case["prefix"]) * (NOPE + DR + V))}
    if op in ("linear", "affine"):
        T, o, i = case["tokens"], case["out_features"], case["in_features"]
        sb = 4 if case.get("scales") == "f32" else 2
        return {"bytes": 2 * T * i + _weight_bytes(case, o, i, case.get("group", 64), sb) +
                (4 if case["y"] == "f32" else 2) * T * o, "flops": 2 * T * o * i}
    if op == "moe":
        T, E, K, o, i = (case[n] for n in ("tokens", "experts", "per_token", "out_features", "in_features"))
        used = E * (1 - (1 - K / E) ** T)  # experts that some token is routed to
        return {"bytes": int(used * _weight_bytes(case, o, i)) + 2 * T * (i + K * o) + 4 * T * K,
                "flops": 2 * T * K * o * i}
    if op == "index":
        S, T, H = case["rows"], case["keys"], case["heads"]
        sel = min(case["topk"], T)
        return {"bytes": 2 * S * H * 128 + 2 * T * 128 + 4 * S * H + 4 * S * T + 4 * S * sel,
                "flops": 2 * S * T * H * 129}
    H = case["heads"]
    ws = [(Q_LORA, HIDDEN), (H * (NOPE + DR), Q_LORA), (R + DR, HIDDEN), (H * (NOPE + V), R), (HIDDEN, H * V)]
    if case["gate"]:
        ws.append((H * V, HIDDEN))
    wb = sum(_weight_bytes(case, o, i) for o, i in ws)
    wf = sum(2 * o * i for o, i in ws)
    if op == "decode_block":
        N = case["ctx"]
        return {"bytes": wb + 2 * N * (R + DR) + 4 * HIDDEN, "flops": wf + 2 * H * N * (2 * R + DR)}
    T, p0 = case["tokens"], case["position"]
    kvb = 2 * H * (NOPE + V) * R
    return {"bytes": wb + 2 * (p0 + 2 * T) * (R + DR) + 4 * T * HIDDEN,
            "flops": T * (wf - kvb) + (T + p0) * kvb + 2 * H * _pairs(T, p0) * (NOPE + DR + V)}


def tolerance(case):
    """About four times the error against 64 bits that the largest cases show."""
    op = case["op"]
    f32 = case.get("out", case.get("y")) == "f32"
    if op in ("linear", "affine", "moe"):
        # one fp32 sum of up to 16384 products (1e-6), or that rounded once to bf16 (1.7e-3)
        return {"rel": 5e-6, "max": 5e-5} if f32 else {"rel": 7e-3, "max": 2e-2}
    if op == "index":
        # scores: sums of 64 fp32 terms (1e-7); ids swap where two scores are closer than that
        return {"rel": 1e-6, "max": 5e-6, "differ": 5e-3}
    if op in ("decode", "sparse"):
        # probabilities go through the second product in bf16 (2.3e-3)
        return {"rel": 9e-3, "max": 4e-2}
    if op == "prefill":
        # keys, values and probabilities in bf16 (2.7e-3); the first queries
        # see few keys, so their outputs are far above the mean square
        return {"rel": 1.1e-2, "max": 4e-1}
    # six bf16 stages, one after the other (6.5e-3)
    return {"rel": 2.5e-2, "max": 2.5e-1}


# ---------------------------------------------------------------- 64 bits
def _dense64(w):
    if isinstance(w, M.DenseWeights):
        return w.weight.double()
    return _dequant64(w.packed, w.scales, w.biases, w.group_size)


def _dequant64(packed, scales, biases, group):
    sh = torch.arange(0, 32, 4, device=packed.device, dtype=torch.int32)
    q = ((packed.unsqueeze(-1) >> sh) & 15).reshape(*packed.shape[:-1], -1)
    s, b = (t.double().repeat_interleave(group, dim=-1) for t in (scales, biases))
    return s * q.double() + b


def _rms64(x, w, eps):
    return w.double() * (x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps))


def _rot64(x, cos, sin):
    """Adjacent pairs of the last axis; cos / sin [positions, half], x [positions, ..., 2 half]."""
    shape = (cos.shape[0],) + (1,) * (x.dim() - 2) + (cos.shape[1],)
    c, s = cos.double().reshape(shape), sin.double().reshape(shape)
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack([e * c - o * s, e * s + o * c], dim=-1).flatten(-2)


def _causal64(q, lat, rope, kv_b, prefix, heads):
    """Eager causal attention: q [T, H, 192], rows [P, ..], kv_b [H * 256, 512]."""
    T = q.shape[0]
    out = torch.empty(T, heads, V, dtype=torch.float64, device=q.device)
    wb = kv_b.reshape(heads, NOPE + V, R)
    step = 512
    for h in range(heads):
        kv = lat @ wb[h].t()
        k = torch.cat([kv[:, :NOPE], rope], dim=1)
        for t0 in range(0, T, step):
            t1 = min(T, t0 + step)
            n = prefix + t1
            s = (q[t0:t1, h] @ k[:n].t()) * SCALE
            hide = torch.arange(n, device=q.device)[None, :] > torch.arange(prefix + t0, n, device=q.device)[:, None]
            out[t0:t1, h] = torch.softmax(s.masked_fill_(hide, float("-inf")), dim=-1) @ kv[:n, NOPE:]
    return out


def exact(case, seed):
    op = case["op"]
    st = prepare(case, seed)
    if op in ("decode", "sparse"):
        q_lat, q_rope, cache, _ws, kw = st["keep"]
        outs = []
        for b in range(case["batch"]):
            rows = cache[b]
            if op == "sparse":
                ids = kw["indices"][b].long()
                rows = rows[ids[ids >= 0]]
            rows = rows.double()
            s = (q_lat[b].double() @ rows[:, :R].t() + q_rope[b].double() @ rows[:, R:].t()) * SCALE
            if kw.get("sinks") is not None:
                s = torch.cat([s, kw["sinks"].double()[:, None]], dim=1)
            outs.append(torch.softmax(s, dim=-1)[:, : rows.shape[0]] @ rows[:, :R])
        out = torch.stack(outs)
        return {"out": out, "status": None} if op == "sparse" else out
    if op == "prefill":
        q, cache, kv_b, _ws = st["keep"]
        c = cache.double()
        return _causal64(q.double(), c[:, :R], c[:, R:], kv_b.double(), case["prefix"], case["heads"])
    if op in ("linear", "affine"):
        return st["x"].double() @ _dense64(st["w"]).t()
    if op == "moe":
        w, ids, x = st["w"], st["ids"].long(), st["x"].double()
        out = torch.empty(*ids.shape, case["out_features"], dtype=torch.float64, device="cuda")
        for e in ids.unique().tolist():
            t, j = (ids == e).nonzero(as_tuple=True)
            out[t, j] = x[t] @ _dequant64(w.packed[e], w.scales[e], w.biases[e], 64).t()
        return out
    if op == "index":
        k = st["k"].double()
        scores = torch.stack([st["w"][s].double() @ (st["q"][s].double() @ k.t()).clamp_(min=0.0)
                              for s in range(case["rows"])])
        return {"scores": scores, "ids": None, "status": None}
    # a block: x -> q, cache rows -> attention -> gate -> output projection
    H = case["heads"]
    w, x, cos, sin, _ws = st["keep"]
    x = x.double().reshape(-1, HIDDEN)
    p0, T = st["first"], x.shape[0]
    h = x if w["input_norm"] is None else _rms64(x, w["input_norm"], 1e-6)
    q = (_rms64(h @ _dense64(w["q_a"]).t(), w["q_a_norm"], 1e-6) @ _dense64(w["q_b"]).t()).reshape(T, H, NOPE + DR)
    kv = h @ _dense64(w["kv_a"]).t()
    key = kv[:, R:]
    if cos is not None:
        q = torch.cat([q[..., :NOPE], _rot64(q[..., NOPE:], cos, sin)], dim=-1)
        key = _rot64(key, cos, sin)
    rows = torch.cat([_rms64(kv[:, :R], w["kv_a_norm"], 1e-6), key], dim=1)
    cache = torch.cat([st["cache"][:p0].double(), rows])
    attn = _causal64(q, cache[:, :R], cache[:, R:], _dense64(w["kv_b"]), p0, H).reshape(T, H * V)
    if case["gate"]:
        attn = attn * torch.sigmoid(h @ _dense64(w["g_proj"]).t())
    out = attn @ _dense64(w["o_proj"]).t()
    return {"out": out.reshape(st["out"].shape), "rows": rows, "cache": cache}
