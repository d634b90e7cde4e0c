"""What this library is timed on: single layers through the drop-in entry points, at the shapes of
the models in lockstep_amd.workloads, from one decode row to a whole prefill.

Kinds of case:
  linear   lockstep_fullstack.w8a8_matmul, bf16 (or binary32) rows in, the same type out, the linear
           every projection of a served model runs: decode batches and prefill chunks
  site     ref_block_v1.linear_dyn, one GEMM site of the golden block (binary32 in and out)
  outlier  lockstep_fullstack.w8a8_outlier_linear, the norm-fed projection with declared outlier
           channels and the online rotation
  head     t16h_lmvariants.Variant.logits, the wide-integer lm_head on the rows of a decode batch
  moe      moe_ref.moe_forward, int8 experts routed from their logits
  moe_mx   moe_ref.moe_forward_mx / moe_forward_mx2, MXFP4 experts routed from their logits

Every result is defined bit by bit, so the tolerance is "exact" throughout.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from lockstep_amd import contract_common as CC
from lockstep_amd import lockstep_fullstack as FS
from lockstep_amd import moe_ref as MR
from lockstep_amd import ref_block_v1 as RB
from lockstep_amd import t16h_lmvariants as TH
from lockstep_amd import workloads as WL

F64 = torch.float64
QKV, O, GATE_UP, DOWN = (WL.QWEN25_7B[n] for n in ("qkv", "o", "gate_up", "down"))
GATE_UP_L, DOWN_L = WL.LLAMA8B["gate_up"], WL.LLAMA8B["down"]
MOE_DIMS = {"qwen3": WL.QWEN3_30B_A3B, "gpt_oss": WL.GPT_OSS_20B}
DT = {"bf16": torch.bfloat16, "f32": torch.float32}


def _linear(M, NK, bias, dtype="bf16"):
    return {"kind": "linear", "M": M, "N": NK[0], "K": NK[1], "bias": bias, "dtype": dtype}


def listed():
    named = {
        # one user's decode step: the QKV projection with its bias, all latency
        "linear_decode_1": _linear(1, QKV, True),
        # a small serving batch on the down projection (long rows, few columns)
        "linear_decode_24": _linear(24, DOWN_L, False),
        # a busy server's decode batch: more rows than a GEMV, fewer than a prefill
        "linear_decode_72": _linear(72, DOWN, False),
        # a ragged prompt chunk through the QKV projection
        "linear_chunk_777": _linear(777, QKV, True),
        # a prefill chunk on the widest projection
        "linear_prefill_2048": _linear(2048, GATE_UP_L, False),
        # the golden block's longest sequence on its down projection (the largest call)
        "site_down_8192": {"kind": "site", "T": 8192, "N": DOWN[0], "K": DOWN[1]},
        # a prompt through a norm-fed projection with declared outlier channels and the rotation
        "outlier_300": {"kind": "outlier", "M": 300, "N": QKV[0], "K": QKV[1], "ko": 16, "rot": True},
        # the 15-bit lm_head for the last rows of a decode batch
        "head_a15w15_8": {"kind": "head", "M": 8, "N": 65536, "K": 3584, "spec": "a15w15"},
        # an MoE layer of a small decode batch: many experts, one or two rows each
        "moe_decode_16": {"kind": "moe", "T": 16, "dims": "qwen3"},
        # the same layer on a ragged prompt, popular and rare experts together
        "moe_prompt_1500": {"kind": "moe", "T": 1500, "dims": "qwen3"},
        # MXFP4 experts for a decode batch
        "moe_mx_decode_40": {"kind": "moe_mx", "T": 40, "dims": "gpt_oss", "blocks": False},
        # and for a prompt
        "moe_mx_prompt_600": {"kind": "moe_mx", "T": 600, "dims": "gpt_oss", "blocks": False},
    }
    return [dict(c, name=n) for n, c in named.items()]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["linear"] * 4 + ["site", "outlier", "head"] + ["moe"] * 2 + ["moe_mx"] * 2)
    if kind == "linear":
        N, K = rng.choice([QKV, O, GATE_UP, DOWN, GATE_UP_L, DOWN_L])
        if rng.random() < 0.3:   # a shard or a cut vocabulary: columns that fill no tile
            N -= rng.randrange(1, N // 2)
        return _linear(_log(rng, 1, 2048), (N, K), rng.random() < 0.4, rng.choice(["bf16", "bf16", "f32"]))
    if kind == "site":
        N, K = rng.choice([QKV, O, DOWN])
        return {"kind": "site", "T": _log(rng, 256, 8192), "N": N, "K": K}
    if kind == "outlier":
        N, K = rng.choice([QKV, O, GATE_UP_L])
        return {"kind": "outlier", "M": _log(rng, 1, 1024), "N": N, "K": K, "ko": rng.randrange(1, 33),
                "rot": rng.random() < 0.7}
    if kind == "head":
        return {"kind": "head", "M": _log(rng, 1, 64), "N": rng.randrange(16384, 65537), "K": rng.choice([3584, 4096]),
                "spec": rng.choice(["a15w15", "a15w15", "a15", "w15", "a11w11"])}
    if kind == "moe":
        dims = rng.choice(["qwen3", "qwen3", "gpt_oss"])
        return {"kind": "moe", "T": _log(rng, 1, 4096 if dims == "qwen3" else 1024), "dims": dims}
    return {"kind": "moe_mx", "T": _log(rng, 1, 1024), "dims": "gpt_oss", "blocks": rng.random() < 0.3}


# ------------------------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _rows(g, M, K, dtype):
    """N(0,1) rows with one value in a thousand at +-20."""
    x = torch.randn((M, K), generator=g, device="cuda")
    hit = torch.rand((M, K), generator=g, device="cuda")
    x = torch.where(hit < 0.0005, -20.0, torch.where(hit > 0.9995, 20.0, x))
    return x.to(dtype)


def _weight(g, N, K):
    w = torch.randint(-127, 128, (N, K), generator=g, device="cuda", dtype=torch.int8)
    ws = torch.rand((N,), generator=g, device="cuda") * 9e-3 + 1e-3
    return w, ws


def _logits(g, T, E, zipf):
    x = torch.randn((T, E), generator=g, device="cuda")
    if zipf:
        rank = torch.randperm(E, generator=g, device="cuda").to(torch.float32)
        x = x - 1.1 * torch.log1p(rank)[None, :]
    return x.to(torch.bfloat16)


def _inputs(case, seed):
    """The raw inputs of a case, as prepare() and exact() both start from them."""
    g, kind = _gen(seed), case["kind"]
    if kind == "linear":
        w, ws = _weight(g, case["N"], case["K"])
        b = torch.randn((case["N"],), generator=g, device="cuda") * 0.1 if case["bias"] else None
        return {"x": _rows(g, case["M"], case["K"], DT[case["dtype"]]), "w": w, "ws": ws, "b": b}
    if kind == "site":
        w = torch.randint(-127, 128, (case["N"], case["K"]), generator=g, device="cuda", dtype=torch.int8)
        return {"x": torch.randn((case["T"], case["K"]), generator=g, device="cuda"), "w": w, "ew": 7}
    if kind == "outlier":
        N, K, ko = case["N"], case["K"], case["ko"]
        w, ws = _weight(g, N, K)
        x = torch.randn((case["M"], K), generator=g, device="cuda") * 3
        oidx = torch.randperm(K, generator=g, device="cuda")[:ko].sort().values.to(torch.int32)
        x[:, oidx.long()] *= 40.0           # what declares a channel an outlier
        wo = (torch.randn((N, ko), generator=g, device="cuda") * 0.05).to(torch.bfloat16)
        return {"x": x.to(torch.bfloat16), "w": w, "ws": ws, "oidx": oidx, "wo": wo}
    if kind == "head":
        W = (torch.randn((case["N"], case["K"]), generator=g, device="cuda") * 0.05).to(torch.bfloat16)
        return {"x": torch.randn((case["M"], case["K"]), generator=g, device="cuda"), "W": W}
    d, T = MOE_DIMS[case["dims"]], case["T"]
    E, H, I = d["E"], d["H"], d["I"]
    s = {"x": torch.randn((T, H), generator=g, device="cuda").to(torch.bfloat16),
         "logits": _logits(g, T, E, kind == "moe")}
    if kind == "moe":
        s["w13"], s["ws13"] = (t.view(E, 2 * I, -1) for t in _weight(g, E * 2 * I, H))
        s["w2"], s["ws2"] = (t.view(E, H, -1) for t in _weight(g, E * H, I))
        return s
    for n, rows, K in (("13", 2 * I, H), ("2", H, I)):
        s["c" + n] = torch.randint(0, 256, (E, rows, K // 2), generator=g, device="cuda", dtype=torch.uint8)
        s["e" + n] = torch.randint(119, 130, (E, rows, K // 32), generator=g, device="cuda", dtype=torch.uint8)
        s["b" + n] = torch.randn((E, rows), generator=g, device="cuda") * 0.1
    return s


def prepare(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    s["kind"] = kind
    if kind == "outlier":
        s["rot"] = case["rot"]
    elif kind == "head":
        s["variant"] = TH.build(case["spec"]).prepare(s.pop("W"))
    elif kind in ("moe", "moe_mx"):
        d = MOE_DIMS[case["dims"]]
        s["k"], s["tab"] = d["k"], CC.table_on(s["x"].device)
        if kind == "moe":
            w13, ws13, w2, ws2 = (s.pop(n) for n in ("w13", "ws13", "w2", "ws2"))
            s["tables"] = MR.ExpertTables([(w13[e].t(), ws13[e, :, 0], w2[e].t(), ws2[e, :, 0])
                                           for e in range(d["E"])])
        else:
            p = {n: s.pop(n) for n in ("c13", "e13", "b13", "c2", "e2", "b2")}
            s["tables"] = MR.ExpertTablesMX([((p["c13"][e], p["e13"][e]), (p["c2"][e], p["e2"][e]), p["b13"][e],
                                              p["b2"][e]) for e in range(d["E"])], packed=True)
            s["forward"] = MR.moe_forward_mx2 if case["blocks"] else MR.moe_forward_mx
    return s


def run(state):
    s, kind = state, state["kind"]
    if kind == "linear":
        return FS.w8a8_matmul(s["x"], s["w"], s["ws"], s["b"])
    if kind == "site":
        return RB.linear_dyn(s["x"], s["w"].t(), s["ew"])
    if kind == "outlier":
        return FS.w8a8_outlier_linear(s["x"], s["oidx"], s["wo"], s["w"], s["ws"], rot=s["rot"])
    if kind == "head":
        return s["variant"].logits(s["x"])
    if kind == "moe":
        return MR.moe_forward(s["x"], None, s["tables"], s["k"], True, s["tab"], 0, MR.act_silu, logits=s["logits"])
    return s["forward"](s["x"], None, s["tables"], s["k"], True, s["tab"], 0, MR.act_swigluoai, logits=s["logits"])


# ------------------------------------------------------------------------------------------ cost
def _active(T, E, k, zipf):
    """Experts that T tokens reach, over a routing drawn as the logits are."""
    r = np.random.default_rng(1)
    x = r.standard_normal((T, E))
    if zipf:
        x = x - 1.1 * np.log1p(r.permutation(E))[None, :]
    return len(np.unique(np.argpartition(-x, k - 1, axis=1)[:, :k]))


def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, K, e = case["M"], case["N"], case["K"], 2 if case["dtype"] == "bf16" else 4
        return {"bytes": N * K + 4 * N * (2 if case["bias"] else 1) + e * M * (K + N), "flops": 2 * M * N * K}
    if kind == "site":
        T, N, K = case["T"], case["N"], case["K"]
        return {"bytes": N * K + 4 * T * (K + N), "flops": 2 * T * N * K}
    if kind == "outlier":
        M, N, K, ko = case["M"], case["N"], case["K"], case["ko"]
        return {"bytes": N * K + 4 * N + 2 * N * ko + 2 * M * (K + N), "flops": 2 * M * N * (K + ko)}
    if kind == "head":
        M, N, K = case["M"], case["N"], case["K"]
        a, w = {"a15w15": (2, 2), "a15": (2, 1), "w15": (1, 2), "a11w11": (2, 2)}[case["spec"]]
        return {"bytes": w * N * K + 4 * N + 4 * M * (K + N), "flops": 2 * a * w * M * N * K}
    d, T = MOE_DIMS[case["dims"]], case["T"]
    E, k, H, I = d["E"], d["k"], d["H"], d["I"]
    per = 3 * I * H + 4 * (2 * I + H) if kind == "moe" else 3 * I * H * 17 // 32 + 4 * (2 * I + H)
    return {"bytes": _active(T, E, k, kind == "moe") * per + 4 * T * H + 2 * T * E, "flops": 6 * T * k * I * H}


def tolerance(case):
    return "exact"


# ------------------------------------------------------------------------------------------ 64 bits
# The quantised operands are the contract's own binary32 values (they are inputs of the integer
# product, not approximations of anything); all that follows them is binary64, unrounded.
def _quant(x, top=127.0):
    x = x.to(torch.float32)
    asc = x.abs().amax(-1, keepdim=True).clamp(min=1e-8) / top
    return (x / asc).round().clamp(-top, top).to(F64), asc.to(F64)


def _hadamard(n):
    h = torch.ones((1, 1), dtype=F64, device="cuda")
    while h.shape[0] < n:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h


def _mm(q, w):
    """q [M, K] @ w [N, K]^T in binary64, the weight widened in column blocks."""
    return torch.cat([q @ p.to(F64).t() for p in w.split(8192)], 1)


_FP4 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _mx_weight(codes, scale):
    tab = torch.tensor(_FP4 + [-v for v in _FP4], dtype=F64, device="cuda")
    v = torch.stack([tab[(codes & 15).long()], tab[(codes >> 4).long()]], -1).reshape(codes.shape[0], -1)
    return v * torch.exp2(scale.to(F64) - 127.0).repeat_interleave(32, 1)


def _block_quant(x):
    b = x.to(torch.float32).to(F64).reshape(x.shape[0], -1, 32)
    ka = torch.ceil(torch.log2(b.abs().amax(-1, keepdim=True).clamp(min=2.0 ** -120) / 127.0))
    return (torch.round(b * torch.exp2(-ka)) * torch.exp2(ka)).reshape(x.shape)


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        q, asc = _quant(s["x"])
        y = _mm(q, s["w"]) * s["ws"].to(F64) * asc
        return y if s["b"] is None else y + s["b"].to(F64)
    if kind == "site":
        ex = 6 - math.floor(math.log2(float(s["x"].abs().max())))
        if float(s["x"].abs().max()) * 2.0 ** ex > 127.0:
            ex -= 1
        q = torch.round(s["x"] * 2.0 ** ex).clamp(-127, 127).to(F64)
        return _mm(q, s["w"]) * 2.0 ** (-ex - s["ew"]), torch.tensor([ex], device="cuda", dtype=torch.int32)
    if kind == "outlier":
        x, oi = s["x"].to(F64), s["oidx"].long()
        ho = x[:, oi]
        x[:, oi] = 0.0
        if case["rot"]:
            x = (x.reshape(-1, 256) @ _hadamard(256)).reshape(x.shape) / 16.0
        q, asc = _quant(x)
        return _mm(q, s["w"]) * s["ws"].to(F64) * asc + ho @ s["wo"].to(F64).t()
    if kind == "head":
        bits = {"a15w15": (15, 15), "a15": (15, 8), "w15": (8, 15), "a11w11": (11, 11)}[case["spec"]]
        q, asc = _quant(s["x"], 2.0 ** (bits[0] - 1) - 1)
        out = []
        for p in s["W"].split(8192):
            wq, ws = _quant(p, 2.0 ** (bits[1] - 1) - 1)
            out.append(q @ wq.t() * ws.t() * asc)
        return torch.cat(out, 1)
    d, T = MOE_DIMS[case["dims"]], case["T"]
    lg = s["logits"].to(F64)
    sel = torch.sort(lg, dim=1, descending=True, stable=True)[1][:, :d["k"]]
    w = torch.softmax(torch.gather(lg, 1, sel), 1)
    y = torch.zeros((T, d["H"]), dtype=F64, device="cuda")
    for e in range(d["E"]):
        t, j = (sel == e).nonzero(as_tuple=True)
        if t.numel() == 0:
            continue
        x = s["x"][t]
        if kind == "moe":
            q, asc = _quant(x)
            v = q @ s["w13"][e].to(F64).t() * s["ws13"][e, :, 0].to(F64) * asc
            gate, up = v.chunk(2, 1)
            q, asc = _quant(torch.nn.functional.silu(gate) * up)
            v = q @ s["w2"][e].to(F64).t() * s["ws2"][e, :, 0].to(F64) * asc
        else:
            def rows(r):
                if case["blocks"]:
                    return _block_quant(r)
                q, asc = _quant(r)
                return q * asc
            v = rows(x) @ _mx_weight(s["c13"][e], s["e13"][e]).t() + s["b13"][e].to(F64)
            gate, up = v.chunk(2, 1)
            gate, up = gate.clamp(max=7.0), up.clamp(-7.0, 7.0)
            v = rows((up + 1.0) * gate * torch.sigmoid(1.702 * gate)) @ _mx_weight(s["c2"][e], s["e2"][e]).t()
            v = v + s["b2"][e].to(F64)
        y.index_add_(0, t, v * w[t, j][:, None])
    return y, None, None
