"""Workloads of the gated-delta-rule library as its users run it, for timing
and for comparing results.

Every case goes through a public entry point: the torch ops of ``gdn_hip``
(prefill, its fused and norm forms, the decode step, the gated RMSNorm, the
causal conv1d) or the packages transformers imports (``fla.ops.gated_delta_rule``
and ``causal_conv1d``).  Head counts are the layer's 16 k-heads and 32 v-heads,
its shards, and the 32/32 heads of the reference harness's grid; head dims are
128.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch
import torch.nn.functional as F

_PKG = Path(__file__).resolve().parents[1] / "qwen-drive-edge-orin_amd"
for _p in (str(_PKG), str(_PKG / "hf")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import gdn_hip  # noqa: E402
from causal_conv1d import causal_conv1d_update  # noqa: E402
from fla.ops.gated_delta_rule import (  # noqa: E402
    chunk_gated_delta_rule, recurrent_gated_delta_rule)

D = 128          # head dim of keys and values
TAPS = 4         # conv taps
EPS = 1e-6
# 8 packed prompts of 512 .. 4096 tokens, 19,861 in all
VARLEN_8 = "1427 3804 2613 3898 660 2279 4069 1111"
# tokens x v-heads of the longest listed prefill: no drawn case exceeds it
MOST_TOKEN_HEADS = 19861 * 32
# (k-heads, v-heads): the layer, its shards over 2, 4 and 8 cards, equal heads
HEADS = ((16, 32), (8, 16), (4, 8), (2, 4), (16, 16), (32, 32), (8, 32))


def listed():
    return [
        # a short prompt, or a turn added to a cached conversation: launches count
        dict(name="prefill_T77", kind="prefill", B=1, T=77, HK=16, HV=32),
        # the planner's prompt, one text layer: the headline workload
        dict(name="prefill_T1141", kind="prefill", B=1, T=1141, HK=16, HV=32),
        # the largest point of the reference harness's grid (two long prompts)
        dict(name="prefill_B2_T3200", kind="prefill", B=2, T=3200, HK=32, HV=32),
        # a serving batch of packed prompts of uneven lengths
        dict(name="varlen_8seq", kind="varlen", lengths=VARLEN_8, HK=16, HV=32),
        # transformers' prefill call: expanded raw q and k, v a slice of the
        # conv's output, the q/k norm left to the kernel
        dict(name="hf_prefill_T1503", kind="hf_prefill", B=1, T=1503, HK=16, HV=32),
        # the TensorRT adapter's whole step on raw fp16 inputs
        dict(name="fused_fp16_T1141", kind="fused", B=1, T=1141, HK=16, HV=32, dtype="float16"),
        # prefill and the gated RMSNorm after it, two medium prompts
        dict(name="prefill_norm_B2_T512", kind="prefill_norm", B=2, T=512, HK=16, HV=32),
        # one decode step of a serving batch
        dict(name="decode_B64", kind="decode", B=64, T=1, HK=16, HV=32),
        # one layer's decode step as transformers calls it (conv update, the
        # recurrent step into a new state, the gated RMSNorm), batched
        dict(name="hf_decode_B24", kind="hf_decode", B=24, HK=16, HV=32),
        # the same for one user: the smallest calls
        dict(name="hf_decode_B1", kind="hf_decode", B=1, HK=16, HV=32),
        # the layer's gated RMSNorm over a prompt
        dict(name="rmsnorm_1141x32", kind="norm", rows=1141 * 32, dv=128, dtype="bfloat16",
             wdtype="bfloat16"),
        # the conv in front of q, k and v over a prompt (8192 channels)
        dict(name="conv_T1141", kind="conv", B=1, T=1141, C=8192, dtype="bfloat16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("prefill", "prefill", "varlen", "hf_prefill", "fused", "prefill_norm",
                       "decode", "hf_decode", "norm", "conv"))
    HK, HV = rng.choice(HEADS)
    if kind in ("prefill", "hf_prefill", "fused", "prefill_norm"):
        B = rng.choice((1, 1, 1, 2, 3, 4))
        c = dict(kind=kind, B=B, T=_log_int(rng, 1, min(8192, MOST_TOKEN_HEADS // (B * HV))),
                 HK=HK, HV=HV)
        if kind == "fused":
            c["dtype"] = rng.choice(("float16", "bfloat16"))
        return c
    if kind == "varlen":
        n = _log_int(rng, 2, 24)
        ls = [_log_int(rng, 1, min(4096, MOST_TOKEN_HEADS // (n * HV))) for _ in range(n)]
        return dict(kind=kind, lengths=" ".join(map(str, ls)), HK=HK, HV=HV)
    if kind == "decode":
        # up to 8 tokens a call: the check of drafted tokens
        return dict(kind=kind, B=_log_int(rng, 1, 96), T=rng.choice((1, 1, 1, 2, 3, 4, 5, 8)),
                    HK=HK, HV=HV)
    if kind == "hf_decode":
        return dict(kind=kind, B=_log_int(rng, 1, 64), HK=HK, HV=HV)
    dt = rng.choice(("bfloat16", "bfloat16", "float16"))
    if kind == "norm":
        return dict(kind=kind, rows=_log_int(rng, 1, 4096) * HV, dv=rng.choice((128, 128, 128, 64, 256)),
                    dtype=dt, wdtype=rng.choice((dt, "float32")))
    return dict(kind=kind, B=rng.choice((1, 1, 1, 2, 4)), T=_log_int(rng, 1, 4096),
                C=(2 * HK + HV) * D, dtype=dt)


# ---------------------------------------------------------------- inputs
class _Rand:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def n(self, *shape):
        return torch.randn(*shape, generator=self.gen, device="cuda")

    def u(self, *shape):
        return torch.rand(*shape, generator=self.gen, device="cuda")


def _l2norm(x):
    return x * torch.rsqrt((x * x).sum(-1, keepdim=True) + EPS)


def _gates(r, B, T, HV):
    """beta in (0, 1); log-decays around -0.3 for the fastest head of a layer
    to around -0.01 for the slowest."""
    shift = 1.0 + 4.0 * r.u(HV)
    return F.logsigmoid(r.n(B, T, HV) + shift), torch.sigmoid(r.n(B, T, HV))


def _lengths(case):
    return [int(x) for x in case["lengths"].split()]


def prepare(case, seed):
    r = _Rand(seed)
    kind = case["kind"]
    ops = gdn_hip.load()
    s = {"kind": kind, "ops": ops}
    if kind == "norm":
        dt, wdt = getattr(torch, case["dtype"]), getattr(torch, case["wdtype"])
        s.update(x=r.n(case["rows"], case["dv"]).to(dt), z=r.n(case["rows"], case["dv"]).to(dt),
                 w=(1 + 0.1 * r.n(case["dv"])).to(wdt))
        return s
    if kind == "conv":
        dt = getattr(torch, case["dtype"])
        C = case["C"]
        s.update(x=r.n(case["B"], case["T"], C).to(dt).transpose(1, 2),
                 w=(0.5 * r.n(C, TAPS)).to(dt))
        return s
    HK, HV = case["HK"], case["HV"]
    bf = torch.bfloat16
    if kind == "hf_decode":
        B, C = case["B"], (2 * HK + HV) * D
        g, beta = _gates(r, B, 1, HV)
        s.update(HK=HK, HV=HV, x=r.n(B, C, 1).to(bf), conv_state=r.n(B, C, TAPS).to(bf),
                 w=(0.5 * r.n(C, TAPS)).to(bf), g=g, beta=beta,
                 state=0.1 * r.n(B, HV, D, D), z=r.n(B * HV, D).to(bf),
                 nw=(1 + 0.1 * r.n(D)).to(bf))
        return s
    if kind == "varlen":
        ls = _lengths(case)
        B, T, N = 1, sum(ls), len(ls)
        cu = [0]
        for x in ls:
            cu.append(cu[-1] + x)
        s["cu"] = torch.tensor(cu, dtype=torch.int32, device="cuda")
    else:
        B, T = case["B"], case["T"]
        N = B
    if kind == "fused":
        dt = getattr(torch, case["dtype"])
        s.update(q=r.n(B, T, HK, D).to(dt), k=r.n(B, T, HK, D).to(dt), v=r.n(B, T, HV, D).to(dt),
                 a=r.n(B, T, HV).to(dt), b=r.n(B, T, HV).to(dt),
                 A_log=torch.log(0.02 + 0.98 * r.u(HV)), dt_bias=(0.5 * r.n(HV)).to(dt),
                 state=0.02 * r.n(B, HV, D, D))
        return s
    g, beta = _gates(r, B, T, HV)
    s.update(g=g, beta=beta, s0=0.02 * r.n(N, HV, D, D))
    if kind == "hf_prefill":
        mixed = r.n(B, T, (2 * HK + HV) * D).to(bf)
        q, k, v = torch.split(mixed, [HK * D, HK * D, HV * D], dim=-1)
        rep = HV // HK
        q, k = (x.reshape(B, T, HK, D) for x in (q, k))
        if rep > 1:
            q, k = q.repeat_interleave(rep, dim=2), k.repeat_interleave(rep, dim=2)
        s.update(q=q, k=k, v=v.reshape(B, T, HV, D))
        return s
    s.update(q=_l2norm(r.n(B, T, HK, D)).to(bf), k=_l2norm(r.n(B, T, HK, D)).to(bf),
             v=r.n(B, T, HV, D).to(bf))
    if kind == "prefill_norm":
        s.update(z=r.n(B, T, HV, D).to(bf), nw=(1 + 0.1 * r.n(D)).to(bf))
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    kind, ops = s["kind"], s["ops"]
    if kind == "prefill":
        return ops.chunk_prefill(s["q"], s["k"], s["v"], s["g"], s["beta"], s["s0"])
    if kind == "varlen":
        return ops.chunk_prefill(s["q"], s["k"], s["v"], s["g"], s["beta"], s["s0"],
                                 cu_seqlens=s["cu"])
    if kind == "hf_prefill":
        return chunk_gated_delta_rule(s["q"], s["k"], s["v"], g=s["g"], beta=s["beta"],
                                      initial_state=s["s0"], output_final_state=True,
                                      use_qk_l2norm_in_kernel=True)
    if kind == "fused":
        o = ops.chunk_prefill_fused(s["q"], s["k"], s["v"], s["a"], s["b"], s["A_log"],
                                    s["dt_bias"], s["state"])
        return o, s["state"]
    if kind == "prefill_norm":
        return ops.chunk_prefill_norm(s["q"], s["k"], s["v"], s["g"], s["beta"], s["z"], s["nw"],
                                      s["s0"], eps=EPS)
    if kind == "decode":
        o = ops.recurrent_step(s["q"], s["k"], s["v"], s["g"], s["beta"], s["s0"])
        return o, s["s0"]
    if kind == "hf_decode":
        HK, HV = s["HK"], s["HV"]
        B = s["x"].shape[0]
        mixed = causal_conv1d_update(s["x"], s["conv_state"], s["w"], None, "silu")
        q, k, v = torch.split(mixed.transpose(1, 2), [HK * D, HK * D, HV * D], dim=-1)
        o, s["state"] = recurrent_gated_delta_rule(
            q.reshape(B, 1, HK, D), k.reshape(B, 1, HK, D), v.reshape(B, 1, HV, D), g=s["g"],
            beta=s["beta"], initial_state=s["state"], output_final_state=True,
            use_qk_l2norm_in_kernel=True)
        y = ops.gated_rmsnorm(o.reshape(-1, D), s["z"], s["nw"], EPS)
        return y, s["state"], s["conv_state"]
    if kind == "norm":
        return ops.gated_rmsnorm(s["x"], s["z"], s["w"], EPS)
    return ops.causal_conv1d_fwd(s["x"], s["w"], None, True)


# ---------------------------------------------------------------- work and tolerance
def work(case):
    kind = case["kind"]
    if kind == "norm":
        n = case["rows"] * case["dv"]
        return {"bytes": 6 * n, "flops": 10 * n}
    if kind == "conv":
        n = case["B"] * case["T"] * case["C"]
        return {"bytes": 4 * n + 2 * TAPS * case["C"], "flops": (2 * TAPS + 4) * n}
    HK, HV = case["HK"], case["HV"]
    state = 4 * HV * D * D
    if kind == "hf_decode":
        B, C = case["B"], (2 * HK + HV) * D
        return {"bytes": B * (2 * state + 2 * C * (2 + 2 * TAPS) + 8 * HV + 8 * HV * D)
                + 2 * C * TAPS, "flops": B * HV * 7 * D * D}
    N = len(_lengths(case)) if kind == "varlen" else case["B"]
    tokens = sum(_lengths(case)) if kind == "varlen" else N * case["T"]
    qk = HV if kind == "hf_prefill" else HK
    gates = 4 * HV if kind == "fused" else 8 * HV
    nbytes = tokens * (2 * D * (2 * qk + 2 * HV) + gates) + 2 * N * state
    if kind == "prefill_norm":
        nbytes += tokens * 2 * D * HV
    if kind == "decode":
        return {"bytes": nbytes, "flops": tokens * HV * 7 * D * D}
    # the dense chunked algorithm, 64-token chunks: five C x C x 128 and three
    # C x 128 x 128 products and C^3 / 3 for the inverse per chunk
    C = 64
    return {"bytes": nbytes,
            "flops": tokens * HV * 2 * (5 * C * D + 3 * D * D + C * C / 3)}


def tolerance(case):
    kind = case["kind"]
    # one rounding of the result to 16 bits, and a tie's neighbour here and there
    if kind in ("norm", "conv"):
        return {"rel": 4e-3}
    # sums of 128 products of bf16 values in fp32, o rounded to bf16
    if kind == "decode":
        return {"rel": 4e-3}
    # several chained roundings to 16 bits (conv, normalised rows, o, the norm)
    if kind in ("hf_decode", "prefill_norm"):
        return {"rel": 1e-2}
    # products of 16-bit operands inside a chunk, o rounded to bf16
    return {"rel": 6e-3}


# ---------------------------------------------------------------- 64-bit results
def _delta_rule(q, k, v, g, beta, S, lengths=None):
    """The token recurrence in 64 bits: q, k [B, T, HK, D], v [B, T, HV, D],
    g, beta [B, T, HV], S [B, HV, D, D]; tokens at or past a row's length
    leave its state alone."""
    rep = v.shape[2] // k.shape[2]
    q, k, v, g, beta, S = (x.double() for x in (q, k, v, g, beta, S))
    o = torch.empty_like(v)
    for t in range(v.shape[1]):
        kt = k[:, t].repeat_interleave(rep, dim=1)
        qt = q[:, t].repeat_interleave(rep, dim=1)
        new = S * g[:, t].exp()[..., None, None]
        delta = (v[:, t] - torch.matmul(kt[:, :, None], new)[:, :, 0]) * beta[:, t, :, None]
        new = new + kt[..., None] * delta[:, :, None]
        o[:, t] = torch.matmul(qt[:, :, None], new)[:, :, 0] * D ** -0.5
        if lengths is None:
            S = new
        else:
            S = torch.where((lengths > t)[:, None, None, None], new, S)
    return o, S


def _norm64(x, z, w):
    x, z, w = x.double(), z.double(), w.double()
    return w * x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * F.silu(z)


def _unit64(x):
    return _l2norm(x.double())


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "norm":
        return _norm64(s["x"], s["z"], s["w"])
    if kind == "conv":
        x, w = s["x"].double(), s["w"].double()
        T = x.shape[2]
        xp = F.pad(x, (TAPS - 1, 0))
        return F.silu(sum(xp[:, :, j:j + T] * w[:, j, None] for j in range(TAPS)))
    if kind == "hf_decode":
        HK, HV = s["HK"], s["HV"]
        B = s["x"].shape[0]
        window = torch.cat([s["conv_state"], s["x"]], dim=2).double()
        mixed = F.silu((window[:, :, -TAPS:] * s["w"].double()).sum(-1))
        q, k, v = torch.split(mixed, [HK * D, HK * D, HV * D], dim=-1)
        o, S = _delta_rule(_unit64(q.reshape(B, 1, HK, D)), _unit64(k.reshape(B, 1, HK, D)),
                           v.reshape(B, 1, HV, D), s["g"], s["beta"], s["state"])
        return _norm64(o.reshape(-1, D), s["z"], s["nw"]), S, window[:, :, -TAPS:]
    if kind == "fused":
        g = -s["A_log"].double().exp() * F.softplus(s["a"].double() + s["dt_bias"].double())
        return _delta_rule(_unit64(s["q"]), _unit64(s["k"]), s["v"], g,
                           torch.sigmoid(s["b"].double()), s["state"])
    if kind == "hf_prefill":
        return _delta_rule(_unit64(s["q"]), _unit64(s["k"]), s["v"], s["g"], s["beta"], s["s0"])
    if kind == "varlen":
        ls = _lengths(case)
        T = max(ls)

        def rows(x):
            out = torch.zeros(len(ls), T, *x.shape[2:], dtype=torch.float64, device=x.device)
            for i, (row, n) in enumerate(zip(x[0].split(ls), ls)):
                out[i, :n] = row
            return out

        o, S = _delta_rule(*(rows(s[n]) for n in ("q", "k", "v", "g", "beta")), s["s0"],
                           torch.tensor(ls, device="cuda"))
        return torch.cat([o[i, :n] for i, n in enumerate(ls)])[None], S
    o, S = _delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"], s["s0"])
    if kind == "prefill_norm":
        return _norm64(o, s["z"], s["nw"]), S
    return o, S
