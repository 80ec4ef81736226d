"""Benchmark of the gated-delta-rule prefill on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu-baseline]

One step = one chunked gated-delta prefill call (q, k, v, g, beta,
initial_state -> o, final_state) at the planner shape B=1, T=1141, HV=32,
HK=16, d=128, bf16 inputs, fp32 state, synthetic seeded data.  Inputs are
resident in HBM before timing starts; successive steps rotate through enough
input copies (> 256 MB) that the Infinity Cache cannot serve them, so the
timed number is the cold one.  The warm (same inputs every step) number and
the secondary workloads (gated RMSNorm, decode step, varlen prefill, causal
conv1d prefill and decode update, the fused raw-input prefill, the prefill
with the gated RMSNorm in its output stage) are
reported in the same JSON line.

Prints ONE JSON line.  `value` is TFLOP/s under the fixed dense FLOP
convention of 182.95 kFLOP per token per v-head.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
for p in (ROOT, ROOT / "qwen-drive-edge-orin_amd", ROOT / "tests"):
    sys.path.insert(0, str(p))

HBM_PEAK_GBS = 8000.0       # MI355X HBM3E, published
MFMA_PEAK_TFLOPS = 2500.0   # MI355X dense fp16/bf16 MFMA, published
MALL_BYTES = 256 << 20


def _bytes(*ts):
    return sum(t.numel() * t.element_size() for t in ts if t is not None)


def whole_call_roofline(flops, algo_bytes, ms):
    """Fractions of the whole call against both bounds, and the attainable
    rate min(MFMA peak, AI x HBM peak) with AI = algorithmic FLOPs / minimum
    unique HBM bytes: the best a call can do when it reads its inputs and
    writes its outputs once at peak bandwidth."""
    tflops = flops / ms / 1e9
    gbs = algo_bytes / ms / 1e6
    ai = flops / algo_bytes
    attain = min(MFMA_PEAK_TFLOPS, ai * HBM_PEAK_GBS / 1e3)
    return {"mfma_frac": round(tflops / MFMA_PEAK_TFLOPS, 4),
            "hbm_gbs": round(gbs, 1), "hbm_frac": round(gbs / HBM_PEAK_GBS, 4),
            "algo_flops": flops, "algo_bytes": algo_bytes,
            "arith_intensity_flop_per_byte": round(ai, 1),
            "ridge_flop_per_byte": round(MFMA_PEAK_TFLOPS * 1e3 / HBM_PEAK_GBS, 1),
            "attainable_tflops": round(attain, 1),
            "attainable_bound": "hbm" if ai * HBM_PEAK_GBS / 1e3 < MFMA_PEAK_TFLOPS else "mfma",
            "attainable_us": round(flops / attain / 1e6, 3),
            "frac_of_attainable": round(tflops / attain, 4)}


# Untimed warm-up before every timed region lasts at least this long: from an
# idle GPU the first ~10 ms of back-to-back calls run several percent slower
# (the T=1141 prefill measured 41.5 us per call over its first 220 calls
# against 38.3 us after).
WARM_S = 0.05


def warm_up(fn, n_sets, warmup):
    """`warmup` untimed calls, then more in batches until WARM_S seconds of
    device-synchronised calls have passed."""
    import time
    import torch

    t0 = time.perf_counter()
    i = 0
    while True:
        for _ in range(max(warmup, 1)):
            fn(i % n_sets)
            i += 1
        torch.cuda.synchronize()
        if time.perf_counter() - t0 >= WARM_S:
            return


def time_calls(fn, n_sets, steps, warmup):
    """HIP-event time of `steps` back-to-back calls fn(i) on the current
    stream, bracketed by device synchronisation, after warm_up; returns ms
    per call."""
    import torch

    warm_up(fn, n_sets, warmup)
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record()
    for i in range(steps):
        fn(i % n_sets)
    end.record()
    torch.cuda.synchronize()
    return start.elapsed_time(end) / steps


def time_graph(fn, n_sets, reps, warmup):
    """ms per call of fn(0) .. fn(n_sets - 1) captured once in a HIP graph and
    replayed `reps` times between two events: back-to-back device execution
    without the host's per-call launch cost, which exceeds a few-us kernel's
    own time.  The ops allocate their outputs and issue no memset."""
    import torch

    for i in range(warmup):
        fn(i % n_sets)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            for i in range(n_sets):
                fn(i)
    torch.cuda.current_stream().wait_stream(stream)
    warm_up(lambda i: graph.replay(), 1, 1)
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record()
    for _ in range(reps):
        graph.replay()
    end.record()
    torch.cuda.synchronize()
    return start.elapsed_time(end) / (reps * n_sets)


def rotation(make, per_set_bytes, dev, min_total=2 * MALL_BYTES, max_sets=64):
    n = max(2, min(max_sets, -(-min_total // max(per_set_bytes, 1))))
    base = [t.to(dev) if hasattr(t, "to") else t for t in make()]
    sets = [base] + [[t.clone() if hasattr(t, "clone") else t for t in base] for _ in range(n - 1)]
    return sets


def bench_prefill(ops, dev, steps, warmup):
    import torch
    import gdn_cases as gc

    q, k, v, g, beta, s0 = gc.prefill_inputs()
    in_bytes = _bytes(q, k, v, g, beta, s0)
    sets = rotation(lambda: (q, k, v, g, beta, s0), in_bytes, dev)
    fn = lambda i: ops.chunk_prefill(*sets[i])  # noqa: E731
    cold_ms = time_calls(fn, len(sets), steps, warmup)
    warm_ms = time_calls(lambda i: ops.chunk_prefill(*sets[0]), 1, steps, warmup)
    T, HV = q.shape[1], v.shape[2]
    flops = gc.flops_prefill(T, HV)
    out_bytes = _bytes(v) + _bytes(s0)  # o (bf16, like v) + final state
    algo_bytes = in_bytes + out_bytes
    return dict(cold_ms=cold_ms, warm_ms=warm_ms, flops=flops, algo_bytes=algo_bytes,
                n_sets=len(sets), T=T, HV=HV)


def bench_prefill_norm(ops, dev, steps, warmup):
    """The prefill with the gated RMSNorm in its output stage
    (chunk_prefill_norm(fused=True)) at T=1141 HV=32, cold inputs, against the
    two steps it replaces (chunk_prefill, then gated_rmsnorm; what
    chunk_prefill_norm runs by default) on the same rotated inputs."""
    import torch
    import gdn_cases as gc

    q, k, v, g, beta, s0 = gc.prefill_inputs()
    gen = torch.Generator().manual_seed(33)
    z = torch.randn(*v.shape, generator=gen).to(torch.bfloat16)
    w = (1 + 0.1 * torch.randn(v.shape[-1], generator=gen)).to(torch.bfloat16)
    per = _bytes(q, k, v, g, beta, s0, z)
    sets = rotation(lambda: (q, k, v, g, beta, s0, z, w), per, dev)
    ms_f = time_calls(lambda i: ops.chunk_prefill_norm(*sets[i][:5], sets[i][6], sets[i][7],
                                                       sets[i][5], fused=True),
                      len(sets), steps, warmup)

    def two(i):
        o, _ = ops.chunk_prefill(*sets[i][:6])
        ops.gated_rmsnorm(o, sets[i][6], sets[i][7], 1e-6)

    ms_2 = time_calls(two, len(sets), steps, warmup)
    return dict(ms_f=ms_f, ms_2=ms_2)


def bench_varlen(ops, dev, steps, warmup):
    import torch
    import gdn_cases as gc

    q, k, v, g, beta, s0, cu = gc.varlen_inputs()
    d = [t.to(dev) for t in (q, k, v, g, beta, s0)]
    cud = cu.to(dev)
    # ~1 GB of inputs and workspace: the first few dozen calls of a process
    # run ~10 % slower (measured 500 against 440 us), so 30 warm-up calls
    warmup = max(warmup, 30)
    ms = time_calls(lambda i: ops.chunk_prefill(*d, cu_seqlens=cud), 1, steps, warmup)
    total = int(cu[-1])
    flops = gc.flops_prefill(total, v.shape[2])
    algo = _bytes(q, k, v, g, beta, s0) + _bytes(v) + _bytes(s0)
    out = dict(ms=ms, tflops=flops / ms / 1e9, gbs=algo / ms / 1e6, tokens=total)
    # the same call with each scan instance forced (deltanet_chunk_prefill_cols):
    # 16 value columns per work-group, and the paired 32 (the library picks the
    # wide 64-column instance here)
    import ctypes as ct
    from gdn_hip import capi

    lib = capi.lib()
    N, HV, HK = len(cu) - 1, v.shape[2], q.shape[2]
    wsb = lib.deltanet_prefill_varlen_live_workspace_size(total, N, HV, 128, 128, 64)
    ws = torch.empty(wsb, dtype=torch.uint8, device=dev)
    o = torch.empty_like(d[2])
    sf = torch.empty(N, HV, 128, 128, dtype=torch.float32, device=dev)
    stream = torch.cuda.current_stream().cuda_stream

    def forced(cols):
        def call(i):
            err = lib.deltanet_chunk_prefill_cols(
                *[t.data_ptr() for t in d[:5]], o.data_ptr(), d[5].data_ptr(), sf.data_ptr(),
                cud.data_ptr(), N, total, HV, HK, ws.data_ptr(), wsb, stream, cols, ct.c_uint(0))
            assert err == 0, err
        return time_calls(call, 1, steps, warmup)

    out["ms_scan16"] = forced(16)
    out["ms_scan32"] = forced(32)
    del ws
    return out


def bench_decode(ops, dev, steps, warmup):
    import gdn_cases as gc

    q, k, v, g, beta, s0 = gc.decode_inputs()
    per = _bytes(q, k, v, g, beta, s0)
    sets = rotation(lambda: (q, k, v, g, beta, s0), per, dev)
    ms = time_graph(lambda i: ops.recurrent_step(*sets[i]), len(sets), max(4, steps // len(sets)), warmup)
    algo = per + _bytes(s0) + _bytes(v)  # state read + written, o written
    return dict(ms=ms, gbs=algo / ms / 1e6, frac=algo / ms / 1e6 / HBM_PEAK_GBS, bytes=algo)


def bench_norm(ops, dev, steps, warmup):
    import gdn_cases as gc

    x, z, w, eps = gc.rmsnorm_inputs()
    per = _bytes(x, z, w)
    sets = rotation(lambda: (x, z, w), per, dev)
    ms = time_graph(lambda i: ops.gated_rmsnorm(sets[i][0], sets[i][1], sets[i][2], eps),
                    len(sets), max(4, steps // len(sets)), warmup)
    algo = per + _bytes(x)
    return dict(ms=ms, gbs=algo / ms / 1e6, frac=algo / ms / 1e6 / HBM_PEAK_GBS, bytes=algo)


def bench_stream(dev, steps, warmup):
    """This library's HBM streaming probe (gdn_stream_probe), graph-replayed over
    rotated buffers, for the two HBM-bound access patterns: read 2 / write 1 over
    the gated RMSNorm's 3 x 9.35 MB, and read + write in place over the decode
    state's 134.2 MB.  Best of plain and non-temporal accesses and three grid
    sizes of the grid-stride form; for read 2 / write 1 also the one-pass form
    in the gated RMSNorm's own launch shape (no loop, 1 to 3 16-byte pieces per
    lane).  GB/s of bytes moved."""
    import torch
    from gdn_hip import capi

    lib = capi.lib()
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    out = {}
    for kind, nb, nbuf in ((0, 1141 * 32 * 128 * 2, 3), (1, 64 * 32 * 128 * 128 * 4, 1)):
        sets = rotation(lambda: [torch.empty(nb, dtype=torch.uint8) for _ in range(nbuf)],
                        nbuf * nb, dev)
        moved = 3 * nb if kind == 0 else 2 * nb
        best = None
        for nt in (0, 1):
            for mult in (4, 8, 16):
                def fn(i, nt=nt, blocks=cus * mult):
                    t = sets[i]
                    a = t[0].data_ptr() if kind == 0 else None
                    b = t[1].data_ptr() if kind == 0 else None
                    err = lib.gdn_stream_probe(kind, nt, a, b, t[-1].data_ptr(), nb, blocks,
                                               torch.cuda.current_stream().cuda_stream)
                    assert err == 0, f"gdn_stream_probe returned {err}"
                ms = time_graph(fn, len(sets), max(4, steps // len(sets)), warmup)
                if best is None or ms < best[0]:
                    best = (ms, nt, mult)
        ms, nt, mult = best
        out[kind] = dict(us=ms * 1e3, gbs=moved / ms / 1e6, nontemporal=nt, blocks_per_cu=mult,
                         bytes=moved)
        if kind == 0:
            once = {}
            for pieces in (1, 2, 3):
                def fn(i, pieces=pieces):
                    t = sets[i]
                    err = lib.gdn_stream_probe(2, 1, t[0].data_ptr(), t[1].data_ptr(),
                                               t[-1].data_ptr(), nb, pieces,
                                               torch.cuda.current_stream().cuda_stream)
                    assert err == 0, f"gdn_stream_probe returned {err}"
                ms1 = time_graph(fn, len(sets), max(4, steps // len(sets)), warmup)
                once[pieces] = dict(us=round(ms1 * 1e3, 2), gbs=round(moved / ms1 / 1e6, 1))
            out["once"] = once
        del sets
    return out


def bench_fused(ops, dev, steps, warmup):
    """The fused prefill on the plugin's raw fp16 inputs (q/k L2 norm, gate
    math, conversions and the in-place state inside the two kernels) at
    T=1141 HV=32 HK=16, against the same step done as the reference adapter
    does it: separate normalisation, conversion and gate passes (here torch
    ops on the GPU), the prefill, the o conversion and a state copy."""
    import torch
    import torch.nn.functional as F
    import gdn_cases as gc

    q, k, v, a, b, A_log, dt_bias, s0 = gc.fused_inputs(20, B=1, T=1141, HK=16, HV=32)
    per = _bytes(q, k, v, a, b, s0)
    sets = rotation(lambda: (q, k, v, a, b, A_log, dt_bias, s0), per, dev)
    ms_f = time_calls(lambda i: ops.chunk_prefill_fused(*sets[i]), len(sets), steps, warmup)

    def l2n(x):
        x = x.float()
        return (x * torch.rsqrt((x * x).sum(dim=-1, keepdim=True) + 1e-6)).to(torch.bfloat16)

    def chain(i):
        # the adapter's separate passes (l2 norm with eps inside the rsqrt,
        # g = -exp(A_log) softplus(a + dt_bias), beta = sigmoid(b))
        qq, kk, vv, aa, bb, Al, dt, st = sets[i]
        qn, kn = l2n(qq), l2n(kk)
        g = -torch.exp(Al.float()) * F.softplus(aa.float() + dt.float())
        beta = torch.sigmoid(bb.float())
        o, sf = ops.chunk_prefill(qn, kn, vv.to(torch.bfloat16), g, beta, st)
        o.to(torch.float16)
        st.copy_(sf)

    ms_c = time_calls(chain, len(sets), max(10, steps // 4), warmup)
    return dict(ms_f=ms_f, ms_c=ms_c)


def bench_hf_lane(ops, dev, steps, warmup):
    """transformers' call into the fla adapter at T=1141, HV=32 (q/k already
    repeat_interleaved to 32 heads, bf16, use_qk_l2norm_in_kernel=True):
    with the q/k normalisation in the prep kernel (graph replay: device time,
    as for the other secondaries; the call launches only this library's two
    kernels), and with it done by torch first (the adapter's path for other
    dtypes or a custom scale; timed eagerly, since torch's reductions are
    kept out of captured graphs, so host launch time can show in it)."""
    import importlib
    import torch
    import gdn_cases as gc

    hf = str(ROOT / "qwen-drive-edge-orin_amd" / "hf")
    sys.path.insert(0, hf)
    try:
        ad = importlib.import_module("fla.ops.gated_delta_rule")
    finally:
        sys.path.remove(hf)
    gen = torch.Generator().manual_seed(5)
    T, HV = 1141, 32
    q = torch.randn(1, T, HV, 128, generator=gen).bfloat16().to(dev)
    k = torch.randn(1, T, HV, 128, generator=gen).bfloat16().to(dev)
    _, _, v, g, beta, s0 = gc.prefill_inputs()
    v, g, beta, s0 = v.to(dev), g.to(dev), beta.to(dev), s0.to(dev)
    call = lambda i: ad.chunk_gated_delta_rule(q, k, v, g, beta, initial_state=s0,  # noqa: E731
                                               output_final_state=True,
                                               use_qk_l2norm_in_kernel=True)
    # 8 calls per captured graph, so the graph launch is amortised as in the
    # other graph-timed workloads (same inputs each call: warm)
    ms_k = time_graph(call, 8, max(4, steps // 16), warmup)
    call_t = lambda i: ad.chunk_gated_delta_rule(q, k, v, g, beta, scale=0.0883883,  # noqa: E731
                                                 initial_state=s0, output_final_state=True,
                                                 use_qk_l2norm_in_kernel=True)
    ms_t = time_calls(call_t, 1, max(10, steps // 4), warmup)
    return dict(ms_k=ms_k, ms_t=ms_t)


def bench_twolevel(ops, dev, reps=10):
    """The two-level chunk-group scan prototype (deltanet_chunk_prefill_twolevel)
    against the plain call on the same warm inputs: the T=1141 HV=32 layer and
    the 8-sequence packed batch at 4 segments per sequence, and one long
    sequence with few heads (B=1 T=16384 HV=4 HK=2) at 8 segments, where the
    plain scan leaves most CUs idle.  Device time from the call's own events
    (median of `reps`), split into prep, pass 1 (B), pass 1 (Phi), combine and
    replay; the serial chain depth (chunks a scan walks in a row) of each."""
    import ctypes as ct
    import torch
    import gdn_cases as gc
    from gdn_hip import capi

    lib = capi.lib()
    hip = _Hip()
    stream = torch.cuda.current_stream().cuda_stream
    cases = []
    q, k, v, g, beta, s0 = gc.prefill_inputs()
    cases.append(("T1141_HV32_4seg", (q, k, v, g, beta, s0), None, 4))
    vq, vk, vv, vg, vb, vs0, cu = gc.varlen_inputs()
    cases.append(("varlen_8seq_4seg", (vq, vk, vv, vg, vb, vs0), cu, 4))
    lq, lk, lv, lg, lb, ls0 = gc.make_gdn_inputs(12, B=1, T=16384, HK=2, HV=4, g_shift=2.0)
    cases.append(("T16384_HV4_8seg", (lq, lk, lv, lg, lb, ls0), None, 8))
    out = {}
    for name, ten, cu_t, segs in cases:
        d = [t.to(dev) for t in ten]
        if cu_t is None:
            N, T = d[0].shape[0], d[0].shape[1]
            cu_p = None
            lens = [T] * N
        else:
            N, T = len(cu_t) - 1, int(cu_t[-1])
            cu_h = (ct.c_int32 * len(cu_t))(*[int(x) for x in cu_t])
            cu_p = ct.cast(cu_h, ct.c_void_p)
            lens = [int(cu_t[i + 1] - cu_t[i]) for i in range(N)]
        HV, HK = d[2].shape[2], d[0].shape[2]
        o = torch.empty_like(d[2])
        sf = torch.empty(N, HV, 128, 128, device=dev)
        wsb = lib.deltanet_prefill_twolevel_workspace_size(cu_p, N, T, HV, segs)
        ws = torch.empty(wsb, dtype=torch.uint8, device=dev)
        evs = hip.events(6)
        parts = []
        for r in range(reps + 2):
            err = lib.deltanet_chunk_prefill_twolevel(
                *[t.data_ptr() for t in d[:5]], o.data_ptr(), d[5].data_ptr(), sf.data_ptr(),
                cu_p, N, T, HV, HK, segs, ws.data_ptr(), wsb, stream, evs, 6)
            assert err == 0, err
            torch.cuda.synchronize()
            if r >= 2:
                parts.append([hip.elapsed_ms(evs[i], evs[i + 1]) * 1e3 for i in range(5)])
        hip.destroy(evs)
        med = [sorted(p[i] for p in parts)[len(parts) // 2] for i in range(5)]
        if cu_t is None:
            plain = lambda i: ops.chunk_prefill(*d)  # noqa: E731
        else:
            cud = cu_t.to(dev)
            plain = lambda i: ops.chunk_prefill(*d, cu_seqlens=cud)  # noqa: E731
        ms_plain = time_calls(plain, 1, reps * 2, 3)
        nch = [(n + 63) // 64 for n in lens]
        seg_len = max(-(-c // min(segs, c)) if c else 0 for c in nch)
        cus = torch.cuda.get_device_properties(dev).multi_processor_count

        def groups(seqs):
            # work-groups of the scan instance that the library chooses
            cols = lib.deltanet_prefill_scan_cols(sum(nch), seqs, HV, HK, cus, 0)
            return -(-seqs * HV // 8) * 8 * (128 // cols)

        nseg = sum(min(segs, c) if c else 1 for c in nch)
        out[name] = {"us_plain": round(ms_plain * 1e3, 2),
                     "us_twolevel": round(sum(med), 2),
                     "us_prep": round(med[0], 2), "us_pass1_B": round(med[1], 2),
                     "us_pass1_Phi": round(med[2], 2), "us_combine": round(med[3], 2),
                     "us_replay": round(med[4], 2),
                     "serial_chunks_plain": max(nch),
                     "serial_chunks_twolevel": 2 * seg_len + max(0, min(segs, max(nch)) - 2),
                     "scan_groups_plain": groups(N),
                     "scan_groups_per_pass_twolevel": groups(nseg)}
        del ws, d
    return out


def bench_conv(ops, dev, steps, warmup):
    """Causal conv1d + SiLU ahead of the recurrence: the prefill form over
    the layer's conv channels (D = 2 * 16 * 128 + 32 * 128 = 8192, T = 1141,
    K = 4, bf16) and the decode update at B = 64 (state of 4 tokens)."""
    import torch

    D, T, K = 8192, 1141, 4
    gen = torch.Generator().manual_seed(3)
    x = torch.randn(1, T, D, generator=gen).bfloat16()
    w = (0.5 * torch.randn(D, K, generator=gen)).bfloat16()
    per = _bytes(x)
    sets = rotation(lambda: (x, w), per, dev)
    ms = time_graph(lambda i: ops.causal_conv1d_fwd(sets[i][0].transpose(1, 2), sets[i][1], None,
                                                    True),
                    len(sets), max(4, steps // len(sets)), warmup)
    algo = 2 * _bytes(x) + _bytes(w)   # x read, y written, weights
    Bd, L = 64, 4
    xt = torch.randn(Bd, 1, D, generator=gen).bfloat16()
    st = torch.randn(Bd, D, L, generator=gen).bfloat16()
    per_d = _bytes(xt, st)
    dsets = rotation(lambda: (xt, st, w), per_d, dev)
    ms_d = time_graph(lambda i: ops.causal_conv1d_update(dsets[i][0].transpose(1, 2), dsets[i][1],
                                                         dsets[i][2], None, True),
                      len(dsets), max(4, steps // len(dsets)), warmup)
    algo_d = 2 * _bytes(xt) + 2 * _bytes(st) + _bytes(w)   # x, y; state read + written
    return dict(ms=ms, gbs=algo / ms / 1e6, frac=algo / ms / 1e6 / HBM_PEAK_GBS,
                ms_d=ms_d, gbs_d=algo_d / ms_d / 1e6, frac_d=algo_d / ms_d / 1e6 / HBM_PEAK_GBS)


# Algorithmic FLOPs per chunk-head of each prefill kernel under the fixed
# convention (C = 64, dk = dv = 128, 2 FLOP per MAC; five C x C x 128
# products, three 64 x 128 x 128 products and C^3/3 MACs of inversion, 182.95
# kFLOP per token per v-head in total), split by where each product runs:
#   prep  K K^T, Q K^T, W = T diag(beta e^c) K, and the inversion
#         = 3 C x C x 128 + C^3/3 = 3.32 MFLOP
#   scan  U = T diag(beta) V, M V_new (two C x C x 128), W S, (Q e^c) S and
#         K~^T V_new (three 64 x 128 x 128) = 8.39 MFLOP
_CC = 2 * 64 * 64 * 128          # one C x C x 128 product
_CD = 2 * 64 * 128 * 128         # one 64 x 128 x 128 product
_INV = 2 * 64 ** 3 // 3
KERNEL_FLOPS_PER_CHUNK_HEAD = {"gdn_prep_kernel": 3 * _CC + _INV,
                               "gdn_scan_kernel": 3 * _CD + 2 * _CC}
assert sum(KERNEL_FLOPS_PER_CHUNK_HEAD.values()) == 5 * _CC + 3 * _CD + _INV


class _Hip:
    """hipEvent_t helpers over libamdhip64 (the events the library records)."""

    def __init__(self):
        import ctypes as ct

        self.ct = ct
        self.rt = ct.CDLL("libamdhip64.so")
        self.rt.hipEventCreate.argtypes = [ct.POINTER(ct.c_void_p)]
        self.rt.hipEventElapsedTime.argtypes = [ct.POINTER(ct.c_float), ct.c_void_p, ct.c_void_p]
        self.rt.hipEventDestroy.argtypes = [ct.c_void_p]
        self.rt.hipEventRecord.argtypes = [ct.c_void_p, ct.c_void_p]

    def record(self, ev, stream):
        assert self.rt.hipEventRecord(ev, stream) == 0

    def events(self, n):
        evs = (self.ct.c_void_p * n)()
        for i in range(n):
            ev = self.ct.c_void_p()
            assert self.rt.hipEventCreate(self.ct.byref(ev)) == 0
            evs[i] = ev
        return evs

    def elapsed_ms(self, a, b):
        ms = self.ct.c_float()
        assert self.rt.hipEventElapsedTime(self.ct.byref(ms), a, b) == 0
        return ms.value

    def destroy(self, evs):
        for e in evs:
            self.rt.hipEventDestroy(e)


def kernel_times(dev, steps, warmup):
    """Average duration of each prefill kernel at T=1141 HV=32, cold: `steps`
    back-to-back launches of that kernel alone (deltanet_chunk_prefill_kernel)
    between two HIP events on the launch stream.  Every launch touches inputs
    and a workspace the previous launches did not: the launches rotate over the
    resident input copies, each with its own workspace, which a full call
    filled beforehand for the scan's launches (the scan reads the records the
    prep of the same inputs wrote)."""
    import torch
    import gdn_cases as gc
    from gdn_hip import capi

    lib = capi.lib()
    hip = _Hip()
    nk = lib.deltanet_prefill_kernel_count()
    names = [lib.deltanet_prefill_kernel_name(i).decode() for i in range(nk)]
    q, k, v, g, beta, s0 = gc.prefill_inputs()
    B, T, HK, D = q.shape
    HV = v.shape[2]
    sets = rotation(lambda: (q, k, v, g, beta, s0), _bytes(q, k, v, g, beta, s0), dev)
    wsb = lib.deltanet_prefill_live_workspace_size(B, T, HV, D, D, 64)
    wss = [torch.empty(wsb, dtype=torch.uint8, device=dev) for _ in sets]
    o = torch.empty_like(sets[0][2])
    sf = torch.empty_like(sets[0][5])
    stream = torch.cuda.current_stream().cuda_stream

    def launch(i, kernel):
        qq, kk, vv, gg, bb, ss = sets[i % len(sets)]
        args = (qq.data_ptr(), kk.data_ptr(), vv.data_ptr(), gg.data_ptr(), bb.data_ptr(),
                o.data_ptr(), ss.data_ptr(), sf.data_ptr(), B, T, HV, HK, D, D, 64,
                wss[i % len(sets)].data_ptr(), wsb, stream)
        err = (lib.deltanet_chunk_prefill(*args, 0) if kernel < 0
               else lib.deltanet_chunk_prefill_kernel(*args, kernel))
        assert err == 0, f"prefill kernel {kernel} returned {err}"

    out = {}
    nch = B * ((T + 63) // 64) * HV
    for j, nm in enumerate(names):
        if j > 0:
            for i in range(len(sets)):
                launch(i, -1)   # every workspace holds its inputs' records
        warm_up(lambda i: launch(i, j), len(sets), warmup)
        ev = hip.events(2)
        hip.record(ev[0], stream)
        for i in range(steps):
            launch(i, j)
        hip.record(ev[1], stream)
        torch.cuda.synchronize()
        out[nm] = dict(ms=hip.elapsed_ms(ev[0], ev[1]) / steps,
                       flops=KERNEL_FLOPS_PER_CHUNK_HEAD[nm] * nch)
        hip.destroy(ev)
    del wss
    return out


def traffic_from_profiles(kernel):
    """HBM bytes per launch of `kernel` (T=1141, HV=32 prefill) from the committed rocprofv3
    --pmc summary (FETCH_SIZE + WRITE_SIZE, calibrated against a copy of
    known size), or None when no summary exists for it."""
    import re

    p = ROOT / "profiles" / f"{kernel}_T1141_HV32_traffic.md"
    if not p.exists():
        return None
    m = re.search(r"^traffic_bytes_per_launch:\s*([0-9.eE+]+)", p.read_text(), flags=re.M)
    return float(m.group(1)) if m else None


def trace_from_profiles():
    """Average duration (µs) of each prefill kernel at T=1141 HV=32 from the committed
    rocprofv3 kernel-trace summary (rows of the plain bf16 instances at this
    workload's grids), or {} when it is absent."""
    import re

    p = ROOT / "profiles" / "gdn_prefill_T1141_HV32_kernel_trace.md"
    if not p.exists():
        return {}
    out = {}
    for m in re.finditer(r"^\| (gdn_prep_kernel<false,0,false(?:,false)?>|"
                         r"gdn_scan_kernel<0,false,false(?:,false)?>) \| \d+ \| "
                         r"([0-9.]+) \|.*\| (\d+)x1 \| \d+ \|$", p.read_text(), flags=re.M):
        name = m.group(1).split("<")[0]
        grid = int(m.group(3))
        if (name == "gdn_prep_kernel" and grid == 576) or (name == "gdn_scan_kernel" and grid == 256):
            out[name] = float(m.group(2))
    return out


def profile_pass(ops, dev):
    """Work for a counter run: cold T=1141 HV=32 prefill calls, then a copy of known
    size (torch.neg over 256 MiB fp32: 256 MiB read + 256 MiB written)."""
    import torch
    import gdn_cases as gc

    q, k, v, g, beta, s0 = gc.prefill_inputs()
    sets = rotation(lambda: (q, k, v, g, beta, s0), _bytes(q, k, v, g, beta, s0), dev)
    for i in range(4):
        ops.chunk_prefill(*sets[(7 * i) % len(sets)])
    torch.cuda.synchronize()
    del sets
    # gated RMSNorm (1141 x 32 x 128) and the decode step (B64 HV32), each on
    # input copies it has not touched before (cold)
    x, z, w, eps = gc.rmsnorm_inputs()
    nsets = rotation(lambda: (x, z, w), _bytes(x, z, w), dev)
    for i in range(4):
        ops.gated_rmsnorm(nsets[(5 * i) % len(nsets)][0], nsets[(5 * i) % len(nsets)][1],
                          nsets[(5 * i) % len(nsets)][2], eps)
    torch.cuda.synchronize()
    del nsets
    dq, dk, dv, dg, db, ds = gc.decode_inputs()
    dsets = rotation(lambda: (dq, dk, dv, dg, db, ds), _bytes(dq, dk, dv, dg, db, ds), dev,
                     max_sets=5)
    for i in range(4):
        ops.recurrent_step(*dsets[i % len(dsets)])
    torch.cuda.synchronize()
    del dsets
    src = torch.ones(64 << 20, dtype=torch.float32, device=dev)
    dst = torch.empty_like(src)
    for _ in range(2):
        torch.neg(src, out=dst)
    torch.cuda.synchronize()
    print("profile pass done: 4 prefill calls (T=1141, HV=32), 4 gated RMSNorm calls "
          "(1141x32x128), 4 decode steps (B64 HV32), 2 x torch.neg over 256 MiB", flush=True)


def _cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for ln in f:
                if ln.startswith("model name"):
                    return ln.split(":", 1)[1].strip()
    except OSError:
        pass
    return None


def _cpu_time(run, budget_s, max_runs=50):
    """One warm-up, then timed calls until >= 3 and the budget is spent;
    median ms."""
    run()
    times = []
    t_start = time.perf_counter()
    while len(times) < 3 or (time.perf_counter() - t_start < budget_s and len(times) < max_runs):
        t0 = time.perf_counter()
        run()
        times.append(time.perf_counter() - t0)
    times.sort()
    return times[len(times) // 2] * 1e3, len(times)


def cpu_baseline(gpu_us=None, budget_s=8.0):
    """The CPU oracle (fp32 torch restatement of the reference's torch path) on
    the same seeded inputs as the GPU runs, on the host cores, in this process.
    `value` is config 4 (the T=1141 HV=32 prefill); the other configs are timed
    beside it: 1 (CPU plumbing), 2 (gated RMSNorm), 3 (decode step) and 5
    (varlen prefill, one call per sequence)."""
    import torch
    import gdn_cases as gc
    from oracle import gdn_oracle as orc

    # the host share of one GPU is at most 16 cores, whatever os.cpu_count() says
    torch.set_num_threads(max(1, min(16, int(os.environ.get("OMP_NUM_THREADS", "16")),
                                     os.cpu_count() or 1)))
    gpu_us = gpu_us or {}
    q, k, v, g, beta, s0 = gc.prefill_inputs()
    ms4, n4 = _cpu_time(lambda: orc.chunk_gated_delta_rule(q, k, v, g, beta, s0,
                                                           dtype=torch.float32), budget_s)
    flops = gc.flops_prefill(q.shape[1], v.shape[2])
    configs = {}

    def row(name, ms, n, sample):
        r = {"ms_per_call": round(ms, 3), "runs": n, "sample": sample}
        if name in gpu_us:
            r["gpu_us"] = gpu_us[name]
            r["speedup"] = round(ms * 1e3 / gpu_us[name], 1)
        configs[name] = r

    row("c4_prefill_T1141_HV32", ms4, n4, "full call")
    pq, pk, pv, pg, pb = gc.plumbing_inputs()[:5]
    ms1, n1 = _cpu_time(lambda: orc.chunk_gated_delta_rule(pq, pk, pv, pg, pb, None,
                                                           dtype=torch.float32), 2.0)
    row("c1_plumbing_T256_H4_d64", ms1, n1, "full call")
    x, z, w, eps = gc.rmsnorm_inputs()
    ms2, n2 = _cpu_time(lambda: orc.gated_rmsnorm(x, z, w, eps), 2.0)
    row("c2_gated_rmsnorm_1141x32x128", ms2, n2, "full call (bf16 I/O, fp32 math)")
    dq, dk, dv, dg, db, ds = gc.decode_inputs()
    ms3, n3 = _cpu_time(lambda: orc.recurrent_gated_delta_rule(dq, dk, dv, dg, db, ds,
                                                               dtype=torch.float32), 3.0,
                        max_runs=10)
    row("c3_decode_B64_HV32", ms3, n3, "full step, state [64,32,128,128] fp32")
    vq, vk, vv, vg, vb, vs0, cu = gc.varlen_inputs()
    ms5, n5 = _cpu_time(lambda: orc.chunk_gated_delta_rule_varlen(vq, vk, vv, vg, vb, cu, vs0,
                                                                  dtype=torch.float32), 3.0,
                        max_runs=5)
    row("c5_varlen_8seq_19861tok", ms5, n5, "8 sequences, one call each")
    return dict(value=round(flops / ms4 / 1e9, 6), unit="TFLOP/s", ms_per_call=round(ms4, 3),
                cores=torch.get_num_threads(), cpu_count=os.cpu_count(), cpu_model=_cpu_model(),
                kind="port",
                sample=f"full prefill call (T=1141, HV=32), fp32 torch CPU oracle, median of {n4}",
                configs=configs)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-secondary", action="store_true")
    ap.add_argument("--profile-pass", action="store_true",
                    help="no timing: 4 cold T=1141 HV=32 prefill calls, then 2 elementwise copies of "
                         "256 MiB (the calibration for rocprofv3 --pmc FETCH_SIZE/WRITE_SIZE)")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU: the gated-delta hot path is built and measured on a "
              "single MI355X (heads shard with no exchange across GPUs); run with --gpus 1",
              file=sys.stderr)
        sys.exit(2)

    import torch
    import gdn_hip

    ops = gdn_hip.load()
    dev = torch.device("cuda:0")
    if args.profile_pass:
        profile_pass(ops, dev)
        return
    pre = bench_prefill(ops, dev, args.steps, args.warmup)
    ms = pre["cold_ms"]
    tflops = pre["flops"] / ms / 1e9
    gbs = pre["algo_bytes"] / ms / 1e6
    line = {
        "metric": "gated-delta prefill µs + TFLOP/s (T=1141,H=32,d=128); % MFMA/HBM roofline",
        "value": round(tflops, 3),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 5),
        "us_per_call": round(ms * 1e3, 2),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (seeded randn; q/k l2-normalised; beta=sigmoid, g=logsigmoid(x+2))",
        "config": {"workload": "chunked gated-delta prefill, one layer", "B": 1, "T": pre["T"],
                   "HV": pre["HV"], "HK": 16, "dk": 128, "dv": 128, "chunk": 64,
                   "inputs": f"rotated over {pre['n_sets']} resident copies (cold)"},
        "warm": {"us_per_call": round(pre["warm_ms"] * 1e3, 2),
                 "tflops": round(pre["flops"] / pre["warm_ms"] / 1e9, 3)},
        "roofline_whole_call": whole_call_roofline(pre["flops"], pre["algo_bytes"], ms),
    }
    kt = kernel_times(dev, args.steps, args.warmup)
    trace = trace_from_profiles()
    # the dominant kernel: the longer one in the committed rocprof kernel
    # trace of this workload (the live timing when no trace is committed)
    dom = max(kt, key=lambda nm: trace.get(nm, kt[nm]["ms"] * 1e3))
    per = {}
    for nm, d in kt.items():
        # achieved / frac from the committed rocprof trace average (each
        # launch's own begin-to-end time); the live back-to-back cold figure
        # beside it (it also counts the launch gaps between kernels)
        live = d["flops"] / d["ms"] / 1e9
        t_us = trace.get(nm)
        ach = d["flops"] / t_us / 1e6 if t_us else live
        per[nm] = {"trace_avg_us": t_us, "achieved": round(ach, 3),
                   "frac": round(ach / MFMA_PEAK_TFLOPS, 5),
                   "us_per_launch_live": round(d["ms"] * 1e3, 2),
                   "achieved_live": round(live, 3), "frac_live": round(live / MFMA_PEAK_TFLOPS, 5),
                   "algo_flops": d["flops"],
                   "algo_flops_per_chunk_head": KERNEL_FLOPS_PER_CHUNK_HEAD[nm],
                   "traffic": traffic_from_profiles(nm)}
    line["roofline"] = {
        "kernel": dom, "bound": "mfma", "achieved": per[dom]["achieved"],
        "peak": MFMA_PEAK_TFLOPS, "unit": "TFLOP/s", "frac": per[dom]["frac"],
        "traffic": per[dom]["traffic"], "trace_avg_us": per[dom]["trace_avg_us"],
        "us_per_launch_live": per[dom]["us_per_launch_live"],
        "frac_live": per[dom]["frac_live"],
        "kernels": per,
    }
    if not args.no_secondary:
        nrm = bench_norm(ops, dev, args.steps, args.warmup)
        dec = bench_decode(ops, dev, max(20, args.steps // 4), args.warmup)
        var = bench_varlen(ops, dev, max(10, args.steps // 10), 5)
        cv = bench_conv(ops, dev, args.steps, args.warmup)
        fu = bench_fused(ops, dev, args.steps, args.warmup)
        pn = bench_prefill_norm(ops, dev, args.steps, args.warmup)
        hl = bench_hf_lane(ops, dev, args.steps, args.warmup)
        sp = bench_stream(dev, args.steps, args.warmup)
        tl = bench_twolevel(ops, dev)
        line["secondary"] = {
            "gated_rmsnorm_1141x32x128": {
                "us": round(nrm["ms"] * 1e3, 2), "GB/s": round(nrm["gbs"], 1),
                "hbm_frac": round(nrm["frac"], 4),
                "frac_of_stream_probe": round(nrm["gbs"] / max(sp[0]["gbs"], max(
                    v["gbs"] for v in sp["once"].values())), 4),
                "frac_of_same_shape_probe": round(nrm["gbs"] / sp["once"][2]["gbs"], 4)},
            "decode_B64_HV32": {"us": round(dec["ms"] * 1e3, 2), "GB/s": round(dec["gbs"], 1),
                          "hbm_frac": round(dec["frac"], 4),
                          "frac_of_stream_probe": round(dec["gbs"] / sp[1]["gbs"], 4)},
            "hbm_stream_probe_read2_write1_3x9.35MB": {
                "us": round(sp[0]["us"], 2), "GB/s": round(sp[0]["gbs"], 1),
                "hbm_frac": round(sp[0]["gbs"] / HBM_PEAK_GBS, 4),
                "nontemporal": sp[0]["nontemporal"], "blocks_per_cu": sp[0]["blocks_per_cu"],
                "one_pass_nontemporal_by_pieces_per_lane": sp["once"]},
            "hbm_stream_probe_rw_in_place_134.2MB": {
                "us": round(sp[1]["us"], 2), "GB/s": round(sp[1]["gbs"], 1),
                "hbm_frac": round(sp[1]["gbs"] / HBM_PEAK_GBS, 4),
                "nontemporal": sp[1]["nontemporal"], "blocks_per_cu": sp[1]["blocks_per_cu"]},
            "varlen_prefill_8seq_19861tok": {"us": round(var["ms"] * 1e3, 2),
                                  "TFLOP/s": round(var["tflops"], 3),
                                  "tokens": var["tokens"],
                                  "us_scan_16col_forced": round(var["ms_scan16"] * 1e3, 2),
                                  "us_scan_32col_forced": round(var["ms_scan32"] * 1e3, 2)},
            "causal_conv1d_silu_1141x8192_k4": {"us": round(cv["ms"] * 1e3, 2),
                                                "GB/s": round(cv["gbs"], 1),
                                                "hbm_frac": round(cv["frac"], 4)},
            "fused_prefill_fp16_raw_T1141_HV32": {"us": round(fu["ms_f"] * 1e3, 2),
                                                  "adapter_chain_us": round(fu["ms_c"] * 1e3, 2)},
            "prefill_gated_rmsnorm_fused_T1141_HV32": {
                "us": round(pn["ms_f"] * 1e3, 2),
                "us_prefill_then_gated_rmsnorm": round(pn["ms_2"] * 1e3, 2)},
            "hf_lane_chunk_gated_delta_rule_T1141_HV32": {
                "us": round(hl["ms_k"] * 1e3, 2),
                "us_torch_l2norm_eager": round(hl["ms_t"] * 1e3, 2)},
            "twolevel_scan_prototype": tl,
            "causal_conv1d_update_B64x8192_k4": {"us": round(cv["ms_d"] * 1e3, 2),
                                                 "GB/s": round(cv["gbs_d"], 1),
                                                 "hbm_frac": round(cv["frac_d"], 4)},
        }
    if not args.no_cpu_baseline:
        gpu_us = {"c4_prefill_T1141_HV32": line["us_per_call"]}
        sec = line.get("secondary", {})
        for key, name in (("gated_rmsnorm_1141x32x128", "c2_gated_rmsnorm_1141x32x128"),
                          ("decode_B64_HV32", "c3_decode_B64_HV32"),
                          ("varlen_prefill_8seq_19861tok", "c5_varlen_8seq_19861tok")):
            if key in sec:
                gpu_us[name] = sec[key]["us"]
        line["cpu_baseline"] = cpu_baseline(gpu_us)
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
