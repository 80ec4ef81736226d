"""GPU parity of the chunked prefill against the CPU oracle.

The oracle runs in fp64 on the same bf16/fp32 input tensors.  Bars:
max |err| <= 2e-2 on o and on the final state (mean error printed), and the
reference harness's random-case bar (row-cos >= 0.999, max-rel < 1e-2 with
denominator floor 0.1; kernels/harness/parity_test.py:188-189).
"""
import pytest
import torch

import gdn_cases as gc
from oracle import gdn_oracle as orc

pytestmark = pytest.mark.gpu


def _run_and_check(ops, dev, q, k, v, g, beta, s0, tag, ref_bar=True, cu=None):
    print(f"[prefill] {tag} q={tuple(q.shape)} v={tuple(v.shape)} s0={'Y' if s0 is not None else 'n'}"
          f" cu={'Y' if cu is not None else 'n'}", flush=True)
    args = [t.to(dev) if t is not None else None for t in (q, k, v, g, beta, s0)]
    if cu is None:
        o, sf = ops.chunk_prefill(*args)
        o_ref, s_ref = orc.chunk_gated_delta_rule(q, k, v, g, beta, s0, dtype=torch.float64)
    else:
        o, sf = ops.chunk_prefill(*args, cu_seqlens=cu.to(dev))
        o_ref, s_ref = orc.chunk_gated_delta_rule_varlen(q, k, v, g, beta, cu, s0,
                                                         dtype=torch.float64)
    torch.cuda.synchronize()
    mo, ms = gc.parity(o, o_ref), gc.parity(sf, s_ref)
    print(f"    o: {gc.fmt(mo)}\n    S: {gc.fmt(ms)}", flush=True)
    gc.assert_abs(mo, what=f"{tag} o")
    gc.assert_abs(ms, what=f"{tag} state")
    if ref_bar:
        gc.assert_ref_bar(mo, what=f"{tag} o")
        gc.assert_ref_bar(ms, what=f"{tag} state")
    return o, sf


def test_prefill_T1141_HV32(ops, dev):
    """B1 T1141 HV32 HK16 d128: ragged 53-row tail chunk, GQA 2:1; also the
    reference's fixture bar (o L2-rel < 3e-3, cos >= 0.9999; state cos >=
    0.9999, max-rel < 1e-3)."""
    q, k, v, g, beta, s0 = gc.prefill_inputs()
    o, sf = _run_and_check(ops, dev, q, k, v, g, beta, s0, tag="prefill T1141 HV32")
    o_ref, s_ref = orc.chunk_gated_delta_rule(q, k, v, g, beta, s0, dtype=torch.float64)
    gc.assert_fixture_bar(o, o_ref, sf, s_ref, what="T1141 HV32")


def test_golden_g128(ops, dev):
    """Committed fixture (tests/golden/g128.npz): fp64 recurrence outputs."""
    from test_golden import g128_inputs

    q, k, v, g, beta, s0, o_ref, s_ref = g128_inputs()
    print(f"[prefill] golden g128 q={tuple(q.shape)} v={tuple(v.shape)}", flush=True)
    o, sf = ops.chunk_prefill(*[t.to(dev) for t in (q, k, v, g, beta, s0)])
    torch.cuda.synchronize()
    mo, ms = gc.parity(o, o_ref), gc.parity(sf, s_ref)
    print(f"    o: {gc.fmt(mo)}\n    S: {gc.fmt(ms)}", flush=True)
    gc.assert_abs(mo, what="g128 o")
    gc.assert_abs(ms, what="g128 state")
    gc.assert_fixture_bar(o, o_ref, sf, s_ref, what="g128")


def test_varlen_8_sequences(ops, dev):
    """8 sequences of seed-7 lengths (sum 19861), independent initial states.
    The workspace (693 MB) exceeds the 256 MB MALL, so the scan reads the
    prep's records back from HBM."""
    q, k, v, g, beta, s0, cu = gc.varlen_inputs()
    o, sf = _run_and_check(ops, dev, q, k, v, g, beta, s0, tag="varlen 8 seqs", cu=cu)
    o_ref, s_ref = orc.chunk_gated_delta_rule_varlen(q, k, v, g, beta, cu, s0, dtype=torch.float64)
    gc.assert_fixture_bar(o, o_ref, sf, s_ref, what="varlen 8 seqs")


@pytest.mark.parametrize("scale", [100.0, 1000.0])
def test_fp16_operand_headroom(ops, dev, scale):
    """The scan's fp16 operands (beta v as an hi / lo pair, the state S rounded
    for the W S product, -W, M, Q, T - I) hold values below 65,504.  With
    unit-norm q / k rows and beta in (0, 1), |W|, |M| and |Q| stay below 1,
    so the limit binds through v and the state: here v and the initial state
    are scaled by 100 and 1000 at the T=1141 HV=32 shape (|v| up to ~5,000,
    |S| growing with it).  o and the final state scale exactly with (v, s0),
    so the bar is the absolute bar times the scale plus the reference
    harness's fixture bar on o / scale and S / scale (its state max-rel
    floors the denominator at 0.1, an absolute size, so it applies in the
    unit domain)."""
    q, k, v, g, beta, s0 = gc.prefill_inputs()
    vs = (v.float() * scale).to(torch.bfloat16)
    ss = s0 * scale
    print(f"[prefill] fp16 headroom: v, s0 x {scale:g}, max|v| {vs.float().abs().max():.1f}",
          flush=True)
    d = [t.to(dev) for t in (q, k, vs, g, beta, ss)]
    o, sf = ops.chunk_prefill(*d, checked=True)
    torch.cuda.synchronize()
    assert torch.isfinite(o.float()).all() and torch.isfinite(sf).all()
    o_ref, s_ref = orc.chunk_gated_delta_rule(q, k, vs, g, beta, ss, dtype=torch.float64)
    mo, ms = gc.parity(o, o_ref), gc.parity(sf, s_ref)
    print(f"    o: {gc.fmt(mo)}\n    S: {gc.fmt(ms)}  max|S| {s_ref.abs().max():.1f}", flush=True)
    gc.assert_abs(mo, what="scaled o", tol=gc.ABS_TOL * scale)
    gc.assert_abs(ms, what="scaled state", tol=gc.ABS_TOL * scale)
    gc.assert_fixture_bar(o.double().cpu() / scale, o_ref / scale, sf.double().cpu() / scale,
                          s_ref / scale, what=f"v x {scale:g}, divided back")


@pytest.mark.parametrize("T", [1, 2, 17, 63, 64, 65, 127, 128, 200])
@pytest.mark.parametrize("B", [1, 2])
def test_small_shapes(ops, dev, T, B):
    q, k, v, g, beta, s0 = gc.make_gdn_inputs(100 + T * 3 + B, B=B, T=T, HK=2, HV=4)
    _run_and_check(ops, dev, q, k, v, g, beta, s0, tag=f"T{T}B{B}")


@pytest.mark.parametrize("hk,hv", [(4, 4), (1, 4), (2, 8), (3, 6)])
def test_head_maps(ops, dev, hk, hv):
    q, k, v, g, beta, s0 = gc.make_gdn_inputs(7 + hk * 10 + hv, B=1, T=150, HK=hk, HV=hv,
                                              with_s0=False)
    _run_and_check(ops, dev, q, k, v, g, beta, None, tag=f"hk{hk}hv{hv}")


@pytest.mark.parametrize("l2_pre", [False, True])
@pytest.mark.parametrize("B", [1, 2])
@pytest.mark.parametrize("S", [128, 512, 3200])
def test_reference_grid(ops, dev, l2_pre, B, S):
    """The reference harness's random grid (kernels/harness/parity_cuda.py:146-153):
    H=32 heads (q/k pre-expanded), q/k = randn/8, g = -0.3 rand, beta = rand."""
    seed = hash((B, S, l2_pre)) % 2 ** 31
    q, k, v, g, beta, s0 = gc.make_reference_inputs(B, S, seed, l2_pre=l2_pre)
    _run_and_check(ops, dev, q, k, v, g, beta, s0, tag=f"grid S{S} B{B} l2={l2_pre}")


def test_reference_grid_init_state(ops, dev):
    """parity_cuda.py:154-156: B=1, S=512 with a random initial state."""
    q, k, v, g, beta, s0 = gc.make_reference_inputs(1, 512, hash((1, 512, False)) % 2 ** 31,
                                                     with_init_state=True)
    _run_and_check(ops, dev, q, k, v, g, beta, s0, tag="grid init")


@pytest.mark.parametrize("B,T,HK,HV,g_shift", [(1, 16384, 2, 4, 2.0), (1, 32768, 1, 2, 4.0),
                                               (2, 8192, 2, 4, 0.0)])
def test_long_sequences(ops, dev, B, T, HK, HV, g_shift):
    """Chains of 128 to 512 chunks, so that error growth over many scan steps
    (the state carried as an fp32 hi accumulation plus a decayed lo part, the
    V_n products on its fp16 copy) shows.  The mean gate is -0.81, -0.18 and
    -0.03 per token for g_shift 0, 2 and 4, so a chunk keeps e^{64 g} ~ 1e-22,
    8e-6 and 0.15 of the state: with g_shift 4 every step adds to a state
    that carries far back."""
    q, k, v, g, beta, s0 = gc.make_gdn_inputs(500 + T + HV, B=B, T=T, HK=HK, HV=HV,
                                              g_shift=g_shift, s0_scale=0.5)
    _run_and_check(ops, dev, q, k, v, g, beta, s0, tag=f"long T{T} B{B} HV{HV} g+{g_shift:g}")


def test_workspace_beyond_the_memory_side_cache(ops, dev):
    """B2 T4096 HV32 HK16: 276 MB of workspace and 204 MB of records, more
    than the memory-side cache keeps beside the inputs, so the prep writes
    them non-temporally; 64 heads with such records, so the wide scan runs."""
    q, k, v, g, beta, s0 = gc.make_gdn_inputs(4096, B=2, T=4096, HK=16, HV=32, g_shift=2.0)
    _run_and_check(ops, dev, q, k, v, g, beta, s0, tag="T4096 B2 HV32 (276 MB workspace)")


def test_reference_grid_long(ops, dev):
    """The reference harness's random distribution (q/k = randn/8, g = -0.3
    rand, beta = rand; parity_cuda.py:146-153) at S=16384, beyond its grid's
    longest case (S=3200): 256 chunks, 32 heads."""
    q, k, v, g, beta, s0 = gc.make_reference_inputs(1, 16384, 16384, l2_pre=True)
    _run_and_check(ops, dev, q, k, v, g, beta, s0, tag="grid S16384")


def test_varlen_edges(ops, dev):
    """Empty, single-token and chunk-boundary lengths in one packed batch."""
    lens = torch.tensor([0, 1, 63, 64, 65, 0, 130, 5])
    q, k, v, g, beta, s0, cu = gc.varlen_inputs(lens)
    o, sf = _run_and_check(ops, dev, q, k, v, g, beta, s0, tag="varlen-edges", cu=cu)
    # empty sequences pass their initial state through unchanged
    assert torch.equal(sf[0].cpu(), s0[0].float())
    assert torch.equal(sf[5].cpu(), s0[5].float())


def test_varlen_equals_per_sequence_calls(ops, dev):
    """Size-independent property at the 8-sequence varlen size: the packed call is bitwise the
    per-sequence fixed-length calls (same chunking, same kernels; the packed call's workspace
    exceeds the MALL, the per-sequence calls' workspaces fit it)."""
    q, k, v, g, beta, s0, cu = gc.varlen_inputs()
    d = [t.to(dev) for t in (q, k, v, g, beta, s0)]
    o, sf = ops.chunk_prefill(*d, cu_seqlens=cu.to(dev))
    for i in range(len(cu) - 1):
        a, b = int(cu[i]), int(cu[i + 1])
        oi, si = ops.chunk_prefill(d[0][:, a:b], d[1][:, a:b], d[2][:, a:b], d[3][:, a:b],
                                   d[4][:, a:b], d[5][i:i + 1])
        assert torch.equal(oi, o[:, a:b]), f"seq {i} o"
        assert torch.equal(si[0], sf[i]), f"seq {i} state"


def test_empty_sequence(ops, dev):
    """T = 0: o is empty and the final state is the initial one (zeros without one)."""
    q, k, v, g, beta, s0 = [t.to(dev) for t in gc.make_gdn_inputs(9, B=2, T=0, HK=2, HV=4)]
    s0 = torch.randn(2, 4, 128, 128, device=dev)
    o, sf = ops.chunk_prefill(q, k, v, g, beta, s0)
    assert o.shape == (2, 0, 4, 128) and torch.equal(sf, s0)
    _, sf0 = ops.chunk_prefill(q, k, v, g, beta, None)
    assert torch.count_nonzero(sf0).item() == 0


@pytest.mark.parametrize("n", [64, 65, 100])
def test_varlen_many_sequences(ops, dev, n):
    """More sequences than the scan's longest-first ordering table holds (64):
    the packed call is still bitwise the per-sequence calls, lengths 0..100."""
    gen = torch.Generator().manual_seed(700 + n)
    lens = torch.randint(0, 101, (n,), generator=gen)
    lens[n // 3] = 0
    q, k, v, g, beta, s0, cu = gc.varlen_inputs(lens)
    print(f"[varlen-many] n={n} tokens={int(lens.sum())}", flush=True)
    d = [t.to(dev) for t in (q, k, v, g, beta, s0)]
    o, sf = ops.chunk_prefill(*d, cu_seqlens=cu.to(dev))
    for i in range(n):
        a, b = int(cu[i]), int(cu[i + 1])
        oi, si = ops.chunk_prefill(d[0][:, a:b], d[1][:, a:b], d[2][:, a:b], d[3][:, a:b],
                                   d[4][:, a:b], d[5][i:i + 1])
        assert torch.equal(oi, o[:, a:b]), f"seq {i} o"
        assert torch.equal(si[0], sf[i]), f"seq {i} state"


def test_gqa_equals_expanded_heads(ops, dev):
    """HK=16 -> HV=32 sharing is bitwise the explicit repeat_interleave."""
    q, k, v, g, beta, s0 = [t.to(dev) for t in gc.prefill_inputs()]
    o1, s1 = ops.chunk_prefill(q, k, v, g, beta, s0)
    o2, s2 = ops.chunk_prefill(q.repeat_interleave(2, 2), k.repeat_interleave(2, 2), v, g, beta, s0)
    assert torch.equal(o1, o2) and torch.equal(s1, s2)


def test_resume_split(ops, dev):
    """Running [0, 640) then [640, T) from the carried state matches one call
    (chunk-aligned split, so the chunking is identical).  Not bitwise: within
    a call the scan keeps the lo part of the state update in a second
    accumulator and adds it at the end, so a resumed call rounds fp16(S + Sc)
    where the single call rounds fp16(S) for the next K S product."""
    q, k, v, g, beta, s0 = [t.to(dev) for t in gc.prefill_inputs()]
    o, sf = ops.chunk_prefill(q, k, v, g, beta, s0)
    t = 640
    oa, sa = ops.chunk_prefill(q[:, :t], k[:, :t], v[:, :t], g[:, :t], beta[:, :t], s0)
    ob, sb = ops.chunk_prefill(q[:, t:], k[:, t:], v[:, t:], g[:, t:], beta[:, t:], sa)
    do = (torch.cat([oa, ob], 1).float() - o.float()).abs().max().item()
    ds = (sb - sf).abs().max().item()
    print(f"[prefill] resume split max|diff| o={do:.3e} state={ds:.3e}", flush=True)
    assert do <= 2e-3 and ds <= 1e-5


def test_debug_views(ops, dev):
    """chunk_prefill_debug's views against the oracle's per-chunk quantities
    (chunk_debug_views, fp64): A, T = (I - A)^-1, T after the diagonal-block
    inversion, M, cumsum(g) and the state at each chunk's start."""
    q, k, v, g, beta, s0 = gc.make_gdn_inputs(11, B=1, T=100, HK=2, HV=4)
    d = [t.to(dev) for t in (q, k, v, g, beta, s0)]
    out = ops.chunk_prefill_debug(*d)
    assert len(out) == 8
    o, sf, Tm, A, cg, Tp, M, Sc = [x.cpu().double() if i > 1 else x for i, x in enumerate(out)]
    o2, sf2 = ops.chunk_prefill(*d)
    assert torch.equal(o, o2) and torch.equal(sf, sf2)
    ref = orc.chunk_debug_views(q, k, v, g, beta, s0, dtype=torch.float64)
    nc = 2
    assert Tm.shape == (nc, 4, 64, 64) and cg.shape == (nc, 4, 64) and Sc.shape == (nc, 4, 128, 128)
    assert torch.allclose(cg, ref["c"], atol=1e-5)
    assert torch.allclose(A, ref["A"], atol=1e-5)
    assert torch.allclose(Tm, ref["T"], atol=1e-5, rtol=1e-4)
    assert torch.allclose(M, ref["M"], atol=1e-5)
    assert torch.allclose(Sc, ref["S"], atol=2e-4)
    # post-leaf: each 16x16 diagonal block inverted, A below them, zero above
    eye = torch.eye(16, dtype=torch.float64)
    for b in range(4):
        blk = slice(16 * b, 16 * b + 16)
        inv = torch.linalg.solve_triangular(eye - ref["A"][..., blk, blk], eye, upper=False,
                                            unitriangular=True)
        assert torch.allclose(Tp[..., blk, blk], inv, atol=1e-5, rtol=1e-4)
    below = torch.tril(torch.ones(64, 64, dtype=torch.bool), -16) & ~torch.block_diag(
        *[torch.ones(16, 16, dtype=torch.bool)] * 4)
    assert torch.allclose(Tp[..., below], ref["A"][..., below], atol=1e-5)
    above = torch.triu(torch.ones(64, 64, dtype=torch.bool), 1) & ~torch.block_diag(
        *[torch.ones(16, 16, dtype=torch.bool)] * 4)
    assert torch.count_nonzero(Tp[..., above]) == 0
