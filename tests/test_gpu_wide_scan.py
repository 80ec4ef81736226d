"""The wide scan instance (two work-groups of 64 value columns per (sequence,
head)) against the 16-column instance, through the C ABI's
deltanet_chunk_prefill_cols: bitwise the same o and final state, since each
compute wave runs the 16-column arithmetic operation for operation.  Lengths
cover no chunk, one chunk, odd and even chunk counts (the two stages of each
operand part) and ragged last chunks."""
import ctypes as ct

import pytest
import torch

import gdn_cases as gc
from gdn_hip import capi

pytestmark = pytest.mark.gpu


def _run(dev, d, cu, cols, o_offset=0):
    lib = capi.lib()
    q, k, v, g, beta, s0 = d
    B, T, HK, D = q.shape
    HV = v.shape[2]
    N = len(cu) - 1 if cu is not None else B
    size = (lib.deltanet_prefill_varlen_live_workspace_size if cu is not None
            else lib.deltanet_prefill_live_workspace_size)
    wsb = size(T, N, HV, D, D, 64) if cu is not None else size(B, T, HV, D, D, 64)
    ws = torch.empty(wsb, dtype=torch.uint8, device=dev)
    o = torch.zeros(v.numel() + 8, dtype=v.dtype, device=dev)
    o = o[o_offset:o_offset + v.numel()].view(v.shape)
    sf = torch.zeros(N, HV, D, D, device=dev)
    cud = cu.to(dev) if cu is not None else None
    print(f"[wide] cols={cols} N={N} T={T} HK={HK} HV={HV}", flush=True)
    err = lib.deltanet_chunk_prefill_cols(
        capi.ptr(q), capi.ptr(k), capi.ptr(v), capi.ptr(g), capi.ptr(beta), o.data_ptr(),
        capi.ptr(s0), sf.data_ptr(), capi.ptr(cud), N, T, HV, HK, ws.data_ptr(), wsb,
        torch.cuda.current_stream().cuda_stream, cols, ct.c_uint(0))
    assert err == capi.HIP_SUCCESS, err
    torch.cuda.synchronize()
    return o, sf


@pytest.mark.parametrize("lens,HK,HV", [
    ([0, 1, 63, 64, 65, 0, 130, 5, 128, 192, 193, 257], 2, 4),
    ([300, 1, 640], 4, 12),
    ([70] * 70, 1, 1),
])
def test_wide_equals_16col_varlen(dev, lens, HK, HV):
    q, k, v, g, beta, s0 = gc.make_gdn_inputs(91, B=1, T=sum(lens), HK=HK, HV=HV, g_shift=2.0)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    s0 = 0.02 * torch.randn(len(lens), HV, 128, 128, generator=torch.Generator().manual_seed(5))
    d = [t.to(dev) for t in (q, k, v, g, beta, s0)]
    o16, s16 = _run(dev, d, cu, 16)
    o, s = _run(dev, d, cu, 128)
    assert torch.equal(o, o16) and torch.equal(s, s16)


@pytest.mark.parametrize("B,T,HK,HV", [(3, 300, 16, 32), (2, 200, 3, 3), (5, 64, 2, 16)])
def test_wide_equals_16col_batch(dev, B, T, HK, HV):
    """Without an initial state too (zeros)."""
    d = [t.to(dev) for t in gc.make_gdn_inputs(17 + B, B=B, T=T, HK=HK, HV=HV, g_shift=2.0)]
    for s0 in (d[5], None):
        o16, s16 = _run(dev, d[:5] + [s0], None, 16)
        o, s = _run(dev, d[:5] + [s0], None, 128)
        assert torch.equal(o, o16) and torch.equal(s, s16)


def test_wide_o_at_an_8_byte_address(dev):
    """o's rows 8 bytes past a 16-byte boundary, all the narrower instances ask for."""
    d = [t.to(dev) for t in gc.make_gdn_inputs(23, B=2, T=130, HK=2, HV=4, g_shift=2.0)]
    o16, s16 = _run(dev, d, None, 16, o_offset=4)
    o, s = _run(dev, d, None, 128, o_offset=4)
    assert o.data_ptr() % 16 == 8
    assert torch.equal(o, o16) and torch.equal(s, s16)


def test_spin_limit_keeps_bounded_waits(dev):
    """Heads for which the library takes the wide instance: a caller's spin
    limit is met by one with bounded waits, and reported."""
    lib = capi.lib()
    d = [t.to(dev) for t in gc.make_gdn_inputs(29, B=5, T=200, HK=8, HV=16, g_shift=2.0)]
    o, sf = torch.empty_like(d[2]), torch.empty_like(d[5])
    wsb = lib.deltanet_prefill_live_workspace_size(5, 200, 16, 128, 128, 64)
    ws = torch.empty(wsb, dtype=torch.uint8, device=dev)
    stream = torch.cuda.current_stream().cuda_stream
    for spin, want in ((0, capi.HIP_ERROR_LAUNCH_TIMEOUT), (1 << 20, capi.HIP_SUCCESS)):
        print(f"[wide] spin={spin} N=5 T=200 HK=8 HV=16", flush=True)
        assert lib.deltanet_chunk_prefill_spin(
            *[capi.ptr(t) for t in d[:5]], o.data_ptr(), d[5].data_ptr(), sf.data_ptr(), 5, 200, 16,
            8, ws.data_ptr(), wsb, stream, ct.c_uint(spin)) == capi.HIP_SUCCESS
        assert lib.deltanet_prefill_status(ws.data_ptr(), wsb, stream) == want


@pytest.mark.parametrize("B,T,HK,HV", [(3, 193, 16, 32), (2, 65, 32, 32), (9, 128, 4, 8)])
def test_wide_raw_rows_as_alone(ops, dev, B, T, HK, HV):
    """Raw q and k (normalised in the kernels) and the fused step's raw bf16
    and fp16 rows: each sequence as alone, where the 16-column scan runs."""
    assert capi.lib().deltanet_prefill_scan_cols(B * ((T + 63) // 64), B, HV, HK, 256, 0) == 64
    one = [slice(b, b + 1) for b in range(B)]
    print(f"[wide] raw rows B={B} T={T} HK={HK} HV={HV}", flush=True)
    d = [t.to(dev) for t in gc.make_gdn_inputs(83, B=B, T=T, HK=HK, HV=HV, g_shift=2.0)]
    o, s = ops.chunk_prefill(*d, qk_l2norm=True)
    for i in one:
        o1, s1 = ops.chunk_prefill(*[t[i] for t in d], qk_l2norm=True)
        assert torch.equal(o[i], o1) and torch.equal(s[i], s1)
    for dtype in (torch.bfloat16, torch.float16):
        q, k, v, a, b, A_log, dt_bias, s0 = [
            t.to(dev) for t in gc.fused_inputs(84, B=B, T=T, HK=HK, HV=HV, dtype=dtype)]
        s = s0.clone()
        o = ops.chunk_prefill_fused(q, k, v, a, b, A_log, dt_bias, s)
        for i in one:
            s1 = s0[i].clone()
            o1 = ops.chunk_prefill_fused(q[i], k[i], v[i], a[i], b[i], A_log, dt_bias, s1)
            assert torch.equal(o[i], o1) and torch.equal(s[i], s1)


def test_wide_noalloc_as_alone(ops, dev):
    """The allocation-free entry on the wide scan (3 x 200 tokens, 32 heads:
    384 chunk-heads, inside its array), each sequence as alone."""
    lib = capi.lib()
    B, T, HK, HV = 3, 200, 16, 32
    d = [t.to(dev) for t in gc.make_gdn_inputs(85, B=B, T=T, HK=HK, HV=HV, g_shift=2.0)]
    o, sf = torch.empty_like(d[2]), torch.empty_like(d[5])
    stream = torch.cuda.current_stream().cuda_stream
    print(f"[wide] noalloc B={B} T={T} HK={HK} HV={HV}", flush=True)
    assert lib.deltanet_chunk_prefill_noalloc(
        *[capi.ptr(t) for t in d[:5]], o.data_ptr(), d[5].data_ptr(), sf.data_ptr(), B, T, HV, HK,
        128, 128, 64, stream) == capi.HIP_SUCCESS
    assert lib.deltanet_prefill_noalloc_status(stream) == capi.HIP_SUCCESS
    for i in (slice(0, 1), slice(1, 2), slice(2, 3)):
        o1, s1 = ops.chunk_prefill(*[t[i] for t in d])
        assert torch.equal(o[i], o1) and torch.equal(sf[i], s1)
