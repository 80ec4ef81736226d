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
