"""The prep's instances by the size of a call's records: first chunk first,
last chunk first (176 to 192 MB, written through) and non-temporal above.  Two
sequences on either side of each border against each sequence alone, whose
half as many records go out first chunk first: bitwise the same.  Raw q and k
(l2norm, fp16 rows) and rows that lie apart have instances of their own."""
import pytest
import torch

import gdn_cases as gc

pytestmark = pytest.mark.gpu

HK, HV = 16, 32
PER_CHUNK = HV * (3 * 6144 + 16384 + 1024) + HK * 2 * 16384   # bytes of records
BORDERS = [(176 << 20) // PER_CHUNK // 2, (192 << 20) // PER_CHUNK // 2]   # chunks a sequence
TS = [64 * c + r for c in BORDERS for r in (0, 1)]   # the last that fits, and one chunk more


def _apart(x):
    return torch.cat([x.flatten(2), x.flatten(2)], 2)[..., :x.shape[2] * 128].unflatten(
        2, (x.shape[2], 128))


@pytest.mark.parametrize("T", TS)
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("apart", [False, True])
def test_two_sequences_as_alone(ops, dev, T, norm, apart):
    q, k, v, g, beta, s0 = [t.to(dev) for t in gc.make_gdn_inputs(T, B=2, T=T, HK=HK, HV=HV,
                                                                  g_shift=2.0)]
    f = _apart if apart else (lambda x: x)
    print(f"[prep order] T={T} norm={norm} apart={apart}", flush=True)
    o, s = ops.chunk_prefill(f(q), f(k), f(v), g, beta, s0, qk_l2norm=norm)
    for b in range(2):
        i = slice(b, b + 1)
        o1, s1 = ops.chunk_prefill(q[i], k[i], v[i], g[i], beta[i], s0[i], qk_l2norm=norm)
        assert torch.equal(o[i], o1) and torch.equal(s[i], s1)


@pytest.mark.parametrize("T", TS)
def test_fused_fp16(ops, dev, T):
    gen = torch.Generator(device=dev).manual_seed(T)
    n = lambda *shape: torch.randn(*shape, generator=gen, device=dev).half()   # noqa: E731
    q, k, v = n(2, T, HK, 128), n(2, T, HK, 128), n(2, T, HV, 128)
    a, b = n(2, T, HV), n(2, T, HV)
    A_log = torch.rand(HV, generator=gen, device=dev).log()
    dt_bias = n(HV)
    s0 = 0.02 * torch.randn(2, HV, 128, 128, generator=gen, device=dev)
    s = s0.clone()
    print(f"[prep order] fused fp16 T={T}", flush=True)
    o = ops.chunk_prefill_fused(q, k, v, a, b, A_log, dt_bias, s)
    for i in (slice(0, 1), slice(1, 2)):
        s1 = s0[i].clone()
        o1 = ops.chunk_prefill_fused(q[i], k[i], v[i], a[i], b[i], A_log, dt_bias, s1)
        assert torch.equal(o[i], o1) and torch.equal(s[i], s1)
