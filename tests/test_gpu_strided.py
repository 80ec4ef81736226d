"""q, k and v read where they lie (slices of one buffer, transposes, expanded
rows, odd offsets) and the decode step into a new state: bitwise what the same
values give from packed tensors and from the in-place step."""
import pytest
import torch

import gdn_cases as gc

pytestmark = pytest.mark.gpu

# forms of one [B, T, H, 128] tensor with the same values
FORMS = {
    "slice": lambda x: torch.cat([x.flatten(2), x.flatten(2)], 2)[..., :x.shape[2] * 128]
    .unflatten(2, (x.shape[2], 128)),
    "odd_offset": lambda x: torch.cat([x.flatten()[:1], x.flatten()])[1:].view(x.shape),
    "odd_stride": lambda x: torch.nn.functional.pad(x.flatten(2), (0, 3))[..., :x.shape[2] * 128]
    .unflatten(2, (x.shape[2], 128)),
    "tokens_first": lambda x: x.transpose(0, 1).contiguous().transpose(0, 1),
    "heads_first": lambda x: x.transpose(1, 2).contiguous().transpose(1, 2),
    "batch_gap": lambda x: torch.cat([x, x[:, :1]], 1)[:, :x.shape[1]],
    "wide_elements": lambda x: torch.stack([x, x], -1)[..., 0],
}


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("B,T,HK,HV", [(1, 77, 2, 4), (2, 130, 4, 4), (3, 1, 1, 2)])
def test_prefill_strided(ops, dev, form, B, T, HK, HV):
    q, k, v, g, beta, s0 = [t.to(dev) for t in gc.make_gdn_inputs(7, B=B, T=T, HK=HK, HV=HV,
                                                                  g_shift=2.0)]
    f = FORMS[form]
    print(f"[strided] prefill {form} B={B} T={T} HK={HK} HV={HV}", flush=True)
    for norm in (False, True):
        o_ref, s_ref = ops.chunk_prefill(q, k, v, g, beta, s0, qk_l2norm=norm)
        o, s = ops.chunk_prefill(f(q), f(k), f(v), g, beta, s0, qk_l2norm=norm)
        assert o.is_contiguous() and torch.equal(o, o_ref) and torch.equal(s, s_ref)


@pytest.mark.parametrize("form", ["slice", "odd_stride"])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("B,T,HK,HV", [(2, 130, 16, 32), (3, 70, 16, 16), (3, 70, 16, 32),
                                       (2, 129, 32, 32)])
def test_prefill_strided_paired_and_wide(ops, dev, form, norm, B, T, HK, HV):
    """More (sequence, head) pairs than 16-column groups fit: the first two
    run the paired scan, the others the wide one, against each sequence alone
    and packed (the 16-column scan).  "slice" is read in place, "odd_stride"
    copied."""
    q, k, v, g, beta, s0 = [t.to(dev) for t in gc.make_gdn_inputs(11, B=B, T=T, HK=HK, HV=HV,
                                                                  g_shift=2.0)]
    f = FORMS[form]
    print(f"[strided] prefill {form} B={B} T={T} HK={HK} HV={HV} norm={norm}", flush=True)
    o, s = ops.chunk_prefill(f(q), f(k), f(v), g, beta, s0, qk_l2norm=norm)
    for b in range(B):
        i = slice(b, b + 1)
        o1, s1 = ops.chunk_prefill(q[i], k[i], v[i], g[i], beta[i], s0[i], qk_l2norm=norm)
        assert torch.equal(o[i], o1) and torch.equal(s[i], s1)


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("lens,HK,HV", [([70, 0, 1], 2, 4), ([65, 130], 16, 32),
                                        ([0, 64, 63, 1, 200, 0], 8, 16)])
def test_prefill_strided_packed_sequences(ops, dev, norm, lens, HK, HV):
    """Ragged and empty sequences in rows of one buffer (16-column, paired and
    wide scan) against the same rows without gaps, a sequence at a time."""
    T = sum(lens)
    q, k, v, g, beta, _ = [t.to(dev) for t in gc.make_gdn_inputs(12, B=1, T=T, HK=HK, HV=HV,
                                                                 g_shift=2.0)]
    s0 = 0.02 * torch.randn(len(lens), HV, 128, 128, generator=torch.Generator().manual_seed(6))
    s0 = s0.to(dev)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    f = FORMS["slice"]
    print(f"[strided] packed sequences {lens} HK={HK} HV={HV} norm={norm}", flush=True)
    o, s = ops.chunk_prefill(f(q), f(k), f(v), g, beta, s0, cu_seqlens=cu.to(dev),
                             qk_l2norm=norm)
    for i in range(len(lens)):
        t = slice(int(cu[i]), int(cu[i + 1]))
        o1, s1 = ops.chunk_prefill(q[:, t], k[:, t], v[:, t], g[:, t], beta[:, t], s0[i:i + 1],
                                   qk_l2norm=norm)
        assert torch.equal(o[:, t], o1) and torch.equal(s[i:i + 1], s1)


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("B,T,HK,HV", [(1, 1, 2, 4), (3, 1, 2, 4), (2, 3, 1, 2)])
def test_decode_strided_and_new_state(ops, dev, form, B, T, HK, HV):
    q, k, v, g, beta, s0 = [t.to(dev) for t in gc.make_gdn_inputs(9, B=B, T=T, HK=HK, HV=HV,
                                                                  g_shift=2.0)]
    f = FORMS[form]
    print(f"[strided] decode {form} B={B} T={T} HK={HK} HV={HV}", flush=True)
    for norm in (False, True):
        s_ref = s0.clone()
        o_ref = ops.recurrent_step(q, k, v, g, beta, s_ref, qk_l2norm=norm)
        s_in = s0.clone()
        o = ops.recurrent_step(f(q), f(k), f(v), g, beta, s_in, qk_l2norm=norm)
        assert torch.equal(o, o_ref) and torch.equal(s_in, s_ref)
        keep = s0.clone()
        o, s = ops.recurrent_step_new(f(q), f(k), f(v), g, beta, keep, qk_l2norm=norm)
        assert torch.equal(o, o_ref) and torch.equal(s, s_ref) and torch.equal(keep, s0)
        s_ref = torch.zeros_like(s0)
        o_ref = ops.recurrent_step(q, k, v, g, beta, s_ref, qk_l2norm=norm)
        o, s = ops.recurrent_step_new(f(q), f(k), f(v), g, beta, None, qk_l2norm=norm)
        assert torch.equal(o, o_ref) and torch.equal(s, s_ref)


def test_decode_new_state_without_tokens(ops, dev):
    q, k, v, g, beta, s0 = [t.to(dev) for t in gc.make_gdn_inputs(9, B=2, T=1, HK=2, HV=4)]
    e = [t[:, :0] for t in (q, k, v, g, beta)]
    o, s = ops.recurrent_step_new(*e, s0)
    assert o.shape == (2, 0, 4, 128) and torch.equal(s, s0) and s.data_ptr() != s0.data_ptr()
    with pytest.raises(RuntimeError):
        ops.recurrent_step_new(*[t[:0] for t in e], s0[:0])


def test_decode_state_at_any_float(ops, dev):
    """The state a contiguous view that starts one float into its buffer."""
    q, k, v, g, beta, s0 = [t.to(dev) for t in gc.make_gdn_inputs(9, B=2, T=2, HK=2, HV=4)]
    s_ref = s0.clone()
    o_ref = ops.recurrent_step(q, k, v, g, beta, s_ref)
    for off in (1, 2, 3):
        s = torch.cat([s0.flatten()[:off], s0.flatten()])[off:].view(s0.shape)
        assert s.data_ptr() % 16 == 4 * off
        o, s_new = ops.recurrent_step_new(q, k, v, g, beta, s)
        assert torch.equal(o, o_ref) and torch.equal(s_new, s_ref) and torch.equal(s, s0)
        o = ops.recurrent_step(q, k, v, g, beta, s)
        assert torch.equal(o, o_ref) and torch.equal(s, s_ref)


@pytest.mark.parametrize("norm", [False, True])
def test_decode_batches_of_2_31_elements(ops, dev, norm):
    """v's batches lie 2^31 elements apart (T HV = 2^24): the second batch as
    it steps alone, in place and into a new state."""
    B, T, HK, HV = 2, 1024, 1, 16384
    print(f"[strided] decode B={B} T={T} HK={HK} HV={HV} norm={norm}", flush=True)
    gen = torch.Generator(device=dev).manual_seed(21)
    kw = dict(generator=gen, device=dev)
    q, k = (torch.randn(B, T, HK, 128, **kw).mul_(0.1).bfloat16() for _ in range(2))
    v = torch.randn(B, T, HV, 128, dtype=torch.bfloat16, **kw)
    g = -torch.rand(B, T, HV, **kw)
    beta = torch.rand(B, T, HV, **kw)
    s0 = torch.randn(B, HV, 128, 128, **kw)
    s1 = s0[1:].clone()
    o1 = ops.recurrent_step(q[1:], k[1:], v[1:], g[1:], beta[1:], s1, qk_l2norm=norm)
    o, s = ops.recurrent_step_new(q, k, v, g, beta, s0, qk_l2norm=norm)
    assert torch.equal(o[1:], o1) and torch.equal(s[1:], s1)
    del o, s
    o = ops.recurrent_step(q, k, v, g, beta, s0, qk_l2norm=norm)
    assert torch.equal(o[1:], o1) and torch.equal(s0[1:], s1)
