"""The library's own choice of the scan instance (value columns per
work-group), on either side of each border, for 256 CUs.  CPU only."""
import pytest

from gdn_hip import capi


def _cols(chunks, n, hv, hk, cus=256, spin=0):
    return capi.lib().deltanet_prefill_scan_cols(chunks, n, hv, hk, cus, spin)


@pytest.mark.parametrize("n,hv,hk,want", [
    (1, 32, 16, 16), (2, 16, 16, 16), (1, 34, 17, 32),   # 16-column groups fit up to 32 heads
    (3, 16, 16, 32), (7, 7, 7, 64),                      # every head its own Q, K^T: wide above 48
    (3, 16, 8, 32), (2, 32, 16, 32), (33, 2, 1, 64),     # else wide above 64
    (8, 32, 16, 64), (1000, 1, 1, 64),
])
def test_heads(n, hv, hk, want):
    assert _cols(n, n, hv, hk) == want


@pytest.mark.parametrize("n,hv,hk", [(2, 32, 16), (7, 8, 4)])
def test_records_past_the_memory_side_cache(n, hv, hk):
    """Above 48 heads the wide instance from 192 MB of records on."""
    per_chunk = hv * (3 * 6144 + 16384 + 1024) + hk * 2 * 16384
    last = (192 << 20) // per_chunk
    assert _cols(last, n, hv, hk) == 32 and _cols(last + 1, n, hv, hk) == 64
    assert _cols(last + 1, 1, hv, hk) == 16   # too few heads


@pytest.mark.parametrize("n,hv,hk", [(3, 32, 16), (2, 32, 32), (64, 32, 16)])
def test_own_spin_limit_keeps_bounded_waits(n, hv, hk):
    assert _cols(1000, n, hv, hk) == 64
    assert _cols(1000, n, hv, hk, spin=1) == 32
    assert _cols(1000, n, hv, hk, spin=1 << 20) == 64   # the library's own limit


def test_refuses():
    assert _cols(1, 0, 2, 2) == -1 and _cols(1, 1, 3, 2) == -1 and _cols(1, 1, 2, 2, cus=0) == -1
