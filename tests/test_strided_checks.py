"""Host checks of the strided entries: refused before any launch (no GPU)."""
import pytest

from gdn_hip import capi

P = 1 << 20   # a 16-byte aligned non-null address, never read


@pytest.mark.parametrize("q,qt,v,vt", [
    (P, 12, P, 256),        # token stride not a multiple of 8 elements
    (P, -8, P, 256),        # negative
    (P, 1 << 31, P, 256),   # beyond 32 bits
    (P + 8, 256, P, 256),   # q not 16-byte aligned
    (P, 256, P + 2, 256),   # v not 16-byte aligned
    (None, 256, P, 256),    # null
])
def test_prefill_strided_refuses(q, qt, v, vt):
    assert capi.lib().deltanet_chunk_prefill_strided(
        q, qt, P, 256, v, vt, P, P, P, None, P, None, 1, 1, 64, 2, 2, 0, P, 1 << 30,
        None) == capi.HIP_ERROR_INVALID_VALUE


@pytest.mark.parametrize("B,T,s_in,qb,v,vt", [
    (1, 1, P, -1, P, 256),          # negative stride
    (1, 1, P, 1 << 31, P, 256),     # beyond 32 bits
    (1, 1, P, 256, P + 4, 256),     # v not 8-byte aligned
    (1, 1, P, 256, P, 6),           # v stride not a multiple of 4
    (0, 1, P, 256, P, 256),         # no batch
    (0, 0, P, 256, P, 256),
    (1, 0, P + 64, 256, P, 256),    # no token: the state cannot move
])
def test_decode_strided_refuses(B, T, s_in, qb, v, vt):
    assert capi.lib().deltanet_recurrent_step_strided(
        P, P, v, P, P, P, s_in, P, B, T, 2, 2, qb, 256, 256, 256, 256, vt, 0,
        None) == capi.HIP_ERROR_INVALID_VALUE


@pytest.mark.parametrize("T,heads,b,t,h", [
    (1, 1, 0, 0, 0),
    (3, 32, 5, 2, 31),
    (524288, 32, 1, 0, 0),          # a batch of 2^31 elements
    (524289, 32, 1, 524288, 31),
    (1024, 16384, 1, 1023, 16383),
    (4096, 8192, 200, 4095, 8191),
])
def test_decode_packed_rows_in_64_bits(T, heads, b, t, h):
    """Batch strides of the packed decode entries, past 2^31 elements too."""
    assert capi.lib().deltanet_recurrent_row_offset(T, heads, b, t, h) == \
        ((b * T + t) * heads + h) * 128
