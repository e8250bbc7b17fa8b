"""The bound of the split-attention tests (helpers.attention_row_bound) on the
CPU: the oracle rounded as a kernel rounds passes it, and a piece of the keys
left out does not, at the lengths those tests use."""
import numpy as np
import pytest

from oracle import oracle as orc

from helpers import assert_rows_close, bits

# rows, keys, keys left out (a decode split, or a piece of a split prefill)
CASES = [(1, 640, 128), (1, 4096, 128), (1, 16384, 128), (1, 70000, 2048), (3, 3000, 128), (32, 6000, 256)]


def attention(q, k, v, dt, rounded):
    """float64 attention of every row over every key; rounded: probabilities
    and result rounded to the 16-bit type, as a kernel does."""
    s = q @ k.T / np.sqrt(q.shape[1])
    p = np.exp(s - s.max(1, keepdims=True))
    l = p.sum(1, keepdims=True)
    if rounded:
        p = orc.to_float(bits(p, dt), dt).astype(np.float64)
    o = p @ v / l
    return orc.to_float(bits(o, dt), dt) if rounded else o


@pytest.mark.parametrize("dt", [orc.HALF, orc.BF16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("rows,keys,piece", CASES)
def test_bound_sees_a_lost_piece(rows, keys, piece, dt):
    r = np.random.default_rng(keys + rows)
    for D in (32, 128):
        q, k, v = (orc.to_float(bits(r.uniform(-1, 1, (n, D)), dt), dt).astype(np.float64)
                   for n in (rows, keys, keys))
        ref = attention(q, k, v, dt, False)
        assert_rows_close(attention(q, k, v, dt, True), ref, dt, "rounded")
        for first in (0, (keys // 2) // piece * piece, keys - piece):
            keep = np.r_[0:first, first + piece:keys]
            with pytest.raises(AssertionError):
                assert_rows_close(attention(q, k[keep], v[keep], dt, True), ref, dt, "piece lost")
        with pytest.raises(AssertionError):
            assert_rows_close(np.zeros_like(ref), ref, dt, "zeros")
        with pytest.raises(AssertionError):
            assert_rows_close(np.full_like(ref, np.nan), ref, dt, "NaN")
