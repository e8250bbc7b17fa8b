"""causal_conv1d over token-contiguous rows that start anywhere: rows cut at
the 16-byte boundary before their first token, against the oracle."""
import numpy as np
import pytest
import torch

import tecoops
from oracle import oracle as orc

from helpers import as_f32, bits, dev, host_bits

pytestmark = pytest.mark.gpu

# sequence lengths: every start offset mod 8 with rows that end just before,
# at and after a vector, segment (512) or group of segments (2048); rows
# shorter than the window beside long ones; short rows (several per wave)
LENGTHS = {
    "long": [2048, 7, 1, 2041, 513, 3, 2055, 505, 2, 4097, 511, 520, 8, 1025, 4091, 9, 300],
    "short": [1, 2, 3, 8, 15, 17, 63, 64, 65, 5, 31, 33, 7, 129, 66, 4, 250],
    # more than 64 sequences in one group of 2048 tokens, some empty
    "many": [1, 2, 3, 0, 9, 4, 1, 1, 30] * 60 + [2100, 1, 2],
}
LENGTHS["mixed"] = LENGTHS["long"] + [5, 1, 12]
# channels: the kernel that runs along the token axis takes all of "short" and
# "many", "mixed" from three channels per CU on, and "long" (over 1024 tokens in
# the mean) not at all
DIMS = {"long": (21, 72), "short": (21, 1400), "many": (21, 400), "mixed": (21, 776)}


@pytest.mark.parametrize("W", [2, 3, 4])
@pytest.mark.parametrize("pad", [0, 1, 8], ids=["packed", "out_off_by_1", "out_off_by_8"])
@pytest.mark.parametrize("big", [False, True], ids=["rows", "axis"])
@pytest.mark.parametrize("kind", sorted(LENGTHS))
def test_rows_at_any_start(kind, big, pad, W):
    """pad: elements that out's rows are longer than x's (1: x and out of a
    row are off the 16-byte boundary by different amounts).  big: channels in
    number (2^20 elements), with which all but "long" run along the token axis."""
    r = np.random.default_rng(60 + W + pad)
    lens, dim = LENGTHS[kind], DIMS[kind][big]
    assert (sum(lens) * dim >= 1 << 20) == big
    B, total = len(lens), sum(lens)
    x, w = bits(r.standard_normal((dim, total))), bits(r.standard_normal((W, dim)) * 0.5)
    st = bits(r.standard_normal((B + 2, W - 1, dim)))
    qsl = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    cidx = r.permutation(B + 2)[:B].astype(np.int32)
    cidx[4] = -7  # skipped
    hinit = (np.arange(B) % 3 != 0).astype(np.int8)
    st_ref = st.copy()
    ref = orc.causal_conv1d(x, w, conv_state=st_ref, query_start_loc=qsl, cache_indices=cidx,
                            has_initial_state=hinit, pad_slot_id=-7, layout="dl")
    buf = torch.full((dim, total + pad), 77.0, dtype=torch.float16, device="cuda")
    out, st_dev = buf[:, :total], dev(st)
    tecoops.causal_conv1d_fn_torch(out, st_dev, dev(x), dev(w), dev(qsl), dev(cidx), dev(hinit), -7)
    torch.cuda.synchronize()
    got = as_f32(out).astype(np.float64)
    # the skipped sequence and the padding stay untouched
    skipped = slice(qsl[4], qsl[5])
    assert (got[:, skipped] == 77).all() and (buf[:, total:] == 77).all()
    # one rounding to fp16 (half an ulp, twice that allowed) and fp32 sums of
    # W products and the activation's exponential, 16 roundings of their size
    big = sum(np.abs(orc.to_float(w)[k])[:, None] for k in range(W)) * np.abs(orc.to_float(x)).max()
    keep = np.ones(total, bool)
    keep[skipped] = False
    err = np.abs(got - ref)[:, keep]
    bound = 2.0 ** -10 * np.abs(ref)[:, keep] + 16 * 2.0 ** -24 * big + 2.0 ** -24
    assert (err <= bound).all(), (err - bound).max()
    assert np.array_equal(host_bits(st_dev), st_ref)


@pytest.mark.parametrize("dim", [1, 5, 768])
@pytest.mark.parametrize("W", [2, 4])
@pytest.mark.parametrize("lens", [[3001, 900], [2, 4101], [3072], [4097, 0]], ids=str)
def test_few_sequences_along_the_axis(lens, W, dim):
    """One or two long sequences of few channels run along the token axis, past
    its groups of 2048 tokens: as a wave per row computes them, which takes the
    sequences one by one in the batched layout, up to one unit of fp16 (the
    kernels' products and sums may be contracted differently, and a result then
    rounds the other way)."""
    g = torch.Generator(device="cuda").manual_seed(W + dim)
    total, B = sum(lens), len(lens)
    x = torch.randn(dim, total, generator=g, device="cuda").half()
    w = torch.randn(W, dim, generator=g, device="cuda").half()
    st = torch.randn(B, W - 1, dim, generator=g, device="cuda").half()
    qsl = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device="cuda")
    ci = torch.arange(B, dtype=torch.int32, device="cuda")
    hi = torch.ones(B, dtype=torch.int8, device="cuda")
    out, got_st = torch.full_like(x, 77.0), st.clone()
    tecoops.causal_conv1d_fn_torch(out, got_st, x, w, qsl, ci, hi, -1)
    want, want_st, at = torch.full_like(x, 77.0), st.clone(), 0
    for b, n in enumerate(lens):
        if n:
            row, o = x[:, at:at + n].contiguous()[None], torch.empty(1, dim, n, dtype=x.dtype, device="cuda")
            tecoops.causal_conv1d(row, w.t(), None, o, want_st, ci[b:b + 1], hi[b:b + 1])
            want[:, at:at + n] = o[0]
        at += n
    torch.cuda.synchronize()
    a, b = out.float(), want.float()
    off = (a - b).abs() > 2.0 ** -10 * b.abs() + 2.0 ** -24
    assert not off.any(), (off.sum(), off.nonzero()[:4], a[off][:4], b[off][:4])
    assert (a != b).float().mean() < 1e-3 and torch.equal(got_st, want_st)
