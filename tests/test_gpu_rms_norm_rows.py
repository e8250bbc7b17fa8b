"""GPU parity of rms_norm with the CPU oracle at the edges of its kernels: a
wave or a workgroup per row, by row width and number of rows, and in place.

Both sum fp32 squares, in different orders: the sums differ by at most D *
2^-24 relative (1e-3 at 16384), rstd by half of that, so the 16-bit result by
at most one unit in the last place of fp16 up to 8192 and of bf16 everywhere.
The residual sum is rounded once on both sides and has to be the same.
"""
import numpy as np
import pytest
import torch

import tecoops
from oracle import oracle as orc

from helpers import bits, dev, host_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [orc.HALF, orc.BF16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("rows,D", [(3, 512), (3, 520), (7, 1000), (2, 4096), (2, 4104), (1, 8192),
                                    (3, 8200), (2, 16384), (2, 16392), (1024, 520), (1025, 520),
                                    (1025, 2040), (1025, 2048), (1025, 4096), (1025, 4104)])
@pytest.mark.parametrize("residual", [False, True], ids=["pure", "add"])
def test_rms_norm_rows(rows, D, residual, dt):
    if dt == orc.HALF and D > 8200:
        pytest.skip("past the bound of one fp16 unit")
    r = np.random.default_rng(rows + D)
    x, w = bits(r.standard_normal((rows, D)), dt), bits(r.uniform(0.5, 1.5, D), dt)
    res = bits(r.standard_normal((rows, D)), dt) if residual else None
    ref, ref_sum = orc.rms_norm(x, w, residual=res, eps=1e-6, dtype=dt)
    xd, wd = dev(x, dt), dev(w, dt)
    out = torch.empty_like(xd)
    rd = dev(res, dt) if residual else None
    # the residual stream is updated in place, as a model does
    tecoops.rms_norm(xd, wd, rd, out, rd, 1e-6)
    torch.cuda.synchronize()
    ulp = np.abs(host_bits(out).astype(np.int32) - ref.astype(np.int32))
    assert ulp.max() <= 1
    if residual:
        assert np.array_equal(host_bits(rd), ref_sum)


@pytest.mark.parametrize("dt", [orc.HALF, orc.BF16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("rows,D", [(1024, 4104), (1025, 4112), (1025, 8192), (1025, 8200), (5120, 4104),
                                    (5121, 4104), (4096, 4096), (4095, 4096), (8192, 4096), (16400, 1024)])
@pytest.mark.parametrize("residual", [False, True], ids=["pure", "add"])
def test_rms_norm_many_rows(rows, D, residual, dt):
    """A wave per row of 4104 to 8192 between 1025 and 5120 rows without residual,
    past the caches from 128 MiB on, in place.  Units are counted on the number line:
    the product of a zero, of which so many values hold some, rounds to fp16 with
    either sign."""
    r = np.random.default_rng(rows + D)
    x, w = bits(r.standard_normal((rows, D)), dt), bits(r.uniform(0.5, 1.5, D), dt)
    res = bits(r.standard_normal((rows, D)), dt) if residual else None
    ref, ref_sum = orc.rms_norm(x, w, residual=res, eps=1e-6, dtype=dt)
    xd, wd = dev(x, dt), dev(w, dt)
    rd = dev(res, dt) if residual else None
    tecoops.rms_norm(xd, wd, rd, xd, rd, 1e-6)
    torch.cuda.synchronize()

    def line(v):
        v = v.astype(np.int32)
        return np.where(v & 0x8000, -(v & 0x7fff), v)

    assert np.abs(line(host_bits(xd)) - line(ref)).max() <= 1
    if residual:
        assert np.array_equal(host_bits(rd), ref_sum)
