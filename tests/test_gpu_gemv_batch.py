"""Weight products of several rows of x (gemv_batch.hip), against the oracle,
at the sizes where its tiling can go wrong: every number of W rows per
workgroup (8 to 128, picked from N and the batch), the row remainders of each,
every number of staged x rows (4 to 64) and the batches around it, slices of
64, K of one 16-byte chunk, K that ends inside a stage, and K parts that are
empty."""
import numpy as np
import pytest
import torch

import tecoops
from oracle import oracle as orc

from helpers import as_f32, bits, dev

pytestmark = pytest.mark.gpu

# N: 8 to 128 rows per workgroup on 256 CUs
SHAPES = [(3, 1, 8), (4, 2041, 136), (5, 2050, 520), (8, 4090, 72), (9, 6007, 200), (16, 301, 4104),
          (17, 11001, 120), (32, 3000, 1032), (33, 20001, 88), (48, 5003, 264), (49, 28003, 72),
          (64, 32765, 40), (65, 1000, 392), (130, 60, 2056), (6, 28672, 256), (12, 32768, 128),
          # up to 8 rows of x: 32, 48 and 64 rows, the last workgroup in part
          (8, 6100, 1160), (3, 4097, 72), (5, 12001, 264), (8, 12288, 128), (8, 14335, 392),
          (4, 12300, 520)]


def _check(y, dt, ref, W, x, what):
    """One rounding of the result (half an ulp, twice that allowed), fp32
    products and sums in any order (K + 8 roundings of the absolute sum), and
    the smallest fp16 step."""
    K = x.shape[1]
    total = np.abs(x) @ np.abs(W).T
    bound = (2.0 ** -10 if dt == orc.HALF else 2.0 ** -7) * np.abs(ref) + \
        (K + 8) * 2.0 ** -24 * total + 2.0 ** -24
    err = np.abs(as_f32(y, dt).astype(np.float64) - ref)
    assert (err <= bound).all(), f"{what}: {err.max()} over the bound by {(err - bound).max()}"


@pytest.mark.parametrize("dt", [orc.HALF, orc.BF16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("B,N,K", SHAPES)
def test_gemv_batch(B, N, K, dt):
    r = np.random.default_rng(40 + B + N + K)
    W, x = bits(r.normal(0, 0.05, (N, K)), dt), bits(r.standard_normal((B, K)), dt)
    y = torch.empty((B, N), dtype=torch.float16 if dt == orc.HALF else torch.bfloat16, device="cuda")
    tecoops.gemv(dev(W, dt), dev(x, dt), y)
    torch.cuda.synchronize()
    _check(y, dt, orc.gemv(W, x, dtype=dt), orc.to_float(W, dt), orc.to_float(x, dt), f"{B}x{N}x{K}")


@pytest.mark.parametrize("B,N,K", [(b, n, k + (8 if k % 16 else 0)) for b, n, k in SHAPES] +
                         [(2, 77, 16), (2, 9000, 272), (4, 8192, 512), (8, 17000, 256)])
def test_gemv_int8_batch(B, N, K):
    r = np.random.default_rng(90 + B + N + K)
    W = r.integers(-127, 128, (N, K), dtype=np.int8)
    s, x = bits(r.uniform(0.001, 0.01, N)), bits(r.standard_normal((B, K)))
    y = torch.empty((B, N), dtype=torch.float16, device="cuda")
    tecoops.gemv_int8(dev(W), dev(s), dev(x), y)
    torch.cuda.synchronize()
    scaled = W.astype(np.float32) * orc.to_float(s)[:, None]
    _check(y, orc.HALF, orc.gemv_int8(W, s, x), scaled, orc.to_float(x), f"{B}x{N}x{K}")


# int8 W with K split over more waves: 8 rows eight ways (from 16 stages of K),
# 32 rows four ways (from 16, up to 4 rows of x 32, where few CUs have work),
# with parts that end early or are empty, and the N and K just outside
@pytest.mark.parametrize("B,N,K", [(2, 9, 4096), (3, 2047, 3856), (4, 2041, 3840), (5, 300, 4112),
                                   (8, 2048, 13824), (7, 100, 7696), (2, 4104, 8192), (4, 5001, 7952),
                                   (3, 6143, 13840), (4, 6145, 8192), (5, 5000, 3856), (8, 6000, 4096),
                                   (6, 4999, 3840), (8, 4500, 12304), (4, 5000, 7936)])
def test_gemv_int8_batch_split_k(B, N, K):
    test_gemv_int8_batch(B, N, K)


@pytest.mark.parametrize("N,K", [(40, 4104), (9000, 136)])
def test_gemv_batch_infinity(N, K):
    """A weight of infinity reaches its own row of y only, as infinity (no
    product of it with a padding zero)."""
    W = torch.full((N, K), 0.01, dtype=torch.float16, device="cuda")
    W[N // 2, K - 1] = float("inf")
    x = torch.full((5, K), 0.5, dtype=torch.float16, device="cuda")
    y = torch.empty((5, N), dtype=torch.float16, device="cuda")
    tecoops.gemv(W, x, y)
    torch.cuda.synchronize()
    want = torch.zeros(5, N, dtype=torch.bool, device="cuda")
    want[:, N // 2] = True
    assert torch.equal(torch.isposinf(y), want) and not torch.isnan(y).any()


def test_gemv_batch_misaligned_output():
    """y on a 2-byte boundary, and N that is no multiple of 4."""
    r = np.random.default_rng(7)
    for N, off in ((64, 1), (63, 0)):
        W, x = bits(r.normal(0, 0.05, (N, 256))), bits(r.standard_normal((5, 256)))
        buf = torch.full((5 * N + 2,), -1.0, dtype=torch.float16, device="cuda")
        y = buf[off:off + 5 * N].view(5, N)
        tecoops.gemv(dev(W), dev(x), y)
        torch.cuda.synchronize()
        _check(y, orc.HALF, orc.gemv(W, x), orc.to_float(W), orc.to_float(x), f"offset {off}")
        assert (buf[:off] == -1).all() and (buf[off + 5 * N:] == -1).all()
