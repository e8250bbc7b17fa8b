"""The number of W rows that a batch product takes per workgroup
(gemv_batch.h), on the CPU: the header built as host C++."""
import ctypes
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "teco-ops_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

SOURCE = """
#include "gemv_batch.h"
extern "C" int rows(int n, int k, int batch, int i8, int cus) {
    return tecoops::gemv_batch_rows(n, k, batch, i8 != 0, cus);
}
extern "C" int staged(int batch) { return tecoops::gemv_batch_staged(batch); }
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rows")
    (d / "rows.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1",
                    "-I", os.path.join(REPO, "include"), "-I", CSRC, "-I", os.path.join(ROCM, "include"),
                    str(d / "rows.cpp"), "-o", str(d / "rows.so")], check=True)
    return ctypes.CDLL(str(d / "rows.so"))


def copied(rule, n, batch, i8, r, cus=256):
    """Bytes per element of K that the busiest CU copies: its share of W and, once
    per workgroup, x."""
    return -(-(-(-n // r)) // cus) * (r * (1 if i8 else 2) + 2 * rule.staged(batch))


@pytest.mark.parametrize("i8", [0, 1], ids=["16bit", "int8"])
@pytest.mark.parametrize("batch", [2, 4, 5, 8, 9, 16, 32, 33, 48, 64])
def test_rows_per_workgroup(rule, batch, i8):
    """A product of fewer rows never costs the busiest CU more than one of more
    rows, and none costs much more than its even share: what a width between
    two sizes cost when rows of W alone were counted."""
    staged = rule.staged(batch)
    before = 0
    for n in range(64, 65537, 8):
        r = rule.rows(n, 4096, batch, i8, 256)
        assert r in (8, 16, 32, 48, 64, 96, 112, 128)
        assert r != 48 or staged <= 8          # the kernels that are built
        assert r >= 32 or not i8 or staged <= 32
        cost = copied(rule, n, batch, i8, r)
        assert cost >= before
        before = cost
        # the even share of W, and x once for every 64 rows of it
        share = n / 256 * (1 if i8 else 2) + 2 * staged * max(1, -(-n // (64 * 256)))
        if n >= 4096:
            assert cost <= 1.85 * share, (n, r, cost, share)


def test_wide_strides(rule):
    """16-bit rows of a multiple of 32 KiB do not take 48 rows, nor 16 in
    several rounds."""
    assert rule.rows(4096, 16384, 3, 0, 256) == 16 and rule.rows(10240, 16384, 3, 0, 256) == 8
    assert rule.rows(12288, 14336, 8, 0, 256) == 48
    assert rule.rows(12288, 16384, 8, 0, 256) == 64
    assert rule.rows(12288, 32768, 8, 0, 256) == 64
    assert rule.rows(12288, 16384, 8, 1, 256) == 48
