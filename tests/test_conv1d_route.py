"""When causal_conv1d's ragged rows run along the token axis
(causal_conv1d.h), on the CPU: the header built as host C++."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "teco-ops_amd", "csrc")
CUS = 256


@pytest.fixture(scope="module")
def along_axis(tmp_path_factory):
    d = tmp_path_factory.mktemp("route")
    (d / "route.cpp").write_text("""#include "causal_conv1d.h"
extern "C" int along_axis(long long batch, long long dim, long long tokens, long long cus) {
    return tecoops::conv1d_along_axis(batch, dim, tokens, cus);
}
""")
    subprocess.run(["g++", "-std=c++17", "-fPIC", "-shared", "-I", CSRC, str(d / "route.cpp"), "-o",
                    str(d / "route.so")], check=True)
    fn = ctypes.CDLL(str(d / "route.so")).along_axis
    fn.argtypes = [ctypes.c_longlong] * 4
    return lambda batch, dim, tokens: bool(fn(batch, dim, tokens, CUS))


@pytest.mark.parametrize("batch,mean", [(8, 2048), (16, 1000), (16, 512), (64, 256), (64, 4096), (512, 40)])
def test_channels_fill_the_chip(along_axis, batch, mean):
    """A workgroup takes a whole channel: with many sequences and fewer
    channels than CUs it would leave CUs idle that a wave per row fills."""
    assert not any(along_axis(batch, dim, batch * mean) for dim in range(1, CUS + 1, 5))


@pytest.mark.parametrize("dim", [1, 64, 512, 4096, 16384])
def test_long_sequences_stay_by_rows(along_axis, dim):
    """Rows of 1024 tokens and more stream as well by themselves, and faster
    where they start on the boundary; few sequences fill the chip otherwise
    only with channels in number."""
    for batch in (3, 4, 8, 16, 64):
        for mean in (1024, 2048, 8192):
            assert not along_axis(batch, dim, batch * mean)
    for batch in (1, 2):
        assert along_axis(batch, dim, 65536) == (batch * dim <= 6 * CUS)


def test_what_gains_runs_along_the_axis(along_axis):
    for batch, dim, tokens in ((16, 4096, 8064), (64, 512, 64 * 256), (512, 4096, 512 * 40), (32, 1024, 29561),
                               (1, 64, 16384), (2, 768, 3901), (32, 2048, 2140)):
        assert along_axis(batch, dim, tokens)


def test_ragged_batches_run_along_the_axis(along_axis):
    """Lengths that are not alike in whole vectors, by their total: many short
    sequences, and longer ones of many channels; not a few tokens, nor few channels
    of long sequences."""
    for batch, dim, tokens in ((44, 6336, 750), (100, 6360, 873), (26, 4840, 831), (7, 2704, 1142), (6, 6544, 3821),
                               (20, 1192, 23715), (52, 360, 14260)):
        assert along_axis(batch, dim, tokens)
    for batch, dim, tokens in ((7, 4520, 434), (8, 4888, 512), (54, 272, 59702), (5, 736, 44727), (99, 216, 17744)):
        assert not along_axis(batch, dim, tokens)
