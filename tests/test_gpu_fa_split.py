"""GPU parity of prefill over split keys (fa_split.hip) with the CPU oracle:
query tiles whose keys are cut into pieces, at the edges of tiles, pieces and
batches, and the calls that run unsplit instead.

Splitting adds one fp32 rounding per piece to a merge of at most 64 pieces
(64 * 2^-24 = 4e-6 of the row's largest term), which is nothing beside the
rounding of the probabilities and the output to 16 bits that the unsplit
kernels have too, so the bound is the one of those, relative to the row
(attention_row_bound): a piece left out of any of these cases is seen.
"""
import math

import numpy as np
import pytest
import torch

import tecoops
from oracle import oracle as orc

from helpers import as_f32, assert_rows_close, dev
from test_gpu_flash_attention import make_inputs, run_gpu, run_reference_entry

pytestmark = pytest.mark.gpu

# (H, Hkv, D, block size, q_lens, cached): uneven chunks with few rows run in
# 4-wave workgroups of 32 to 128 rows, many rows in 12-wave ones of 96 to 384.
CHUNKS = [1, 33, 0, 64, 7, 130]
CACHED = [5000, 700, 90, 0, 4111, 2600]
CASES = [
    (8, 2, 128, 16, CHUNKS, CACHED),
    (8, 2, 128, 24, CHUNKS, CACHED),         # uniform pages of 8 rows
    (8, 2, 64, 16, CHUNKS, CACHED),
    (8, 2, 96, 16, CHUNKS, CACHED),
    (4, 2, 128, 16, CHUNKS, CACHED),         # two heads per tile
    (4, 2, 64, 32, CHUNKS, CACHED),
    (3, 3, 128, 16, CHUNKS, CACHED),         # one head per tile
    (3, 3, 96, 16, CHUNKS, CACHED),
    (8, 2, 128, 16, [192], [6001]),          # one sequence, whole 12-wave tiles
    (8, 2, 128, 24, [193], [6000]),
    (8, 2, 64, 16, [191], [6000]),
    (8, 2, 96, 8, [190], [5999]),
    (4, 2, 128, 16, [385], [6000]),
    (1, 1, 64, 16, [769], [6000]),
    (8, 1, 128, 16, [96, 96], [8000, 7999]),  # two groups of heads per kv head
    (8, 2, 128, 16, [9] * 64, [40 * i for i in range(64)]),   # the largest batch split
    (8, 2, 128, 16, [9] * 65, [40 * i for i in range(65)]),   # one more: unsplit
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"H{c[0]}/{c[1]}-D{c[2]}-bs{c[3]}-B{len(c[4])}-q{max(c[4])}")
@pytest.mark.parametrize("causal", [True, False], ids=["causal", "full"])
def test_split_prefill(case, causal):
    H, Hkv, D, bs, q_lens, cached = case
    kv = [a + b for a, b in zip(q_lens, cached)]
    dt = orc.BF16 if (H + bs) % 16 else orc.HALF
    q, kc, vc, bt = make_inputs(H * D + bs, H, Hkv, D, bs, q_lens, kv, dtype=dt)
    got = run_gpu(q, kc, vc, bt, q_lens, kv, dt, causal=causal)
    ref = orc.flash_attention(q, kc, vc, bt, q_lens, kv, causal=causal, dtype=dt)
    assert_rows_close(got, ref, dt, what="split prefill")
    if causal:  # lengths per sequence, the reference's entry point
        assert_rows_close(run_reference_entry(q, kc, vc, bt, q_lens, kv, max(q_lens), max(kv), dt),
                          ref, dt, what="split prefill (q_seq_lens)")


@pytest.mark.parametrize("q_lens,kv", [([40, 200], [6000, 30]), ([64, 64, 64], [0, 5000, 1]),
                                       ([300, 20], [4096, 0])],
                         ids=["kv_shorter_than_q", "empty_kv", "last_empty"])
def test_split_prefill_short_contexts(q_lens, kv):
    """Sequences with fewer keys than rows, or none, beside a split one."""
    q, kc, vc, bt = make_inputs(len(kv), 8, 2, 128, 16, q_lens, kv, dtype=orc.BF16)
    got = run_gpu(q, kc, vc, bt, q_lens, kv, orc.BF16)
    ref = orc.flash_attention(q, kc, vc, bt, q_lens, kv, dtype=orc.BF16)
    assert_rows_close(got, ref, orc.BF16, what="split prefill")


@pytest.mark.parametrize("max_q,max_k", [(0, 0), (16, 0), (9, 100000)])
def test_split_prefill_hints(max_q, max_k):
    """The hints choose the route; the pieces come from the lengths."""
    kv = [a + b for a, b in zip(CHUNKS, CACHED)]
    q, kc, vc, bt = make_inputs(3, 8, 2, 128, 16, CHUNKS, kv, dtype=orc.BF16)
    got = run_gpu(q, kc, vc, bt, CHUNKS, kv, orc.BF16, max_q=max_q, max_k=max_k)
    assert_rows_close(got, orc.flash_attention(q, kc, vc, bt, CHUNKS, kv, dtype=orc.BF16), orc.BF16,
                      what="hints")


def run_entry(entry, inputs, q_lens, kv, dt, ws=None):
    """tecoopsFlashAttentionEx with workspace `ws`, or ...NoAlloc."""
    from tecoops import _lib
    q, kc, vc, bt = (dev(a, dt) for a in inputs)
    cu = dev(np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32))
    kl, out = dev(np.array(kv, np.int32)), torch.empty_like(q)
    code = _lib.DATA_HALF if dt == orc.HALF else _lib.DATA_BFLOAT16
    with tecoops._Desc(bt, _lib.DATA_INT32) as btd, tecoops._Desc(q, code) as qd, \
            tecoops._Desc(kc, code) as kd, tecoops._Desc(vc, code) as vd, \
            tecoops._Desc(out, code) as od:
        args = [tecoops._handle(out.device), max(q_lens), max(kv), None, cu.data_ptr(), kl.data_ptr(), btd,
                bt.data_ptr(), qd, q.data_ptr(), kd, kc.data_ptr(), vd, vc.data_ptr(), od, out.data_ptr(),
                1.0 / math.sqrt(q.shape[2]), 1]
        _lib.call(entry, *args, *([ws.data_ptr()] if entry.endswith("Ex") else []))
    torch.cuda.synchronize()
    return as_f32(out, dt)


# (H, Hkv, q_lens, cached, whether keys are cut).  The last two: one sequence
# more than a split call may have, and contexts too short to cut.
ROUTES = [(8, 2, CHUNKS, CACHED, True), (3, 3, CHUNKS, CACHED, True),
          (8, 2, [9] * 64, [40 * i for i in range(64)], True),
          (8, 2, [9] * 65, [40 * i for i in range(65)], False), (8, 2, [30, 64], [100, 90], False)]


@pytest.mark.parametrize("case", ROUTES, ids=["chunks", "one_head", "B64", "B65", "short"])
def test_split_is_taken(case):
    """The allocation-free entry point never splits.  Where the eager call runs
    the same kernel (4 waves), its output has the same bits if and only if it
    cut no keys: a cut rounds the probabilities beside other running maxima."""
    H, Hkv, q_lens, cached, cut = case
    kv = [a + b for a, b in zip(q_lens, cached)]
    inputs = make_inputs(17, H, Hkv, 128, 16, q_lens, kv, dtype=orc.HALF, dist="normal")
    got = run_gpu(*inputs, q_lens, kv, orc.HALF)
    unsplit = run_entry("tecoopsFlashAttentionNoAlloc", inputs, q_lens, kv, orc.HALF)
    assert (not np.array_equal(got, unsplit)) == cut


def test_split_many_tiles():
    """More than 64 query tiles in one sequence, whose pieces are found 64
    tiles at a time: beside many short chunks it keeps to 32-row tiles."""
    q_lens, cached = [5] * 24 + [2150], [90] * 24 + [5000]
    kv = [a + b for a, b in zip(q_lens, cached)]
    q, kc, vc, bt = make_inputs(18, 4, 1, 128, 16, q_lens, kv, dtype=orc.BF16)
    got = run_gpu(q, kc, vc, bt, q_lens, kv, orc.BF16)
    assert_rows_close(got, orc.flash_attention(q, kc, vc, bt, q_lens, kv, dtype=orc.BF16), orc.BF16,
                      what="many tiles")


def prefill_call(seed):
    kv = [a + b for a, b in zip(CHUNKS, CACHED)]
    q, kc, vc, bt = make_inputs(seed, 8, 2, 128, 16, CHUNKS, kv, dtype=orc.BF16)
    cu = dev(np.concatenate([[0], np.cumsum(CHUNKS)]).astype(np.int32))
    args = (dev(q, orc.BF16), dev(kc, orc.BF16), dev(vc, orc.BF16), max(CHUNKS), cu, max(kv), None,
            dev(np.array(kv, np.int32)), 1.0 / math.sqrt(128), True, None, dev(bt), False,
            torch.zeros(q.shape, dtype=torch.bfloat16, device="cuda"))
    return args, orc.flash_attention(q, kc, vc, bt, CHUNKS, kv, dtype=orc.BF16)


@pytest.mark.parametrize("front", ["tecoops", "torch.ops"])
def test_split_prefill_streams(front):
    """Calls in turn on ten streams through one handle, which keeps scratch
    for eight: the others run unsplit, and none waits for another's buffer."""
    fn = tecoops.flash_attn_varlen_func if front == "tecoops" else \
        torch.ops.tecoops.flash_attn_varlen_func
    runs = [prefill_call(70 + i) for i in range(10)]
    streams = [torch.cuda.Stream() for _ in runs]
    torch.cuda.synchronize()
    for _ in range(2):
        for (args, _), st in zip(runs, streams):
            with torch.cuda.stream(st):
                fn(*args)
    torch.cuda.synchronize()
    for i, (args, ref) in enumerate(runs):
        assert_rows_close(as_f32(args[-1], orc.BF16), ref, orc.BF16, what=f"stream {i}")


@pytest.mark.parametrize("front", ["tecoops", "torch.ops"])
def test_prefill_captured(front):
    """A prefill that is split when called is captured unsplit, without the
    handle's scratch, and replays beside eager calls that use it."""
    fn = tecoops.flash_attn_varlen_func if front == "tecoops" else \
        torch.ops.tecoops.flash_attn_varlen_func
    args, ref = prefill_call(90)
    other, oref = prefill_call(91)
    fn(*args)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn(*args)
    for _ in range(3):
        args[-1].zero_()
        other[-1].zero_()
        graph.replay()
        fn(*other)
        torch.cuda.synchronize()
        assert_rows_close(as_f32(args[-1], orc.BF16), ref, orc.BF16, what="replay")
        assert_rows_close(as_f32(other[-1], orc.BF16), oref, orc.BF16, what="eager between replays")


def test_caller_workspace_prefill_is_unsplit():
    """A caller's workspace is sized for decode: a prefill leaves it alone and
    runs as the entry point that never splits."""
    kv = [a + b for a, b in zip(CHUNKS, CACHED)]
    inputs = make_inputs(5, 8, 2, 128, 16, CHUNKS, kv, dtype=orc.HALF, dist="normal")
    ws = torch.full((4096,), 0xA5, dtype=torch.uint8, device="cuda")
    got = run_entry("tecoopsFlashAttentionEx", inputs, CHUNKS, kv, orc.HALF, ws)
    assert np.array_equal(got, run_entry("tecoopsFlashAttentionNoAlloc", inputs, CHUNKS, kv, orc.HALF))
    assert (ws == 0xA5).all()
    assert_rows_close(got, orc.flash_attention(*inputs, CHUNKS, kv, dtype=orc.HALF), orc.HALF, what="workspace")
