"""GPU parity of split-KV decode with the CPU oracle where few sequences are
split down to one 128-key tile, and where the partials are merged by several
rows of lanes at once.

A row's partials are merged with one fp32 rounding each (at most 1024 splits *
2^-24 = 6e-5 of its largest term), which is nothing beside the 16-bit rounding
of probabilities and output, so the bound is the one of those, relative to the
row (attention_row_bound): a split left out of any of these cases is seen.
"""
import pytest

from oracle import oracle as orc

from helpers import assert_rows_close
from test_gpu_flash_attention import make_inputs, run_gpu, run_gpu_workspace

pytestmark = pytest.mark.gpu

# (H, Hkv, D, block size, kv lengths, q length)
CASES = [
    (8, 2, 128, 16, [512], 1),                     # one split
    (8, 2, 128, 16, [513], 1),                     # 128 keys each, the last of one
    (8, 2, 128, 16, [1, 127, 128, 129, 0, 640], 1),
    (32, 8, 128, 16, [2048, 2049, 4096, 255], 1),  # 512 workgroups of 256 keys
    (32, 32, 128, 16, [700, 300, 511, 90], 1),     # 128 keys would pass two per CU
    (8, 1, 128, 16, [16384], 1),                   # 128 splits by 8 rows of lanes
    (8, 1, 128, 16, [70000], 1),                   # 2048 keys and the rest
    (4, 1, 64, 24, [3000, 17], 3),                 # several rows per column group
    (6, 2, 96, 16, [2500, 5000], 2),               # 8 of 10 rows of lanes in use
    (8, 2, 32, 16, [9000, 1], 1),
    (4, 2, 160, 16, [3000, 1100], 2),
    (32, 1, 192, 8, [4097, 600], 1),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"H{c[0]}/{c[1]}-D{c[2]}-B{len(c[4])}-k{max(c[4])}")
@pytest.mark.parametrize("dt", [orc.HALF, orc.BF16], ids=["fp16", "bf16"])
def test_decode_short_splits(case, dt):
    H, Hkv, D, bs, kv, rows = case
    q_lens = [rows] * len(kv)
    q, kc, vc, bt = make_inputs(H + D + len(kv), H, Hkv, D, bs, q_lens, kv, dtype=dt)
    ref = orc.flash_attention(q, kc, vc, bt, q_lens, kv, dtype=dt)
    assert_rows_close(run_gpu(q, kc, vc, bt, q_lens, kv, dt), ref, dt, what="handle's scratch")
    # the splits that a sequence lacks are never written: NaN there stays out
    got = run_gpu_workspace(q, kc, vc, bt, q_lens, kv, dt, 0xFF)
    assert_rows_close(got, ref, dt, what="caller's workspace")
