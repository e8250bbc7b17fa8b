"""The workspace that the torch op allocates for a decode on the GPU."""
import pytest
import torch

import tecoops  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,Hkv,keys,splits", [(32, 8, 1657, 7), (32, 32, 1657, 2), (8, 1, 4096, 32)])
def test_decode_workspace_is_of_its_kv_heads(H, Hkv, keys, splits):
    """A split's partials are a float per head, row and dim, and two more per
    head and row; sized for the worst number of kv heads, they were twice that."""
    batch, D, block = 8, 128, 16
    pages = -(-keys // block)
    kc = torch.zeros(pages, Hkv, block, D, dtype=torch.float16, device="cuda")
    q = torch.zeros(batch, H, D, dtype=torch.float16, device="cuda")
    out = torch.empty_like(q)
    table = torch.arange(pages, dtype=torch.int32, device="cuda").repeat(batch, 1)
    starts = torch.arange(batch + 1, dtype=torch.int32, device="cuda")
    lens = torch.full((batch,), keys, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    torch.ops.tecoops.flash_attn_varlen_func(q, kc, kc, 1, starts, keys, None, lens, 1.0, True, None,
                                             table, False, out)
    torch.cuda.synchronize()
    used = torch.cuda.max_memory_allocated() - before
    need = batch * H * splits * (D + 2) * 4
    assert need <= used <= need + 1024  # 256 spare bytes, whole allocation units
