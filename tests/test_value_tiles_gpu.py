"""Values of a prompt into a paged cache through tiles of 64 rows: 16-byte reads of rows and reads of one value (odd sizes, strides and
addresses), tiles that are not full, slots out of order and left out.  Values are copied: exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows", [65, 128, 131, 300])
@pytest.mark.parametrize("vdim,vpad,extra,offset", [(64, 64, 0, 0), (128, 128, 8, 8), (128, 128, 8, 1), (128, 128, 3, 0),
                                                    (40, 64, 0, 0), (20, 32, 4, 4), (33, 64, 0, 0)])
def test_values(rows, vdim, vpad, extra, offset, dtype):
    import light_vllm_amd._custom_ops  # noqa: F401
    amd = torch.ops._C_amd
    heads = kv_heads = 2
    dim, block = 64, 16
    g = torch.Generator().manual_seed(rows + vdim)
    width = 2 * heads * dim + kv_heads * vdim
    # q, k and v are columns of one matrix, `offset` values from an aligned address, `extra` between rows
    flat = torch.randn(rows * (width + extra) + offset, generator=g).to(dtype).to(DEV)
    all_rows = flat[offset:].view(rows, width + extra)
    q, k, v = all_rows[:, :heads * dim], all_rows[:, heads * dim:2 * heads * dim], all_rows[:, 2 * heads * dim:width]
    blocks = (rows + block - 1) // block + 3
    # most slots consecutive, as a prompt's; the last third shuffled; every seventh row of that left out
    slots = torch.arange(rows) + 5
    third = rows * 2 // 3
    slots[third:] = slots[third:][torch.randperm(rows - third, generator=g)]
    slots[third::7] = -1
    x = 16 // flat.element_size()
    kc = torch.zeros(blocks, kv_heads, dim // x, block, x, dtype=dtype, device=DEV)
    vc = torch.zeros(blocks, kv_heads, vpad, block, dtype=dtype, device=DEV)
    want = torch.zeros(blocks * block, kv_heads, vpad, dtype=dtype)
    ok = slots >= 0
    want[slots[ok], :, :vdim] = v.cpu().view(rows, kv_heads, vdim)[ok]
    amd.qk_norm_cache(q, k, v, torch.ones(dim, device=DEV), torch.ones(dim, device=DEV), 1e-5, heads, kv_heads, kc, vc, slots.to(DEV))
    got = vc.cpu().permute(0, 3, 1, 2).reshape(blocks * block, kv_heads, vpad)
    assert torch.equal(got, want)
