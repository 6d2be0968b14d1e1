"""The history write: both quantisations in one launch, hardware e4m3 codes.

Codes and scales are compared byte for byte with the CPU oracle (index K) and
with the pack alone, whose codes are those of the oracle too, over row counts
around the block sizes (16 index rows, 4 tokens) and rows that take the
software encoding (an infinity, a NaN) beside rows that do not.
"""
import pytest
import torch

from oracle import quantize as oquant

pytestmark = pytest.mark.gpu
DEVICE = "cuda:0"


def special_rows(rows, width, seed):
    gen = torch.Generator().manual_seed(seed)
    # Magnitudes over the range of bf16, so that codes reach subnormals, both
    # ends of the clamp and both ends of the scales.
    x = torch.randn(rows, width, generator=gen) * torch.exp2(
        torch.randint(-30, 100, (rows, 1), generator=gen).float())
    x[0] = 0.0
    x[rows // 2, 5] = float("inf")
    x[rows // 3, 7] = float("nan")
    x[rows - 1, 1:] = -0.0
    x[rows - 1, 0] = 3.3e38
    return x.to(torch.bfloat16)


def oracle_rows(x):
    codes, scales = oquant.quantize_index(x.float().numpy())
    return torch.from_numpy(codes), torch.from_numpy(scales).reshape(-1).view(torch.int32)


@pytest.mark.parametrize("rows", [1, 3, 4, 5, 15, 16, 17, 63, 65, 1001])
def test_history_codes_match_the_oracle(rows):
    from cxldsagr_amd import attention
    from cxldsagr_amd.layer import DSALayer

    k, kv = special_rows(rows, 128, rows), special_rows(rows, 576, rows + 1)
    layer = DSALayer(1024 + 128, device=DEVICE)
    layer.write_history(k[:1].to(DEVICE), kv[:1].to(DEVICE))  # an odd offset for the rest
    layer.write_history(k.to(DEVICE), kv.to(DEVICE))
    assert layer.written == rows + 1
    codes, scales = oracle_rows(k)
    assert torch.equal(layer.index_keys[1:rows + 1].view(torch.uint8).cpu(), codes)
    assert torch.equal(layer.index_scales[1:rows + 1].view(torch.int32).cpu(), scales)

    codes, scales = oracle_rows(kv[:, :512].reshape(-1, 128))
    pages = -(-(rows + 1) // 64)
    packed = torch.zeros_like(layer.kv_cache)
    attention.pack_kv_fp8(kv[:1].to(DEVICE), packed, layer.page_table)
    attention.pack_kv_fp8(kv.to(DEVICE), packed, layer.page_table, token_offset=1)
    assert torch.equal(layer.kv_cache.view(torch.uint8), packed.view(torch.uint8))
    table = layer.page_table[:pages].cpu().long()
    records = packed.cpu().view(torch.uint8).reshape(packed.shape[0], -1)[table]
    records = records.reshape(-1, 656)[1:rows + 1]
    assert torch.equal(records[:, :512].reshape(-1, 128), codes)
    assert torch.equal(records[:, 512:528].reshape(-1, 4).contiguous().view(torch.int32).reshape(-1),
                       scales)


def test_history_rows_that_are_no_plain_matrix():
    """Strided rows are taken, rows without a unit stride are refused, as the
    separate quantiser has it."""
    from cxldsagr_amd.layer import DSALayer

    gen = torch.Generator().manual_seed(5)
    wide = torch.randn(20, 130, generator=gen).to(torch.bfloat16).to(DEVICE)
    kv = torch.randn(20, 576, generator=gen).to(torch.bfloat16).to(DEVICE)
    a, b = DSALayer(64, device=DEVICE), DSALayer(64, device=DEVICE)
    a.write_history(wide[:, 1:129], kv)
    b.write_history(wide[:, 1:129].contiguous(), kv)
    assert torch.equal(a.index_keys.view(torch.uint8), b.index_keys.view(torch.uint8))
    with pytest.raises(ValueError):
        DSALayer(128, device=DEVICE).write_history(
            torch.zeros(128, 128, dtype=torch.bfloat16, device=DEVICE).t(),
            torch.zeros(128, 576, dtype=torch.bfloat16, device=DEVICE))
