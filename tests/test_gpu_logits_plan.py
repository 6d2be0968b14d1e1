"""The logits launcher's key splits and work-group order: a score does not
depend on the rows it is computed with, so every batch equals, bit for bit,
the same rows in batches of one query group."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# Query groups that do not divide the CUs, more than one round of work-groups,
# key counts off the 128-key stage and below one stage.
@pytest.mark.parametrize("rows,columns", [(17, 17), (100, 5001), (129, 130), (200, 16584),
                                          (340, 9000), (4100, 4200)])
def test_scores_do_not_depend_on_the_batch(gpu, rows, columns):
    from cxldsagr_amd import indexer

    gen = torch.Generator(device=gpu).manual_seed(rows)
    q8, _ = indexer.quantize_index(torch.randn(rows, 64, 128, generator=gen, device=gpu).bfloat16())
    k8, ks = indexer.quantize_index(torch.randn(columns, 128, generator=gen, device=gpu).bfloat16())
    w = torch.randn(rows, 64, generator=gen, device=gpu) / 8
    ks = ks[:, 0].contiguous()
    start = columns - rows
    whole = indexer.logits(q8, k8, w, ks, start, _pad_to_stride=True)
    for i in {0, rows // 2 // 16 * 16, (rows - 1) // 16 * 16}:
        part = indexer.logits(q8[i:i + 16].contiguous(), k8, w[i:i + 16].contiguous(), ks, start + i,
                              _pad_to_stride=True)
        assert torch.equal(whole[i:i + 16].view(torch.int32), part.view(torch.int32)), i
    values, ids = indexer.exact_topk(whole[:, :columns], 2048)
    got = indexer.select_topk(q8, k8, w, ks, start, 2048)
    assert torch.equal(got[1], ids) and torch.equal(got[0].view(torch.int32), values.view(torch.int32))
