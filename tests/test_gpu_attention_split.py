"""The split form of sparse MLA (scores and values in two launches, taken for
the rows after the last full round of work-groups) gives the bits of the
one-launch kernel, which the C entries without a workspace run."""

import pytest
import torch

pytestmark = pytest.mark.gpu

SCALE = 576**-0.5


def _one_launch(q, cache, table, kv, ids, n_tokens, scale):
    from cxldsagr_amd import _native

    out = torch.empty(*q.shape[:2], 512, dtype=q.dtype, device=q.device)
    if kv is None:
        _native.call("dsa_sparse_mla_fp8_paged", _native.ptr(q), q.shape[0], q.shape[1],
                     _native.ptr(cache), cache.shape[0], _native.ptr(table), n_tokens,
                     _native.ptr(ids), ids.shape[1], scale, _native.ptr(out),
                     _native.stream_of(q.device))
    else:
        _native.call("dsa_sparse_mla_bf16", _native.ptr(q), q.shape[0], q.shape[1],
                     _native.ptr(kv), kv.shape[0], _native.ptr(ids), ids.shape[1], scale,
                     _native.ptr(out), _native.stream_of(q.device))
    return out


# Rows around the bounds of the rule (an eighth and a quarter of a round of 256
# work-groups, one row past a full round), selections around its shortest and
# longest, off the 32-key block, the 64-key step and the 256-key round.
@pytest.mark.parametrize("rows,heads,selected", [
    (1, 128, 2048), (1, 64, 321), (2, 192, 1000), (16, 128, 2047), (17, 128, 545),
    (32, 128, 2048), (33, 128, 700), (64, 64, 1025), (65, 64, 320), (129, 128, 640),
    (160, 128, 351), (161, 128, 352), (3, 128, 319), (3, 128, 2049), (5, 64, 511),
    # Both sides of the selections at which it begins to be the faster form.
    (8, 128, 320), (9, 128, 320), (9, 128, 321), (16, 128, 384), (16, 128, 385), (17, 128, 448),
    (17, 128, 449), (17, 128, 513), (32, 128, 960), (160, 128, 961), (64, 64, 962), (21, 192, 1000),
])
def test_split_form_has_the_bits_of_one_launch(gpu, rows, heads, selected):
    from cxldsagr_amd.attention import pack_kv_fp8, sparse_mla, sparse_mla_fp8_paged

    gen = torch.Generator(device=gpu).manual_seed(rows * 4096 + selected)
    tokens = 5000
    pages = (tokens + 63) // 64
    kv = torch.randn(tokens, 576, generator=gen, device=gpu).bfloat16()
    table = torch.randperm(pages, generator=gen, device=gpu).int()
    cache = torch.zeros(pages, 64, 656, dtype=torch.uint8, device=gpu)
    pack_kv_fp8(kv, cache, table)
    q = torch.randn(rows, heads, 576, generator=gen, device=gpu).bfloat16()
    q[-1] *= 16  # peaked scores: the running max rises block after block
    ids = torch.randint(0, tokens, (rows, selected), generator=gen, device=gpu).int()
    # Padding: tails of every length in the last rows, holes and whole blocks,
    # an empty row, a row of out-of-range ids, an infinite record.
    keep = torch.randint(0, selected + 1, (rows, 1), generator=gen, device=gpu)
    tail = torch.arange(selected, device=gpu) >= keep
    ids[1::3] = torch.where(tail, -1, ids)[1::3]
    ids[0, 32:128] = -1
    ids[0, ::7] = -1
    if rows > 2:
        ids[1] = -1
        ids[2] = tokens + 5
    if rows > 3:
        kv[7, 100] = float("inf")
        ids[3, selected // 2] = 7
    paged = sparse_mla_fp8_paged(q, cache, table, ids, SCALE, n_tokens=tokens)
    flat = sparse_mla(q, kv, ids, SCALE)
    for got, records in ((paged, None), (flat, kv)):
        want = _one_launch(q, cache, table, records, ids, tokens, SCALE)
        torch.cuda.synchronize()
        same = (got.view(torch.int16) == want.view(torch.int16)) | (got.isnan() & want.isnan())
        assert bool(same.all())


def test_negative_and_zero_scales_take_one_launch(gpu):
    """The split form skips a block by its -inf maximum, which holds for
    positive scales only; others run as without a workspace."""
    from cxldsagr_amd.attention import sparse_mla

    gen = torch.Generator(device=gpu).manual_seed(3)
    kv = torch.randn(900, 576, generator=gen, device=gpu).bfloat16()
    q = torch.randn(4, 64, 576, generator=gen, device=gpu).bfloat16()
    ids = torch.randint(0, 900, (4, 640), generator=gen, device=gpu).int()
    for scale in (-SCALE, 0.0):
        want = _one_launch(q, None, None, kv, ids, 0, scale)
        assert torch.equal(sparse_mla(q, kv, ids, scale).view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("heads", [64, 192])
def test_rows_that_end_in_padding_equal_their_short_selections(gpu, heads):
    """Rows stop at their last id in range: a full round of rows whose ids end
    at every edge of the 64-key step has, row by row, the bits of the same ids
    without the padding (-1, or ids past the records)."""
    from cxldsagr_amd.attention import sparse_mla

    gen = torch.Generator(device=gpu).manual_seed(11)
    rows, selected, tokens = 256 if heads == 64 else 85, 300, 1000
    kv = torch.randn(tokens, 576, generator=gen, device=gpu).bfloat16()
    q = torch.randn(rows, heads, 576, generator=gen, device=gpu).bfloat16()
    ids = torch.randint(0, tokens, (rows, selected), generator=gen, device=gpu).int()
    ends = [0, 1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 192, 255, 256, 257, 299, 300]
    for r in range(rows):
        ids[r, ends[r % len(ends)]:] = -1 if r % 2 else tokens
    got = sparse_mla(q, kv, ids, SCALE)
    for r in range(len(ends)):
        end = ends[r]
        want = (sparse_mla(q[r:r + 1], kv, ids[r:r + 1, :end].contiguous(), SCALE)[0] if end
                else torch.zeros_like(got[r]))
        assert torch.equal(got[r].view(torch.int16), want.view(torch.int16)), end


@pytest.mark.parametrize("heads", [64, 192])
def test_paged_rows_that_end_in_padding(gpu, heads):
    """The same over the fp8 paged cache, whose rows stop by a look-ahead of
    their own: -1, ids past n_tokens (the page table covers more) and ids on
    pages outside the cache, which do not stop a row. The oracle of the
    dequantised records has the same rows (tolerance: a bf16 output and P)."""
    import numpy as np

    from cxldsagr_amd.attention import pack_kv_fp8, sparse_mla_fp8_paged
    from oracle import kv_fp8 as okv
    from oracle import sparse_mla as omla

    gen = torch.Generator(device=gpu).manual_seed(12)
    rows, selected, tokens, pages = 256 if heads == 64 else 85, 300, 1000, 16
    kv = torch.randn(tokens, 576, generator=gen, device=gpu).bfloat16()
    table = torch.randperm(pages, generator=gen, device=gpu).int()
    cache = torch.zeros(pages, 64, 656, dtype=torch.uint8, device=gpu)
    pack_kv_fp8(kv, cache, table)
    records = okv.logical_records(cache.cpu().numpy(), table.cpu().numpy(), tokens)
    table = torch.cat((table, torch.zeros(4, dtype=torch.int32, device=gpu)))
    table[3], table[7] = pages, -1  # outside the cache
    outside = torch.zeros(tokens, dtype=torch.bool, device=gpu)
    outside[192:256] = outside[448:512] = True
    q = torch.randn(rows, heads, 576, generator=gen, device=gpu).bfloat16()
    ids = torch.randint(0, tokens, (rows, selected), generator=gen, device=gpu).int()
    ids[:, 5::11] = 200  # on a page outside
    ends = [0, 1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 192, 255, 256, 257, 299, 300]
    fills = [-1, tokens, 470]
    for r in range(rows):
        ids[r, ends[r % len(ends)]:] = fills[r % 3]
    got = sparse_mla_fp8_paged(q, cache, table, ids, SCALE, n_tokens=tokens)
    for r in range(54):  # every end with every filling
        end = ends[r % len(ends)]
        want = (sparse_mla_fp8_paged(q[r:r + 1], cache, table, ids[r:r + 1, :end].contiguous(),
                                     SCALE, n_tokens=tokens)[0] if end else torch.zeros_like(got[r]))
        assert torch.equal(got[r].view(torch.int16), want.view(torch.int16)), (r, end)
    valid = (ids >= 0) & (ids < tokens)
    valid &= ~outside[ids.clamp(0, tokens - 1).long()]
    sample = list(range(0, 54, 5))
    _, ref = omla.sparse_mla(q[sample].float().cpu().numpy(), records,
                             torch.where(valid, ids, -1)[sample].cpu().numpy(), SCALE)
    np.testing.assert_allclose(got[sample].float().cpu().numpy(), ref, atol=4e-3, rtol=2e-2)


@pytest.mark.parametrize("fewer,more,heads,selected", [(12, 16, 128, 2048), (26, 32, 128, 2048),
                                                       (24, 32, 128, 1024), (24, 32, 64, 2048)])
def test_fewer_rows_take_no_longer(gpu, fewer, more, heads, selected):
    """The score launch's runs fit one round of work-groups for every row count
    (fewer rows had taken 1.10 to 1.13 times as long as more, and take 0.90 to 0.92)."""
    from cxldsagr_amd.attention import sparse_mla

    gen = torch.Generator(device=gpu).manual_seed(1)
    kv = torch.randn(20000, 576, generator=gen, device=gpu).bfloat16()

    def call(rows):
        q = torch.randn(rows, heads, 576, generator=gen, device=gpu).bfloat16()
        ids = torch.randint(0, 20000, (rows, selected), generator=gen, device=gpu).int()
        return lambda: sparse_mla(q, kv, ids, SCALE)

    calls, best = [call(fewer), call(more)], [float("inf")] * 2
    for fn in calls:
        fn()
    for _ in range(9):
        for i, fn in enumerate(calls):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record()
            for _ in range(30):
                fn()
            end.record()
            torch.cuda.synchronize()
            best[i] = min(best[i], begin.elapsed_time(end))
    assert best[0] < 1.04 * best[1], best
