"""The candidate top-k's one-sort path for rows stored in full (at most 8,192
columns) and its value buckets, against the unfused operators bit for bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(gpu, rows, columns, seed):
    from cxldsagr_amd import indexer

    gen = torch.Generator(device=gpu).manual_seed(seed)
    q8, _ = indexer.quantize_index(torch.randn(rows, 64, 128, generator=gen, device=gpu).bfloat16())
    k8, ks = indexer.quantize_index(torch.randn(columns, 128, generator=gen, device=gpu).bfloat16())
    w = torch.randn(rows, 64, generator=gen, device=gpu) / 8
    return q8, k8, w, ks[:, 0].contiguous(), gen


def _check(q8, k8, w, ks, start, topk, bounds=None):
    from cxldsagr_amd import indexer

    columns = len(k8)
    scores = indexer.logits(q8, k8, w, ks, start, _bounds=bounds, _pad_to_stride=True)
    values, ids = indexer.exact_topk(scores[:, :columns], topk)
    got_values, got_ids = indexer.select_topk(q8, k8, w, ks, start, topk, _bounds=bounds)
    torch.cuda.synchronize()
    assert torch.equal(got_ids, ids)
    # (A non-finite value has id -1; its own bits may be another's.)
    same = got_values.view(torch.int32) == values.view(torch.int32)
    assert bool((same | (~got_values.isfinite() & ~values.isfinite())).all())


@pytest.mark.parametrize("rows,columns,topk", [
    (1, 1, 2048), (2, 2, 1), (5, 63, 64), (40, 2047, 2048), (33, 2048, 2048), (33, 2049, 2048),
    (7, 4096, 2048), (300, 5000, 777), (3, 8191, 2048), (3, 8192, 2048), (3, 8193, 2048),
    (40, 8200, 2048), (16, 200, 2048), (16, 201, 2048), (17, 200, 2048), (3, 130, 7),
])
def test_short_rows_equal_unfused(gpu, rows, columns, topk):
    q8, k8, w, ks, _ = _inputs(gpu, rows, columns, columns)
    _check(q8, k8, w, ks, columns - rows, topk)


@pytest.mark.parametrize("columns", [3000, 20000])
def test_rows_whose_threshold_is_negative_or_extreme(gpu, columns):
    """Weights all negative (every score below zero), all equal scores, a span
    too large or too small to scale, infinite and NaN scores, signed zeros."""
    rows = 12
    q8, k8, w, ks, gen = _inputs(gpu, rows, columns, 7)
    w[0] = -w[0].abs()
    w[1] = -w[1].abs() + 0.01
    w[2] = 0.0
    w[3] = -0.0
    w[4] *= 1e37
    w[5] *= 1e-38
    w[6, 0] = float("inf")
    w[7, 0] = float("nan")
    w[8] = 1e-3
    _check(q8, k8, w, ks, columns - rows, 2048)
    ks = ks.clone()
    ks[::5] = 0.0
    ks[1] = float("inf")
    ks[2] = float("nan")
    _check(q8, k8, w, ks, columns - rows, 2048)


def test_short_rows_with_bounds(gpu):
    """Ragged [starts, ends) windows, empty ones among them."""
    rows, columns = 24, 6000
    q8, k8, w, ks, gen = _inputs(gpu, rows, columns, 3)
    ends = torch.randint(0, columns + 1, (rows,), generator=gen, device=gpu).int()
    starts = (ends - torch.randint(0, 4000, (rows,), generator=gen, device=gpu).int()).clamp_min(0)
    starts[0], ends[0] = 0, columns
    starts[1], ends[1] = 500, 500
    starts[2], ends[2] = 700, 100
    _check(q8, k8, w, ks, columns - rows, 2048, (starts, ends))
