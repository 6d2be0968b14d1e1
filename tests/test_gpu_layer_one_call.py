"""The layer's one-call indexer (``indexer.layer_select``) against the separate
operators: same ids, same cache writes, for every layout the layer takes."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _strided(t):
    return torch.stack((t, t), dim=-1)[..., 0]


def _offset(t):
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    flat[1:] = t.reshape(-1)
    return flat[1:].view(t.shape)


@pytest.mark.parametrize("layout", ["plain", "strided", "offset"])
@pytest.mark.parametrize("history,rows,topk,kv_format", [
    (0, 1, 2048, "fp8_paged"), (70, 5, 64, "bf16"), (9000, 33, 2048, "fp8_paged"),
    (9000, 16, 1, "bf16"),
])
def test_layer_equals_separate_operators(gpu, layout, history, rows, topk, kv_format):
    from cxldsagr_amd import attention, indexer
    from cxldsagr_amd.layer import DSALayer

    change = {"plain": lambda t: t, "strided": _strided, "offset": _offset}[layout]
    gen = torch.Generator(device=gpu).manual_seed(history + rows)

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=gpu)

    tokens = history + rows
    index_q, index_k = randn(rows, 64, 128).bfloat16(), randn(tokens, 128).bfloat16()
    weights, q, kv = randn(rows, 64) / 8, randn(rows, 64, 576).bfloat16(), randn(tokens, 576).bfloat16()
    layer = DSALayer(tokens, device=gpu, heads=64, topk=topk, kv_format=kv_format)
    layer.write_history(index_k[:history], kv[:history])
    out, selection = layer.forward(change(index_q), change(index_k[history:].clone()),
                                   change(weights), change(q), change(kv[history:].clone()))

    q8, _, folded = indexer.quantize_index_folded(index_q, weights)
    k8, ks = indexer.quantize_index(index_k)
    _, ids = indexer.select_topk(q8, k8, folded, ks[:, 0].contiguous(), history, topk)
    assert torch.equal(selection.token_ids, ids)
    assert torch.equal(layer.index_keys.view(torch.uint8), k8.view(torch.uint8))
    assert torch.equal(layer.index_scales, ks[:, 0])
    if kv_format == "bf16":
        assert torch.equal(layer.records, kv)
        want = attention.sparse_mla(q, kv, ids, layer.scale)
    else:
        want = attention.sparse_mla_fp8_paged(q, layer.kv_cache, layer.page_table, ids, layer.scale,
                                              n_tokens=tokens)
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    assert layer.written == tokens


def test_refused_inputs_stay_refused(gpu):
    from cxldsagr_amd.layer import DSALayer

    def step(rows, kv_rows=None, topk=2048):
        layer = DSALayer(128, device=gpu, heads=64, topk=topk)
        bf16 = {"dtype": torch.bfloat16, "device": gpu}
        n = rows if kv_rows is None else kv_rows
        return layer.forward(torch.zeros(rows, 64, 128, **bf16), torch.zeros(rows, 128, **bf16),
                             torch.zeros(rows, 64, device=gpu), torch.zeros(rows, 64, 576, **bf16),
                             torch.zeros(n, 576, **bf16))

    for args in ((0,), (129,), (4, 3), (4, None, 0), (4, None, 2049)):
        with pytest.raises(ValueError):
            step(*args)
