"""The indexer's calls of several launches refuse bad buffers before the first
of them: it already writes the workspace (floors) and, in a layer step, the
caches."""

import ctypes

import pytest
import torch

from cxldsagr_amd import _native

ROWS, POSITION, TOPK = 3, 500, 64
COLUMNS = POSITION + ROWS


def _size(name, *args):
    size = ctypes.c_int64()
    _native.call(name, *args, ctypes.byref(size))
    return size.value


def _layer_args(address, stream):
    """dsa_layer_indexer_fp8's arguments by name; ``address(name, bytes)``
    gives each buffer's."""
    scratch = _size("dsa_layer_indexer_scratch_bytes", ROWS, COLUMNS, TOPK)
    workspace = _size("dsa_indexer_select_workspace_bytes", ROWS, COLUMNS, 0)
    return {
        "q": address("q", ROWS * 64 * 256), "rows": ROWS, "weights": address("weights", ROWS * 256),
        "k": address("k", ROWS * 256), "kv": address("kv", ROWS * 1152),
        "page_table": address("page_table", 32), "pages": 8,
        "cache": address("cache", 8 * 64 * 656), "index_keys": address("index_keys", COLUMNS * 128),
        "index_scales": address("index_scales", COLUMNS * 4), "position": POSITION, "topk": TOPK,
        "indices": address("indices", ROWS * TOPK * 4), "scores": address("scores", ROWS * 512 * 4),
        "scratch": address("scratch", scratch), "scratch_bytes": scratch,
        "workspace": address("workspace", workspace), "workspace_bytes": workspace, "stream": stream,
    }


def _select_args(address, stream):
    """The same for dsa_indexer_select_fp8."""
    workspace = _size("dsa_indexer_select_workspace_bytes", ROWS, COLUMNS, 0)
    return {
        "q": address("q", ROWS * 64 * 128), "k": address("k", COLUMNS * 128),
        "weights": address("weights", ROWS * 256), "kscale": address("kscale", COLUMNS * 4),
        "starts": None, "ends": None, "query_start": POSITION, "rows": ROWS, "columns": COLUMNS,
        "q_fold": address("q_fold", ROWS * 2048), "scores": address("scores", ROWS * 512 * 4),
        "topk": TOPK, "values": address("values", ROWS * TOPK * 4),
        "indices": address("indices", ROWS * TOPK * 4), "out_ld": TOPK,
        "workspace": address("workspace", workspace), "workspace_bytes": workspace, "stream": stream,
    }


def _refused(name, args):
    """Variants of valid arguments that the call must refuse."""
    if name == "dsa_indexer_select_fp8":
        return [
            {"workspace_bytes": args["workspace_bytes"] - 1}, {"workspace_bytes": 0},
            {"workspace": None}, {"workspace": args["workspace"] + 16}, {"scores": None},
            {"indices": None}, {"values": None}, {"out_ld": TOPK - 1}, {"topk": 0}, {"topk": 2049},
            {"q": None}, {"q_fold": args["q_fold"] + 4}, {"query_start": POSITION + 1},
            {"ends": args["kscale"]}, {"columns": 2**26},
        ]
    return [
        {"workspace_bytes": args["workspace_bytes"] - 1}, {"workspace_bytes": 0},
        {"workspace": None}, {"workspace": args["workspace"] + 16}, {"scores": None},
        {"scratch_bytes": args["scratch_bytes"] - 1}, {"scratch": args["scratch"] + 8},
        {"indices": None}, {"rows": 0}, {"rows": 2**31}, {"position": -1}, {"position": 2**31},
        {"position": 2**62}, {"topk": 2049}, {"index_keys": args["index_keys"] + 8},
        {"q": None}, {"cache": args["cache"] + 8}, {"pages": 7},
    ]


CALLS = {"dsa_layer_indexer_fp8": _layer_args, "dsa_indexer_select_fp8": _select_args}


def _refuses(name, args, change):
    with pytest.raises(ValueError):
        _native.call(name, *{**args, **change}.values())


@pytest.mark.parametrize("name", CALLS)
@pytest.mark.skipif(torch.cuda.is_available(), reason="addresses that no device may see")
def test_calls_refuse_before_any_launch(name):
    """Without a device a launch is an error of another kind."""
    args = CALLS[name](lambda buffer, size: 1 << 20, None)
    for change in _refused(name, args):
        _refuses(name, args, change)


@pytest.mark.gpu
@pytest.mark.parametrize("name", CALLS)
def test_refused_calls_write_nothing(gpu, name):
    buffers = {}

    def address(buffer, size):
        buffers[buffer] = torch.full((size + 256,), 0x5A, dtype=torch.uint8, device=gpu)
        return buffers[buffer].data_ptr()

    args = CALLS[name](address, _native.stream_of(gpu))
    for change in _refused(name, args):
        _refuses(name, args, change)
    torch.cuda.synchronize()
    for buffer, content in buffers.items():
        assert bool((content == 0x5A).all()), buffer
