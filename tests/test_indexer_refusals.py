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


def _refused(args):
    """Variants of valid arguments that the call must refuse."""
    return [
        {"workspace_bytes": args["workspace_bytes"] - 1}, {"workspace_bytes": 0},
        {"workspace": None}, {"workspace": args["workspace"] + 16}, {"scores": None},
        {"scratch_bytes": args["scratch_bytes"] - 1}, {"scratch": args["scratch"] + 8},
        {"indices": None}, {"rows": 0}, {"rows": 2**31}, {"position": -1}, {"position": 2**31},
        {"position": 2**62}, {"topk": 2049}, {"index_keys": args["index_keys"] + 8},
        {"q": None}, {"cache": args["cache"] + 8}, {"pages": 7},
    ]


def _refuses(args, change):
    with pytest.raises(ValueError):
        _native.call("dsa_layer_indexer_fp8", *{**args, **change}.values())


@pytest.mark.skipif(torch.cuda.is_available(), reason="addresses that no device may see")
def test_layer_indexer_refuses_before_any_launch():
    """Without a device a launch is an error of another kind."""
    args = _layer_args(lambda name, size: 1 << 20, None)
    for change in _refused(args):
        _refuses(args, change)


@pytest.mark.gpu
def test_refused_layer_calls_write_nothing(gpu):
    buffers = {}

    def address(name, size):
        buffers[name] = torch.full((size + 256,), 0x5A, dtype=torch.uint8, device=gpu)
        return buffers[name].data_ptr()

    args = _layer_args(address, _native.stream_of(gpu))
    for change in _refused(args):
        _refuses(args, change)
    torch.cuda.synchronize()
    for name, buffer in buffers.items():
        assert bool((buffer == 0x5A).all()), name
