"""Which sparse MLA calls take the split form (those that need a workspace): on
256 CUs (the count taken where no device is visible) the split form must be the
faster one, so no call of a short selection over many rows."""

import pytest

from cxldsagr_amd import _native


def _needs_workspace(rows, heads, selected):
    return _native.size_of("dsa_sparse_mla_workspace_bytes", None, rows, heads, selected) > 0


# The times of both forms on which the line rests, us (fp8 records): split, wide.
@pytest.mark.parametrize("rows,heads,selected,split,wide", [
    (16, 128, 320, 21.8, 18.2), (24, 128, 320, 24.6, 18.5), (32, 128, 320, 26.7, 18.5),
    (32, 64, 320, 21.8, 18.4), (64, 64, 320, 26.9, 18.8), (16, 128, 384, 21.8, 20.2),
    (32, 128, 512, 27.1, 24.4), (64, 64, 512, 28.0, 24.6), (24, 128, 640, 29.5, 28.2),
    (32, 128, 640, 32.2, 28.4), (36, 128, 2048, 78.4, 71.4), (44, 128, 2048, 84.5, 72.1),
    (64, 128, 2048, 83.3, 73.1), (96, 64, 2048, 90.9, 73.2), (32, 192, 2048, 90.8, 71.8),
    (4, 128, 2048, 34.3, 71.2), (16, 128, 2048, 42.9, 71.9), (32, 128, 2048, 54.2, 71.6),
    (64, 64, 2048, 58.7, 72.6), (16, 128, 448, 21.4, 22.3), (4, 128, 384, 18.6, 20.2),
    (20, 128, 768, 28.3, 32.1), (28, 128, 1024, 35.2, 40.0), (32, 128, 1024, 37.2, 39.9),
    (10, 192, 512, 22.7, 24.2), (128 + 16, 128, 448, 21.4, 22.3), (28, 128, 832, 36.4, 34.0),
    (32, 128, 832, 38.0, 34.0), (64, 64, 832, 38.5, 34.3), (21, 192, 832, 37.7, 34.2),
    (32, 128, 896, 38.1, 36.0), (24, 128, 704, 29.6, 30.2), (24, 128, 1024, 34.4, 39.8),
])
def test_the_faster_form_is_taken(rows, heads, selected, split, wide):
    if _native.torch.cuda.is_available():
        pytest.skip("the plan follows the visible device's CU count")
    assert _needs_workspace(rows, heads, selected) == (split < wide)
