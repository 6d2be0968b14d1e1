"""Sparse MLA takes an ``out`` that is 8-byte aligned: no store of the kernels
may be compiled for more, and such an output has the bits of an aligned one."""

import re
import shutil
import subprocess

import pytest

from cxldsagr_amd.csrc import build

SCALE = 576**-0.5


@pytest.mark.skipif(shutil.which("hipcc") is None and not build.Path("/opt/rocm/bin/hipcc").exists(),
                    reason="needs hipcc")
def test_stores_of_out_claim_no_more_than_eight_bytes(tmp_path):
    source, ir = build.HERE / "sparse_mla.hip", tmp_path / "sparse_mla.ll"
    subprocess.run([build.hipcc(), *build.FLAGS, *build.SOURCE_FLAGS[source.name], "-w",
                    "--cuda-device-only", "-S", "-emit-llvm", str(source), "-o", str(ir)],
                   check=True, capture_output=True)
    # The kernels whose only global stores are those of `out`.
    claims, kernel = {}, ""
    for line in ir.read_text().splitlines():
        if line.startswith("define"):
            kernel = next((k for k in ("sparse_mla_fwd", "mla_values") if k in line), "")
        elif kernel and re.match(r"\s*store .*addrspace\(1\)", line):
            claims.setdefault(kernel, set()).add(int(re.search(r"align (\d+)", line)[1]))
    assert set(claims) == {"sparse_mla_fwd", "mla_values"}
    assert max(max(c) for c in claims.values()) <= 8, claims


# The wide form, the split form (with 64 and with 128 dims per work-group), both.
@pytest.mark.gpu
@pytest.mark.parametrize("rows,heads,selected", [(3, 64, 100), (2, 128, 2048), (32, 128, 1024),
                                                 (130, 128, 600)])
@pytest.mark.parametrize("fp8", [True, False])
def test_an_eight_byte_aligned_out_has_the_same_bits(gpu, rows, heads, selected, fp8):
    import torch

    from cxldsagr_amd import _native, attention

    gen = torch.Generator(device=gpu).manual_seed(rows)
    tokens = 3000
    kv = torch.randn(tokens, 576, generator=gen, device=gpu).bfloat16()
    q = torch.randn(rows, heads, 576, generator=gen, device=gpu).bfloat16()
    ids = torch.randint(-1, tokens, (rows, selected), generator=gen, device=gpu).int()
    flat = torch.full((rows * heads * 512 + 8,), 7.0, dtype=torch.bfloat16, device=gpu)
    out = flat[4:-4].view(rows, heads, 512)
    assert out.data_ptr() % 16 == 8
    if fp8:
        pages = (tokens + 63) // 64
        table = torch.randperm(pages, generator=gen, device=gpu).int()
        cache = torch.zeros(pages, 64, 656, dtype=torch.uint8, device=gpu)
        attention.pack_kv_fp8(kv, cache, table)
        attention.sparse_mla_fp8_paged(q, cache, table, ids, SCALE, n_tokens=tokens, _out=out)
        want = attention.sparse_mla_fp8_paged(q, cache, table, ids, SCALE, n_tokens=tokens)
    else:
        workspace = attention._workspace(q, selected)
        _native.call("dsa_sparse_mla_bf16_ws", _native.ptr(q), rows, heads, _native.ptr(kv), tokens,
                     _native.ptr(ids), selected, SCALE, _native.ptr(out), _native.ptr(workspace),
                     0 if workspace is None else workspace.numel(), _native.stream_of(gpu))
        want = attention.sparse_mla(q, kv, ids, SCALE)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    assert bool((flat[:4] == 7.0).all()) and bool((flat[-4:] == 7.0).all())
