"""Gated products of 9 to 128 rows by the kernel that shares the activations, in tiles of eight gate and eight up rows and of
either (csrc/gemm_bf16.hip), against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# rows: ends of the blocks of 16; outputs: fewer tiles than compute units, one tile to some and five to all, and six (tiles of
# either); K: two k-steps less than a chunk of ten, one chunk, a chunk and a part
@pytest.mark.parametrize("m", [9, 16, 17, 48, 49, 64, 65, 128])
@pytest.mark.parametrize("n,k", [(48, 512), (4112, 640), (10240, 704), (10256, 128)])
def test_gated_rows(m, n, k):
    from ctypes import c_float, c_int

    from qwen3_runtime_amd.ops.hip import BF16, HipOps, _ptr, _stream

    ops, g = HipOps(), torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(2 * n, k, generator=g) * k ** -0.5).to(torch.bfloat16).cuda()
    scale = torch.rand(m, generator=g).cuda()
    sums = x.double() @ w.double().T
    off = (x.double().abs() @ w.double().abs().T) * (k + 16) * 2.0 ** -24 + sums.abs() * 2.0 ** -8  # the sums' own, and rounded to bfloat16
    gate, up = sums.split(n, 1)
    gate_off, up_off = off.split(n, 1)
    want = gate * torch.sigmoid(gate) * up
    allowed = 1.1 * gate_off * (up.abs() + up_off) + gate.abs() * up_off + want.abs() * 2.0 ** -7  # silu's slope is at most 1.1
    for rows in (None, scale):
        out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
        ops._check(ops.lib, ops.lib.qrt_gated_gemm_bf16(_ptr(x), _ptr(w), _ptr(out), BF16, c_int(m), c_int(n), c_int(k), c_int(1), c_int(0),
                                                        c_float(0.0), _ptr(rows), _stream()))
        by = 1.0 if rows is None else rows.double()[:, None]
        assert ((out.double() - want * by).abs() <= allowed * by).all()
