"""The FP4Linear projection where its tiles can go wrong: each tile shape, ragged rows and rows at a tile's edge, feature
counts whose tiles are no multiple of 8, K ranges shorter than a workgroup's waves.

Held against float64 sums of the two parities: half a bf16 spacing (at most 2^-8 of the value) for each of the three
roundings, and 2^-20 of sum |x w| for the float32 sums, as the projection tests allow."""

from __future__ import annotations

import pytest
import torch

from qwen38_amd import ext
from qwen38_amd.quant import dequantize_mxfp4, quantize_mxfp4


@pytest.mark.gpu
@pytest.mark.parametrize(
    "rows, k, n",
    [
        (1, 256, 256),  # 32 x 32 features x tokens; four K-steps over eight waves
        (33, 1280, 768),
        (255, 768, 1024),
        (32, 1024, 16640),  # 64 x 32
        (7, 256, 16640),  # 260 tiles of 64: more than CUs, at few rows
        (50, 2304, 5120),
        (65, 512, 5120),  # 64 x 64
        (100, 320 * 4, 4864),
        (64, 256, 14336),
        (129, 768, 16640),  # 128 x 64; 130 feature tiles
        (200, 5120, 5120),
        (513, 256, 4352),
    ],
)
def test_planes_match_float64(gpu, rows, k, n):
    print(f"rows {rows} k {k} n {n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(rows + k + n)
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    w[:, 32:64] *= 50.0  # blocks with different scales
    x = torch.randn(rows, k, generator=g, device="cuda").to(torch.bfloat16)
    packed = quantize_mxfp4(w)
    wd, xd = dequantize_mxfp4(*packed).double(), x.double()
    got = ext.fp4_linear(x, *ext.pack_weight_fp4(*packed), n).double()
    even, odd = (xd[:, p::2] @ wd[:, p::2].T for p in (0, 1))
    bound = 2.0**-8 * (even.abs() + odd.abs() + got.abs()) + 2.0**-20 * (xd.abs() @ wd.abs().T)
    off = (got - (even + odd)).abs()
    assert bool((off <= bound).all()), float((off / bound).max())
