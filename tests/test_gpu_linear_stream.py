"""The weight-streaming projection (up to 128 tokens) where its schedule can go wrong: K ranges shorter than a workgroup's
waves, tiles left over beyond a multiple of the CUs split in K, four-wave workgroups, ragged tokens; e4m3 and MXFP4.

Held against float64: half a bf16 ulp of the result for its rounding, plus 2^-20 of sum |x w| for the float32 sums (as the
projection tests allow; measured about 1e-8). Finishing the split tiles by recomputing their parts gives the same bits, in
every form that splits."""

from __future__ import annotations

import ctypes

import pytest
import torch

from qwen38_amd import ext
from qwen38_amd.quant import dequantize_e4m3, dequantize_mxfp4, quantize_e4m3, quantize_mxfp4, round_e5m2


def inputs(rows, k, n, mx):
    g = torch.Generator(device="cuda").manual_seed(rows * 31 + k + n)
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    w[:, :32] *= 50.0  # groups with different scales
    x = torch.randn(rows, k, generator=g, device="cuda").to(torch.bfloat16)
    packed = quantize_mxfp4(w) if mx else quantize_e4m3(w)
    return x, packed, (dequantize_mxfp4 if mx else dequantize_e4m3)(*packed).double()


def check(got, x, wd):
    xq = round_e5m2(x).double()
    exact, bound = xq @ wd.T, (xq.abs() @ wd.abs().T) * 2.0**-20
    ulp = torch.exp2(torch.floor(torch.log2(exact.abs().clamp_min(2.0**-126))) - 7)
    off = (got.double() - exact).abs() - bound
    assert bool((off <= ulp * 0.5).all()), float((off / ulp).max())


@pytest.mark.gpu
@pytest.mark.parametrize("mx", [False, True])
@pytest.mark.parametrize(
    "rows, k, n",
    [
        (1, 256, 256),  # 4 tiles of 4 K-steps: most waves have none
        (32, 768, 512),  # 12 K-steps over 8 waves
        (33, 4352, 256),  # 4 tiles split 4 ways
        (5, 1280, 16640),  # 256 whole tiles and 4 left over
        (64, 512, 16640),
        (17, 320 * 4, 33280),  # 520 tiles: four-wave workgroups, 8 left over
        (61, 17408, 5120),  # 80 tiles split 3 ways
        (65, 256, 256),  # two blocks of 64 tokens
        (100, 1280, 16640),  # 520 tiles, not eight of a block at a time: four-wave workgroups, 8 left over
        (128, 17408, 5120),
        (97, 5120, 4864),  # 152 tiles
    ],
)
def test_streamed_projection(gpu, rows, k, n, mx):
    x, packed, wd = inputs(rows, k, n, mx)
    if mx:
        check(ext.mxfp4_linear(x, *ext.pack_weight_fp4(*packed), n), x, wd)
        return
    tiles, scales = ext.pack_weight(*packed)
    got = ext.fp8_linear(x, tiles, scales, n)
    check(got, x, wd)
    again = ext.fp8_linear_mfma(x, tiles, scales, n, "bf16", recompute=True)
    assert torch.equal(got.view(torch.int16), again.view(torch.int16))
    scratch = ext.linear_scratch(rows, k)
    for _ in range(2):  # the arrival counters are zero again after a call
        assert torch.equal(ext.fp8_linear(x, tiles, scales, n, scratch), got)


@pytest.mark.gpu
@pytest.mark.parametrize("rows, k, inter", [(1, 256, 256), (32, 1024, 16640), (20, 1280, 128 * 17)])
def test_streamed_gate_up(gpu, rows, k, inter):
    """The SwiGLU pair against the plain projection of the same interleaved weight: its own roundings applied to it."""
    x, packed, _ = inputs(rows, k, 2 * inter, False)
    tiles, scales = ext.pack_weight(*packed)
    from qwen38_amd.steps import act_tiles_to_rows

    got = act_tiles_to_rows(ext.mlp_up(x, rows, k, tiles, scales, inter), 32, inter)[:rows].float()
    y = ext.fp8_linear(x, tiles, scales, 2 * inter).reshape(rows, inter // 32, 2, 32)
    gate, up = y[:, :, 0].reshape(rows, inter), y[:, :, 1].reshape(rows, inter)
    want = round_e5m2(gate * torch.sigmoid(gate) * up).float()
    # The sums are the same numbers in both, but for tiles split differently (their float32 sums, and so a bf16 rounding,
    # may fall the other way) and the sigmoid's last bit: an e5m2 step, a quarter of the value at most, at few values.
    assert float((got != want).float().mean()) <= 2e-3
    assert bool(((got - want).abs() <= 0.26 * want.abs() + 2.0**-16).all())


@pytest.mark.gpu
@pytest.mark.parametrize("k, n", [(256, 256), (3072, 1024), (5120, 4352)])
def test_streamed_sums_of_128_tokens(gpu, k, n):
    """The float32 sums (the split-K form's, one part): 2^-20 of sum |x w|."""
    x, packed, wd = inputs(128, k, n, False)
    xq = round_e5m2(x).double()
    off = (ext.fp8_linear_f32(x, *ext.pack_weight(*packed), n).double() - xq @ wd.T).abs()
    assert bool((off <= (xq.abs() @ wd.abs().T) * 2.0**-20).all())


class GemmArgs(ctypes.Structure):
    """csrc/kernels.h: the launcher's argument block."""

    _fields_ = (
        [(n, ctypes.c_void_p) for n in ("w", "ws", "act")] + [(n, ctypes.c_int) for n in ("K", "N", "T", "Tpad")]
        + [("out0", ctypes.c_void_p), ("ld0", ctypes.c_int), ("n0", ctypes.c_int), ("out1", ctypes.c_void_p), ("ld1", ctypes.c_int)]
        + [("part", ctypes.c_void_p), ("fix", ctypes.c_void_p), ("fix_floats", ctypes.c_size_t), ("counters", ctypes.c_void_p)]
        + [(n, ctypes.c_int) for n in ("counters_n", "cus", "splits_max", "recompute", "splits", "w4", "f8")]
    )


@pytest.mark.gpu
@pytest.mark.parametrize("mx", [False, True])
@pytest.mark.parametrize("rows, epi", [(17, 0), (64, 0), (100, 0), (17, 1)])
def test_recomputed_parts_give_the_same_bits(gpu, rows, epi, mx):
    """Finishing a split tile from its parts' sums and by computing them again (as when they ran on another XCD): bf16
    outputs and the SwiGLU pair, e4m3 and MXFP4. 68 tiles of 64 features, split three ways (136 in blocks of 64 tokens; of
    which, at 100 CUs, 36 are left over and split in two)."""
    k, n = 4352, 4352
    x, packed, _ = inputs(rows, k, n, mx)
    tiles, scales = (ext.pack_weight_fp4 if mx else ext.pack_weight)(*packed)
    scratch = ext.linear_scratch(rows, k)
    (ext.mxfp4_linear if mx else ext.fp8_linear)(x, tiles, scales, n, scratch)
    tpad = 32 if rows <= 32 else 64 if rows <= 64 else 128
    base, counters = scratch.data_ptr(), scratch.data_ptr() + tpad * k
    outs = [torch.zeros(rows, n, dtype=torch.bfloat16, device="cuda") if epi == 0 else torch.zeros(tpad * n // 2, dtype=torch.uint8, device="cuda") for _ in range(2)]
    launch = gpu["_Z8q38_gemmRK8GemmArgsiPiP12ihipStream_t"]
    torch.cuda.synchronize()
    for recompute, out in enumerate(outs):
        a = GemmArgs(w=tiles.data_ptr(), ws=scales.data_ptr(), act=base, K=k, N=n, T=rows, Tpad=tpad, out0=out.data_ptr(), ld0=n, n0=n,
                     fix=counters + 65536 * 8, fix_floats=2 * 256 * 65536, counters=counters, counters_n=65536, cus=100 if rows > 64 else 256,
                     recompute=recompute, w4=int(mx))
        assert launch(ctypes.byref(a), epi, None, ctypes.c_void_p(0)) == 0
    torch.cuda.synchronize()
    assert bool((outs[0] != 0).any()) and torch.equal(outs[0].view(torch.uint8), outs[1].view(torch.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [17, 64, 100])
@pytest.mark.parametrize("cus", [8, 20, 36, 250, 255, 304])
def test_any_number_of_cus(gpu, rows, cus):
    """The schedule asks for no multiple of 8 compute units (a partition or another part of the chip): bf16 outputs with
    tiles left over and split, and float32 sums."""
    k, n = 4352, 4352
    x, packed, wd = inputs(rows, k, n, False)
    tiles, scales = ext.pack_weight(*packed)
    scratch = ext.linear_scratch(rows, k)
    ext.fp8_linear(x, tiles, scales, n, scratch)  # leaves x's tiles at the start of the scratch, its counters zero
    tpad = 32 if rows <= 32 else 64 if rows <= 64 else 128
    base, counters = scratch.data_ptr(), scratch.data_ptr() + tpad * k
    out = torch.empty(rows, n, dtype=torch.bfloat16, device="cuda")
    part = torch.empty(tpad, n, device="cuda")
    a = GemmArgs(w=tiles.data_ptr(), ws=scales.data_ptr(), act=base, K=k, N=n, T=rows, Tpad=tpad, out0=out.data_ptr(), ld0=n, n0=n,
                 part=part.data_ptr(), fix=counters + 65536 * 8, fix_floats=2 * 256 * 65536, counters=counters, counters_n=65536, cus=cus,
                 splits_max=1)
    launch = gpu["_Z8q38_gemmRK8GemmArgsiPiP12ihipStream_t"]
    torch.cuda.synchronize()
    for epi in (0, 2):
        assert launch(ctypes.byref(a), epi, None, ctypes.c_void_p(0)) == 0
    torch.cuda.synchronize()
    check(out, x, wd)
    xq = round_e5m2(x).double()
    assert bool(((part[:rows].double() - xq @ wd.T).abs() <= (xq.abs() @ wd.abs().T) * 2.0**-20).all())


@pytest.mark.gpu
def test_streamed_parts_of_96_tokens_match_the_oracle(gpu):
    """The MTP step of 24 rows x 4 tokens, whose projections are summed from several workgroups' parts: per row within the
    2e-2 that the step's one layer is held to."""
    from oracle import model as om
    from qwen38_amd import synth
    from qwen38_amd.config import tiny_config
    from qwen38_amd.generate import mtp_step_inputs
    from qwen38_amd.steps import Engine, MTPStep
    from scenario import oracle_weights

    cfg, b, k, s, seed = tiny_config(1), 24, 4, 128, 29
    context = [(7 * r) % 120 for r in range(b)]
    values = dict((sp.name, v) for sp, v in synth.make_all(synth.model_specs(cfg), seed))
    engine = Engine(cfg, b, k, s, mtp=True)
    engine.load(values.items())
    mst = synth.kv_states(cfg, b, s, context, seed, "mtp")
    engine.set_kv(engine.mtp_layer, mst["k_cache"], mst["v_cache"])
    mi = mtp_step_inputs(cfg, context, k, s, torch.bfloat16, [True] * b)
    mi["position"] = torch.as_tensor(context, dtype=torch.int32)
    hidden = synth.hidden_states((b, k, cfg.hidden_size), seed, "stream.hidden")
    embeds = values["embed_tokens"][torch.randint(0, cfg.vocab_size, (b, k), generator=torch.Generator().manual_seed(seed))]
    out = MTPStep(engine)(hidden=hidden, inputs_embeds=embeds, **mi).cpu().float().flatten(1)
    want = om.mtp_forward(cfg, oracle_weights(values, cfg)[1], mst, hidden, embeds, mi["cos"], mi["sin"], mi["position"], mi["active"])
    want = want.float().flatten(1)
    assert float(((out - want).norm(dim=1) / want.norm(dim=1)).max()) <= 2e-2
