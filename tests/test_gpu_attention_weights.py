"""The softmax weights of the chunked and the prefill attention at the small end of float32, where the two exponentials that
form them must not lose values: positions 88 below the row's maximum weigh e^-88 = 6.05e-39, below 2^-126, and with
values of 3e35 they are all of the row's output (the other positions' values are zero)."""

from __future__ import annotations

import math

import pytest
import torch

from probe_layer import probe_config, probe_hidden, probe_rows, probe_weights
from qwen38_amd.generate import batch_step_inputs, prefill_inputs
from qwen38_amd.steps import Engine, StepGraph


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["decode", "prefill"])
def test_weights_below_the_smallest_normal_number(gpu, form):
    cfg, seq, start, chunk = probe_config(), 2048, 1500, 32  # above 1,024 positions decode takes the chunked kernels
    engine = Engine(cfg, 1, 1, seq, mtp=False, prefill_chunk=chunk)
    engine.load(probe_weights(cfg).items())
    k, v = (torch.zeros(1, 2, seq, 256, dtype=torch.bfloat16) for _ in range(2))
    k[:, :, 1:start, 64] = -88.0  # position 0 scores 0: the maximum from the first block on
    v[:, :, 1:start] = 3e35
    engine.set_kv(0, k, v)
    step = StepGraph(engine)
    if form == "decode":
        out = step(inputs_embeds=probe_hidden(1, 1, cfg), **batch_step_inputs(cfg, [start], seq, torch.bfloat16))[0]
    else:
        out = step(inputs_embeds=probe_hidden(1, chunk, cfg), **prefill_inputs(cfg, 0, start, chunk, chunk, torch.bfloat16))[0]
    got = probe_rows(out)[:, 1].cpu()
    # The step's own tokens score 0 too: token t's weights sum to t + 2. Four heads, each times a half.
    want = 4 * 0.5 * (start - 1) * math.exp(-88.0) * float(v[0, 0, 1, 0]) / (2 + torch.arange(len(got)).float())
    off = (got / want.unsqueeze(-1) - 1).abs().max()
    print(f"{form}: token 0 {float(got[0].min()):.4f} .. {float(got[0].max()):.4f}, expected {float(want[0]):.4f}, off {float(off):.3f}")
    # o_proj's inputs round to e5m2 (an eighth); a bf16 weight below 2^-126 is a multiple of 2^-133, 1 % here.
    assert float(off) <= 0.125 + 0.02
