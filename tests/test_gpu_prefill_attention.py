"""The prefill attention over ranges of positions: chunks whose 64-token tiles, 32-position sub-blocks, ranges and blocks of
2048 end at every kind of edge, one attention layer of the small model against the CPU oracle from the same inputs.

The layer rounds the inputs of its out, gate/up and down projections to e5m2, so a last-bit difference before one (the
float32 sums' order; over several blocks the sums are not rounded to bf16 at each block's end, as the reference's are)
moves the few inputs next to a boundary by an e5m2 step, an eighth to a quarter of the value. d of n inputs moved shift
a projection's output by about 0.2 sqrt(d / n): one of 1,024 by 6e-3, ten by 2e-2, so a token may be off by 1e-2 with a
single flip and by 6e-2 with several in each of the three (the layer tests measure up to 1e-1 at the 27B widths). Held:
6e-2 per token and, over all tokens, the 2e-2 of the layer outputs. A wrong position, weight or token moves whole rows by
far more.
"""

from __future__ import annotations

import pytest
import torch

from oracle import model as om
from qwen38_amd import synth
from qwen38_amd.config import FULL, tiny_config, with_layers
from qwen38_amd.generate import prefill_inputs
from qwen38_amd.quant import encode_kv
from qwen38_amd.steps import Engine, StepGraph
from scenario import oracle_weights


@pytest.mark.gpu
@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize(
    "seq, chunk, start, n_valid",
    [
        (64, 32, 0, 1),  # one sub-block, one token
        (512, 96, 0, 96),  # half a tile at the end, no cached positions
        (512, 64, 37, 60),  # a cached end inside a sub-block
        (2112, 160, 1920, 160),  # cached positions and chunk in two blocks, the chunk cut at 2048
        (4160, 256, 3001, 250),  # two cached blocks, one and a half thousand positions between cache end and chunk block
        (2048, 128, 1900, 128),  # the cache a whole number of blocks
    ],
)
def test_a_chunk_sees_every_position_it_should(gpu, kv, seq, chunk, start, n_valid):
    cfg = with_layers(tiny_config(1), (FULL,))
    values = dict((sp.name, v) for sp, v in synth.make_all(synth.model_specs(cfg, mtp=False, head=False), 3))
    layers, _, _ = oracle_weights({**values, **dict((sp.name, v) for sp, v in synth.make_all(synth.head_specs(cfg), 3))}, cfg)
    batch, slot = 2, 1
    engine = Engine(cfg, batch, 1, seq, mtp=False, prefill_chunk=chunk, kv_cache_format=kv)
    engine.load(values.items())
    st = synth.kv_states(cfg, batch, seq, [0, start], 3, "kv")
    if kv == "fp8":
        ks, vs = synth.kv_scales(cfg, 3, "kv")
        st = {"k_cache": encode_kv(st["k_cache"], ks), "v_cache": encode_kv(st["v_cache"], vs), "k_scale": ks, "v_scale": vs}
        engine.set_kv_scales(0, ks, vs)
    engine.set_kv(0, st["k_cache"], st["v_cache"])
    x = synth.hidden_states((1, chunk, cfg.hidden_size), 3, "x")
    pi = prefill_inputs(cfg, slot, start, n_valid, chunk, torch.bfloat16)
    got = StepGraph(engine)(inputs_embeds=x, **pi).float().cpu()[0, :n_valid]
    want = om.step_prefill(cfg, [layers[0]], [st], x, pi["cos"], pi["sin"], pi["slot"], pi["start"], pi["n_valid"]).float()[0, :n_valid]
    per_token = (got - want).norm(dim=-1) / want.norm(dim=-1)
    whole = float((got - want).norm() / want.norm())
    print(f"all tokens {whole:.2e}, worst token {float(per_token.max()):.2e}")
    assert whole <= 2e-2 and float(per_token.max()) <= 6e-2
