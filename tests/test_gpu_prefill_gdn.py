"""The gated delta rule's prefill in chunks of 32 tokens, at the edges of its chunks and head groups: one gated-delta layer of
small shapes against the CPU oracle from the same inputs, with a number of value heads per key head that leaves the last
group of four partly empty, one, and more than one group.

The oracle runs the rule in pieces of up to 128 tokens in float32, this build in pieces of 32; both are float32 sums in
another order, so outputs differ where a bf16 or e5m2 rounding falls the other way. An e5m2 step at one of n inputs of a
projection is an eighth to a quarter of that input, about 0.2 / sqrt(n) of the output: 6e-3 at 1,024 inputs. Held: 6e-2 per
token (several such steps in each of three projections), 2e-2 over all tokens, 1e-2 for the states.
"""

from __future__ import annotations

from dataclasses import replace

import pytest
import torch

from oracle import model as om
from qwen38_amd import synth
from qwen38_amd.config import LINEAR, tiny_config, with_layers
from qwen38_amd.generate import prefill_inputs
from qwen38_amd.steps import Engine, StepGraph
from scenario import oracle_weights


@pytest.mark.gpu
@pytest.mark.parametrize(
    "key_heads, value_heads, chunk, start, n_valid",
    [
        (4, 8, 32, 0, 1),  # one token of one chunk, a new row
        (4, 8, 32, 32, 32),
        (8, 8, 64, 64, 33),  # one value head per key head; the padding starts inside the second chunk
        (2, 8, 96, 32, 95),  # four value heads per key head: one whole group
        (1, 8, 128, 96, 128),  # eight: two groups
        (8, 24, 160, 5, 129),  # three, as the 27B layer
    ],
)
def test_a_chunk_of_the_delta_rule(gpu, key_heads, value_heads, chunk, start, n_valid):
    cfg = replace(with_layers(tiny_config(1), (LINEAR,)), linear_num_key_heads=key_heads, linear_num_value_heads=value_heads)
    values = dict((sp.name, v) for sp, v in synth.make_all(synth.model_specs(cfg, mtp=False, head=False), 4))
    layers, _, _ = oracle_weights({**values, **dict((sp.name, v) for sp, v in synth.make_all(synth.head_specs(cfg), 4))}, cfg)
    batch, slot = 2, 1
    engine = Engine(cfg, batch, 1, 512, mtp=False, prefill_chunk=chunk)
    engine.load(values.items())
    st = synth.gdn_states(cfg, batch, 1, 4, "s")
    engine.set_gdn(0, st)
    x = synth.hidden_states((1, chunk, cfg.hidden_size), 4, "x")
    pi = prefill_inputs(cfg, slot, start, n_valid, chunk, torch.bfloat16)
    got = StepGraph(engine)(inputs_embeds=x, **pi).float().cpu()[0, :n_valid]
    mine = {k: engine.gdn_state(0)[k].float().cpu() for k in ("recurrent_state", "conv_state")}
    before = {k: st[k].clone() for k in mine}
    # The oracle's pieces are as long as the call allows and must divide it: a multiple of 32 tokens, in pieces of 32.
    om_chunk, om.DELTA_CHUNK = om.DELTA_CHUNK, 32
    try:
        want = om.step_prefill(cfg, [layers[0]], [st], x, pi["cos"], pi["sin"], pi["slot"], pi["start"], pi["n_valid"]).float()[0, :n_valid]
    finally:
        om.DELTA_CHUNK = om_chunk
    per_token = (got - want).norm(dim=-1) / want.norm(dim=-1)
    whole = float((got - want).norm() / want.norm())
    print(f"all tokens {whole:.2e}, worst token {float(per_token.max()):.2e}")
    assert whole <= 2e-2 and float(per_token.max()) <= 6e-2
    for key, value in mine.items():
        ref = st[key].float()
        err = float((value[slot] - ref[slot]).norm() / ref[slot].norm())
        print(f"{key} {err:.2e}")
        assert err <= 1e-2
        assert torch.equal(value[1 - slot], before[key][1 - slot].float())
