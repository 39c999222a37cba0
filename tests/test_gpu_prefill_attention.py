"""The prefill attention over ranges of positions: chunks whose 64-token tiles, 32-position sub-blocks, ranges and blocks of
2048 end at every kind of edge, one attention layer of the small model against the CPU oracle from the same inputs.

The layer rounds the inputs of its out, gate/up and down projections to e5m2, so a last-bit difference before one (the
float32 sums' order) moves the few inputs next to a boundary by an e5m2 step, an eighth to a quarter of the value. d of n inputs moved shift
a projection's output by about 0.2 sqrt(d / n): one of 1,024 by 6e-3, ten by 2e-2, so a token may be off by 1e-2 with a
single flip and by 6e-2 with several in each of the three (the layer tests measure up to 1e-1 at the 27B widths). Held:
6e-2 per token and, over all tokens, the 2e-2 of the layer outputs. That sees a wrong weight or token, and a wrong position
where there are few; over a long context one sub-block is a hundredth of a row, and the layer of probe_layer.py shows
each position by itself.
"""

from __future__ import annotations

import pytest
import torch

from oracle import model as om
from probe_layer import probe_config, probe_hidden, probe_rows, probe_weights
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


def probe_engine(heads, kv, seq, chunk, v, v_scale):
    """The probe layer with zero keys and values v in its cache."""
    cfg = probe_config(heads)
    engine = Engine(cfg, 1, 1, seq, mtp=False, prefill_chunk=chunk, kv_cache_format=kv)
    engine.load(probe_weights(cfg).items())
    k = torch.zeros_like(v)
    if kv == "fp8":
        scales = torch.ones(1, dtype=torch.bfloat16), torch.tensor([v_scale], dtype=torch.bfloat16)
        engine.set_kv_scales(0, *scales)
        k, v = (encode_kv(t, s) for t, s in zip((k, v), scales))
    engine.set_kv(0, k, v)
    return cfg, engine


@pytest.mark.gpu
@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize(
    "heads, seq, chunk, start",
    [
        (8, 4160, 32, 4096),  # each block in parts
        (8, 8256, 64, 4100),  # a third cached block of four positions
        (8, 10240, 512, 8192),  # a block per item
        (32, 8256, 1024, 4100),  # two
        (32, 17408, 1024, 16384),  # five
    ],
)
def test_each_block_is_rounded_to_bf16(gpu, kv, heads, seq, chunk, start):
    """blocked_attention rounds each block's weights x V to bf16. With equal scores every weight is one, so values of 2^14,
    one of them 2^15, over the first block sum to 2,049 x 2^14, which rounds to 2,048 x 2^14, and the second block's
    -2^14 cancel that: dim 0 is exactly zero, and 2^14 / (start + t + 1) without the rounding. Dim 1 is one everywhere."""
    v = torch.zeros(1, 2, seq, 256, dtype=torch.bfloat16)
    v[0, 1, :2048, 0], v[0, 1, 5, 0], v[0, 1, 2048:4096, 0] = 2.0**14, 2.0**15, -(2.0**14)
    v[0, 1, :start, 1] = 256.0
    cfg, engine = probe_engine(heads, kv, seq, chunk, v, 256.0)
    pi = prefill_inputs(cfg, 0, start, chunk, chunk, torch.bfloat16)
    got = probe_rows(StepGraph(engine)(inputs_embeds=probe_hidden(1, chunk, cfg), **pi))[0, :, 1].cpu()
    share = start / (start + 1 + torch.arange(chunk).float())
    print(f"dim 0 {float(got[:, 0].abs().max())}, unrounded {heads / 2 * 0.5 * 2.0**14 / start:.2f}", flush=True)
    assert bool((got[:, 0] == 0).all())
    assert bool(((got[:, 1] / (heads / 2 * 0.5 * 256.0 * share) - 1).abs() <= 0.13).all())  # e5m2: an eighth


@pytest.mark.gpu
@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize(
    "heads, seq, chunk, start",
    [
        (8, 4160, 256, 3001),  # a cached end inside a sub-block, parts of blocks
        (8, 4160, 96, 4064),  # the chunk ends the cache
        (12, 2112, 160, 1920),  # the chunk cut at 2,048; wave tiles of two token groups in a workgroup
        (8, 10240, 256, 8200),
        (32, 6208, 256, 4097),
    ],
)
def test_every_position_counts_once(gpu, kv, heads, seq, chunk, start):
    """With equal scores a row is the mean of the values. 256 probed cached positions (the edges of 32-position sub-blocks,
    of blocks and of the cached range among them) each hold 1.05 x start in a dim of their own: every one shows as the e5m2
    value 0.5 in every head, half of it gated. Each of the chunk's tokens holds 32 in its own dim: seen from itself on."""
    edges = {p for e in range(0, start + 1, 2048) for p in (e - 1, e, e + 31) if 0 <= p < start} | {0, start - 1}
    more = [p for i in range(0, start, 32) for p in (i, min(i + 31, start - 1)) if p not in edges]
    g = torch.Generator().manual_seed(start)
    probes = sorted(edges) + [more[i] for i in torch.randperm(len(more), generator=g).tolist()]
    probes = torch.tensor(list(dict.fromkeys(probes))[:256])
    v = torch.zeros(1, 2, seq, 256, dtype=torch.bfloat16)
    v[0, 1, probes, torch.arange(len(probes))] = 1.05 * start
    cfg, engine = probe_engine(heads, kv, seq, chunk, v, 1.05 * start / 128)
    pi = prefill_inputs(cfg, 0, start, chunk, chunk, torch.bfloat16)
    got = probe_rows(StepGraph(engine)(inputs_embeds=probe_hidden(1, chunk, cfg), **pi))[0].cpu()
    # 0.525 start / (start + t + 1) lies between 0.469 and 0.5625 (the bounds of what rounds to 0.5) for t up to 0.11 start.
    near = torch.arange(chunk) < 0.1 * start
    cached = got[near][:, 1, : len(probes)]
    wrong = (cached != heads / 2 * 0.5).nonzero()
    assert len(wrong) == 0, [(int(t), int(probes[i]), float(cached[t, i])) for t, i in wrong[:5]]
    t = torch.arange(chunk).float()
    mine, sees = got[:, 0, :chunk], torch.ones(chunk, chunk).tril().bool()
    assert bool((mine[~sees] == 0).all())
    # 16 / (start + t + 1) a head within e5m2's eighth (and e4m3's sixteenth for the own values through an FP8 cache).
    off = (mine / (heads / 2 * 16 / (start + 1 + t)).unsqueeze(-1) - 1).abs()[sees]
    assert float(off.max()) <= (0.13 if kv == "bf16" else 0.2)
