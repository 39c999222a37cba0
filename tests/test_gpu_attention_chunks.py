"""The chunked attention where the chunk a wave scores is longer than its shortest: 256 and 512 positions (a batch with
enough (row, KV head) pairs over a long cache), at 6, 24 and 48 query rows per KV head, with contexts at the edges of
chunks and of blocks of 16 positions, bf16 and FP8 caches.

Four rows, each 64 times in the batch: the four against the oracle, per row within the 2e-2 that one layer of the MTP
step is held to (bf16 stages; a wrong chunk, maximum or position is far outside it), and every copy, which other
workgroups compute, bit for bit its first."""

from __future__ import annotations

import dataclasses

import pytest
import torch

from oracle import model as om
from qwen38_amd import synth
from qwen38_amd.config import tiny_config
from qwen38_amd.generate import mtp_step_inputs
from qwen38_amd.quant import encode_kv
from qwen38_amd.steps import Engine, MTPStep
from scenario import oracle_weights

COPIES = 64


@pytest.mark.gpu
@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize(
    "k, s, context",
    [
        (1, 6144, [6142, 1537, 2048, 1039]),  # chunks of 512; decode's query rows
        (4, 6144, [6139, 2561, 5632, 1100]),
        (4, 3104, [3099, 1281, 1040, 2047]),  # chunks of 256, the cache's end inside one
        (8, 3104, [3095, 1793, 1281, 2559]),  # two query tiles
    ],
)
def test_long_chunks_match_the_oracle(gpu, k, s, context, kv):
    print(f"k {k} s {s} kv {kv}", flush=True)
    cfg = dataclasses.replace(tiny_config(1), num_attention_heads=12)
    rows, seed = len(context), 23
    values = dict((sp.name, v) for sp, v in synth.make_all(synth.model_specs(cfg), seed))
    _, mtp_w, _ = oracle_weights(values, cfg)
    engine = Engine(cfg, rows * COPIES, k, s, mtp=True, kv_cache_format=kv)
    engine.load(values.items())
    mst = synth.kv_states(cfg, rows, s, context, seed, "mtp")
    if kv == "fp8":
        ks, vs = synth.kv_scales(cfg, seed, "mtp")
        mst = {"k_cache": encode_kv(mst["k_cache"], ks), "v_cache": encode_kv(mst["v_cache"], vs), "k_scale": ks, "v_scale": vs}
        engine.set_kv_scales(engine.mtp_layer, ks, vs)
    many = lambda t: t.cuda().repeat(COPIES, *[1] * (t.dim() - 1))  # noqa: E731
    engine.set_kv(engine.mtp_layer, many(mst["k_cache"]), many(mst["v_cache"]))
    mi = mtp_step_inputs(cfg, context, k, s, torch.bfloat16, [True] * rows)
    mi["position"] = torch.as_tensor(context, dtype=torch.int32)
    hidden = synth.hidden_states((rows, k, cfg.hidden_size), seed, "attn.hidden")
    ids = torch.randint(0, cfg.vocab_size, (rows, k), generator=torch.Generator().manual_seed(seed))
    embeds = values["embed_tokens"][ids]

    out = MTPStep(engine)(hidden=many(hidden), inputs_embeds=many(embeds), **{n: many(t) for n, t in mi.items()}).cpu()
    want = om.mtp_forward(cfg, mtp_w, mst, hidden, embeds, mi["cos"], mi["sin"], mi["position"], mi["active"])
    out = out.reshape(COPIES, *want.shape)
    assert torch.equal(out, out[:1].expand_as(out))
    err = (out[0].float() - want.float()).flatten(1).norm(dim=1) / want.float().flatten(1).norm(dim=1)
    print(f"row_rel {err.tolist()}", flush=True)
    assert float(err.max()) <= 2e-2
