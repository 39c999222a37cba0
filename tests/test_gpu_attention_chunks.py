"""The chunked attention where the chunk a wave scores is longer than its shortest: 256 and 512 positions (a batch with
enough (row, KV head) pairs over a long cache), at 6, 24 and 48 query rows per KV head, with contexts at the edges of
chunks and of blocks of 16 positions, bf16 and FP8 caches.

Four rows, each 64 times in the batch: the four against the oracle, per row within the 2e-2 that one layer of the MTP
step is held to (bf16 stages; a wrong chunk or maximum is far outside it), and every copy, which other workgroups
compute, bit for bit its first. A block of 16 positions is a few thousandths of such a row: the layer of probe_layer.py
shows one position of each by itself."""

from __future__ import annotations

import dataclasses

import pytest
import torch

from oracle import model as om
from probe_layer import probe_config, probe_hidden, probe_rows, probe_weights
from qwen38_amd import synth
from qwen38_amd.config import tiny_config
from qwen38_amd.generate import mtp_step_inputs, verify_inputs
from qwen38_amd.quant import encode_kv
from qwen38_amd.steps import Engine, MTPStep, VerifyStep
from scenario import oracle_weights

COPIES = 64


FORMS = [
    (1, 6144, [6142, 1537, 2048, 1039]),  # chunks of 512; decode's query rows
    (4, 6144, [6139, 2561, 5632, 1100]),
    (4, 3104, [3099, 1281, 1040, 2047]),  # chunks of 256, the cache's end inside one
    (8, 3104, [3095, 1793, 1281, 2559]),  # two query tiles
]


@pytest.mark.gpu
@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("k, s, context", FORMS)
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


@pytest.mark.gpu
@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("copies", [1, 64])  # alone: the shortest chunks, several splits of a row
@pytest.mark.parametrize("k, s, context", FORMS)
def test_every_block_counts_once(gpu, k, s, context, copies, kv):
    """With equal scores a row is the mean of the values. One position of each block of 16 (its first, last or another) holds
    1.03 x context in a dim of its own: each shows as the e5m2 value 0.5 in every head, half of it gated. The step's own
    tokens hold 32 each in their own dim: seen from themselves on."""
    print(f"k {k} s {s} copies {copies} kv {kv}", flush=True)
    cfg, rows, heads = probe_config(12), len(context), 12
    engine = Engine(cfg, rows * copies, k, s, mtp=False, kv_cache_format=kv)
    engine.load(probe_weights(cfg).items())
    v = torch.zeros(rows, 2, s, 256, dtype=torch.bfloat16)
    room = [(0, d) for d in range(8, 256)] + [(1, d) for d in range(256)]
    g, probes = torch.Generator().manual_seed(k * s), []
    for r, n in enumerate(context):
        blocks = (n + 15) // 16
        off = torch.randint(0, 16, (blocks,), generator=g)
        at = [min(16 * b + (0, 15, int(off[b]))[b % 3], n - 1) for b in range(blocks)]
        probes.append([(h, d, p) for (h, d), p in zip(room, at)])
        assert len(probes[r]) == blocks
        for h, d, p in probes[r]:
            v[r, h, p, d] = 1.03 * n
    kc = torch.zeros_like(v)
    if kv == "fp8":
        scales = torch.ones(1, dtype=torch.bfloat16), torch.tensor([1.03 * max(context) / 128], dtype=torch.bfloat16)
        engine.set_kv_scales(0, *scales)
        kc, v = (encode_kv(t, sc) for t, sc in zip((kc, v), scales))
    engine.set_kv(0, kc.cuda().repeat(copies, 1, 1, 1), v.cuda().repeat(copies, 1, 1, 1))
    inputs = verify_inputs(cfg, context, k, s, torch.bfloat16, [True] * rows, [0] * rows)
    many = lambda t: t.cuda().repeat(copies, *[1] * (t.dim() - 1))  # noqa: E731
    out = VerifyStep(engine)(inputs_embeds=many(probe_hidden(rows, k, cfg)), **{n: many(t) for n, t in inputs.items()})
    out = out.reshape(copies, rows, k, -1)
    assert torch.equal(out, out[:1].expand_as(out))
    got = probe_rows(out[0]).cpu()
    for r, n in enumerate(context):
        # 0.515 within e4m3's sixteenth (FP8) and bf16's 2^-8 for the weight: between 0.469 and 0.5625, which round to 0.5.
        wrong = [(p, got[r, :, h, d].tolist()) for h, d, p in probes[r] if not bool((got[r, :, h, d] == heads / 2 * 0.5).all())]
        assert not wrong, (n, wrong[:5])
        sees, t = torch.ones(k, k).tril().bool(), torch.arange(k).float()
        mine = got[r, :, 0, :k]
        assert bool((mine[~sees] == 0).all())
        off = (mine / (heads / 2 * 16 / (n + 1 + t)).unsqueeze(-1) - 1).abs()[sees]
        assert float(off.max()) <= (0.14 if kv == "bf16" else 0.2)
