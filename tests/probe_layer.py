"""A full-attention layer of the small model's shapes whose output shows its attention value by value: every query is 16 in
dim 64 and zero elsewhere (so a key scores its own dim 64), the step's own keys are zero, sigmoid(gate) is a half, the MLP
adds nothing, and output 256 v + d is the sum over the query heads of KV head v of dim d of their rows. Token t of a row
is one-hot (feature 512 + t), and its own value is 32 in dim t of KV head 0, zero in KV head 1."""

from __future__ import annotations

from dataclasses import replace

import torch

from qwen38_amd import synth
from qwen38_amd.config import FULL, tiny_config, with_layers
from qwen38_amd.quant import quantize_e4m3


def probe_config(query_heads: int = 8):
    return replace(with_layers(tiny_config(1), (FULL,)), num_attention_heads=query_heads)


def probe_weights(cfg) -> dict:
    hidden, hd, hq, hkv = cfg.hidden_size, cfg.head_dim, cfg.num_attention_heads, cfg.num_key_value_heads
    assert (hidden, hd, hkv) == (1024, 256, 2)
    q = torch.zeros(hq, 2, hd, hidden)
    q[:, 0, 64] = 1.0
    v = torch.zeros(hkv, hd, hidden)
    v[0, torch.arange(hd), 512 + torch.arange(hd)] = 1.0
    o = torch.zeros(hidden, hq, hd)
    for h in range(hq):
        o[h // (hq // hkv) * hd + torch.arange(hd), h, torch.arange(hd)] = 1.0
    made = {"q_proj": q.reshape(-1, hidden), "v_proj": v.reshape(-1, hidden), "o_proj": o.reshape(hidden, -1)}
    values = {}
    for sp in synth.model_specs(cfg, mtp=False, head=False):
        w = made.get(sp.name.rsplit(".", 1)[-1], torch.zeros(sp.shape))
        values[sp.name] = quantize_e4m3(w) if sp.kind == "fp8" else w.to(torch.bfloat16)
    return values


def probe_hidden(rows: int, tokens: int, cfg) -> torch.Tensor:
    x = torch.zeros(rows, tokens, cfg.hidden_size)
    x[:, torch.arange(tokens), 512 + torch.arange(tokens) % 512] = 1.0
    return x.to(torch.bfloat16)


def probe_rows(out: torch.Tensor) -> torch.Tensor:
    """The layer's output as [..., KV head, dim]: the heads' summed attention rows times a half."""
    return out[..., :512].float().reshape(*out.shape[:-1], 2, 256)
