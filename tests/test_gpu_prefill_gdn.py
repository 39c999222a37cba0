"""The gated delta rule's prefill in chunks of 32 tokens, at the edges of its chunks and head groups: one gated-delta layer of
small shapes against the CPU oracle from the same inputs, with a number of value heads per key head that leaves the last
group of four partly empty, one, and more than one group.

The oracle runs the rule in pieces of up to 128 tokens in float32, this build in pieces of 32; both are float32 sums in
another order, so outputs differ where a bf16 or e5m2 rounding falls the other way. An e5m2 step at one of n inputs of a
projection is an eighth to a quarter of that input, about 0.2 / sqrt(n) of the output: 6e-3 at 1,024 inputs. Held: 6e-2 per
token (several such steps in each of three projections), 2e-2 over all tokens, 1e-2 for the states.
"""

from __future__ import annotations

import ctypes
from dataclasses import replace

import pytest
import torch

from oracle import model as om
from qwen38_amd import synth
from qwen38_amd.config import LINEAR, tiny_config, with_layers
from qwen38_amd.generate import prefill_inputs
from qwen38_amd.quant import quantize_e4m3
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


class PrefillGdnArgs(ctypes.Structure):
    """csrc/kernels.h: the launcher's argument block."""

    _fields_ = (
        [(n, ctypes.c_int) for n in ("L", "Hk", "Hv", "C", "rows")]
        + [(n, ctypes.c_void_p) for n in ("slot", "start", "n_valid", "qkv", "z", "gate_part")]
        + [("gate_groups", ctypes.c_int)]
        + [(n, ctypes.c_void_p) for n in ("a_log", "dt_bias", "conv_w", "norm_w", "state", "conv", "qn", "kn", "v", "decay", "pt", "o", "act")]
        + [("eps", ctypes.c_float)]
    )


@pytest.mark.gpu
def test_the_chunks_matrices_are_rounded_once(gpu):
    """P_ts = e^(c_t - c_s) q_t . k_s and T = (I + beta k . k)^-1 of every chunk against 64 bits from the kernel's own q, k and
    beta, without decay (A_log = -inf): an entry of P is its exact sum rounded once, 2^-24 of it, where a float32 chain of
    128 products is off by 128 x 2^-24 of its terms at worst."""
    L, Hk, Hv, D = 96, 2, 8, 128
    C, rep, g = 2 * Hk * D + Hv * D, Hv // Hk, torch.Generator(device="cuda").manual_seed(5)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    ints = lambda v: torch.tensor([v], dtype=torch.int32, device="cuda")  # noqa: E731
    zeros = lambda n: torch.zeros(n, device="cuda")  # noqa: E731
    bf = lambda t: t.to(torch.bfloat16)  # noqa: E731
    t = {
        "slot": ints(0), "start": ints(0), "n_valid": ints(L), "qkv": bf(rand(L, C)), "z": bf(rand(L, Hv * D)),
        "gate_part": rand(L, 2 * Hv), "a_log": bf(torch.full((Hv,), -torch.inf, device="cuda")), "dt_bias": bf(zeros(Hv)),
        "conv_w": bf(rand(C, 4) * 0.5), "norm_w": bf(zeros(D)), "state": bf(zeros(Hv * D * D)), "conv": bf(zeros(C * 3)),
        "qn": zeros(L * Hk * D), "kn": zeros(L * Hk * D), "v": bf(zeros(L * Hv * D)), "decay": zeros(L * Hv * 3),
        "pt": zeros(L * Hv * 2 * 32), "o": bf(zeros(L * Hv * D)), "act": torch.zeros(L * Hv * D, dtype=torch.uint8, device="cuda"),
    }
    a = PrefillGdnArgs(L=L, Hk=Hk, Hv=Hv, C=C, rows=1, gate_groups=1, eps=1e-6, **{n: v.data_ptr() for n, v in t.items()})
    launch = gpu["_Z15q38_gdn_prefillRK14PrefillGdnArgsP12ihipStream_t"]
    torch.cuda.synchronize()
    assert launch(ctypes.byref(a), ctypes.c_void_p(0)) == 0
    torch.cuda.synchronize()
    heads = lambda n: t[n].view(L // 32, 32, Hk, D).double().permute(0, 2, 1, 3).repeat_interleave(rep, 1).contiguous()  # noqa: E731
    q, k, beta = heads("qn"), heads("kn"), t["decay"].view(L // 32, Hv, 3, 32)[:, :, 0].double()
    pt = t["pt"].view(L // 32, Hv, 2, 32, 32).double()
    want = (q @ k.transpose(-1, -2).contiguous()).tril()
    off = (pt[:, :, 1] - want).abs()
    print(f"P off by at most {float((off / want.abs().clamp_min(1e-30)).max()):.2e}, rms {float(off.norm() / want.norm()):.2e}")
    assert bool((off <= 2.0**-24 * want.abs() * (1 + 1e-6)).all())
    inverse = torch.linalg.inv(torch.eye(32, device="cuda", dtype=torch.float64) + (k @ k.transpose(-1, -2).contiguous()).tril(-1) * beta.unsqueeze(-1))
    # Forward substitution in float32: 32 products and sums per entry.
    assert float((pt[:, :, 0] - inverse).norm() / inverse.norm()) <= 32 * 2.0**-24


def gdn_layer_run(change, x, n_valid):
    """A chunk of x (row 0 from position 0) through one gated-delta layer whose weights `change` edits: output, final state."""
    cfg = with_layers(tiny_config(1), (LINEAR,))
    values = dict((sp.name, v) for sp, v in synth.make_all(synth.model_specs(cfg, mtp=False, head=False), 4))
    change(values)
    engine = Engine(cfg, 1, 1, 512, mtp=False, prefill_chunk=x.shape[1])
    engine.load(values.items())
    pi = prefill_inputs(cfg, 0, 0, n_valid, x.shape[1], torch.bfloat16)
    out = StepGraph(engine)(inputs_embeds=x, **pi).cpu()[0]
    return out, engine.gdn_state(0)["recurrent_state"].cpu()[0]


@pytest.mark.gpu
@pytest.mark.parametrize("at, n_valid", [(0, 96), (5, 96), (47, 96), (63, 96), (70, 64)])  # the last: in the padding
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_a_token_that_is_not_finite_leaves_the_earlier_ones(gpu, at, n_valid, value):
    x = synth.hidden_states((1, 96, 1024), 4, "x")
    want, _ = gdn_layer_run(lambda values: None, x, n_valid)
    x[0, at] = value
    got, state = gdn_layer_run(lambda values: None, x, n_valid)
    assert torch.equal(got[:at], want[:at])
    assert not bool(got[at:].isfinite().all(-1).any()) or at >= n_valid
    assert not bool(state.isfinite().any())


@pytest.mark.gpu
def test_a_value_that_is_not_finite_leaves_the_other_dims(gpu):
    """One dim of one value head, infinite at token 40 of 96: that column of the head's state is lost, every other one and
    every earlier token's output are what they are without it."""
    x = synth.hidden_states((1, 96, 1024), 4, "x")
    x[..., 7] = 0.0
    x[0, 40, 7] = 16.0
    head, dim, name = 3, 77, "layers.0.linear_attn.in_proj_qkv"

    def change(scale):
        def edit(values):
            row = torch.zeros(1, 1024)
            row[0, 7] = scale
            coded, scales = quantize_e4m3(row)
            channel = 2 * 4 * 128 + head * 128 + dim
            values[name][0][channel], values[name][1][channel] = coded[0], scales[0]

        return edit

    want, clean = gdn_layer_run(change(0.0), x, 96)
    got, state = gdn_layer_run(change(2.0**126), x, 96)
    assert torch.equal(got[:40], want[:40])
    lost = torch.zeros(state.shape, dtype=torch.bool)  # [value head, key dim, value dim]
    lost[head, :, dim] = True
    assert torch.equal(state[~lost], clean[~lost]) and not bool(state[lost].isfinite().any())


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [(40,), (33, 34, 60), (0, 31, 32, 95)])
@pytest.mark.parametrize("far", [2.0**20, 2.0**60, 2.0**100])
def test_a_decay_to_nothing_is_one_however_far(gpu, tokens, far):
    """e^g is zero from g = -104 down: the state restarts at such a token, and the decays after it keep their digits."""
    x = synth.hidden_states((1, 96, 1024), 4, "x")
    x[..., 7] = 0.0
    x[0, list(tokens), 7] = 30.0

    def change(weight):
        def edit(values):
            values["layers.0.linear_attn.in_proj_a"][:, 7] = weight  # times about 20: g is below -300
            values["layers.0.linear_attn.A_log"].zero_()

        return edit

    want, clean = gdn_layer_run(change(16.0), x, 96)
    got, state = gdn_layer_run(change(far), x, 96)
    assert bool(want.isfinite().all()) and torch.equal(got, want) and torch.equal(state, clean)


@pytest.mark.gpu
def test_an_infinite_decay_is_a_decay_to_nothing(gpu):
    x = synth.hidden_states((1, 96, 1024), 4, "x")

    def change(log):
        def edit(values):
            values["layers.0.linear_attn.A_log"].fill_(log)
            values["layers.0.linear_attn.dt_bias"].fill_(2.0)

        return edit

    want, clean = gdn_layer_run(change(6.0), x, 96)  # below -400 at every token
    got, state = gdn_layer_run(change(100.0), x, 96)  # e^100 is infinite
    assert bool(want.isfinite().all()) and torch.equal(got, want) and torch.equal(state, clean)
