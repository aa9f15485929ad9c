"""What a user of this package has it do, as cases that can be timed and compared.

Seven kinds of work, all through the package's public entry points and under ``torch.no_grad()`` (the kernels have no
backward), on random weights and activations:

``layer_prefill``  ``CausalSelfAttention.prefill`` over a prompt: projections, norm, RoPE, windowed attention
``attention``      ``ops.prefill_attention`` on q, k, v that the caller already has (with or without RoPE, documents)
``layer_step``     ``CausalSelfAttention.step``: one new token per sequence against a layer's ring cache
``model_step``     ``core.step`` / ``core.GraphedStep``: one new token per sequence through a stack of attention layers
``kda``            ``chunk_kda`` on the caller's tensors, a batch of sequences or sequences packed along T
``kda_layer``      ``KimiLinearSelfAttention.forward`` / ``prefill`` over a batch of prompts
``kda_step``       ``KimiLinearSelfAttention.step``: one new token per sequence, state updated in place

The listed sizes are those of the repository's configurations and of its benchmark and tests;
``draw`` covers the ranges around them, ragged lengths included.
"""
from __future__ import annotations

import math

import torch

from daisy_amd import (CausalSelfAttention, KimiLinearSelfAttention, KVCache, WindowMask, build_window_mask, chunk_kda, core,
                       doc_start_from_ids, fused_kda_gate, norm, ops)

DEVICE = "cuda:0"
EOS = 0                # token id that opens a document
NEW_TOKENS = 64        # a decode case generates this many tokens from its position before it starts over
LARGEST_FLOPS = 1.76e13


# ---------------------------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------------------------
def listed():
    return [
        # The plumbing configuration: one small layer over a short sequence. Launches and host time are all there is.
        dict(name="prefill_plumbing", kind="layer_prefill", B=1, T=256, H=4, D=64, window=128, docs=0, ve=False),
        # A chat prompt of odd length in front of the generator, one layer of the 12-head shape, value embeddings mixed in.
        dict(name="prefill_prompt_777", kind="layer_prefill", B=1, T=777, H=12, D=128, window=8192, docs=0, ve=True),
        # The windowed prefill configuration, as the module a model calls: the ordinary prefill of a batch.
        dict(name="prefill_batch8_4096", kind="layer_prefill", B=8, T=4096, H=8, D=128, window=1024, docs=0, ve=False),
        # A long packed training / evaluation row of several documents, head dim 64, keys rotated by the call.
        dict(name="attention_documents", kind="attention", B=1, T=20001, H=16, D=64, window=4096, docs=7, rope=True),
        # The long-context configuration, full causal: the largest call there is.
        dict(name="attention_full_65536", kind="attention", B=1, T=65536, H=16, D=128, window=0, docs=0, rope=False),
        # One token of one sequence through a layer, fp16 ring (the generator's default dtype): the smallest decode call.
        dict(name="step_layer_b1", kind="layer_step", B=1, H=12, D=128, window=8192, pos=8300, ring="float16", ve=False),
        # The decode configuration: 64 sequences, a wrapped ring of 4096 rows. Reading the cache is all there is.
        dict(name="step_layer_b64", kind="layer_step", B=64, H=16, D=128, window=4096, pos=8192, ring="bfloat16", ve=False),
        # The generator's regime at its best: one sequence, 12 layers, the step recorded once and replayed per token.
        dict(name="step_model_b1_recorded", kind="model_step", L=12, B=1, H=12, D=128, window=8192, pos=8292, vocab=8192, recorded=True),
        # The KDA configuration: fp32 log-decays, final state wanted.
        dict(name="kda_b4_8192", kind="kda", B=4, T=8192, H=16, Dk=128, Dv=128, packed=0, g="float32"),
        # A padded batch packed along T (seven sequences of unequal length), narrow heads, bf16 log-decays of the layer's gate.
        dict(name="kda_packed_6001", kind="kda", B=1, T=6001, H=12, Dk=64, Dv=64, packed=7, g="bfloat16"),
        # The KDA layer over a batch of long rows: projections, convolutions, gate, delta rule, gated norm.
        dict(name="kda_layer_b4_8192", kind="kda_layer", B=4, T=8192, H=16, Dk=128, prompt=False),
        # A decode step of the KDA layer for a batch of sequences.
        dict(name="kda_step_b64", kind="kda_step", B=64, H=16, Dk=128),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_once(rng):
    kind = rng.choice(["layer_prefill", "layer_prefill", "attention", "attention", "layer_step", "layer_step", "model_step",
                       "kda", "kda", "kda_layer", "kda_step"])
    D = rng.choice([64, 128, 128])
    if kind == "layer_prefill":
        H = rng.choice([4, 6, 8, 12, 16])
        return dict(kind=kind, B=_log_int(rng, 1, 16), T=_log_int(rng, 32, 16384), H=H, D=D, window=_log_int(rng, 128, 8192),
                    docs=rng.choice([0, 0, 3]), ve=rng.random() < 0.5)
    if kind == "attention":
        return dict(kind=kind, B=_log_int(rng, 1, 8), T=_log_int(rng, 500, 65536), H=rng.choice([4, 8, 12, 16]), D=D,
                    window=rng.choice([0, _log_int(rng, 256, 8192), _log_int(rng, 256, 8192)]), docs=rng.choice([0, 0, rng.randint(2, 9)]),
                    rope=rng.random() < 0.5)
    if kind == "layer_step":
        W = _log_int(rng, 512, 8192)
        return dict(kind=kind, B=_log_int(rng, 1, 64), H=rng.choice([4, 8, 12, 16]), D=D, window=W, pos=_log_int(rng, 64, 2 * W),
                    ring=rng.choice(["float16", "bfloat16"]), ve=rng.random() < 0.3)
    if kind == "model_step":
        W = _log_int(rng, 512, 8192)
        return dict(kind=kind, L=rng.randint(3, 12), B=_log_int(rng, 1, 16), H=rng.choice([8, 12]), D=D, window=W,
                    pos=_log_int(rng, 64, 2 * W), vocab=8 * _log_int(rng, 128, 6288), recorded=rng.random() < 0.6)
    if kind == "kda":
        packed = rng.choice([0, 0, rng.randint(2, 16)])
        return dict(kind=kind, B=1 if packed else _log_int(rng, 1, 8), T=_log_int(rng, 100, 16384), H=rng.choice([4, 8, 12, 16]),
                    Dk=rng.choice([64, 128, 128]), Dv=rng.choice([64, 128, 128]), packed=packed, g=rng.choice(["float32", "bfloat16"]))
    if kind == "kda_layer":
        return dict(kind=kind, B=_log_int(rng, 1, 8), T=_log_int(rng, 64, 8192), H=rng.choice([4, 8, 12, 16]),
                    Dk=rng.choice([64, 128, 128]), prompt=rng.random() < 0.5)
    return dict(kind=kind, B=_log_int(rng, 1, 64), H=rng.choice([8, 12, 16]), Dk=rng.choice([64, 128, 128]))


def _memory(case):
    """Rough size of a state with its outputs, in elements."""
    if case["kind"] in ("layer_step", "model_step"):
        return 2 * case.get("L", 1) * case["B"] * case["H"] * case["window"] * case["D"]
    return 8 * case["B"] * case.get("T", 64) * case["H"] * case.get("D", case.get("Dk", 128))


def draw(rng):
    """One more case of the ranges above; none costs more than the largest listed one."""
    while True:
        case = _draw_once(rng)
        if case["kind"] == "layer_prefill" and case["B"] > 1:
            case["docs"] = 0                     # one mask serves a batch: documents come with one row
        if case["kind"] == "attention" and case["B"] > 1:
            case["docs"] = 0
        if case["docs"] if "docs" in case else False:
            case["docs"] = min(case["docs"], max(case["T"] // 64, 1))
        if case["kind"] in ("kda", "kda_layer", "layer_prefill") and case["B"] * case["T"] > 40000:
            continue
        if work(case)["flops"] <= 0.9 * LARGEST_FLOPS and _memory(case) <= 1.1e9:
            return case


# ---------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------
def _randn(g, *shape, dtype=torch.bfloat16, scale=1.0):
    return (torch.randn(*shape, generator=g, device=DEVICE) * scale).to(dtype)


def _doc_starts(T, docs):
    """First positions of ``docs`` documents of unequal length in a row of T tokens (the same for every seed)."""
    return sorted({0} | {int(T * (i / docs) ** 1.3) for i in range(1, docs)}) if docs else [0]


def _token_row(T, docs):
    ids = torch.ones(T, dtype=torch.long, device=DEVICE)
    starts = [s for s in _doc_starts(T, docs) if s > 0]
    if starts:
        ids[torch.tensor(starts, device=DEVICE)] = EOS
    return ids


def _pairs(T, window, docs):
    """Visible (query, key) pairs of one row: causal, at most ``window`` keys, inside the query's document."""
    bounds = _doc_starts(T, docs) + [T]
    total = 0
    for a, b in zip(bounds, bounds[1:]):
        n = b - a
        w = n if window <= 0 else min(window, n)
        total += w * (w + 1) // 2 + (n - w) * w
    return total


def _attention_layer(case, g, max_len):
    dim = case["H"] * case["D"]
    with torch.device(DEVICE):
        attn = CausalSelfAttention(dim, case["H"], case["D"], receives_ve=bool(case.get("ve")), layer_idx=0, max_seq_len=max_len)
    with torch.no_grad():
        attn.qkvo_w.copy_(_randn(g, 4, dim, dim, scale=0.02))
    return attn.eval()


def _random_cache(case, g, layers):
    cache = KVCache(L=layers, B=case["B"], H=case["H"], W=case["window"], D=case["D"], device=DEVICE,
                    dtype=getattr(torch, case.get("ring", "bfloat16")))
    for store in (cache.k, cache.v):     # normalised rows, as a model writes them
        for i in range(layers):
            store[i].copy_(norm(_randn(g, *store.shape[1:])))
    cache.t = case["pos"]
    return cache


class _Block(torch.nn.Module):
    """The attention part of a model's block, pre-norm with a residual."""

    def __init__(self, attn):
        super().__init__()
        self.attn = attn

    def step(self, x, ve, x0, k_ctx, v_ctx, pos, window):
        y, k, v = self.attn.step(norm(x), k_ctx, v_ctx, pos, ve, window)
        return x + y, k, v


class _Stack(torch.nn.Module):
    """A stack of attention layers with the attributes that ``core.step`` walks."""

    def __init__(self, case, g):
        super().__init__()
        dim = case["H"] * case["D"]
        self.embed = torch.nn.Embedding(case["vocab"], dim, device=DEVICE, dtype=torch.bfloat16)
        self.lm_head_w = torch.nn.Parameter(_randn(g, case["vocab"], dim, scale=0.02))
        with torch.no_grad():
            self.embed.weight.copy_(_randn(g, case["vocab"], dim))
        self.blocks = torch.nn.ModuleList([_Block(_attention_layer(case, g, 2 * case["window"] + 256)) for _ in range(case["L"])])
        self.skip_map, self.skip_weights, self.ve_module_map = {}, None, {}
        self.window_size = self.attn_window_size = case["window"]
        self.attn_num_heads, self.attn_head_dim = case["H"], case["D"]
        self.eos_token_id = EOS


def _kda_layer(case, seed, max_len):
    torch.manual_seed(seed)
    with torch.device(DEVICE):
        layer = KimiLinearSelfAttention(case["H"] * case["Dk"], case["H"], max_seq_len=max_len, head_dim=case["Dk"])
    return layer.eval()


@torch.no_grad()
def prepare(case, seed):
    kind = case["kind"]
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    s = dict(case=case)
    if kind == "layer_prefill":
        B, T, dim = case["B"], case["T"], case["H"] * case["D"]
        s["attn"] = _attention_layer(case, g, T)
        s["x"] = _randn(g, B, T, dim)
        s["ve"] = _randn(g, B, T, dim) if case["ve"] else None
        s["mask"] = (build_window_mask(_token_row(T, case["docs"]), case["window"], EOS) if case["docs"]
                     else WindowMask(case["window"]))
    elif kind == "attention":
        B, T, H, D = (case[n] for n in "BTHD")
        s["qkv"] = [_randn(g, B, T, H, D) for _ in range(3)]
        s["kw"] = dict(window=case["window"] or None)
        if case["docs"]:
            s["kw"]["doc_start"] = doc_start_from_ids(_token_row(T, case["docs"]), EOS)
        if case["rope"]:
            freq = (1 / 10000.0) ** torch.linspace(0, 1, D // 2, device=DEVICE)
            theta = torch.outer(torch.arange(T, device=DEVICE, dtype=torch.float32), freq)
            s["kw"].update(cos=theta.cos(), sin=theta.sin())
    elif kind == "layer_step":
        s["attn"] = _attention_layer(case, g, case["pos"] + NEW_TOKENS + 1)
        s["cache"] = _random_cache(case, g, 1)
        s["x"] = _randn(g, case["B"], 1, case["H"] * case["D"])
        s["ve"] = _randn(g, case["B"], 1, case["H"] * case["D"]) if case["ve"] else None
    elif kind == "model_step":
        s["model"] = _Stack(case, g).eval()
        s["cache"] = _random_cache(case, g, case["L"])
        s["tokens"] = torch.randint(1, case["vocab"], (case["B"],), generator=g, device=DEVICE)
        if case["recorded"]:
            s["step"] = core.GraphedStep(s["model"], s["cache"])
            s["step"](s["tokens"])           # records; the recorded step then starts from the case's position
            s["cache"].t = case["pos"]
        else:
            s["step"] = lambda tokens, m=s["model"], c=s["cache"]: core.step(m, tokens, c)
    elif kind == "kda":
        B, T, H, Dk, Dv = case["B"], case["T"], case["H"], case["Dk"], case["Dv"]
        silu = torch.nn.functional.silu
        s["q"], s["k"], s["v"] = silu(_randn(g, B, T, H, Dk)), silu(_randn(g, B, T, H, Dk)), silu(_randn(g, B, T, H, Dv))
        if case["g"] == "float32":
            s["g"] = torch.nn.functional.logsigmoid(torch.randn(B, T, H, Dk, generator=g, device=DEVICE))
        else:                                # what the layer's gate makes of its input at its initial parameters
            a_log = torch.log(1 + 15 * torch.rand(H, generator=g, device=DEVICE))
            s["g"] = fused_kda_gate(_randn(g, B, T, H * Dk), a_log, Dk, torch.zeros(H * Dk, device=DEVICE))
        s["beta"] = torch.sigmoid(torch.randn(B, T, H, generator=g, device=DEVICE))
        s["kw"] = dict(output_final_state=True, use_qk_l2norm_in_kernel=True)
        if case["packed"]:
            s["kw"]["cu_seqlens"] = torch.tensor(_doc_starts(T, case["packed"]) + [T], dtype=torch.int32, device=DEVICE)
    elif kind == "kda_layer":
        s["layer"] = _kda_layer(case, seed, case["T"])
        s["x"] = _randn(g, case["B"], case["T"], case["H"] * case["Dk"])
    else:
        s["layer"] = _kda_layer(case, seed, 8192)
        s["layer"].prefill(_randn(g, case["B"], 64, case["H"] * case["Dk"]), None)
        s["x"] = _randn(g, case["B"], 1, case["H"] * case["Dk"])
    return s


# ---------------------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------------------
@torch.no_grad()
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "layer_prefill":
        return s["attn"].prefill(s["x"], s["ve"], attn_mask=s["mask"])
    if kind == "attention":
        return ops.prefill_attention(*s["qkv"], **s["kw"])
    if kind == "layer_step":
        cache = s["cache"]
        if cache.t >= case["pos"] + NEW_TOKENS:
            cache.t = case["pos"]
        ring = cache.ring(0)
        out = s["attn"].step(s["x"], ring, ring, cache.t, s["ve"], case["window"])
        cache.advance()
        return out + (cache.k, cache.v)
    if kind == "model_step":
        cache = s["cache"]
        if cache.t >= case["pos"] + NEW_TOKENS:
            cache.t = case["pos"]
        logits = s["step"](s["tokens"])
        return logits, cache.k, cache.v
    if kind == "kda":
        return chunk_kda(s["q"], s["k"], s["v"], s["g"], s["beta"], **s["kw"])
    layer = s["layer"]
    if kind == "kda_layer":
        if not case["prompt"]:
            return layer(s["x"], None)
        layer.reset_history()
        y, _, _ = layer.prefill(s["x"], None)
        return [y] + layer.state_tensors()
    y, _, _ = layer.step(s["x"], None, None, 64, None, None)
    return [y] + layer.state_tensors()


# ---------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------
def _attn_step_work(case):
    """One attention layer's step: weights and live cache rows once."""
    B, dim = case["B"], case["H"] * case["D"]
    rows = min(case["pos"] + 1, case["window"])
    nbytes = 2 * (4 * dim * dim + 2 * B * rows * dim + 2 * B * dim + 2 * B * dim)
    return nbytes, 8 * B * dim * dim + 4 * B * rows * dim


def work(case):
    kind = case["kind"]
    if kind in ("layer_prefill", "attention"):
        B, T, H, D = (case[n] for n in "BTHD")
        n, dim = B * T * H * D, H * D
        flops = 4 * D * B * H * _pairs(T, case["window"], case["docs"])
        if kind == "attention":
            return {"bytes": 2 * n * (5 if case["rope"] else 4) + (4 * T * D if case["rope"] else 0), "flops": flops}
        # x in, y, k and v out, the four weight matrices
        return {"bytes": 2 * n * (5 if case["ve"] else 4) + 8 * dim * dim, "flops": flops + 8 * B * T * dim * dim}
    if kind == "layer_step":
        nbytes, flops = _attn_step_work(case)
        return {"bytes": nbytes, "flops": flops}
    if kind == "model_step":
        dim = case["H"] * case["D"]
        nbytes, flops = _attn_step_work(case)
        return {"bytes": case["L"] * nbytes + 2 * case["vocab"] * dim + 4 * case["B"] * case["vocab"],
                "flops": case["L"] * flops + 2 * case["B"] * case["vocab"] * dim}
    B, H, Dk = case["B"], case["H"], case["Dk"]
    if kind == "kda":
        n, Dv = B * case["T"] * H, case["Dv"]
        states = case["packed"] or B
        return {"bytes": n * (2 * (2 * Dk + 2 * Dv) + Dk * (4 if case["g"] == "float32" else 2) + 4) + 4 * states * H * Dk * Dv,
                "flops": 7 * n * Dk * Dv}
    # A KDA layer: four square projections, two low-rank pairs through one head's width, beta; the state of the recurrence.
    dim = H * Dk
    weights = 4 * dim * dim + 4 * dim * Dk + H * dim
    if kind == "kda_layer":
        n = B * case["T"]
        state = 4 * B * H * Dk * Dk + 2 * 3 * B * dim * 4 if case["prompt"] else 0
        return {"bytes": 2 * weights + 2 * 2 * n * dim + state, "flops": 2 * n * weights + 7 * n * dim * Dk}
    return {"bytes": 2 * weights + 4 * B * dim + 2 * 4 * B * H * Dk * Dk + 2 * 2 * 3 * B * dim * 4,
            "flops": 2 * B * weights + 7 * B * dim * Dk}


def tolerance(case):
    # bf16 operands, probabilities and outputs with fp32 accumulation; a stack of layers rounds its residual stream
    # to bf16 at every layer.
    return {"rel": 2e-2 if case["kind"] == "model_step" else 1e-2}
