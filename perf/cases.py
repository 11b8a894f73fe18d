"""The work that a user of the library has it do, as cases that can be timed and checked.

Six kinds, each one pass through public entry points of qm38.Runtime:

  linear   one Q4 projection                                   q4_project
  layer    a layer's projections: QKV with the SwiGLU pair in  q4_project_set, q4_project
           one same-input set, then down
  attend   decode attention of a ragged batch                  attn_prepare, gqa_attention_q8
  prompt   causal attention of new rows over a cache           attn_prepare, gqa_attention_q8_prefill
  delta    Gated DeltaNet over new rows, then a decode step    deltanet_prefill(_with_snapshots), deltanet_step
  tokens   whole tokens through a hybrid block to the logits   decode_layers, residual_rmsnorm, q4_project

Every pass can be repeated on its state: attention passes move the caches back
to their cached length first (as a program does that drops draft tokens), and
DeltaNet passes start from a state that they do not modify, or from a recorded
verification image.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "qwen38-metal_amd"))
import qm38  # noqa: E402

DEV = "cuda:0"
EPS = 1e-6
FLT_MIN = 1.1754943508222875e-38

# The sizes of the repository's benchmark: hidden, MLP and fused QKV widths of
# a 27B-class layer; its attention and DeltaNet heads.
HIDDEN, INTER, QKV = 5120, 17408, 10240
VOCAB = 32768
CONV = 4

_RT = None


def _runtime():
    """One runtime for the program, on torch's stream."""
    global _RT
    if _RT is None:
        _RT = qm38.Runtime(0)
    _RT.set_stream(torch.cuda.current_stream())
    return _RT


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # The smallest call: one square projection of one token, where the
        # launch and its latency count.
        dict(name="linear_1", kind="linear", rows=1, width=4096, out=4096),
        # One decoding request: the projections of a layer for one token.
        dict(name="layer_1", kind="layer", rows=1, hidden=HIDDEN, inter=INTER, qkv=QKV),
        # Concurrent requests or drafted tokens: a few rows share the weights.
        dict(name="layer_5", kind="layer", rows=5, hidden=HIDDEN, inter=INTER, qkv=QKV),
        # A short prompt, or the ragged end of a long one.
        dict(name="layer_77", kind="layer", rows=77, hidden=HIDDEN, inter=INTER, qkv=QKV),
        # A long prompt's chunk.
        dict(name="layer_2048", kind="layer", rows=2048, hidden=HIDDEN, inter=INTER, qkv=QKV),
        # One request decoding at a long context.
        dict(name="attend_32k", kind="attend", heads=64, kv_heads=8, head_dim=128, lengths="32768"),
        # Eight requests of very different ages in one decode batch.
        dict(name="attend_ragged", kind="attend", heads=64, kv_heads=8, head_dim=128,
             lengths="4096,32768,131071,777,65536,32001,4096,1"),
        # Verification of a few drafted tokens at a long context, with the wide
        # heads (256) and a group of six query heads.
        dict(name="prompt_5_on_20001", kind="prompt", heads=24, kv_heads=4, head_dim=256, rows=5, cached=20001),
        # A prompt's second chunk.
        dict(name="prompt_2048_on_4096", kind="prompt", heads=64, kv_heads=8, head_dim=128, rows=2048, cached=4096),
        # Verification of drafted tokens with state images, back to an accepted
        # one, and on with a decode step.
        dict(name="delta_5", kind="delta", key_heads=16, value_heads=32, head_dim=128, rows=5, images=True),
        # A long prompt's chunk and the first token after it.
        dict(name="delta_2048", kind="delta", key_heads=16, value_heads=32, head_dim=128, rows=2048, images=False),
        # A request goes on after dropped draft tokens: two whole tokens through
        # three DeltaNet layers and a full-attention layer to their logits.
        dict(name="tokens_2", kind="tokens", tokens=2, cached=4096, graph=False),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "layer", "layer", "layer", "attend", "attend", "prompt", "prompt",
                       "prompt", "delta", "delta", "tokens"])
    if kind == "linear":
        width, out = 64 * _log_int(rng, 4, INTER // 64), _log_int(rng, 32, VOCAB)
        rows = min(_log_int(rng, 1, 2048), int(1.2e12 / (2 * width * out)))
        return dict(kind=kind, rows=rows, width=width, out=out)
    if kind == "layer":
        return dict(kind=kind, rows=_log_int(rng, 1, 2048), hidden=64 * _log_int(rng, 16, HIDDEN // 64),
                    inter=64 * _log_int(rng, 32, INTER // 64), qkv=_log_int(rng, 1024, QKV))
    if kind in ("attend", "prompt"):
        heads, kv_heads, head_dim = rng.choice([(64, 8, 128), (24, 4, 256), (16, 2, 128), (8, 8, 64)])
        if kind == "attend":
            lengths = [_log_int(rng, 1, 65536) for _ in range(rng.randint(1, 8))]
            return dict(kind=kind, heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                        lengths=",".join(map(str, lengths)))
        rows, cached = _log_int(rng, 2, 2048), _log_int(rng, 1, 65536) - 1
        # No more than the listed long prompt's products.
        cached = min(cached, int(3.4e11 / (4 * heads * head_dim * rows)) - rows // 2)
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, head_dim=head_dim, rows=rows, cached=max(0, cached))
    if kind == "delta":
        key_heads, value_heads = rng.choice([(16, 32), (16, 32), (8, 16), (4, 4)])
        rows = _log_int(rng, 2, 2047)
        return dict(kind=kind, key_heads=key_heads, value_heads=value_heads, head_dim=128, rows=rows,
                    images=rows <= 8)
    return dict(kind=kind, tokens=rng.randint(1, 4), cached=_log_int(rng, 16, 16384), graph=rng.random() < 0.5)


# ---------------------------------------------------------------------------
# Inputs, made from the seed alone
# ---------------------------------------------------------------------------
class _Maker:
    """Draws of one seed, in a fixed order."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV)
        self.gen.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.gen, device=DEV) * std

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.gen, device=DEV) * (hi - lo) + lo

    def bf16(self, *shape, std=1.0):
        return self.normal(*shape, std=std).to(torch.bfloat16)

    def q4(self, out, width):
        """Uniform nibbles, scales such that a projection of unit activations
        is about 1, biases around -7.5 scales (MLX affine)."""
        words = torch.randint(-2 ** 31, 2 ** 31, (out, width // 8), generator=self.gen, device=DEV, dtype=torch.int32)
        unit = 1.0 / (4.6 * math.sqrt(width))
        scales = self.uniform(0.5 * unit, 1.5 * unit, out, width // 64).to(torch.bfloat16)
        biases = (scales.float() * self.uniform(-8.0, -7.0, out, width // 64)).to(torch.bfloat16)
        return words, scales, biases

    def norm(self, n):
        return 1.0 + self.normal(n, std=0.1)

    def delta_weights(self, c):
        kh, vh, d = c["key_heads"], c["value_heads"], c["head_dim"]
        channels = 2 * kh * d + vh * d
        # Decays from a wide range of time constants, as trained layers have.
        a_log = torch.log(self.uniform(1.0, 16.0, vh))
        dt = torch.exp(self.uniform(math.log(1e-3), math.log(1e-1), vh))
        return dict(conv=self.normal(channels, CONV, std=0.5), a_log=a_log, dt_bias=torch.log(torch.expm1(dt)),
                    norm=self.norm(d))

    def delta_state(self, c):
        kh, vh, d = c["key_heads"], c["value_heads"], c["head_dim"]
        return self.normal(2 * kh * d + vh * d, CONV - 1), self.normal(vh, d, d, std=0.2)

    def delta_rows(self, c, rows):
        kh, vh, d = c["key_heads"], c["value_heads"], c["head_dim"]
        return (self.normal(rows, 2 * kh * d + vh * d), self.normal(rows, vh * d), self.normal(rows, vh),
                self.normal(rows, vh))


def _cache_rows(seed, sequence, tokens, kv_heads, head_dim):
    """The K and V rows that fill one cache, in blocks of up to 8192 tokens."""
    m = _Maker(seed * 64 + sequence + 1)
    done = 0
    while done < tokens:
        n = min(8192, tokens - done)
        yield n, m.normal(n, kv_heads, head_dim), m.normal(n, kv_heads, head_dim)
        done += n


def _cache(rt, seed, sequence, tokens, room, kv_heads, head_dim):
    """A cache that holds `tokens` tokens, with room for more, filled by the
    cheapest causal pass (one query head per KV head)."""
    kv = rt.create_q8_kv_state(kv_heads, head_dim)
    kv.reserve(tokens + room)
    kv.truncate(0)
    for n, k, v in _cache_rows(seed, sequence, tokens, kv_heads, head_dim):
        q = torch.zeros((n, kv_heads, head_dim), dtype=torch.bfloat16, device=DEV)
        rt.gqa_attention_q8_prefill(kv, q, None, k, v, kv_heads, n, torch.empty_like(q))
    return kv


def _rotary(head_dim):
    """Partial rotary (a quarter of the head) with interleaved M-RoPE axes."""
    rotary = head_dim // 4
    return qm38.RopeConfig(head_dim, rotary, 1e7, rotary // 6, rotary // 6, 1)


def _positions(m, first):
    """uint32 [3][rows] axis positions: text rows, a few of them off the diagonal as image rows are."""
    base = torch.tensor(first, dtype=torch.int64, device=DEV)
    shift = torch.randint(0, 3, (2, len(first)), generator=m.gen, device=DEV)
    return torch.cat([base[None], base[None] + shift]).to(torch.int32).contiguous()


def _lengths(case):
    return [int(t) for t in case["lengths"].split(",")]


def _attention_inputs(case, seed):
    """(maker's draws) of the rows that a pass of attend / prompt works on."""
    m = _Maker(seed)
    h, kvh, d = case["heads"], case["kv_heads"], case["head_dim"]
    first = _lengths(case) if case["kind"] == "attend" else list(range(case["cached"], case["cached"] + case["rows"]))
    r = len(first)
    return dict(rows=r, qg=m.bf16(r, h, 2 * d), k=m.bf16(r, kvh, d), v=m.normal(r, kvh, d), q_norm=m.norm(d),
                k_norm=m.norm(d), pos=_positions(m, first))


BLOCK = dict(key_heads=16, value_heads=32, head_dim=128)
BLOCK_HEADS, BLOCK_KV, BLOCK_D = 64, 8, 128
BLOCK_LAYERS = ("linear", "linear", "linear", "full")


def _block_inputs(case, seed):
    """Weights of the block and the head, states and the tokens' embedding rows."""
    m = _Maker(seed)
    val = BLOCK["value_heads"] * BLOCK["head_dim"]
    channels = 2 * BLOCK["key_heads"] * BLOCK["head_dim"] + val
    layers = []
    for kind in BLOCK_LAYERS:
        L = dict(kind=kind, in_norm=m.norm(HIDDEN), post_norm=m.norm(HIDDEN), gate=m.q4(INTER, HIDDEN),
                 up=m.q4(INTER, HIDDEN), down=m.q4(HIDDEN, INTER))
        if kind == "linear":
            L.update(qkv=m.q4(channels, HIDDEN), z=m.q4(val, HIDDEN), b=m.q4(BLOCK["value_heads"], HIDDEN),
                     a=m.q4(BLOCK["value_heads"], HIDDEN), out=m.q4(HIDDEN, val), dn=m.delta_weights(BLOCK),
                     state=m.delta_state(BLOCK), draft=m.delta_rows(BLOCK, 3))
        else:
            L.update(q=m.q4(2 * BLOCK_HEADS * BLOCK_D, HIDDEN), k=m.q4(BLOCK_KV * BLOCK_D, HIDDEN),
                     v=m.q4(BLOCK_KV * BLOCK_D, HIDDEN), o=m.q4(HIDDEN, BLOCK_HEADS * BLOCK_D),
                     q_norm=m.norm(BLOCK_D), k_norm=m.norm(BLOCK_D))
        layers.append(L)
    return dict(layers=layers, norm=m.norm(HIDDEN), head=m.q4(VOCAB, HIDDEN),
                rows=m.normal(case["tokens"], HIDDEN))


# ---------------------------------------------------------------------------
# What a program has in hand
# ---------------------------------------------------------------------------
def _job(q4, out):
    return qm38.Runtime.job(*q4, out)


def _empty(*shape, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=dtype, device=DEV)


def _delta_objects(rt, c, w, state):
    """DeltaNet weights and a state that holds `state`."""
    cfg = qm38.DnConfig(c["key_heads"], c["value_heads"], c["head_dim"], c["head_dim"], CONV)
    weights = rt.create_deltanet_weights(cfg, *(w[n].cpu().numpy() for n in ("conv", "a_log", "dt_bias", "norm")))
    st = weights.create_state()
    st.write(*(t.cpu().numpy() for t in state))
    return weights, st


def prepare(case, seed):
    rt = _runtime()
    kind = case["kind"]
    s = dict(case=case, rt=rt)
    if kind == "linear":
        m = _Maker(seed)
        s.update(job=_job(m.q4(case["out"], case["width"]), case["out"]), x=m.bf16(case["rows"], case["width"]),
                 y=_empty(case["rows"], case["out"]))
    elif kind == "layer":
        m = _Maker(seed)
        M, K, I, N = case["rows"], case["hidden"], case["inter"], case["qkv"]
        s.update(x=m.bf16(M, K), qkv=_job(m.q4(N, K), N), gate=_job(m.q4(I, K), I), up=_job(m.q4(I, K), I),
                 down=_job(m.q4(K, I), K), qkv_out=_empty(M, N), h=_empty(M, I), y=_empty(M, K))
    elif kind in ("attend", "prompt"):
        a = _attention_inputs(case, seed)
        r, h, kvh, d = a["rows"], case["heads"], case["kv_heads"], case["head_dim"]
        s.update(a, rope=_rotary(d), q=_empty(r, h, d), gate=_empty(r, h, d), o=_empty(r, h, d),
                 kr=_empty(r, kvh, d, dtype=torch.float32))
        if kind == "attend":
            s["caches"] = [_cache(rt, seed, i, n, 1, kvh, d) for i, n in enumerate(_lengths(case))]
        else:
            s["caches"] = [_cache(rt, seed, 0, case["cached"], r, kvh, d)]
    elif kind == "delta":
        m = _Maker(seed)
        rows, width = case["rows"], case["value_heads"] * case["head_dim"]
        weights, source = _delta_objects(rt, case, m.delta_weights(case), m.delta_state(case))
        s.update(weights=weights, source=source, state=source.clone(), new=m.delta_rows(case, rows),
                 step=m.delta_rows(case, 1), out=_empty(rows, width, dtype=torch.float32),
                 step_out=_empty(1, width, dtype=torch.float32))
        if case["images"]:
            # Room for two images at the least: a one-row set is exchanged, not copied.
            s["images"] = weights.create_snapshots(max(2, rows - 1))
    else:
        s.update(_prepare_tokens(rt, case, seed))
    return s


class _Raw:
    """fp32 device memory of the library, as torch takes it in."""

    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f4", data=(ptr, False), version=2)


def _prepare_tokens(rt, case, seed):
    b = _block_inputs(case, seed)
    val = BLOCK["value_heads"] * BLOCK["head_dim"]
    descs, rolls, keep = [], [], []
    for L in b["layers"]:
        if L["kind"] == "linear":
            weights, st = _delta_objects(rt, BLOCK, L["dn"], L["state"])
            images = weights.create_snapshots(2)
            rt.deltanet_prefill_with_snapshots(weights, None, st, images, *L["draft"], 3, EPS,
                                               _empty(3, val, dtype=torch.float32))
            rolls.append((images, st))
            out = {n: _job(L[n], L[n][0].shape[0]) for n in ("qkv", "z", "b", "a", "out", "gate", "up", "down")}
            descs.append(qm38.DecodeLinearLayer(L["in_norm"].data_ptr(), L["post_norm"].data_ptr(), out["qkv"],
                                                out["z"], out["b"], out["a"], out["out"], weights.handle.value,
                                                st.handle.value, out["gate"], out["up"], out["down"]))
            keep.append((weights, out))
        else:
            kv = _cache(rt, seed, 0, case["cached"], case["tokens"], BLOCK_KV, BLOCK_D)
            out = {n: _job(L[n], L[n][0].shape[0]) for n in ("q", "k", "v", "o", "gate", "up", "down")}
            descs.append(qm38.DecodeFullLayer(L["in_norm"].data_ptr(), L["post_norm"].data_ptr(), out["q"], out["k"],
                                              out["v"], out["o"], L["q_norm"].data_ptr(), L["k_norm"].data_ptr(),
                                              BLOCK_HEADS, _rotary(BLOCK_D), kv.handle.value, out["gate"], out["up"],
                                              out["down"]))
            keep.append(out)
    state = rt.create_decode_state(HIDDEN)
    graph = qm38.DecodeGraph(rt, state, descs, EPS) if case["graph"] else None
    return dict(b=b, keep=keep, descs=descs, rolls=rolls, kv=kv, state=state, graph=graph,
                hidden=torch.as_tensor(_Raw(state.hidden_ptr, HIDDEN), device=DEV), head=_job(b["head"], VOCAB),
                x=_empty(1, HIDDEN), logits=_empty(case["tokens"], VOCAB))


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s):
    return _RUN[s["case"]["kind"]](s, s["case"], s["rt"])


def _run_linear(s, c, rt):
    rt.q4_project([s["job"]], s["x"], c["width"], c["rows"], [s["y"]])
    return s["y"]


def _run_layer(s, c, rt):
    rt.q4_project_set([s["qkv"], s["gate"]], [None, s["up"]], s["x"], c["hidden"], c["rows"], [s["qkv_out"], s["h"]])
    rt.q4_project([s["down"]], s["h"], c["inter"], c["rows"], [s["y"]])
    return dict(qkv=s["qkv_out"], h=s["h"], y=s["y"])


def _prepare_rows(s, c, rt):
    rt.attn_prepare(s["rope"], s["rows"], c["heads"], c["kv_heads"], s["qg"], s["k"], s["q_norm"], s["k_norm"], EPS,
                    s["q"], s["gate"], s["kr"], positions=s["pos"])


def _run_attend(s, c, rt):
    for kv, n in zip(s["caches"], _lengths(c)):
        kv.truncate(n)
    _prepare_rows(s, c, rt)
    rt.gqa_attention_q8(s["caches"], s["q"], s["gate"], s["kr"], s["v"], c["heads"], s["o"])
    return dict(q=s["q"], gate=s["gate"], k=s["kr"], o=s["o"])


def _run_prompt(s, c, rt):
    s["caches"][0].truncate(c["cached"])
    _prepare_rows(s, c, rt)
    rt.gqa_attention_q8_prefill(s["caches"][0], s["q"], s["gate"], s["kr"], s["v"], c["heads"], s["rows"], s["o"])
    return dict(q=s["q"], gate=s["gate"], k=s["kr"], o=s["o"])


def _accepted(c):
    """The image that verification goes back to: the state after this row."""
    return (c["rows"] - 1) // 2


def _run_delta(s, c, rt):
    if c["images"]:
        rt.deltanet_prefill_with_snapshots(s["weights"], s["source"], s["state"], s["images"], *s["new"], c["rows"],
                                           EPS, s["out"])
        if _accepted(c) < c["rows"] - 1:
            s["images"].restore(_accepted(c), s["state"])
    else:
        rt.deltanet_prefill(s["weights"], s["state"], *s["new"], c["rows"], EPS, s["out"], source=s["source"])
    rt.deltanet_step(s["weights"], s["state"], *s["step"], EPS, s["step_out"])
    return dict(out=s["out"], step=s["step_out"])


def _run_tokens(s, c, rt):
    for images, st in s["rolls"]:
        images.restore(1, st)
    s["kv"].truncate(c["cached"])
    for t in range(c["tokens"]):
        p = c["cached"] + t
        s["hidden"].copy_(s["b"]["rows"][t])  # the token's embedding row
        if s["graph"]:
            s["graph"].run(p)
        else:
            rt.decode_layers(s["state"], s["descs"], p, EPS)
        rt.residual_rmsnorm(s["state"].hidden_ptr, None, s["b"]["norm"], 1, HIDDEN, EPS, s["x"])
        rt.q4_project([s["head"]], s["x"], HIDDEN, 1, [s["logits"][t]])
    return dict(logits=s["logits"])


_RUN = dict(linear=_run_linear, layer=_run_layer, attend=_run_attend, prompt=_run_prompt, delta=_run_delta,
            tokens=_run_tokens)


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _q4_bytes(out, width):
    return out * width // 2 + 4 * out * (width // 64)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, K, N = case["rows"], case["width"], case["out"]
        return dict(bytes=_q4_bytes(N, K) + 2 * M * (K + N), flops=2 * M * N * K)
    if kind == "layer":
        M, K, I, N = case["rows"], case["hidden"], case["inter"], case["qkv"]
        return dict(bytes=_q4_bytes(N, K) + 2 * _q4_bytes(I, K) + _q4_bytes(K, I) + 2 * M * (K + N + I + K),
                    flops=2 * M * (N * K + 3 * I * K))
    if kind in ("attend", "prompt"):
        h, kvh, d = case["heads"], case["kv_heads"], case["head_dim"]
        if kind == "attend":
            rows = len(_lengths(case))
            held = sum(_lengths(case))
            seen = held + rows
        else:
            rows, held = case["rows"], case["cached"]
            seen = rows * held + rows * (rows + 1) // 2
        # The caches read and appended to; q with its gate, k and v in; q, gate, k and o out.
        return dict(bytes=(held + rows) * kvh * (2 * d + 8) + rows * (2 * h * 2 * d + kvh * (2 * d + 4 * d + 4 * d)
                                                                     + 3 * 2 * h * d),
                    flops=4 * h * d * seen)
    if kind == "delta":
        return _delta_work(case, case["rows"] + 1, images=case["rows"] - 1 if case["images"] else 0)
    t = case["tokens"]
    val = BLOCK["value_heads"] * BLOCK["head_dim"]
    channels = 2 * BLOCK["key_heads"] * BLOCK["head_dim"] + val
    mlp = 3 * INTER * HIDDEN
    linear = HIDDEN * (channels + val + 2 * BLOCK["value_heads"]) + val * HIDDEN
    full = HIDDEN * (2 * BLOCK_HEADS * BLOCK_D + 2 * BLOCK_KV * BLOCK_D) + BLOCK_HEADS * BLOCK_D * HIDDEN
    elements = sum(mlp + (linear if kind == "linear" else full) for kind in BLOCK_LAYERS) + VOCAB * HIDDEN
    d = _delta_work(BLOCK, t)
    n = BLOCK_LAYERS.count("linear")
    seen = t * case["cached"] + t * (t + 1) // 2
    return dict(bytes=t * (elements * 9 // 16 + 2 * VOCAB) + n * d["bytes"] + seen * BLOCK_KV * (2 * BLOCK_D + 8),
                flops=2 * t * elements + n * d["flops"] + 4 * BLOCK_HEADS * BLOCK_D * seen)


def _delta_work(c, rows, images=0):
    kh, vh, d = c["key_heads"], c["value_heads"], c["head_dim"]
    channels = 2 * kh * d + vh * d
    state = 4 * (vh * d * d + channels * (CONV - 1))
    return dict(bytes=(2 + images) * state + 4 * channels * CONV + 4 * rows * (channels + 2 * vh * d + 2 * vh),
                flops=7 * rows * vh * d * d)


# ---------------------------------------------------------------------------
# How far another correct implementation may be off, and the values themselves
# ---------------------------------------------------------------------------
def tolerance(case):
    """About four times what the passes were seen to be off from exact()."""
    if case["kind"] == "delta":
        return dict(rel=3e-5, max=1e-3)  # fp32 sums, chunked ones on split operands: 2e-7 .. 5e-6
    if case["kind"] == "tokens":
        return dict(rel=2.4e-2, max=0.2)  # the bf16 roundings of four layers: 6e-3
    return dict(rel=9e-3, max=0.04)  # one or two bf16 roundings: 1.7e-3 .. 2.4e-3


def _dense(q4):
    """The affine matrix in 64 bits: scale * nibble + bias."""
    words, scales, biases = q4
    shifts = torch.arange(0, 32, 4, device=DEV, dtype=torch.int32)
    q = (words[..., None] >> shifts & 15).reshape(words.shape[0], -1).double()
    return torch.addcmul(biases.double().repeat_interleave(64, 1), q, scales.double().repeat_interleave(64, 1))


def _project(x, q4, step=8192):
    return torch.cat([x @ _dense(tuple(t[i:i + step] for t in q4)).T for i in range(0, q4[0].shape[0], step)], -1)


def _mlp_in(x, gate, up, step=8192):
    return torch.cat([torch.nn.functional.silu(x @ _dense(tuple(t[i:i + step] for t in gate)).T)
                      * (x @ _dense(tuple(t[i:i + step] for t in up)).T) for i in range(0, gate[0].shape[0], step)], -1)


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, pos, head_dim):
    """x [rows][heads][d], pos [3][rows]: the first quarter of the head turns,
    frequency i about the axis that M-RoPE gives it."""
    rope = _rotary(head_dim)
    half = rope.rotary_dim // 2
    axis = [1 if i % 3 == 1 and i // 3 < rope.mrope_section1 else 2 if i % 3 == 2 and i // 3 < rope.mrope_section2
            else 0 for i in range(half)]
    freq = torch.tensor([rope.rope_theta ** (-2.0 * i / rope.rotary_dim) for i in range(half)], dtype=torch.float64,
                        device=DEV)
    angle = pos.double()[axis].T * freq  # [rows][half]
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    a, b = x[..., :half], x[..., half:2 * half]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., 2 * half:]], -1)


def _q8(x):
    """Rows as the cache holds them: absmax / 127 scales, half away from zero."""
    x = x.float()
    scale = (x.abs().amax(-1, keepdim=True) / 127.0).clamp_min(FLT_MIN)
    v = (x / scale).clamp(-127, 127)
    return (v.sign() * (v.abs() + 0.5).floor()).double() * scale.double()


def _attention(q, gate, keys, values, start):
    """q, gate [rows][H][d]; keys, values [T][KVH][d]; row i sees the first start + i + 1 tokens."""
    rows, h, d = q.shape
    T, kvh, _ = keys.shape
    g = h // kvh
    o = torch.empty_like(q)
    step = max(1, (1 << 26) // (g * T))
    for j in range(kvh):
        kj, vj = keys[:, j].contiguous(), values[:, j].contiguous()
        for i in range(0, rows, step):
            n = min(step, rows - i)
            s = (q[i:i + n, j * g:(j + 1) * g].reshape(-1, d) @ kj.T).reshape(n, g, T) / math.sqrt(d)
            ahead = torch.arange(T, device=DEV) > torch.arange(start + i, start + i + n, device=DEV)[:, None]
            p = s.masked_fill_(ahead[:, None], -math.inf).softmax(-1)
            o[i:i + n, j * g:(j + 1) * g] = (p.reshape(-1, T) @ vj).reshape(n, g, d)
    return o * torch.sigmoid(gate)


def _cached_rows(seed, sequence, tokens, kvh, d):
    rows = [(_q8(k), _q8(v)) for _, k, v in _cache_rows(seed, sequence, tokens, kvh, d)]
    empty = torch.empty((0, kvh, d), dtype=torch.float64, device=DEV)
    return [torch.cat([empty] + [r[i] for r in rows]) for i in (0, 1)]


class _Delta:
    """The recurrence in 64 bits, one token after the other."""

    def __init__(self, c, w, state):
        self.c = c
        self.w = {n: t.float().double() for n, t in w.items()}
        self.hist, self.S = (t.double().clone() for t in state)

    def token(self, qkv, z, b, a):
        kh, vh, d = self.c["key_heads"], self.c["value_heads"], self.c["head_dim"]
        window = torch.cat([self.hist, qkv.double()[:, None]], 1)
        self.hist = window[:, 1:].clone()
        x = torch.nn.functional.silu((window * self.w["conv"]).sum(1))
        q, k, v = x[:kh * d].reshape(kh, d), x[kh * d:2 * kh * d].reshape(kh, d), x[2 * kh * d:].reshape(vh, d)
        q = (q * torch.rsqrt(q.square().mean(-1, keepdim=True) + EPS) / d).repeat_interleave(vh // kh, 0)
        k = (k * torch.rsqrt(k.square().mean(-1, keepdim=True) + EPS) / math.sqrt(d)).repeat_interleave(vh // kh, 0)
        decay = torch.exp(-torch.exp(self.w["a_log"]) * torch.nn.functional.softplus(a.double() + self.w["dt_bias"]))
        self.S = self.S * decay[:, None, None]
        delta = (v - (self.S * k[:, None]).sum(-1)) * torch.sigmoid(b.double())[:, None]
        self.S = self.S + delta[..., None] * k[:, None]
        o = (self.S * q[:, None]).sum(-1)
        zz = z.double().reshape(vh, d)
        return (_rms(o, self.w["norm"]) * torch.nn.functional.silu(zz)).reshape(-1)

    def rows(self, new, keep=None):
        """(outputs, the state after row `keep`)."""
        out, kept = [], None
        for t in range(new[0].shape[0]):
            out.append(self.token(*(x[t] for x in new)))
            if t == keep:
                kept = (self.hist, self.S)
        return torch.stack(out), kept


def exact(case, seed):
    kind = case["kind"]
    m = _Maker(seed)
    if kind == "linear":
        q4 = m.q4(case["out"], case["width"])
        return _project(m.bf16(case["rows"], case["width"]).double(), q4)
    if kind == "layer":
        M, K, I, N = case["rows"], case["hidden"], case["inter"], case["qkv"]
        x = m.bf16(M, K).double()
        qkv, gate, up, down = m.q4(N, K), m.q4(I, K), m.q4(I, K), m.q4(K, I)
        h = _mlp_in(x, gate, up)
        return dict(qkv=_project(x, qkv), h=h, y=_project(h, down))
    if kind in ("attend", "prompt"):
        kvh, d = case["kv_heads"], case["head_dim"]
        a = _attention_inputs(case, seed)
        q = _rope(_rms(a["qg"][..., :d].double(), a["q_norm"]), a["pos"], d)
        k = _rope(_rms(a["k"].double(), a["k_norm"]), a["pos"], d)
        gate = a["qg"][..., d:].double()
        if kind == "prompt":
            ck, cv = _cached_rows(seed, 0, case["cached"], kvh, d)
            o = _attention(q, gate, torch.cat([ck, _q8(k)]), torch.cat([cv, _q8(a["v"])]), case["cached"])
        else:
            o = torch.empty_like(q)
            for i, n in enumerate(_lengths(case)):
                ck, cv = _cached_rows(seed, i, n, kvh, d)
                o[i:i + 1] = _attention(q[i:i + 1], gate[i:i + 1], torch.cat([ck, _q8(k[i:i + 1])]),
                                        torch.cat([cv, _q8(a["v"][i:i + 1])]), n)
        return dict(q=q, gate=gate, k=k, o=o)
    if kind == "delta":
        net = _Delta(case, m.delta_weights(case), m.delta_state(case))
        new, step = m.delta_rows(case, case["rows"]), m.delta_rows(case, 1)
        out, kept = net.rows(new, _accepted(case) if case["images"] else None)
        if kept is not None:
            net.hist, net.S = kept
        return dict(out=out, step=net.rows(step)[0])
    return _exact_tokens(case, seed)


def _exact_tokens(case, seed):
    b = _block_inputs(case, seed)
    nets = []
    for L in b["layers"]:
        if L["kind"] == "linear":
            nets.append(_Delta(BLOCK, L["dn"], L["state"]))
            _, (nets[-1].hist, nets[-1].S) = nets[-1].rows(L["draft"], 1)
        else:
            nets.append(_cached_rows(seed, 0, case["cached"], BLOCK_KV, BLOCK_D))
    logits = []
    for t in range(case["tokens"]):
        hidden = b["rows"][t].double()[None]
        pos = torch.full((3, 1), case["cached"] + t, dtype=torch.int32, device=DEV)
        for i, L in enumerate(b["layers"]):
            x = _rms(hidden, L["in_norm"])
            if L["kind"] == "linear":
                y = nets[i].token(*(_project(x, L[n])[0] for n in ("qkv", "z", "b", "a")))[None]
                hidden = hidden + _project(y, L["out"])
            else:
                qg = _project(x, L["q"]).reshape(1, BLOCK_HEADS, 2 * BLOCK_D)
                q = _rope(_rms(qg[..., :BLOCK_D], L["q_norm"]), pos, BLOCK_D)
                k = _rope(_rms(_project(x, L["k"]).reshape(1, BLOCK_KV, BLOCK_D), L["k_norm"]), pos, BLOCK_D)
                v = _project(x, L["v"]).reshape(1, BLOCK_KV, BLOCK_D)
                nets[i] = [torch.cat([c, _q8(n)]) for c, n in zip(nets[i], (k, v))]
                o = _attention(q, qg[..., BLOCK_D:], *nets[i], case["cached"] + t)
                hidden = hidden + _project(o.reshape(1, -1), L["o"])
            x = _rms(hidden, L["post_norm"])
            hidden = hidden + _project(_mlp_in(x, L["gate"], L["up"]), L["down"])
        logits.append(_project(_rms(hidden, b["norm"]), b["head"])[0])
    return dict(logits=torch.stack(logits))
