"""The rollout path's work, case by case: what a program that generates Gemma 4 rollouts has this
framework do, through its public entry points.

Kinds of case:
- ``decode``: one decode step's attention (append one token per row, attend) over several layers'
  caches, replayed from a HIP graph as the generation loop replays its step; ring (sliding) and
  linear (global) caches, from one interactive sequence to ragged 32768-slot rows;
- ``prefill``: causal / sliding-window attention of (left-padded) prompts;
- ``append``: the q/k norms, RoPE and cache writes of a prompt chunk;
- ``mlp``: a decode batch's MLP (gate/up + gated GELU, down projection, residual norms);
- ``draw``: the LM head and the next token's draw over the whole vocabulary;
- ``step``: one decode step of the 30-layer E2B-like model, replayed from a HIP graph, to its logits;
- ``prompt``: the model's prefill of left-padded prompts, to the first token's logits and the caches.

``exact`` restates each in 64-bit torch, with no code of the framework.
"""

from __future__ import annotations

import importlib
import importlib.util
import math
import sys
import weakref
from pathlib import Path

import torch

PKG = "gemma4_posttrain_jax_amd"
if PKG not in sys.modules:  # the package directory's name is no Python identifier
    _dir = Path(__file__).resolve().parent.parent / "gemma4-posttrain-jax_amd"
    _spec = importlib.util.spec_from_file_location(PKG, _dir / "__init__.py", submodule_search_locations=[str(_dir)])
    _pkg = importlib.util.module_from_spec(_spec)
    sys.modules[PKG] = _pkg
    _spec.loader.exec_module(_pkg)
_lib = importlib.import_module(PKG + "._lib")
kernels = importlib.import_module(PKG + ".kernels")
kvcache = importlib.import_module(PKG + ".kvcache")
config = importlib.import_module(PKG + ".config")
model = importlib.import_module(PKG + ".model")
sampler = importlib.import_module(PKG + ".sampler")

DEV = "cuda"
BF16 = torch.bfloat16
EPS = 1e-6
SOFTCAP = 30.0
QK_SCALE = 0.25  # q / k norm weights: scores of order 1, as trained q / k norms give
APPEND_FLAGS = (_lib.G4_APPEND_NORM_Q | _lib.G4_APPEND_ROPE_Q | _lib.G4_APPEND_NORM_K | _lib.G4_APPEND_ROPE_K
                | _lib.G4_APPEND_NORM_V)

# the E2B-like decoder of the benchmark: 30 layers, 4 sliding : 1 global, the last 10 sharing K/V
E2B = dict(
    vocab_size=262144, hidden_size=2048, intermediate_size=8192, num_hidden_layers=30, num_attention_heads=8,
    num_key_value_heads=2, head_dim=256, global_head_dim=256,
    layer_types=(["sliding_attention"] * 4 + ["full_attention"]) * 6, sliding_window=512, num_kv_shared_layers=10,
    hidden_size_per_layer_input=0, final_logit_softcapping=SOFTCAP,
)


def listed() -> list[dict]:
    return [
        # one interactive sequence: the sliding layers of a decode step, latency-bound
        dict(name="decode_single", kind="decode", batch=1, heads=2, group=4, dim=256, ring=True, capacity=512, lo=700,
             hi=701, pad=0, layers=12),
        # the benchmark's sliding-window decode: 64 rows over rings that have wrapped
        dict(name="decode_ring", kind="decode", batch=64, heads=2, group=4, dim=256, ring=True, capacity=512, lo=1536,
             hi=2048, pad=0, layers=8),
        # the benchmark's long-context decode: ragged rows of up to 32768 slots
        dict(name="decode_long", kind="decode", batch=16, heads=2, group=4, dim=256, ring=False, capacity=32768,
             lo=1024, hi=32768, pad=0, layers=1),
        # the benchmark's long-prompt prefill, a global layer
        dict(name="prefill_global", kind="prefill", batch=8, seq=4096, heads=2, group=4, dim=256, window=0, pad=0),
        # a batch of left-padded prompts of different lengths, a sliding layer; no round sizes
        dict(name="prefill_window", kind="prefill", batch=11, seq=1999, heads=2, group=4, dim=256, window=512,
             pad=1500),
        # a stock configuration's global layer (head dim 512) over left-padded prompts
        dict(name="prefill_wide", kind="prefill", batch=4, seq=1024, heads=2, group=4, dim=512, window=0, pad=256),
        # the rollout batch's prompts: one sliding layer's norms, RoPE and cache writes
        dict(name="append_prompt", kind="append", batch=256, seq=256, heads=2, group=4, dim=256, ring=True,
             capacity=512),
        # the MLP of one layer at the reference harness's smallest decode batch
        dict(name="mlp_rows", kind="mlp", rows=32, hidden=2048, ffn=8192),
        # the rollout's draw: temperature 1 over the full vocabulary, inside the LM head
        dict(name="draw_full", kind="draw", rows=256, vocab=262144, hidden=2048, temperature=1.0, top_k=0, top_p=1.0),
        # the reference harness's default draw: top-k 50, at its batch of 64
        dict(name="draw_top_k", kind="draw", rows=64, vocab=262144, hidden=2048, temperature=1.0, top_k=50, top_p=1.0),
        # a decode step of the rollout batch, half way through its completions
        dict(name="step_rollout", kind="step", batch=256, length=512, capacity=768, pad=64),
        # the prompts of one GRPO step, left-padded
        dict(name="prompt_model", kind="prompt", batch=16, seq=512, new=64, pad=300),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng) -> dict:
    kind = rng.choices(["decode", "prefill", "append", "mlp", "draw", "step", "prompt"], [4, 4, 2, 2, 3, 1, 1])[0]
    if kind == "decode":
        heads, group, dim = rng.choice([1, 2, 4]), rng.choice([1, 2, 4, 8]), rng.choice([128, 256, 256, 512])
        ring = rng.random() < 0.5
        capacity = rng.choice([128, 512, 512, 1024]) if ring else _log_int(rng, 48, 32768)
        most = (16 * 32768 * 2 * 256) // (capacity * heads * dim)  # values in one layer's keys
        batch = _log_int(rng, 1, max(1, min(256, most)))
        hi = _log_int(rng, capacity // 2, 4 * capacity) if ring else rng.randint(capacity // 2, capacity)
        lo = rng.randint(max(1, hi // 8), hi - 1)
        layers = max(1, min(8, most // batch))
        return dict(kind=kind, batch=batch, heads=heads, group=group, dim=dim, ring=ring, capacity=capacity, lo=lo,
                    hi=hi, pad=rng.choice([0, lo // 2]), layers=layers)
    if kind == "prefill":
        heads, group, dim = rng.choice([1, 2, 4]), rng.choice([1, 2, 4, 8]), rng.choice([128, 256, 256, 512])
        seq = _log_int(rng, 16, 4096 if dim < 512 else 1536)
        most = (8 * 4096 * 4096 * 2 * 4 * 256) // (seq * seq * heads * group * dim * (1 if dim < 512 else 6))
        batch = _log_int(rng, 1, max(1, min(64, most)))
        window = rng.choice([0, 512, 512, 1024]) if dim < 512 else 0
        return dict(kind=kind, batch=batch, seq=seq, heads=heads, group=group, dim=dim, window=window,
                    pad=rng.choice([0, seq // 4, seq // 2]))
    if kind == "append":
        heads, group, dim = rng.choice([1, 2, 4]), rng.choice([1, 2, 4]), rng.choice([128, 256, 256, 512])
        seq = _log_int(rng, 8, 4096)
        most = (256 * 256 * 2 * 6 * 256) // (seq * heads * (group + 2) * dim)
        ring = rng.random() < 0.6
        return dict(kind=kind, batch=_log_int(rng, 1, max(1, min(256, most))), seq=seq, heads=heads, group=group,
                    dim=dim, ring=ring, capacity=rng.choice([128, 512]) if ring else seq + rng.randint(1, 512))
    if kind == "mlp":
        return dict(kind=kind, rows=_log_int(rng, 1, 256), hidden=64 * rng.randint(8, 48), ffn=512 * rng.randint(4, 24))
    if kind == "draw":
        top_k = rng.choice([0, 0, 50, rng.randint(1, 256)])
        return dict(kind=kind, rows=_log_int(rng, 1, 256), vocab=128 * rng.randint(256, 2048),
                    hidden=128 * rng.randint(4, 16), temperature=rng.choice([1.0, 0.7]), top_k=top_k,
                    top_p=rng.choice([1.0, 0.95]) if top_k else 1.0)
    if kind == "step":
        length = rng.randint(64, 700)
        return dict(kind=kind, batch=_log_int(rng, 1, 256), length=length, capacity=768,
                    pad=rng.choice([0, length // 3]))
    seq = _log_int(rng, 24, 1024)
    return dict(kind=kind, batch=_log_int(rng, 1, max(1, 8192 // seq)), seq=seq, new=rng.randint(8, 128),
                pad=rng.choice([0, seq // 2]))


# --- what a program has in hand ------------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, scale: float = 1.0, dtype=BF16) -> torch.Tensor:
    """N(0, scale^2) values, made in bf16 (the large caches stay one allocation)."""

    return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, scale, generator=g)


def _left_pads(g, batch: int, most: int) -> torch.Tensor:
    """Left padding per row, uniform in [0, most] (the longest prompt of a batch has none)."""

    pads = torch.randint(0, most + 1, (batch,), device=DEV, generator=g)
    pads[0] = 0
    return pads


def _rotary(pos: torch.Tensor, dim: int, theta: float, fraction: float = 1.0) -> tuple[torch.Tensor, torch.Tensor]:
    """f64 cos / sin ``[..., dim]`` of the positions, the first ``fraction`` of the dims rotating."""

    n = int(fraction * dim // 2)
    freq = theta ** (-torch.arange(0, 2 * n, 2, dtype=torch.float64, device=pos.device) / dim)
    freq = torch.cat([freq, freq.new_zeros(dim // 2 - n)])
    angle = pos.double()[..., None] * torch.cat([freq, freq])
    return angle.cos(), angle.sin()


def _decode_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    B, H, R, D = case["batch"], case["heads"], case["group"], case["dim"]
    layers = []
    for _ in range(case["layers"]):
        layer = kvcache.new_layer_cache(B, H, D, case["capacity"], case["ring"], BF16, DEV)
        layer.key.normal_(0.0, QK_SCALE, generator=g)
        layer.value_t.normal_(generator=g)
        layers.append(layer)
    q_pos = torch.randint(case["lo"], case["hi"], (B,), device=DEV, generator=g, dtype=torch.int32)
    width = case["hi"] if case["ring"] else case["capacity"]
    pads = _left_pads(g, B, case["pad"])
    mask = torch.arange(width, device=DEV)[None, :] >= pads[:, None]
    n = case["layers"]
    return dict(layers=layers, q_pos=q_pos, mask=mask, window=case["capacity"] if case["ring"] else 0,
                q=_randn(g, n, B, H, R, D, scale=QK_SCALE), k=_randn(g, n, B, H, D, scale=QK_SCALE),
                v=_randn(g, n, B, H, D))


def _prefill_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    B, S, H, R, D = case["batch"], case["seq"], case["heads"], case["group"], case["dim"]
    slots = kvcache.slot_stride_for(S)
    mask = torch.arange(S, device=DEV)[None, :] >= _left_pads(g, B, case["pad"])[:, None]
    return dict(q=_randn(g, B, S, H, R, D, scale=QK_SCALE),
                k=_randn(g, *kvcache.key_shape(B, H, slots, D), scale=QK_SCALE),
                vt=_randn(g, B, H, slots // 8, D, 8), mask=mask)


def _append_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    B, S, H, R, D = case["batch"], case["seq"], case["heads"], case["group"], case["dim"]
    rows = _randn(g, B, S, (R + 2) * H * D)  # one layer's q/k/v projection output
    cos, sin = _rotary(torch.arange(S, device=DEV).expand(B, S), D, 1e4)
    chunk = kvcache.slot_stride_for(S)
    return dict(
        q=rows[..., : H * R * D].view(B, S, H, R, D), k=rows[..., H * R * D: H * (R + 1) * D].view(B, S, H, D),
        v=rows[..., H * (R + 1) * D:].view(B, S, H, D), cos=cos.float().contiguous(), sin=sin.float().contiguous(),
        qw=(QK_SCALE * (1 + 0.1 * _randn(g, D, dtype=torch.float32))).to(BF16),
        kw=(QK_SCALE * (1 + 0.1 * _randn(g, D, dtype=torch.float32))).to(BF16),
        layer=kvcache.new_layer_cache(B, H, D, min(case["capacity"], S + 64) if case["ring"] else case["capacity"],
                                      case["ring"], BF16, DEV),
        q_out=torch.empty((B, S, H, R, D), dtype=BF16, device=DEV),
        # a ring layer's chunk keeps its own K/V for the prefill attention (zeroed, as the model's)
        k_out=torch.zeros(kvcache.key_shape(B, H, chunk, D), dtype=BF16, device=DEV) if case["ring"] else None,
        vt_out=torch.zeros((B, H, chunk // 8, D, 8), dtype=BF16, device=DEV) if case["ring"] else None)


def _mlp_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    T, M, F = case["rows"], case["hidden"], case["ffn"]
    return dict(h=_randn(g, T, M), x=_randn(g, T, M), gate_up=_randn(g, 2 * F, M, scale=0.02),
                down=_randn(g, M, F, scale=0.02), post=(1 + _randn(g, M, scale=0.1)), nxt=(1 + _randn(g, M, scale=0.1)),
                scalar=torch.ones(1, dtype=torch.float32, device=DEV))


def _draw_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    return dict(x=_randn(g, case["rows"], case["hidden"]),
                embed=_randn(g, case["vocab"], case["hidden"], scale=2.0 / math.sqrt(case["hidden"])),
                key=torch.randint(-2**31, 2**31 - 1, (2,), device=DEV, generator=g).to(torch.int32))


class _Weights:
    """The E2B-like model's weights and their packed form, loaded once and kept, as a program does."""

    live: "weakref.WeakValueDictionary[str, _Weights]" = weakref.WeakValueDictionary()

    def __init__(self) -> None:
        self.cfg = cfg = config.config_from_hf(E2B)
        g = _gen(20240)
        M, F, D, H = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim, cfg.num_key_value_heads
        R = cfg.num_attention_heads // H
        norm = lambda n, v=1.0: model.RMSNormParams(torch.full((n,), v, dtype=BF16, device=DEV))  # noqa: E731
        w = lambda *shape: _randn(g, *shape, scale=0.02)  # noqa: E731
        layers = []
        for i in range(cfg.num_hidden_layers):
            own = i < cfg.num_hidden_layers - cfg.num_kv_shared_layers
            att = model.AttentionParams(w(M, R, H, D), w(M, H, D) if own else None, w(M, H, D) if own else None,
                                        w(R, H, D, M), norm(D, QK_SCALE), norm(D, QK_SCALE) if own else None)
            layers.append(model.DecoderLayerParams(norm(M), att, norm(M), norm(M),
                                                   model.MLPParams(w(M, F), w(M, F), w(F, M)), norm(M), None,
                                                   torch.ones((), dtype=BF16, device=DEV)))
        self.params = model.Gemma4TextParams(w(cfg.vocab_size, M), None, None, None, tuple(layers), norm(M))
        self.packed = model.pack_weights(self.params, cfg)

    @classmethod
    def get(cls) -> "_Weights":
        held = cls.live.get("e2b")
        if held is None:
            held = cls.live["e2b"] = cls()
        return held


def _step_inputs(case: dict, seed: int) -> dict:
    weights = _Weights.get()
    cfg, g, B, n = weights.cfg, _gen(seed), case["batch"], case["length"]
    cache = kvcache.init_kv_cache(cfg, B, case["capacity"], BF16, DEV)
    for layer in cache.layers:
        if layer is not None:
            layer.key.normal_(0.0, QK_SCALE, generator=g)
            layer.value_t.normal_(generator=g)
    pads = _left_pads(g, B, case["pad"])
    slots = torch.arange(case["capacity"], device=DEV)[None, :]
    cache.key_mask.copy_((slots >= pads[:, None]) & (slots < n))
    return dict(weights=weights, cache=cache._replace(length=n),
                tok=torch.randint(0, cfg.vocab_size, (B,), device=DEV, generator=g).to(torch.int32),
                pos=(n - pads).to(torch.int32), active=torch.ones((B, 1), dtype=torch.bool, device=DEV),
                slot=torch.full((B,), n, dtype=torch.int32, device=DEV))


def _prompt_inputs(case: dict, seed: int) -> dict:
    weights, g = _Weights.get(), _gen(seed)
    B, S = case["batch"], case["seq"]
    return dict(weights=weights, ids=torch.randint(0, weights.cfg.vocab_size, (B, S), device=DEV, generator=g).to(torch.int32),
                mask=torch.arange(S, device=DEV)[None, :] >= _left_pads(g, B, case["pad"])[:, None])


_INPUTS = dict(decode=_decode_inputs, prefill=_prefill_inputs, append=_append_inputs, mlp=_mlp_inputs, draw=_draw_inputs,
               step=_step_inputs, prompt=_prompt_inputs)


def _decode_pass(s: dict) -> list:
    return [kernels.decode_attention(layer, s["q"][i], s["mask"], q_pos=s["q_pos"], window=s["window"],
                                     out=s["out"][i], new_k=s["k"][i], new_v=s["v"][i])
            for i, layer in enumerate(s["layers"])]


def _step_pass(s: dict) -> torch.Tensor:
    w = s["weights"]
    return model.forward_gemma4_lm(w.params, s["tok"][:, None], s["pos"][:, None], config=w.cfg,
                                   attention_mask=s["active"], kv_cache=s["cache"], cache_mode="append",
                                   logits_to_keep=1, write_pos=s["slot"]).logits


def _capture(s: dict, run_pass) -> None:
    """The step as a HIP graph (``s["graph"]``, its outputs ``s["result"]``), after one eager pass."""

    _lib.init_device(torch.cuda.current_device())
    run_pass(s)
    torch.cuda.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.cuda.graph(s["graph"], stream=side):
        s["result"] = run_pass(s)
    torch.cuda.current_stream().wait_stream(side)


def prepare(case: dict, seed: int) -> dict:
    s = _INPUTS[case["kind"]](case, seed)
    s["case"] = case
    if case["kind"] == "decode":
        s["out"] = torch.empty_like(s["q"])
        _capture(s, _decode_pass)
    elif case["kind"] == "step":
        _capture(s, _step_pass)
    return s


def run(s: dict):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        s["graph"].replay()
        return [s["out"], [(c.key, c.value_t) for c in s["layers"]]]
    if kind == "step":
        s["graph"].replay()
        return [s["result"], [(c.key, c.value_t) for c in s["cache"].layers if c is not None]]
    if kind == "prefill":
        return kernels.prefill_attention(s["q"], s["k"], s["vt"], s["mask"], window=case["window"])
    if kind == "append":
        kernels.kv_append(s["layer"], s["k"], s["v"], write_pos=0, flags=APPEND_FLAGS, eps=EPS, q=s["q"],
                          q_out=s["q_out"], q_norm_weight=s["qw"], k_norm_weight=s["kw"], rope_cos=s["cos"],
                          rope_sin=s["sin"], k_out=s["k_out"], vt_out=s["vt_out"])
        return [s["q_out"], s["layer"].key, s["layer"].value_t, s["k_out"], s["vt_out"]]
    if kind == "mlp":
        act = kernels.linear_gelu(s["h"], s["gate_up"])
        parts = kernels.linear_partials(act, s["down"], ksplit=model.DOWN_KSPLIT)
        return kernels.residual_norm_splitk(parts, s["post"], s["x"], scalar=s["scalar"], next_weight=s["nxt"], eps=EPS)
    if kind == "draw":
        if not case["top_k"]:
            return kernels.lm_head_sample(s["x"], s["embed"], softcap=SOFTCAP, temperature=case["temperature"],
                                          key=s["key"], split_key=False)
        logits = kernels.lm_head(s["x"], s["embed"])
        token, logp = kernels.sample_top_k(logits, softcap=SOFTCAP, temperature=case["temperature"],
                                           top_k=case["top_k"], top_p=case["top_p"], key=s["key"], split_key=False)
        return [logits, token, logp]
    w = s["weights"]
    out = sampler.prefill(w.params, w.cfg, s["ids"], s["mask"], max_new_tokens=case["new"])
    return [out.logits, [(c.key, c.value_t) for c in out.kv_cache.layers if c is not None]]


# --- the work of a pass ------------------------------------------------------------------------------


def _pairs(seq: int, window: int, pad: int) -> float:
    """Mean number of (query, key) pairs of one head over left pads uniform in [0, pad]."""

    def of(n: int) -> int:
        w = min(window, n) if window else n
        return w * (w + 1) // 2 + (n - w) * w

    pads = [round(i * pad / 16) for i in range(17)] if pad else [0]
    return sum(of(seq - p) for p in pads) / len(pads)


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "decode":
        B, H, R, D = case["batch"], case["heads"], case["group"], case["dim"]
        slots = [p + 1 - case["pad"] / 2 for p in range(case["lo"], case["hi"])]
        if case["ring"]:
            slots = [min(n, case["capacity"]) for n in slots]
        valid = sum(slots) / len(slots) * B * H
        return {"bytes": case["layers"] * 2 * (2 * valid * D + 2 * B * H * R * D + 4 * B * H * D),
                "flops": case["layers"] * 4 * valid * R * D}
    if kind == "prefill":
        B, S, H, R, D = case["batch"], case["seq"], case["heads"], case["group"], case["dim"]
        return {"bytes": 2 * B * S * H * D * (2 * R + 2),
                "flops": 4 * B * H * R * D * _pairs(S, case["window"], case["pad"])}
    if kind == "append":
        B, S, H, R, D = case["batch"], case["seq"], case["heads"], case["group"], case["dim"]
        kept = min(S, case["capacity"]) if case["ring"] else S
        rows = 2 * S * (R + 2) + 2 * kept + (2 * S if case["ring"] else 0) - 2 * S
        return {"bytes": 2 * B * H * D * rows + 8 * B * S * D, "flops": 10 * B * S * H * (R + 2) * D}
    if kind == "mlp":
        T, M, F = case["rows"], case["hidden"], case["ffn"]
        return {"bytes": 2 * (3 * M * F + 4 * T * M), "flops": 6 * T * M * F}
    if kind == "draw":
        T, V, M = case["rows"], case["vocab"], case["hidden"]
        logits = 2 * T * V if case["top_k"] else 0
        return {"bytes": 2 * (V + T) * M + logits, "flops": 2 * T * V * M}
    cfg = config.config_from_hf(E2B)
    M, F, V, L = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size, cfg.num_hidden_layers
    HD, KD = cfg.num_attention_heads * cfg.head_dim, cfg.num_key_value_heads * cfg.head_dim
    own = L - cfg.num_kv_shared_layers
    weights = L * (2 * M * HD + 3 * M * F) + own * 2 * M * KD
    B = case["batch"]
    if kind == "step":
        n = case["length"] + 1 - case["pad"] / 2
        slots = sum(min(n, cfg.sliding_window) if t == config.SLIDING else n for t in cfg.layer_types)
        return {"bytes": 2 * (weights + V * M + 2 * B * slots * KD + B * V),
                "flops": 2 * B * (weights + V * M) + 4 * B * slots * HD}
    tokens = B * (case["seq"] - case["pad"] / 2)
    pairs = sum(_pairs(case["seq"], cfg.sliding_window if t == config.SLIDING else 0, case["pad"])
                for t in cfg.layer_types)
    cache = 2 * B * own * KD * case["seq"]
    return {"bytes": 2 * (weights + V * M + cache + B * V + tokens * M),
            "flops": 2 * tokens * weights + 2 * B * V * M + 4 * B * pairs * HD}


# --- tolerances ------------------------------------------------------------------------------------------

# About four times what another order of the sums shows (the kernels' other split choices, the down
# projection over 4 K ranges instead of 8, f32 library products, attention in f32 torch with the same
# rounding points): single bf16 roundings that fall the other way, rel 2e-5 .. 8e-5 and max 0.008 in one
# kernel; rel 0.015 .. 0.019 and max 0.15 (logits), 0.1 (caches) after 30 layers.
_TOLERANCE = {
    "decode": {"rel": 3e-4, "max": 0.03},
    "prefill": {"rel": 3e-4, "max": 0.03},
    "append": {"rel": 1e-4, "max": 0.03},
    "mlp": {"rel": 2e-4, "max": 0.03},
    "draw": {"rel": 1e-3, "max": 0.05, "differ": 0.01},
    "step": {"rel": 0.07, "max": 0.6},
    "prompt": {"rel": 0.08, "max": 0.4},
}


def tolerance(case: dict):
    return dict(_TOLERANCE[case["kind"]])


# --- 64-bit restatement ----------------------------------------------------------------------------------


def _slots_of_keys(kt: torch.Tensor) -> torch.Tensor:
    """The stored key layout -> ``[B, H, slots, D]``: blocks (32-slot chunk, 32 dims, half) of 16 lanes
    x 32 dims, lane 4 a + c of half b holding slot 8 a + 4 b + c of the chunk."""

    B, H, C, N, _, _, kr = kt.shape
    return kt.reshape(B, H, C, N, 2, 4, 4, kr).permute(0, 1, 2, 5, 4, 6, 3, 7).reshape(B, H, C * 32, N * kr)


def _keys_of_slots(k: torch.Tensor) -> torch.Tensor:
    B, H, S, D = k.shape
    t = k.reshape(B, H, S // 32, 4, 2, 4, D // 32, 32).permute(0, 1, 2, 6, 4, 3, 5, 7)
    return t.reshape(B, H, S // 32, D // 32, 2, 16, 32)


def _slots_of_values(vt: torch.Tensor) -> torch.Tensor:
    """Values in groups of 8 slots, each group dim-major -> ``[B, H, slots, D]``."""

    B, H, G, D, _ = vt.shape
    return vt.transpose(3, 4).reshape(B, H, G * 8, D)


def _values_of_slots(v: torch.Tensor) -> torch.Tensor:
    B, H, S, D = v.shape
    return v.reshape(B, H, S // 8, 8, D).transpose(3, 4)


def _attend64(q, k, v, valid):
    """softmax over the valid keys (over all of them where a row has none): q ``[N, D]``, k / v
    ``[T, D]``, valid ``[N, T]``."""

    scores = (q @ k.T).masked_fill(~valid, torch.finfo(torch.float64).min)
    return torch.softmax(scores, -1) @ v


def _exact_decode(case: dict, seed: int):
    s = _decode_inputs(case, seed)
    B, H, D, C = case["batch"], case["heads"], case["dim"], case["capacity"]
    outs, caches = [], []
    slot = torch.arange(C, device=DEV)
    for i, layer in enumerate(s["layers"]):
        k, v = _slots_of_keys(layer.key).clone(), _slots_of_values(layer.value_t).clone()
        rows = torch.empty((B, H, case["group"], D), dtype=torch.float64, device=DEV)
        for b in range(B):
            p = int(s["q_pos"][b])
            k[b, :, p % C if case["ring"] else p], v[b, :, p % C if case["ring"] else p] = s["k"][i, b], s["v"][i, b]
            held = slot + torch.div(p - slot, C, rounding_mode="floor") * C if case["ring"] else slot
            ok = (held >= 0) & (held <= p) & s["mask"][b, held.clamp(0, s["mask"].shape[1] - 1)]
            for h in range(H):
                rows[b, h] = _attend64(s["q"][i, b, h].double(), k[b, h, :C].double(), v[b, h, :C].double(),
                                       ok[None].expand(case["group"], C))
        outs.append(rows)
        caches.append((_keys_of_slots(k), _values_of_slots(v)))
    return [torch.stack(outs), caches]


def _exact_prefill(case: dict, seed: int):
    s = _prefill_inputs(case, seed)
    B, S, H, R, D = s["q"].shape
    k, v = _slots_of_keys(s["k"])[:, :, :S], _slots_of_values(s["vt"])[:, :, :S]
    at = torch.arange(S, device=DEV)
    seen = at[None, :] <= at[:, None]
    if case["window"]:
        seen &= at[None, :] > at[:, None] - case["window"]
    out = torch.empty((B, S, H, R, D), dtype=torch.float64, device=DEV)
    for b in range(B):
        ok = seen & s["mask"][b][None, :]
        for h in range(H):
            for r in range(R):
                out[b, :, h, r] = _attend64(s["q"][b, :, h, r].double(), k[b, h].double(), v[b, h].double(), ok)
    return out


def _norm64(x, w=None):
    y = x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt()
    return y if w is None else y * w.double()


def _rope64(x, cos, sin):
    a, b = x.chunk(2, -1)
    return x * cos + torch.cat([-b, a], -1) * sin


def _exact_append(case: dict, seed: int):
    s = _append_inputs(case, seed)
    cos, sin = s["cos"].double(), s["sin"].double()
    q = _rope64(_norm64(s["q"].double(), s["qw"]), cos[:, :, None, None], sin[:, :, None, None])
    k = _rope64(_norm64(s["k"].double(), s["kw"]), cos[:, :, None], sin[:, :, None]).transpose(1, 2)
    v = _norm64(s["v"].double()).transpose(1, 2)
    B, H, S, D = k.shape
    layer = s["layer"]
    last = min(S, layer.capacity)
    at = torch.arange(S - last, S, device=DEV) % layer.capacity
    slots = lambda t, n, to: t.new_zeros((B, H, n, D)).index_copy_(2, to, t[:, :, -len(to):])  # noqa: E731
    whole = torch.arange(S, device=DEV)
    chunk = kvcache.slot_stride_for(S)
    return [q, _keys_of_slots(slots(k, layer.slot_stride, at)), _values_of_slots(slots(v, layer.slot_stride, at)),
            _keys_of_slots(slots(k, chunk, whole)) if case["ring"] else None,
            _values_of_slots(slots(v, chunk, whole)) if case["ring"] else None]


def _gelu64(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _exact_mlp(case: dict, seed: int):
    s = _mlp_inputs(case, seed)
    g, u = (s["h"].double() @ s["gate_up"].double().T).chunk(2, -1)
    x = s["x"].double() + _norm64((_gelu64(g) * u) @ s["down"].double().T, s["post"])
    return [x, _norm64(x, s["nxt"])]


def _threefry64(k0: int, k1: int, flat: torch.Tensor) -> torch.Tensor:
    """threefry2x32-20 (Salmon et al. 2011) of the 64-bit counters ``flat``, its two words xored: JAX's
    partitionable random bits."""

    low = 0xFFFFFFFF
    ks = (k0, k1, k0 ^ k1 ^ 0x1BD11BDA)
    x0, x1 = ((flat >> 32) + ks[0]) & low, ((flat & low) + ks[1]) & low
    for i in range(5):
        for r in ((13, 15, 26, 6), (17, 29, 16, 24))[i % 2]:
            x0 = (x0 + x1) & low
            x1 = (((x1 << r) | (x1 >> (32 - r))) & low) ^ x0
        x0, x1 = (x0 + ks[(i + 1) % 3]) & low, (x1 + ks[(i + 2) % 3] + i + 1) & low
    return x0 ^ x1


def _gumbel64(key: torch.Tensor, first: int, rows: int, cols: int) -> torch.Tensor:
    """Gumbel noise of rows ``first`` .. ``first + rows`` of a ``cols``-wide draw: the uniform from the top
    23 bits, floored at the smallest normal float."""

    k0, k1 = (int(w) & 0xFFFFFFFF for w in key)
    flat = torch.arange(first * cols, (first + rows) * cols, device=DEV, dtype=torch.int64)
    u = (_threefry64(k0, k1, flat) >> 9).double() * 2.0 ** -23
    return -(-u.clamp_min(2.0 ** -126).log()).log().reshape(rows, cols)


def _exact_draw(case: dict, seed: int):
    """The logits' two roundings to bf16 (the product's and the soft-cap's) are part of what is drawn
    from, so they are kept: the token is then the same up to ties."""

    s = _draw_inputs(case, seed)
    logits, tokens, logps = [], [], []
    embed = s["embed"].double()
    for first in range(0, case["rows"], 16):
        raw = s["x"][first: first + 16].double() @ embed.T
        x = ((raw.to(BF16).double() / SOFTCAP).tanh() * SOFTCAP).to(BF16).double()
        scores, ids = x / case["temperature"], None
        if case["top_k"]:
            scores, ids = torch.sort(scores, dim=-1, descending=True, stable=True)
            scores, ids = scores[:, : case["top_k"]], ids[:, : case["top_k"]]
            mass = torch.softmax(scores, -1)
            before = torch.cumsum(mass, -1) - mass
            scores = scores.masked_fill((before >= case["top_p"]) & (before > 0), -math.inf)
        token = (scores + _gumbel64(s["key"], first, *scores.shape)).argmax(-1, keepdim=True)
        token = token if ids is None else ids.gather(1, token)
        tokens.append(token[:, 0].to(torch.int32))
        logps.append(torch.log_softmax(x, -1).gather(1, token)[:, 0])
        if case["top_k"]:
            logits.append(raw)
    return ([torch.cat(logits)] if case["top_k"] else []) + [torch.cat(tokens), torch.cat(logps)]


def _model64(weights: _Weights, ids, pos, attend) -> torch.Tensor:
    """The decoder in 64 bits up to the final norm; ``attend(layer, q, k, v)`` attends q ``[B, S, H, R, D]``
    (k / v ``[B, S, H, D]``, None on a layer that shares another's)."""

    cfg, p = weights.cfg, weights.params
    scale = float(torch.tensor(math.sqrt(cfg.hidden_size), dtype=BF16))
    x = p.embed_tokens[ids.long()].double() * scale
    rot = {config.SLIDING: _rotary(pos, cfg.head_dim, cfg.rope_theta_sliding),
           config.FULL: _rotary(pos, cfg.global_head_dim, cfg.rope_theta_full, cfg.full_partial_rotary_factor)}
    for i, lp in enumerate(p.layers):
        a = lp.attention
        cos, sin = rot[cfg.layer_types[i]]
        h = _norm64(x, lp.input_norm.weight)
        M, R, H, D = a.q_proj.shape
        q = (h @ a.q_proj.double().reshape(M, -1)).reshape(*h.shape[:2], R, H, D).transpose(2, 3)
        q = _rope64(_norm64(q, a.q_norm.weight), cos[:, :, None, None], sin[:, :, None, None])
        k = v = None
        if a.k_proj is not None:
            k = (h @ a.k_proj.double().reshape(M, -1)).reshape(*h.shape[:2], H, D)
            k = _rope64(_norm64(k, a.k_norm.weight), cos[:, :, None], sin[:, :, None])
            v = _norm64((h @ a.v_proj.double().reshape(M, -1)).reshape(*h.shape[:2], H, D))
        o = attend(i, q, k, v).transpose(2, 3).reshape(*h.shape[:2], -1) @ a.o_proj.double().reshape(-1, M)
        x = x + _norm64(o, lp.post_attention_norm.weight)
        h = _norm64(x, lp.pre_feedforward_norm.weight)
        act = _gelu64(h @ lp.mlp.gate_proj.double()) * (h @ lp.mlp.up_proj.double())
        x = (x + _norm64(act @ lp.mlp.down_proj.double(), lp.post_feedforward_norm.weight)) * lp.layer_scalar.double()
    return _norm64(x, p.final_norm.weight)


def _source_layers(cfg) -> list[int]:
    """The layer whose K/V each layer reads: itself, or the last one of its type that has its own."""

    own = cfg.num_hidden_layers - cfg.num_kv_shared_layers
    last = {t: max(i for i in range(own) if cfg.layer_types[i] == t) for t in set(cfg.layer_types)}
    return [i if i < own else last[t] for i, t in enumerate(cfg.layer_types)]


def _logits64(weights: _Weights, hidden) -> torch.Tensor:
    raw = hidden.reshape(-1, hidden.shape[-1]) @ weights.params.embed_tokens.double().T
    return ((raw / SOFTCAP).tanh() * SOFTCAP).reshape(*hidden.shape[:2], -1)


def _exact_step(case: dict, seed: int):
    s = _step_inputs(case, seed)
    weights, cache, n = s["weights"], s["cache"], case["length"]
    source, held, written = _source_layers(weights.cfg), {}, {}

    def attend(i, q, k, v):
        layer = cache.layers[source[i]]
        C = layer.capacity
        if k is not None:
            held.clear()  # two layers' worth of 64-bit keys at most
            at = n % C
            kk, vv = _slots_of_keys(layer.key)[:, :, :C].double(), _slots_of_values(layer.value_t)[:, :, :C].double()
            kk[:, :, at], vv[:, :, at] = k[:, 0], v[:, 0]
            held[i] = kk, vv
            written[i] = (k[:, 0], v[:, 0])
        elif source[i] not in held:
            kk, vv = _slots_of_keys(layer.key)[:, :, :C].double(), _slots_of_values(layer.value_t)[:, :, :C].double()
            kk[:, :, n % C], vv[:, :, n % C] = written[source[i]]
            held[source[i]] = kk, vv
        kk, vv = held[source[i]]
        slot = torch.arange(C, device=DEV)
        pos = slot + torch.div(n - slot, C, rounding_mode="floor") * C if layer.ring else slot
        ok = (pos >= 0) & (pos <= n) & (cache.key_mask[:, pos.clamp(0)] | (pos == n))
        scores = torch.matmul(q[:, 0], kk.transpose(2, 3).contiguous())
        scores = scores.masked_fill(~ok[:, None, None, :], torch.finfo(torch.float64).min)
        return torch.matmul(torch.softmax(scores, -1), vv)[:, None]

    hidden = _model64(weights, s["tok"][:, None], s["pos"][:, None], attend)
    return [_logits64(weights, hidden), [(None, None) for c in cache.layers if c is not None]]


def _exact_prompt(case: dict, seed: int):
    s = _prompt_inputs(case, seed)
    weights, mask = s["weights"], s["mask"]
    cfg, S = weights.cfg, case["seq"]
    source, held = _source_layers(cfg), {}
    at = torch.arange(S, device=DEV)

    def attend(i, q, k, v):
        if k is not None:
            held[i] = (k, v)
        k, v = held[source[i]]
        seen = at[None, :] <= at[:, None]
        if cfg.layer_types[i] == config.SLIDING:
            seen = seen & (at[None, :] > at[:, None] - cfg.sliding_window)
        out = torch.empty_like(q)
        for b in range(q.shape[0]):
            ok = seen & mask[b][None, :]
            for h in range(q.shape[2]):
                for r in range(q.shape[3]):
                    out[b, :, h, r] = _attend64(q[b, :, h, r], k[b, :, h], v[b, :, h], ok)
        return out

    pos = (mask.cumsum(-1) - 1).clamp_min(0)
    hidden = _model64(weights, s["ids"], pos, attend)
    own = cfg.num_hidden_layers - cfg.num_kv_shared_layers
    return [_logits64(weights, hidden[:, -1:]), [(None, None) for _ in range(own)]]


_EXACT = dict(decode=_exact_decode, prefill=_exact_prefill, append=_exact_append, mlp=_exact_mlp, draw=_exact_draw,
              step=_exact_step, prompt=_exact_prompt)


def exact(case: dict, seed: int):
    return _EXACT[case["kind"]](case, seed)
