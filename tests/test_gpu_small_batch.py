"""Small decode batches: the kernels and dispatch lines that only few rows reach, at the edges of their
ranges (the larger batches are covered beside each kernel's own tests)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gemma4_posttrain_jax_amd import _lib, kernels
from gemma4_posttrain_jax_amd import config as C
from gemma4_posttrain_jax_amd import model as M
from gemma4_posttrain_jax_amd import sampler as SMP
from gemma4_posttrain_jax_amd.kvcache import new_layer_cache
from gemma4_posttrain_jax_amd.model import rotary_tables
from oracle import g4_oracle as O
from test_gpu_decode_prep import PREP_CFG
from test_gpu_kernels import _decode_case

pytestmark = pytest.mark.gpu

APPEND_FLAGS = (_lib.G4_APPEND_NORM_Q | _lib.G4_APPEND_ROPE_Q | _lib.G4_APPEND_NORM_K | _lib.G4_APPEND_ROPE_K
                | _lib.G4_APPEND_NORM_V)


# 32 / 34 pairs: the last count whose scores launch runs 2-wave workgroups and the first that does not;
# 512 / 513 slots: the one-launch kernel's longest row and the first that only two launches take
@pytest.mark.parametrize("B,D,ring,cap", [(1, 256, True, 512), (16, 256, True, 512), (17, 256, False, 512),
                                          (1, 256, False, 513), (66, 256, True, 512), (16, 128, False, 700),
                                          (17, 512, False, 33), (2, 512, False, 1024)])
def test_decode_few_pairs_automatic(device, B, D, ring, cap):
    rng = np.random.default_rng(B + D + cap)
    q_pos = rng.integers(cap, 3 * cap, B) if ring else rng.integers(0, cap, B)
    km = np.ones((B, max(cap, int(q_pos.max()) + 1)), bool)
    km[0, : int(q_pos[0]) // 2] = False  # a left-padded row
    _decode_case(device, O.BF16, B=B, H=2, R=4, D=D, cap=cap, ring=ring, window=cap if ring else 0, q_pos=q_pos,
                 key_mask=km, fused=True, seed=cap + B)


@pytest.mark.parametrize("R,ring,cap", [(4, True, 512), (1, False, 768), (16, True, 100)])
def test_fused_preparation_of_one_row(device, R, ring, cap):
    """One row (its batch stride is arbitrary) through the fused preparation: bit for bit the append and
    the attention run separately."""

    B, H, D = 1, 2, 256
    g = torch.Generator(device="cuda").manual_seed(R + cap)
    qkv = torch.randn((B, 1, (H * R + 2 * H) * D), device="cuda", generator=g).to(torch.bfloat16)
    q = qkv[..., :H * R * D].view(B, 1, H, R, D)
    k = qkv[..., H * R * D:(H * R + H) * D].view(B, 1, H, D)
    v = qkv[..., (H * R + H) * D:].view(B, 1, H, D)
    layers = [new_layer_cache(B, H, D, cap, ring, torch.bfloat16, device) for _ in range(2)]
    layers[0].key.normal_(generator=g)
    layers[0].value_t.normal_(generator=g)
    layers[1].key.copy_(layers[0].key)
    layers[1].value_t.copy_(layers[0].value_t)
    pos = cap + 7 if ring else cap - 1
    q_pos = torch.full((B,), pos, dtype=torch.int32, device=device)
    km = torch.ones((B, pos + 1), dtype=torch.bool, device=device)
    w = [(1 + 0.1 * torch.randn(D, device="cuda", generator=g)).to(torch.bfloat16) for _ in range(2)]
    inv = (1.0 / (10000.0 ** (torch.arange(0, D, 2, device="cuda", dtype=torch.float32) / D))).contiguous()
    cos, sin = rotary_tables(inv, q_pos[:, None])
    q_out = torch.empty((B, 1, H, R, D), dtype=torch.bfloat16, device=device)
    window = cap if ring else 0
    kernels.kv_append(layers[1], k, v, write_pos=q_pos, flags=APPEND_FLAGS, q=q, q_out=q_out, q_norm_weight=w[0],
                      k_norm_weight=w[1], rope_cos=cos, rope_sin=sin)
    want = kernels.decode_attention(layers[1], q_out.view(B, H, R, D), km, q_pos=q_pos, window=window,
                                    num_splits=_lib.G4_DECODE_TWO_PASS)
    got = kernels.decode_attention_fused(layers[0], q[:, 0], km, q_pos=q_pos, window=window, k_raw=k[:, 0],
                                         v_raw=v[:, 0], q_norm_weight=w[0], k_norm_weight=w[1], rope_cos=cos[:, 0],
                                         rope_sin=sin[:, 0], eps=1e-6, flags=APPEND_FLAGS)
    for a, b in ((got, want), (layers[0].key, layers[1].key), (layers[0].value_t, layers[1].value_t)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


# rows at the edges of the row groups and of the tile choice, K ranges that leave waves without a line
# (64, 192), that do not divide among the waves (576) and that fill every slot; the bars as in
# test_gpu_linear: half a bf16 ulp of the f32-accumulated sum (the split sums are not rounded), and for the
# gated GELU the roundings of g, u and the product
@pytest.mark.parametrize("rows", [1, 16, 17, 33, 64, 65, 128, 192])
@pytest.mark.parametrize("n,k", [(64, 64), (128, 192), (320, 576), (3072, 2048), (4096, 640), (8256, 192)])
def test_few_row_linear(device, rows, n, k):
    g = torch.Generator(device="cuda").manual_seed(rows + n + k)
    x = torch.randn((rows, k), device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn((n, k), device="cuda", generator=g) * k ** -0.5).to(torch.bfloat16)
    ref = x.double() @ w.double().T
    slack = 2.0 ** -20 * (x.double().abs() @ w.double().abs().T)  # f32 sums of k products in any order
    out = torch.full((rows, n + 8), float("nan"), device="cuda", dtype=torch.bfloat16)
    y = kernels.linear(x, w, out=out[:, :n])
    assert torch.all((y.double() - ref).abs() <= ref.abs() * 2.0 ** -8 + slack)
    assert torch.isnan(out[:, n:].float()).all()  # columns past n untouched
    if k % 192 == 0:
        parts = kernels.linear_partials(x, w, ksplit=3)
        assert torch.all((parts.double().sum(0) - ref).abs() <= slack)
    gate, up = (t.to(torch.bfloat16).double() for t in ref.chunk(2, -1))
    want = torch.nn.functional.gelu(gate, approximate="tanh") * up
    got = kernels.linear_gelu(x, w).double()
    # g and u one rounding apart at most (2^-8 relative each, gelu'(g) <= 1.13 and gelu(g) ~ g / 2 below)
    bar = 2.0 ** -7 * (want.abs() + 1.2 * gate.abs() * up.abs()) + 2.0 * slack.chunk(2, -1)[0] * up.abs() + 1e-6
    assert torch.all((got - want).abs() <= bar)


@pytest.mark.parametrize("n,k,rows", [(4096, 192, 64), (36864, 4160, 56)])
def test_many_columns_keep_the_order_of_their_sums(device, n, k, rows):
    """Many columns: the streaming kernel's last batch and the ring kernel's first give a row the same bits."""

    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn((rows + 1, k), device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn((n, k), device="cuda", generator=g) * k ** -0.5).to(torch.bfloat16)
    for call in (kernels.linear, kernels.linear_gelu):
        few, more = call(x[:rows], w), call(x, w)
        assert int((few.view(torch.int16) != more[:rows].view(torch.int16)).sum()) == 0
    ref = x.double() @ w.double().T
    slack = 2.0 ** -20 * (x.double().abs() @ w.double().abs().T)
    assert torch.all((kernels.linear(x, w).double() - ref).abs() <= ref.abs() * 2.0 ** -8 + slack)


# the last batch of each row shape (64, 128, 256 rows per workgroup) and the first of the next
@pytest.mark.parametrize("rows", [1, 63, 64, 65, 128, 129])
@pytest.mark.parametrize("vocab,hidden", [(128, 32), (1280, 96)])
def test_lm_head_row_shapes(device, rows, vocab, hidden):
    """Logits within the bf16 rounding of their f32 sums; the draw on them equals sample_tokens' on the
    stored logits, token for token, at T = 1, another temperature and greedy (logp: f32 sums in another
    order, the reference's 2e-6)."""

    g = torch.Generator(device="cuda").manual_seed(rows + vocab)
    x = torch.randn((rows, hidden), device="cuda", generator=g).to(torch.bfloat16)
    embed = (torch.randn((vocab, hidden), device="cuda", generator=g) * 0.5).to(torch.bfloat16)
    logits = kernels.lm_head(x, embed)
    ref = x.double() @ embed.double().T
    slack = 2.0 ** -20 * (x.double().abs() @ embed.double().abs().T)
    assert torch.all((logits.double() - ref).abs() <= ref.abs() * 2.0 ** -8 + slack)
    key = torch.tensor([5, 6], dtype=torch.int32, device=device)
    for temperature in (1.0, 0.6, 0.0):
        args = dict(softcap=30.0, temperature=temperature, key=key, split_key=False)
        tok, logp = kernels.lm_head_sample(x, embed, **args)
        want_tok, want_logp = kernels.sample_tokens(logits, **args)
        assert torch.equal(tok, want_tok)
        assert torch.all((logp - want_logp).abs() <= 2e-6)


def test_step_with_norm_weights_at_odd_offsets(device, monkeypatch):
    """A graphed step whose q / k norm weights are views at odd offsets of one buffer: the logits of the step
    with weights of their own and the append run separately, bit for bit."""

    cfg = C.config_from_hf(PREP_CFG)
    params = M.params_from_numpy(O.init_params(O.config_from_hf(PREP_CFG), seed=5, dtype=O.BF16, std=0.03, norm_std=0.05,
                                               layer_scalar_min=0.8), cfg, dtype=torch.bfloat16, device=device)

    def moved(norm):
        return norm and M.RMSNormParams(torch.cat([norm.weight[:1], norm.weight])[1:])

    layers = [lp._replace(attention=lp.attention._replace(q_norm=moved(lp.attention.q_norm), k_norm=moved(lp.attention.k_norm)))
              for lp in params.layers]
    ids = torch.arange(24, dtype=torch.int32, device=device).view(2, 12) + 3
    mask = torch.ones_like(ids, dtype=torch.bool)
    active = torch.ones(2, dtype=torch.bool, device=device)
    logits = []
    for p in (params._replace(layers=tuple(layers)), params):
        out = SMP.prefill(p, cfg, ids, mask, max_new_tokens=4)
        engine = SMP.GraphedDecodeStep(p, cfg, out.kv_cache)
        logits.append(engine.step(ids[:, 0], mask.sum(-1, dtype=torch.int32), active).clone())
        monkeypatch.setattr(M, "_fused_decode_prep", lambda *args: False)
    assert torch.equal(logits[0], logits[1])


@pytest.mark.parametrize("moved", ["embed", "hidden"])
def test_lm_head_fallback_takes_any_offset(device, moved):
    """Logits of a vocabulary that the LM-head kernel does not take (no multiple of 128), from operands that
    start at an odd element of a larger buffer: within the bf16 rounding of their f32 sums."""

    g = torch.Generator(device="cuda").manual_seed(7)
    rows, vocab, hidden = 3, 192, 64
    x = torch.randn((rows * hidden + 1,), device="cuda", generator=g).to(torch.bfloat16)[int(moved == "hidden"):]
    e = torch.randn((vocab * hidden + 1,), device="cuda", generator=g).to(torch.bfloat16)[int(moved == "embed"):]
    x, e = x[: rows * hidden].view(rows, 1, hidden), e[: vocab * hidden].view(vocab, hidden)
    ref = x[:, 0].double() @ e.double().T
    slack = 2.0 ** -20 * (x[:, 0].double().abs() @ e.double().abs().T)
    got = M.forward_lm_head(e, x, None)[:, 0].double()
    assert torch.all((got - ref).abs() <= ref.abs() * 2.0 ** -8 + slack)


# both sides of each line of _native_proj_k: (rows, N, K) that it takes, and the first beyond
@pytest.mark.parametrize("rows,n,k,native", [
    (24, 4096, 5376, True), (25, 4096, 5376, False), (32, 4096, 4096, True), (33, 4096, 4096, False),
    (64, 4096, 2048, True), (65, 4096, 2048, False), (16, 8256, 2112, True), (17, 8256, 2112, False),
    (16, 192, 16384, True), (17, 192, 16384, False), (32, 192, 8192, True), (33, 192, 8192, False),
    (64, 192, 5376, True), (65, 192, 5376, False), (128, 1088, 4096, True), (129, 1088, 4096, False),
    (192, 1152, 2048, True), (192, 1152, 2112, False), (192, 2560, 4096, True), (193, 2560, 4096, False),
    (128, 2816, 640, True), (129, 2816, 640, False), (192, 3072, 640, True)])
def test_projection_routes(device, rows, n, k, native):
    """A projection takes the few-row GEMM where that was measured faster, the library's product beyond;
    either within the bf16 rounding of its f32 sums."""

    g = torch.Generator(device="cuda").manual_seed(rows + n)
    x = torch.randn((rows, k), device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn((n, k), device="cuda", generator=g) * k ** -0.5).to(torch.bfloat16)
    assert M._native_proj(x, w) is native
    ref = x.double() @ w.double().T
    slack = 2.0 ** -20 * (x.double().abs() @ w.double().abs().T)  # f32 sums of k products in any order
    assert torch.all((M._proj(x, w).double() - ref).abs() <= ref.abs() * 2.0 ** -8 + slack)


def test_lm_head_fallback_keeps_its_derivatives(device):
    """Logits of a vocabulary that the LM-head kernel does not take (no multiple of 128) are the library's
    product wherever a derivative or a transform follows them: reverse and forward mode, vmap."""

    g = torch.Generator(device="cuda").manual_seed(9)
    x = torch.randn((4, 1, 64), device="cuda", generator=g).to(torch.bfloat16)
    e = torch.randn((192, 64), device="cuda", generator=g).to(torch.bfloat16)
    want = M.forward_lm_head(e, x, None)
    with torch.no_grad():
        assert M._native_proj(x[:, 0].contiguous(), e)
    for operand in (x, e):
        with torch.enable_grad():  # other tests turn gradients off for the process
            leaf = operand.clone().requires_grad_()
            logits = M.forward_lm_head(leaf if operand is e else e, leaf if operand is x else x, None)
            (grad,) = torch.autograd.grad(logits.float().sum(), leaf)
        ref = e.float().sum(0).expand(4, 1, 64) if operand is x else x.float().sum((0, 1)).expand(192, 64)
        assert torch.allclose(grad.float(), ref, rtol=2.0 ** -7, atol=2.0 ** -4)
    tangent = torch.ones_like(x)
    value, jvp = torch.func.jvp(lambda h: M.forward_lm_head(e, h, None), (x,), (tangent,))
    assert torch.allclose(jvp.float(), M.forward_lm_head(e, tangent, None).float(), rtol=2.0 ** -7, atol=2.0 ** -4)
    assert torch.allclose(value.float(), want.float(), rtol=2.0 ** -7, atol=2.0 ** -4)
    stacked = torch.func.vmap(lambda h: M.forward_lm_head(e, h[None], None)[0])(x)
    assert torch.allclose(stacked.float(), want.float(), rtol=2.0 ** -7, atol=2.0 ** -4)
