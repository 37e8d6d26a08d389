"""Prefill-sized appends (one token per wave) against the same tokens appended one at a time, bit for bit:
head counts that leave a remainder of the vectors a wave loads together, each flag by itself, q or k/v
absent, chunks with a partial last tile, a ring smaller than a tile."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gemma4_posttrain_jax_amd import _lib, kernels
from gemma4_posttrain_jax_amd.kvcache import new_layer_cache
from gpu_util import bits

pytestmark = pytest.mark.gpu

NORM_Q, ROPE_Q = _lib.G4_APPEND_NORM_Q, _lib.G4_APPEND_ROPE_Q
NORM_K, ROPE_K, NORM_V = _lib.G4_APPEND_NORM_K, _lib.G4_APPEND_ROPE_K, _lib.G4_APPEND_NORM_V
ALL = NORM_Q | ROPE_Q | NORM_K | ROPE_K | NORM_V


@pytest.mark.parametrize("D", [128, 256, 512])
@pytest.mark.parametrize("H,R,S,cap,ring,start,flags,with_q,with_kv", [
    (1, 1, 8, 8, True, 0, ALL, True, True),
    (3, 3, 13, 24, True, 5, ALL, True, True),
    (2, 4, 17, 5, True, 3, ALL, True, True),
    (3, 1, 16, 40, False, 8, ALL, False, True),
    (1, 5, 9, 9, False, 0, ROPE_K | NORM_V, True, True),
    (2, 2, 8, 64, False, 16, NORM_Q | ROPE_Q, True, False),
    (1, 6, 24, 64, False, 1, NORM_K, True, True),
    (2, 1, 16, 16, True, 16, ROPE_Q, True, True),
])
def test_tiles_match_single_tokens(device, D, H, R, S, cap, ring, start, flags, with_q, with_kv):
    g = torch.Generator(device=device).manual_seed(D + S)
    B, td = 2, torch.bfloat16
    randn = lambda *shape: torch.empty(shape, dtype=td, device=device).normal_(generator=g)  # noqa: E731
    rows = randn(B, S, (R + 2) * H * D)
    q = rows[..., : H * R * D].view(B, S, H, R, D)
    k = rows[..., H * R * D: H * (R + 1) * D].view(B, S, H, D)
    v = rows[..., H * (R + 1) * D:].view(B, S, H, D)
    # cos / sin of a row's two halves differ, as the entry point allows
    cos, sin = (torch.empty((B, S, D), device=device).uniform_(-1, 1, generator=g) for _ in range(2))
    qw, kw = randn(D), randn(D)

    def append(layer, a, b, pos):
        cut = slice(a, b)
        q_out = torch.zeros((B, b - a, H, R, D), dtype=td, device=device)
        args = dict(flags=flags, eps=1e-6, q_norm_weight=qw, rope_cos=cos[:, cut].contiguous(),
                    rope_sin=sin[:, cut].contiguous())
        if not with_kv:
            kernels.prepare_q(q[:, cut], q_out, **args)
        else:
            kernels.kv_append(layer, k[:, cut], v[:, cut], write_pos=pos, k_norm_weight=kw,
                              **(dict(q=q[:, cut], q_out=q_out) if with_q else {}), **args)
        return q_out

    tiled, single = (new_layer_cache(B, H, D, cap, ring, td, device) for _ in range(2))
    q_tiled = append(tiled, 0, S, start)
    q_single = torch.cat([append(single, s, s + 1, start + s) for s in range(S)], 1)
    np.testing.assert_array_equal(bits(q_tiled), bits(q_single))
    np.testing.assert_array_equal(bits(tiled.key), bits(single.key))
    np.testing.assert_array_equal(bits(tiled.value_t), bits(single.value_t))
