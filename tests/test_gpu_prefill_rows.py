"""Prefill attention on the LDS-staged kernels where rows and grids can go wrong: rows without a valid key
(pads, whole rows), key masks whose first valid key lies anywhere in a chunk, holes, and the grid sizes
at which the number of column blocks per wave changes."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gemma4_posttrain_jax_amd import kernels
from gemma4_posttrain_jax_amd.kvcache import group_keys, group_values
from gpu_util import to_np
from oracle import g4_oracle as O

pytestmark = pytest.mark.gpu


def _check(device, B, S, H, R, D, window, key_mask, rows, seed):
    """q and k scaled so that scores are of order 1: the outputs (|o| < 4) then differ from the oracle's
    only by the rounding of probabilities and outputs, each at most half a bf16 ulp (2^-9 relative), plus
    the f32 sums: below 2e-2."""

    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g)  # noqa: E731
    q = (rnd(B, S, H, R, D) * D ** -0.25).to(torch.bfloat16)
    Sp = (S + 63) // 64 * 64
    k = (rnd(B, H, Sp, D) * D ** -0.25).to(torch.bfloat16)
    v = rnd(B, H, Sp, D).to(torch.bfloat16)
    km = torch.from_numpy(key_mask).to(device)
    out = to_np(kernels.prefill_attention(q, group_keys(k), group_values(v), km, window=window))
    masks = O.make_qk_masks(key_mask, window if window else 1 << 30, 0, S)[O.SLIDING]
    for b in rows:
        want = O.attention_core(to_np(q[b:b + 1]).transpose(0, 1, 3, 2, 4), to_np(k[b:b + 1, :, :S]).transpose(0, 2, 1, 3),
                                to_np(v[b:b + 1, :, :S]).transpose(0, 2, 1, 3), masks[b:b + 1], O.BF16)
        err = np.abs(out[b] - want.transpose(0, 1, 3, 2, 4)[0]).max()
        assert err <= 2e-2, f"row {b}: max |out - oracle| = {err}"


@pytest.mark.parametrize("D", [128, 256, 512])
@pytest.mark.parametrize("window", [0, 40])
def test_prefill_masked_rows(device, D, window):
    """Left pads that end on, before and after a chunk's and a workgroup's edge, every key masked, one
    valid key, and holes, one wider than the window."""

    S = 161
    pads = [0, 1, 31, 32, 33, 64, 65, 128, 160, 161]
    key_mask = np.arange(S)[None, :] >= np.array(pads + [0, 5])[:, None]
    key_mask[-2, 40:100] = False
    key_mask[-1, 6:160] = False
    _check(device, len(key_mask), S, 1, 4, D, window, key_mask, range(len(key_mask)), D + window)


# workgroups at two blocks per wave (64 positions at head dim 256, 32 at 512, R = 4): at and beyond 256
# (causal) and 128 (windowed)
@pytest.mark.parametrize("D,B,S,window", [(256, 32, 256, 0), (256, 32, 257, 0), (512, 32, 128, 0), (512, 32, 129, 0),
                                          (256, 16, 256, 70), (256, 16, 257, 70), (512, 16, 128, 70),
                                          (512, 16, 129, 70), (256, 8, 17, 0)])
def test_prefill_block_count_lines(device, D, B, S, window):
    key_mask = np.ones((B, S), bool)
    key_mask[1, : S // 2] = False
    _check(device, B, S, 2, 4, D, window, key_mask, (0, 1, B - 1), S + D)


@pytest.mark.parametrize("D,R", [(512, 1), (512, 16), (256, 16), (256, 1)])
def test_prefill_group_sizes_padded(device, D, R):
    key_mask = np.ones((2, 100), bool)
    key_mask[1, :37] = False
    _check(device, 2, 100, 2, R, D, 0, key_mask, (0, 1), D + R)


@pytest.mark.parametrize("D", [128, 256, 512])
@pytest.mark.parametrize("S", [33, 161, 1999])
def test_prefill_keyless_rows_sum_in_key_order(device, D, S):
    """A row without a valid key averages all S values, summed in key order: bit for bit the last row of the
    same values under scores that are all equal (q = 0: probabilities of 1 / S on every key)."""

    g = torch.Generator(device="cuda").manual_seed(D + S)
    H, R, Sp = 2, 4, (S + 63) // 64 * 64
    k = torch.randn((1, H, Sp, D), device="cuda", generator=g).to(torch.bfloat16).expand(2, H, Sp, D)
    v = torch.randn((1, H, Sp, D), device="cuda", generator=g).to(torch.bfloat16).expand(2, H, Sp, D)
    q = torch.zeros((2, S, H, R, D), device="cuda", dtype=torch.bfloat16)
    km = torch.tensor([[True], [False]], device=device).expand(2, S).contiguous()
    out = kernels.prefill_attention(q, group_keys(k.contiguous()), group_values(v.contiguous()), km, window=0)
    differ = int((out[1].view(torch.int16) != out[0, S - 1].view(torch.int16)).sum())
    assert differ == 0


def test_prefill_head_dim_512_probabilities(device):
    """The bf16 probabilities themselves: scores that are exact in bf16 (one nonzero dim, q = 1), a few near 0
    that make every row's sum another and the others 45 .. 80 below, and one-hot values, so that output dim j
    is key j's probability.
    Against the 64-bit softmax rounded once: an f32 exp, sum and division within 2.5 ulp (3e-7) cross a bf16
    rounding boundary (at least 2^-8 of the value apart) for a share of at most 3e-7 * 2^8 = 7.7e-5 of them;
    the rounding of x log2(e) alone (up to 2.6e-6 there, half of it on average) gives three times that."""

    B, H, D = 64, 8, 512
    S = D
    g = torch.Generator(device="cuda").manual_seed(3)
    k0 = (torch.rand((B, H, S), device="cuda", generator=g) * -35 - 45).to(torch.bfloat16)
    k0[..., 0] = 0
    k0[..., 1:9] = -2 * torch.rand((B, H, 8), device="cuda", generator=g).to(torch.bfloat16)
    k = torch.zeros((B, H, S, D), device="cuda", dtype=torch.bfloat16)
    k[..., 0] = k0
    q = torch.zeros((B, S, H, 1, D), device="cuda", dtype=torch.bfloat16)
    q[..., 0] = 1
    v = torch.eye(S, device="cuda", dtype=torch.bfloat16).expand(B, H, S, D).contiguous()
    km = torch.ones((B, S), dtype=torch.bool, device=device)
    got = kernels.prefill_attention(q, group_keys(k), group_values(v), km, window=0)[:, -1, :, 0]  # [B, H, key]
    want = torch.softmax(k0.double(), -1).to(torch.bfloat16)
    share = float((got != want).float().mean())
    print(f"share of probabilities that round the other way: {share:.2e}")
    assert torch.all((got.double() - want.double()).abs() <= want.double() * 2.0 ** -7)
    assert share <= 7.7e-5


# a grid whose workgroups hold two column blocks per wave, its heads one by one with one block: head dim 128 at
# 512 two-block workgroups of more than 1024 tokens, beyond 16000 keys, and head dim 256 beyond 256
@pytest.mark.parametrize("D,B,S,H,R,window", [(128, 4, 2048, 4, 4, 0), (128, 1, 16001, 8, 1, 0), (128, 1, 16001, 8, 1, 600),
                                              (256, 5, 1025, 4, 4, 0)])
def test_prefill_block_counts_agree(device, D, B, S, H, R, window):
    """Rows do not depend on how many column blocks a workgroup holds: bit for bit the same; and the last
    position within 2e-2 of 64 bits (the rounding of probabilities and outputs, |o| < 4)."""

    g = torch.Generator(device="cuda").manual_seed(S + D)
    Sp = (S + 63) // 64 * 64
    q = (torch.randn((B, S, H, R, D), device="cuda", generator=g) * D ** -0.25).to(torch.bfloat16)
    k = (torch.randn((B, H, Sp, D), device="cuda", generator=g) * D ** -0.25).to(torch.bfloat16)
    v = torch.randn((B, H, Sp, D), device="cuda", generator=g).to(torch.bfloat16)
    km = torch.ones((B, S), dtype=torch.bool, device=device)
    km[0, :40] = False
    kk, vv = group_keys(k), group_values(v)
    out = kernels.prefill_attention(q, kk, vv, km, window=window)
    for b in range(B):
        for h in range(H):
            one = kernels.prefill_attention(q[b:b + 1, :, h:h + 1].contiguous(), kk[b:b + 1, h:h + 1].contiguous(),
                                            vv[b:b + 1, h:h + 1].contiguous(), km[b:b + 1], window=window)
            assert int((one.view(torch.int16) != out[b:b + 1, :, h:h + 1].view(torch.int16)).sum()) == 0
    seen = km & (torch.arange(S, device=device) > S - 1 - window if window else True)
    scores = torch.matmul(q[:, -1].double(), k[:, :, :S].double().transpose(2, 3).contiguous())
    want = torch.matmul(torch.softmax(scores.masked_fill(~seen[:, None, None], float("-inf")), -1), v[:, :, :S].double())
    assert float((out[:, -1].double() - want).abs().max()) <= 2e-2
