"""The counting top-k draw (bf16 rows of at least 4096 columns) on rows that its scheme bends or does not
fit, which the general kernel then draws: against the oracle, token for token."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gemma4_posttrain_jax_amd import kernels
from test_gpu_sampling import _key, _top_k_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,top_k", [(4096, 1), (4096, 256), (4104, 50), (131072, 50)])
@pytest.mark.parametrize("cap", [None, 30.0, 1.5])
def test_top_k_counting_rows(device, V, top_k, cap):
    """Tied maxima across the cut, all values equal (a counter past 65535 at 131072 columns), more ties
    than candidate slots, saturated soft-caps (at cap 1.5 every |logit| above 12 scores the same: many
    logits tied with the k-th), zeros of both signs, -inf columns, negative rows."""

    rng = np.random.default_rng(V + top_k)
    rows = np.empty((9, V), np.float32)
    rows[0] = rng.standard_normal(V) * 3
    rows[1] = 0.25
    rows[2] = np.round(rng.standard_normal(V)) / 2
    rows[3] = rng.uniform(20, 4000, V)  # over 1024 distinct bf16 values, all saturated at cap 1.5
    rows[4] = np.where(rng.random(V) < 0.5, 0.0, -0.0)
    rows[5] = -np.abs(rng.standard_normal(V)) - 100
    rows[6] = rng.standard_normal(V) * 1e-6
    rows[7] = -50.0
    rows[7, -top_k:] = rng.standard_normal(top_k)
    rows[8] = rng.standard_normal(V)
    rows[8, ::3] = -np.inf if cap is None else -1e30
    _top_k_case(device, 9, V, 1.0, top_k, 1.0, cap=cap, logits=rows)
    _top_k_case(device, 9, V, 0.7, top_k, 0.9, cap=cap, logits=rows, seed=5)


def test_top_k_counting_rows_with_nan(device):
    """A row with NaNs (either sign) beside ordinary ones: the ordinary rows' draws do not change, and the
    NaN row draws what the general kernel draws from the same values (its f32 form)."""

    V = 8192
    x = torch.randn((4, V), device=device, generator=torch.Generator(device="cuda").manual_seed(3)).to(torch.bfloat16)
    args = dict(softcap=None, temperature=1.0, top_k=20, top_p=1.0, split_key=False)
    want = kernels.sample_top_k(x, key=_key([1, 2], device), **args)
    x[1, 7] = float("nan")
    x[1, 9] = -float("nan")
    got = kernels.sample_top_k(x, key=_key([1, 2], device), **args)
    general = kernels.sample_top_k(x.float(), key=_key([1, 2], device), **args)
    keep = [0, 2, 3]
    assert torch.equal(got[0][keep], want[0][keep]) and torch.equal(got[1][keep], want[1][keep])
    assert torch.equal(got[0], general[0])
    assert torch.equal(got[1].isnan(), general[1].isnan())
