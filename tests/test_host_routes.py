"""Which native call the Python front end makes, and what it refuses, on the CPU: the launching entry points
are replaced by recorders, the host-side ones are the library's."""

from __future__ import annotations

import ctypes

import pytest
import torch

from gemma4_posttrain_jax_amd import _lib, kernels, model
from gemma4_posttrain_jax_amd.kvcache import new_layer_cache

HOST_FUNCTIONS = ("g4_decode_workspace_size", "g4_linear_workspace_size", "g4_lm_head_sample_workspace_size")


class _Recorder:
    def __init__(self, native):
        self.native, self.calls = native, []

    def __getattr__(self, name):
        if name in HOST_FUNCTIONS:
            return getattr(self.native, name)

        def launch(args, *rest):
            copy = type(args._obj)()
            ctypes.pointer(copy)[0] = args._obj
            self.calls.append((name, copy))
            return _lib.G4_OK

        return launch


@pytest.fixture
def recorder(monkeypatch):
    rec = _Recorder(_lib.lib())
    monkeypatch.setattr(_lib, "lib", lambda: rec)
    monkeypatch.setattr(kernels, "_ptr", lambda t: None if t is None else t.data_ptr())
    monkeypatch.setattr(kernels, "_stream", lambda: None)
    return rec


def _decode(pairs, D=256, cap=512, **kw):
    layer = new_layer_cache(pairs, 1, D, cap, True, torch.bfloat16, "cpu")
    q = torch.zeros((pairs, 1, 4, D), dtype=torch.bfloat16)
    mask = torch.ones((pairs, cap), dtype=torch.bool)
    kernels.decode_attention(layer, q, mask, q_pos=cap - 1, window=cap, **kw)


@pytest.mark.parametrize("pairs", [1, 2, 32, 129, 192, 255])
def test_no_alloc_decode_shares_no_scratch_where_none_is_needed(recorder, pairs):
    """Rows of at most 512 slots over fewer than 256 pairs have a path without a workspace: a no-alloc call
    takes it (the library's per-device scratch would tie calls on different streams together); a call that
    may allocate takes the two-launch path."""

    _decode(pairs, no_alloc=True)
    _decode(pairs)
    (name, a), (_, b) = recorder.calls
    assert name == "g4_decode_attention_noalloc"
    assert a.num_splits == 0 and recorder.native.g4_decode_workspace_size(ctypes.byref(a)) == 0
    assert b.num_splits == _lib.G4_DECODE_TWO_PASS and b.workspace and b.workspace_bytes > 0


@pytest.mark.parametrize("cache", [dict(B=1), dict(H=1), dict(H=4), dict(D=128)])
def test_fused_decode_refuses_a_cache_of_another_shape(recorder, cache):
    """The step's fused attention refuses what its two calls, the append and the attention, refuse: a cache
    whose rows, kv heads or head dim are not the query's (the kernels would index past it)."""

    B, H, R, D = 2, 2, 4, 256
    shape = dict(dict(B=B, H=H, D=D), **cache)
    layer = new_layer_cache(shape["B"], shape["H"], shape["D"], 64, False, torch.bfloat16, "cpu")
    rows = torch.zeros((B, (R + 2) * H * D), dtype=torch.bfloat16)
    args = dict(q_pos=torch.zeros(B, dtype=torch.int32), window=0, k_raw=rows[:, R * H * D:-H * D].view(B, H, D),
                v_raw=rows[:, -H * D:].view(B, H, D), q_norm_weight=None, k_norm_weight=None,
                rope_cos=torch.zeros(B, D), rope_sin=torch.zeros(B, D), eps=1e-6, flags=0)
    with pytest.raises(ValueError, match="does not match"):
        kernels.decode_attention_fused(layer, rows[:, : R * H * D].view(B, H, R, D), torch.ones((B, 64), dtype=torch.bool),
                                       **args)
    assert not recorder.calls


@pytest.mark.parametrize("D", [128, 256, 512])
def test_norm_weights_at_any_offset_take_the_append(recorder, D):
    """The q / k norm weights may start anywhere (a view into a flat parameter buffer): the fused preparation
    reads D / 64 of them in one access and refuses such a start, the append takes it."""

    layer = new_layer_cache(1, 1, D, 64, False, torch.bfloat16, "cpu")
    x, flat = torch.zeros((1, 1, 8), dtype=torch.bfloat16), torch.ones(D + 8, dtype=torch.bfloat16)
    for offset, takes in ((0, True), (1, False), (D // 64, True)):
        for norms in ((flat[offset:][:D], None), (flat[:D], flat[offset:][:D])):
            assert model._fused_decode_prep(x, 1, D, layer, norms) is takes
            prep = _lib.G4DecodePrep(q_raw=256, k_raw=256, v_raw=256, in_row_stride=3 * D, q_norm_weight=norms[0].data_ptr(),
                                     k_norm_weight=norms[1].data_ptr() if norms[1] is not None else None, rope_cos=256,
                                     rope_sin=256, eps=1e-6, flags=0)
            a = _lib.G4DecodeArgs(dtype=_lib.G4_DTYPE_BF16, kind=_lib.G4_CACHE_LINEAR, batch=1, kv_heads=1, group=1,
                                  head_dim=D, capacity=64, slot_stride=64, key_mask=256, key_mask_stride=64, cache_k=256,
                                  cache_vt=256, cache_k_w=256, out=256, num_splits=0,
                                  prep=ctypes.cast(ctypes.pointer(prep), ctypes.c_void_p))
            # refused before any launch, or only for its missing workspace
            want = _lib.G4_ERR_WORKSPACE if takes else _lib.G4_ERR_INVALID
            assert recorder.native.g4_decode_attention(ctypes.byref(a), None) == want
