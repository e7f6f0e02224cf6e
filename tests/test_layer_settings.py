"""The packed layer half of the one-call forwards follows the settings it was
packed from, not only the tensors: scale, clip ratios and window sizes are read
from the configuration at every step, as the reference's forward reads them
(oscar_ascend/backend.py:150-189, 239-319)."""
import dataclasses
from types import SimpleNamespace as NS

import pytest
import torch

from oscar_amd import synthetic
from oscar_amd.kernels import quant
from tests.test_gpu_backend import make_impl

D = 256


@pytest.mark.parametrize("change", [dict(k_clip_ratio=0.9), dict(v_clip_ratio=0.5), dict(sink_tokens=96),
                                    dict(recent_tokens=10), dict(scale=0.125)])
def test_layer_half_is_rebuilt_when_a_setting_changes(change):
    impl = make_impl(2, 1, sink=32, recent=48)
    caches = [torch.zeros(4, 32, 1, D, dtype=torch.int8) for _ in range(2)]
    impl._set_caches(caches)
    rk, rv = synthetic.rotations(D, 1)
    layer = NS(layer_name="model.layers.0.self_attn.attn", _oscar_rots=(rk, rv), _oscar_rvT=rv.t().contiguous(),
               _oscar_rot_ops=(rk, rv, None, None))
    impl._layer_rots = lambda layer, dev: layer._oscar_rots
    first = impl._mtp_layer(layer, caches, torch.device("cpu"))
    # the same settings by value, and the same half
    impl._oscar_cfg = dataclasses.replace(impl._oscar)
    assert impl._mtp_layer(layer, caches, torch.device("cpu")) is first
    if "scale" in change:
        impl.scale = change["scale"]
    else:
        impl._oscar_cfg = dataclasses.replace(impl._oscar, **change)
    a, cfg = impl._mtp_layer(layer, caches, torch.device("cpu")).args, impl._oscar
    assert (a.clip_index_k, a.clip_index_v, a.sink_eff, a.recent, a.scale) == (
        quant.clip_index(cfg.k_clip_ratio, D), quant.clip_index(cfg.v_clip_ratio, D), cfg.sink_tokens // 32 * 32,
        cfg.recent_tokens, impl.scale)          # (powers of two: exact in the struct's float)


def test_rotations_of_any_stride(monkeypatch):
    # a transposed view, as the fp32 products of the general route take it
    impl = make_impl(2, 1, sink=0, recent=0)
    caches = [torch.zeros(4, 32, 1, D, dtype=torch.int8) for _ in range(2)]
    impl._set_caches(caches)
    monkeypatch.setattr(quant, "rotation_operand", lambda R: R.contiguous())
    rk, rv = synthetic.rotations(D, 1)
    layer = NS(layer_name="model.layers.0.self_attn.attn", _oscar_rots=(rk.t(), rv.t()))
    dev = torch.device("cpu")
    half = impl._mtp_layer(layer, caches, dev)
    for got, want in zip(half.tensors, (rk.t(), rv.t(), rv)):
        assert got.is_contiguous() and torch.equal(got, want)
    assert impl._mtp_layer(layer, caches, dev) is half
