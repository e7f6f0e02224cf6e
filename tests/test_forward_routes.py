"""Which forwards are one library call: up to the rows that the library's own
fp32 rotation takes as quickly as the general route's products."""
from types import SimpleNamespace as NS

import pytest
import torch

from oscar_amd import backend
from tests.test_gpu_backend import make_impl

D = 256


def _impl(monkeypatch, hq, taken):
    impl = make_impl(hq, 1, staging=0)
    impl.key_cache = impl.value_cache = torch.zeros(2, 32, 1, D, dtype=torch.int8)
    impl._mtp_layer = impl._layer_rots = lambda *a: None
    for name in ("decode_only_forward", "step_forward"):
        monkeypatch.setattr(backend.step, name, lambda *a, name=name: taken.append(name) or True)
    monkeypatch.setattr(backend._lib, "stream_handle", lambda dev: 0)
    return impl


@pytest.mark.parametrize("hq,B,history,one_call", [(64, 64, 1500, True), (64, 65, 1500, False), (64, 65, 512, True),
                                                   (64, 128, 512, True), (64, 129, 10, False)])
def test_decode_only(monkeypatch, hq, B, history, one_call):
    taken = []
    impl = _impl(monkeypatch, hq, taken)
    md = NS(query_start_loc_cpu=list(range(B + 1)), seq_lens_list=[history] * B,
            block_tables=torch.zeros(B, 1, dtype=torch.int32))
    q = torch.zeros(B, hq * D, dtype=torch.bfloat16)
    assert impl._decode_only_step(NS(), q, None, md, torch.empty_like(q)) is one_call
    assert taken == ["decode_only_forward"] * one_call


@pytest.mark.parametrize("shorts,one_call", [(128, True), (129, False)])
def test_short_requests_beside_a_long_one(monkeypatch, shorts, one_call):
    taken, hq = [], 16
    impl = _impl(monkeypatch, hq, taken)
    lengths = [17] + [16] * shorts
    qsl = [0]
    for n in lengths:
        qsl.append(qsl[-1] + n)
    N = qsl[-1]
    md = NS(num_actual_tokens=N, query_start_loc_cpu=qsl, seq_lens_list=[40] * len(lengths),
            slot_mapping=torch.zeros(N, dtype=torch.int64), block_tables=torch.zeros(len(lengths), 2, dtype=torch.int32))
    q = torch.zeros(N, hq, D, dtype=torch.bfloat16)
    kv = torch.zeros(N, 1, D, dtype=torch.bfloat16)
    layer = NS(_oscar_rot_ops=(None,) * 4, _oscar_rvT_op=None)
    assert impl._long_step(layer, q, kv, kv, None, md, torch.empty_like(q)) is one_call
    assert taken == ["step_forward"] * one_call
