"""The reads of one request over fp32 rows by whole row blocks of 128 or 256 rows
and by equal shares, on both sides of the rules that choose between them,
against the oracle's dense read in fp32 (bar of the prefill kernel: |gpu -
oracle| <= 2e-2 + 2^-8 |oracle|).
"""
import pytest
import torch

from oscar_amd.kernels import _lib, prefill
from oscar_amd.kernels.quant import cache_geometry
from tests.scenarios import decode_case
from tests.test_gpu_prefill_split import _close, _want

pytestmark = pytest.mark.gpu
D = 256


# 128-row blocks that are short of, exactly and over full (21 / 22 tokens of group
# 6, 128 / 129 of group 1, 8 of group 16), and 256-row blocks (42 / 43, 256 / 257);
# several kv heads; 128-row blocks of more than a round of the CUs, where 256 rows
# are taken without a workspace (128 heads of one kv head, half a block at the
# end); histories of as many key blocks as whole row blocks are read with a
# workspace (none, two), and of more, which shares are.
@pytest.mark.parametrize("hq,hk,new", [(6, 1, 21), (6, 1, 22), (6, 1, 42), (6, 1, 43), (1, 1, 128), (1, 1, 129),
                                       (1, 1, 256), (1, 1, 257), (16, 1, 8), (16, 2, 33), (4, 4, 200), (64, 8, 40),
                                       (128, 1, 501)])
@pytest.mark.parametrize("hist", [0, 33, 900])
@pytest.mark.parametrize("window", [False, True])
def test_both_entries(device, hq, hk, new, hist, window):
    bs = 32
    case = decode_case([hist], [new], hq=hq, hk=hk, bs=bs, seed=hist + new, window=window, sink=bs, recent=40)
    L = case.layer
    rows = case.rotated()
    want = _want(case, 0, *rows, hk)
    q, k, v, kc, vc, bt = (t.to(device) for t in (*rows, L.k_cache, L.v_cache, case.bt[0]))
    stage = tuple(t.to(device).contiguous() for t in L.stage()) if window else None
    got = prefill.prefill_continuation(q, k, v, kc, vc, bt, hist, L.scale, stage)
    out = torch.full((new + 1, hq, D), 7.0, device=device)
    _, pages, kst, vst = cache_geometry(kc, vc)
    sk, sv, owner = stage if window else (None, None, None)
    _lib.call("oscar_prefill_continuation", *map(_lib.ptr, (q, k, v)), new, hq, hk, D, _lib.ptr(kc), _lib.ptr(vc), bs,
              pages, *kst, *vst, _lib.ptr(bt), bt.numel(), hist, _lib.ptr(sk), _lib.ptr(sv), _lib.ptr(owner),
              owner.shape[0] if window else 0, L.scale, _lib.ptr(out), _lib.stream_handle(out.device))
    torch.cuda.synchronize()
    _close(got.cpu(), want)
    _close(out[:new].cpu(), want)
    assert (out[new:] == 7.0).all()
