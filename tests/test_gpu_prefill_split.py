"""The prefill read's row blocks, shares and operand tiles at their edges,
against the oracle's dense read in fp32 (bar of the prefill kernel:
|gpu - oracle| <= 2e-2 + 2^-8 |oracle|, the bf16 contract plus half a bf16 ulp;
the bf16 outputs of whole requests after R_v^T likewise).

A workgroup takes 256 (token, head) rows and walks 32-key blocks; equal shares
of all row blocks' key blocks may cut a row block anywhere.  (Reads of fp32 rows
with few rows or keys take whole blocks of 128 rows: tests/test_gpu_prefill_whole.py
has both at their edges.)
"""
import ctypes

import pytest
import torch

from oracle import attention as oatt
from oracle import store as ostore
from oscar_amd.kernels import _lib, prefill, quant
from oscar_amd.kernels.quant import cache_geometry
from tests.scenarios import decode_case

pytestmark = pytest.mark.gpu
D = 256


def _want(case, i, q, k, v, hk):
    L = case.layer
    a, b = case.qsl[i], case.qsl[i + 1]
    hist = case.seqs[i] - (b - a)
    if hist:
        kc, vc = ostore.full_dequant_ref(L.k_cache, L.v_cache, case.bt[i], hist, hk, D)
        if L.stage() is not None:
            kc, vc = L.arena.splice(case.bt[i], hist, kc, vc)
    else:
        kc = vc = torch.zeros(0, hk, D)
    return oatt.prefill_ref(q[a:b], k[a:b], v[a:b], kc, vc, L.scale, hk, D)


def _close(got, want):
    assert torch.isfinite(got).all()
    err = (got - want).abs()
    assert (err <= 2e-2 + 2.0 ** -8 * want.abs()).all(), f"max abs err {err.max().item():.3e}"


# group 6: 42 tokens are 252 rows, 43 are 258; group 1: 256 / 257 rows, whose
# last tokens see up to eight more key blocks than the first; 31 / 32 / 33
# cached tokens and new tokens are one key block less, exactly and more one.
@pytest.mark.parametrize("hq,hk,hist,new,bs", [
    (6, 1, 0, 17, 128), (6, 1, 31, 42, 32), (6, 1, 32, 43, 32), (6, 1, 33, 86, 64), (6, 1, 2000, 32, 128),
    (1, 1, 100, 256, 32), (1, 1, 64, 257, 64), (16, 1, 65, 33, 128), (12, 2, 700, 65, 128), (4, 4, 1, 130, 32),
    (6, 1, 6000, 21, 128)])
@pytest.mark.parametrize("window", [False, True])
def test_tile_edges_split_and_whole(device, hq, hk, hist, new, bs, window):
    case = decode_case([hist], [new], hq=hq, hk=hk, bs=bs, seed=hist + new, window=window, sink=bs, recent=40)
    L = case.layer
    q, k, v = case.rotated()
    want = _want(case, 0, q, k, v, hk)
    dev = [t.to(device) for t in (q, k, v, L.k_cache, L.v_cache, case.bt[0])]
    stage = L.stage()
    dstage = None if stage is None else tuple(t.to(device).contiguous() for t in stage)
    got = prefill.prefill_continuation(*dev, hist, L.scale, dstage)
    torch.cuda.synchronize()
    _close(got.cpu(), want)
    # the entry without a workspace: one workgroup per row block, fp32 rows read in place
    out = torch.full_like(got, float("nan"))
    kc, vc = dev[3], dev[4]
    gbs, pages, kst, vst = cache_geometry(kc, vc)
    sk, sv, owner = dstage if dstage is not None else (None, None, None)
    _lib.call("oscar_prefill_continuation", *map(_lib.ptr, dev[:3]), new, hq, hk, D, _lib.ptr(kc), _lib.ptr(vc), gbs,
              pages, *kst, *vst, _lib.ptr(dev[5]), dev[5].numel(), hist, _lib.ptr(sk), _lib.ptr(sv), _lib.ptr(owner),
              0 if owner is None else owner.shape[0], L.scale, _lib.ptr(out), _lib.stream_handle(out.device))
    torch.cuda.synchronize()
    _close(out.cpu(), want)


# Several requests in one launch (more than one launch holds in the last),
# adjacent and with short requests between them; rows of others stay as they
# are.
@pytest.mark.parametrize("hist,new,hq,hk", [
    ([0, 300, 31], [40, 100, 17], 6, 1), ([500, 40, 0, 64], [33, 4, 64, 20], 12, 2), ([7] * 50, [17] * 50, 6, 1)])
def test_requests_of_a_step_in_one_launch(device, hist, new, hq, hk):
    case = decode_case(hist, new, hq=hq, hk=hk, seed=len(hist), window=True, sink=128, recent=64)
    L = case.layer
    q, k, v = case.rotated()
    reqs = [(case.qsl[i], n, h, i) for i, (h, n) in enumerate(zip(hist, new)) if n > 16]
    ops = [quant.rotation_operand(r.to(device)) for r in (L.R_k, L.R_v, L.R_v.t().contiguous())]
    stage = tuple(t.to(device).contiguous() for t in L.stage())
    out = torch.full((case.qsl[-1], hq, D), 7.0, dtype=torch.bfloat16, device=device)
    prefill.prefill_rotated(case.q.to(device), case.k.to(device), case.v.to(device), reqs, *ops,
                            L.k_cache.to(device), L.v_cache.to(device), case.bt.to(device), L.scale, out, stage)
    torch.cuda.synchronize()
    got = out.cpu().float()
    for i, n in enumerate(new):
        a, b = case.qsl[i], case.qsl[i + 1]
        if n <= 16:
            assert (got[a:b] == 7.0).all()
        else:
            _close(got[a:b], _want(case, i, q, k, v, hk) @ L.R_v.t())


def test_workspace_is_checked(device):
    lib = _lib.load()
    need = lib.oscar_prefill_workspace_bytes(300, 6, 1, 1000)
    assert need > 0 and lib.oscar_prefill_workspace_bytes(300, 5, 2, 1000) == 0
    z = torch.zeros(300, 6, D, device=device)
    kc = torch.zeros(16, 128, 1, D, dtype=torch.int8, device=device)
    bt = torch.arange(16, dtype=torch.int32, device=device)
    ws = torch.empty(need, dtype=torch.uint8, device=device)
    bs, pages, kst, vst = cache_geometry(kc, kc)

    def run(size):
        return lib.oscar_prefill_continuation_split(
            z.data_ptr(), z.data_ptr(), z.data_ptr(), 300, 6, 1, D, kc.data_ptr(), kc.data_ptr(), bs, pages, *kst,
            *vst, bt.data_ptr(), 16, 1000, None, None, None, 0, ctypes.c_float(0.1), z.data_ptr(), ws.data_ptr(),
            size, _lib.stream_handle(z.device))
    assert run(need - 1) == -3


@pytest.mark.parametrize("split", [False, True])
def test_rows_of_less_alignment_than_a_load(device, split):
    # V slots 67 bytes apart from an odd address, an output and an arena that
    # start 4 bytes past a 16-byte line: the same results as aligned ones.
    hq, hk, hist, new, bs = 6, 1, 300, 45, 32
    case = decode_case([hist], [new], hq=hq, hk=hk, bs=bs, seed=8, window=True, sink=bs, recent=40)
    L = case.layer
    q, k, v = (t.to(device) for t in case.rotated())
    kc, vc, bt = L.k_cache.to(device), L.v_cache.to(device), case.bt[0].to(device)
    sk, sv, owner = (t.to(device).contiguous() for t in L.stage())
    pages = kc.shape[0]
    packed = torch.zeros(1 + pages * bs * 67, dtype=torch.int8, device=device)
    packed[1:].view(pages, bs, 67)[:, :, :64] = vc[:, :, 0, :64]
    shifted = [torch.zeros(t.numel() + 1, dtype=torch.float32, device=device) for t in (sk, sv)]
    for s, t in zip(shifted, (sk, sv)):
        s[1:] = t.reshape(-1)
    gbs, _, kst, vst = cache_geometry(kc, vc)
    lib = _lib.load()
    ws = torch.empty(lib.oscar_prefill_workspace_bytes(new, hq, hk, hist), dtype=torch.uint8, device=device)

    def run(vptr, vst, skp, svp, out):
        args = (*map(_lib.ptr, (q, k, v)), new, hq, hk, D, _lib.ptr(kc), vptr, gbs, pages, *kst, *vst, _lib.ptr(bt),
                bt.numel(), hist, skp, svp, _lib.ptr(owner), owner.shape[0], L.scale, out.data_ptr())
        stream = _lib.stream_handle(out.device)
        if split:
            _lib.call("oscar_prefill_continuation_split", *args, _lib.ptr(ws), ws.numel(), stream)
        else:
            _lib.call("oscar_prefill_continuation", *args, stream)
        torch.cuda.synchronize()
        return out.cpu()

    n = new * hq * D
    want = run(vc.data_ptr(), vst, sk.data_ptr(), sv.data_ptr(), torch.zeros(n, device=device))
    got = run(packed.data_ptr() + 1, (bs * 67, 67, 64), shifted[0].data_ptr() + 4, shifted[1].data_ptr() + 4,
              torch.zeros(n + 1, device=device)[1:])
    assert torch.equal(got, want)
    _close(want.view(new, hq, D), _want(case, 0, *case.rotated(), hk))
