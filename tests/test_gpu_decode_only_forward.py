"""oscar_decode_only_forward (bf16 query to model-domain output in one call)
against the oracle's DecodeOnly read.

The read's bar is 1e-3 of the largest rotated output (the DecodeOnly read's
own tests); R_v^T turns an error e in every rotated feature into at most
e sum_f |R_fc|, and a bf16 output adds half an ulp, at most 2^-8 |out|.
"""
import pytest
import torch

from oracle import attention as oatt
from oscar_amd.kernels import _lib, quant, staging, step
from tests.scenarios import decode_case

pytestmark = pytest.mark.gpu
D = 256


# 1, 2 and 4 query vectors per rotation workgroup (at most 512, 2048 and more
# vectors, with and without a remainder), more items than one launch carries,
# an empty history, both bounds paths (groups of at most 8 heads, and more).
@pytest.mark.parametrize("hist,hq,hk", [([1000], 6, 1), ([300, 0, 63], 5, 1), ([40] * 86 + [7], 6, 2),
                                        ([33] * 150, 16, 1), ([4097, 129], 12, 4)])
@pytest.mark.parametrize("window,out_dtype,strided", [(True, torch.bfloat16, False), (False, torch.float32, True)])
def test_against_the_oracle(device, hist, hq, hk, window, out_dtype, strided):
    B = len(hist)
    case = decode_case(hist, [1] * B, hq=hq, hk=hk, bs=32, seed=B + hq, window=window, sink=32, recent=64, staging=256,
                       pool_pages=sum((h + 32) // 32 for h in hist) + 5)
    L = case.layer
    seqs = [s - 1 for s in case.seqs]           # the history alone: nothing of the last step is written
    g = torch.Generator().manual_seed(B)
    q = torch.randn(B, hq, D, generator=g).to(torch.bfloat16)
    arena = (L.arena.stage_k, L.arena.stage_v, L.arena.owner, L.arena.sink_eff, L.recent) if window else None
    rot = oatt.decode_only_ref(q.float() @ L.R_k, L.k_cache, L.v_cache, case.bt, seqs, L.scale, hk, D, arena).double()
    R = L.R_v.t().double()
    want = (rot @ R).reshape(B, -1)
    bound = (1e-3 * rot.abs().max() * R.abs().sum(0)).repeat(hq).expand(B, -1)
    if out_dtype == torch.bfloat16:
        bound = bound + 2.0 ** -8 * (want.abs() + bound)
    stage = None
    if window:
        images = staging.stage_images(L.arena.stage_k, L.arena.stage_v)
        stage = tuple(t.to(device) for t in (L.arena.stage_k, L.arena.stage_v, L.arena.owner, *images))
    ml = step.MtpLayer(L.R_k.to(device), L.R_v.to(device), L.R_v.t().contiguous().to(device), L.k_cache.to(device),
                       L.v_cache.to(device), hq, hk, quant.clip_index(L.clip_k, D), quant.clip_index(L.clip_v, D),
                       L.scale, stage, L.arena.sink_eff if window else 0, L.recent)
    width = hq * D
    dq = q.to(device).reshape(B, width)
    buf = torch.full((B + 1, width + (8 if strided else 0)), 3.0, dtype=out_dtype, device=device)
    if strided:
        wide = torch.zeros(B, width + 3, dtype=torch.bfloat16, device=device)
        wide[:, :width] = dq
        dq = wide[:, :width]
    assert step.decode_only_forward(ml, dq, case.bt.to(device), seqs, buf[:, :width],
                                    _lib.stream_handle(torch.device(device)))
    torch.cuda.synchronize()
    got = buf[:B, :width].cpu().double()
    assert ((got - want).abs() <= bound).all(), ((got - want).abs() - bound).max().item()
    assert (buf[B:] == 3.0).all() and (buf[:, width:] == 3.0).all()
