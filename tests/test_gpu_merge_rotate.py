"""The rotated merge's row groups at their edges, against the plain merge's
fp32 rows rotated in fp64.

Both merges combine the same partials, so they differ by fp32 rounding only.
With u = 2^-24, P partials and vmax the largest |V| a row can hold, each
combined feature is off by at most (P + 4) u vmax in either merge, and a
256-term fp32 product adds 256 u sum_f |o_f R_fc|; a bf16 output adds half an
ulp (8 significant bits: at most 2^-8 |out|).
"""
import pytest
import torch

from oracle import store as ostore
from oscar_amd.kernels import decode
from tests.scenarios import decode_case

pytestmark = pytest.mark.gpu
D = 256


# Rows (tokens x query heads) of one row per block (64 is the most), two (128 in
# quarters, 256 in halves), four (512) and eight, at their last counts and more; groups that do
# not divide the rows per block; several row tiles per request (16 tokens x 6
# heads); requests without tokens; more items than one launch carries; 257
# partials, which eight rows per block do not take.
@pytest.mark.parametrize("hist,new,hq,hk,tiles,gap", [
    ([700], [16], 4, 1, 0, False), ([700], [13], 5, 1, 0, True), ([300, 5], [16, 16], 4, 2, 0, False),
    ([40, 3000, 0], [16, 11, 16], 3, 3, 0, True), ([2000, 9, 77, 0], [16] * 4, 4, 1, 0, False),
    ([20] * 6, [16] * 5 + [6], 3, 1, 0, True), ([0, 5000] * 3, [16, 12] * 3, 3, 1, 0, False), ([130] * 8, [16] * 8, 4, 1, 0, False),
    ([515, 0, 33] * 3, [16, 1, 16] * 3, 6, 1, 0, True), ([64] * 33, [16] * 33, 6, 2, 0, False),
    ([90] * 70, [2] * 70, 12, 2, 0, False), ([32768] + [10] * 40, [4] * 41, 6, 1, 4, False)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_row_groups(device, hist, new, hq, hk, tiles, gap, out_dtype):
    case = decode_case(hist, new, hq=hq, hk=hk, bs=128, seed=len(hist) + hq, window=False)
    L = case.layer
    q, k, v = (t.to(device) for t in case.rotated())
    qsl, seqs, bt = case.qsl, case.seqs, case.bt
    if gap:                                   # a request without tokens in front and one behind the first
        qsl = [0, 0, qsl[1]] + qsl[1:]
        seqs = [9, seqs[0], 20] + seqs[1:]
        bt = torch.cat([bt[:1], bt[:1], bt[:1], bt[1:]])
    rvt = L.R_v.t().contiguous()
    args = (q, k, v, L.k_cache.to(device), L.v_cache.to(device), bt.to(device), qsl, seqs, L.scale)
    n = q.shape[0]
    plain = decode.plan(*args, tiles_per_split=tiles).launch()
    out = torch.full((n + 2, hq * D), 5.0, dtype=out_dtype, device=device)
    decode.plan(*args, tiles_per_split=tiles, out=out[:n], out_rotation=rvt.to(device)).launch()
    torch.cuda.synchronize()
    o, r = plain.cpu().double(), rvt.double()
    want = (o @ r).reshape(n, -1)
    got = out[:n].cpu().double()
    vmax = v.abs().max().item()
    for i, h in enumerate(hist):
        if h:
            vmax = max(vmax, ostore.full_dequant_ref(L.k_cache, L.v_cache, case.bt[i], h, hk, D)[1].abs().max().item())
    parts = (max(hist) + 127) // 128 + 1
    bound = 2.0 ** -24 * (256 * (o.abs() @ r.abs()) + 2 * (parts + 4) * vmax * r.abs().sum(0)).reshape(n, -1)
    if out_dtype == torch.bfloat16:
        bound = bound + 2.0 ** -8 * (want.abs() + bound)
    assert ((got - want).abs() <= bound).all(), ((got - want).abs() - bound).max().item()
    assert (out[n:] == 5.0).all()
