"""The prefill read's output pass (merge of a row block's pieces, R_v^T, bf16)
at its pieces' counts, against the oracle's dense read in fp32, bar of the
prefill kernel: |gpu - oracle| <= 2e-2 + 2^-8 |oracle|.
"""
import pytest
import torch

from oscar_amd.kernels import prefill, quant
from tests.scenarios import decode_case
from tests.test_gpu_prefill_split import _close, _want

pytestmark = pytest.mark.gpu
D = 256


# Row blocks of one piece (a share holds them whole), of 2 to 8, of 9 to 16, of
# more beside many that are whole (all in the pass), and of more than 16 on
# average (merged before it); rows that do not fill 4, 32 or 256; two kv heads.
@pytest.mark.parametrize("hist,new,hq,hk", [
    ([0], [17], 1, 1), ([40, 0], [21, 87], 3, 1), ([600], [260], 6, 1), ([700, 64], [130, 100], 12, 2),
    ([3000], [170], 6, 1), ([9000, 0], [43, 1400], 6, 1), ([5000], [18], 6, 1)])
def test_piece_counts(device, hist, new, hq, hk):
    case = decode_case(hist, new, hq=hq, hk=hk, seed=sum(new), window=True, sink=128, recent=64)
    L = case.layer
    q, k, v = case.rotated()
    reqs = [(case.qsl[i], n, h, i) for i, (h, n) in enumerate(zip(hist, new))]
    ops = [quant.rotation_operand(r.to(device)) for r in (L.R_k, L.R_v, L.R_v.t().contiguous())]
    stage = tuple(t.to(device).contiguous() for t in L.stage())
    out = torch.full((case.qsl[-1] + 1, hq, D), 7.0, dtype=torch.bfloat16, device=device)
    qp = torch.cat([case.q, case.q[:1]]).to(device)
    prefill.prefill_rotated(qp, case.k.to(device), case.v.to(device), reqs[::-1], *ops, L.k_cache.to(device),
                            L.v_cache.to(device), case.bt.to(device), L.scale, out, stage)
    torch.cuda.synchronize()
    got = out.cpu().float()
    for i in range(len(new)):
        _close(got[case.qsl[i]:case.qsl[i + 1]], _want(case, i, q, k, v, hk) @ L.R_v.t())
    assert (got[case.qsl[-1]:] == 7.0).all()
