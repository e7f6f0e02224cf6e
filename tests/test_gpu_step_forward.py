"""oscar_step_forward (one call for a step with long requests) against the
general route's separate calls on the same state.

Bytes written and long requests' rows come from the same kernels on the same
inputs: equal.  Short requests' rows are each within the paged read's bf16 bar
(2e-2 + 2^-8 |out|) of the exact read, so within twice that of each other.
"""
from types import SimpleNamespace as NS

import pytest
import torch

from oscar_amd import synthetic
from tests.scenarios import metadata
from tests.test_gpu_backend import make_impl

pytestmark = pytest.mark.gpu
D = 256


def _requests(spec):
    return [tuple(int(x) for x in r.split("@")) for r in spec.split(",")]


# new@history.  Both kinds, in one and in several runs; only long; a request
# without tokens; more runs (70) than one rotation launch and more long
# requests than one prefill launch carry; more request lengths (2 x 500 + 1)
# than travel with the seat-winner pass, more short ones than one read; a
# write of at most 2048 vectors (fp32 rotation) and of more.
@pytest.mark.parametrize("spec,hq,hk,bs", [
    ("4@300,40@100,1@0,16@33", 6, 1, 64), ("0@9,77@500,17@0", 8, 2, 32), ("1100@130,3@700,0@64,2@5", 6, 1, 32),
    (",".join(["17@5,1@40"] * 70), 4, 1, 32), (",".join(["18@0"] + ["2@31"] * 499), 3, 1, 32)])
@pytest.mark.parametrize("window", [True, False])
def test_against_the_general_route(device, spec, hq, hk, bs, window):
    reqs = _requests(spec)
    B, N = len(reqs), sum(n for n, _ in reqs)
    pages = [(n + h + bs - 1) // bs or 1 for n, h in reqs]
    perm = synthetic.page_permutation(sum(pages) + 3, 5)
    bt = torch.zeros(B, max(pages), dtype=torch.int32)
    at = 0
    for i, p in enumerate(pages):
        bt[i, :p] = perm[at:at + p]
        at += p
    rots = [r.to(device) for r in synthetic.rotations(D, 3)]
    total = sum(h for _, h in reqs)
    hk_, hv_ = synthetic.kv(max(total, 1), hk, D, seed=1)
    hslots = torch.cat([synthetic.slots_for(bt[i], 0, h, bs) for i, (_, h) in enumerate(reqs)])
    k, v = (t.to(torch.bfloat16).to(device) for t in synthetic.kv(N + 2, hk, D, seed=2))
    q = synthetic.queries(N + 2, hq, D, seed=3).to(torch.bfloat16).to(device)
    qsl = [0]
    for n, _ in reqs:
        qsl.append(qsl[-1] + n)
    slots = torch.cat([synthetic.slots_for(bt[i], h, n, bs) for i, (n, h) in enumerate(reqs)])
    md = metadata(slots, qsl, [n + h for n, h in reqs], bt)
    md.num_actual_tokens = N
    md = NS(**{**vars(md), "slot_mapping": slots.to(device), "block_tables": bt.to(device)})

    def run(general):
        impl = make_impl(hq, hk, sink=bs, recent=48, staging=8192 if window else 0)
        layer = NS(layer_name="model.layers.1.self_attn.attn", _oscar_rots=tuple(rots))
        caches = [torch.zeros(sum(pages) + 3, bs, hk, D, dtype=torch.int8, device=device) for _ in range(2)]
        impl.do_kv_cache_update(layer, hk_[:total].to(torch.bfloat16).to(device),
                                hv_[:total].to(torch.bfloat16).to(device), caches, hslots.to(device))
        if general:
            impl._long_step = lambda *a: False
        else:
            impl._read = None                       # the step must not need it
        out = impl.forward(layer, q, k, v, caches, md, output=torch.full((N + 3, hq, D), 7.0, dtype=torch.bfloat16,
                                                                         device=device))
        torch.cuda.synchronize()
        arena = [layer._oscar_stage_k, layer._oscar_stage_v, layer._oscar_slot_owner, layer._oscar_stage_kimg,
                 layer._oscar_stage_vimg] if window else []
        return out.cpu().float(), [t.cpu() for t in caches + arena]

    (got, state), (want, wstate) = run(False), run(True)
    for a, b in zip(state, wstate):
        assert torch.equal(a, b)
    for i, (n, _) in enumerate(reqs):
        a, b = got[qsl[i]:qsl[i + 1]], want[qsl[i]:qsl[i + 1]]
        if n > 16:
            assert torch.equal(a, b), i
        else:
            assert ((a - b).abs() <= 2 * (2e-2 + 2.0 ** -8 * b.abs())).all(), (i, (a - b).abs().max().item())
    assert (got[N:N + 2] == 0).all() and (got[N + 2:] == 7.0).all()
