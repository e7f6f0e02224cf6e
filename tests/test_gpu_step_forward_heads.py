"""The short requests of oscar_step_forward with several kv heads, many splits
and chunked reads, against the oracle's read (oracle/attention.py, restating
oscar_ascend/kernels/paged_attention.py:41-64) of the caches and the arena that
the step left.

Bar: the paged read's, 1e-3 of the output scale per rotated-domain element, so
sqrt(256) 1e-3 scale per row in the 2-norm, which R_v^T preserves, plus the
bf16 cast's half ulp (2^-8 relative at most).
"""
from types import SimpleNamespace as NS

import pytest
import torch

from oracle import attention as oatt
from oscar_amd import synthetic
from tests.scenarios import metadata
from tests.test_gpu_backend import make_impl

pytestmark = pytest.mark.gpu
D = 256


def _run(device, reqs, hq, hk, bs, window):
    """One forward of new@history requests over histories written by
    do_kv_cache_update: (bf16 output, rotated q / k / v, caches, arena or None,
    block table, qsl, seqs, scale, R_v), all on the host."""
    B, N = len(reqs), sum(n for n, _ in reqs)
    pages = [(n + h + bs - 1) // bs for n, h in reqs]
    perm = synthetic.page_permutation(sum(pages), 5)
    bt = torch.zeros(B, max(pages), dtype=torch.int32)
    at = 0
    for i, p in enumerate(pages):
        bt[i, :p] = perm[at:at + p]
        at += p
    Rk, Rv = synthetic.rotations(D, 3)
    hist = [(i, h) for i, (_, h) in enumerate(reqs) if h]
    hk_, hv_ = synthetic.kv(sum(h for _, h in hist), hk, D, seed=1)
    hslots = torch.cat([synthetic.slots_for(bt[i], 0, h, bs) for i, h in hist])
    k, v = synthetic.kv(N, hk, D, seed=2)
    q = synthetic.queries(N, hq, D, seed=3)
    qsl = [0]
    for n, _ in reqs:
        qsl.append(qsl[-1] + n)
    seqs = [n + h for n, h in reqs]
    slots = torch.cat([synthetic.slots_for(bt[i], h, n, bs) for i, (n, h) in enumerate(reqs) if n])
    md = metadata(slots, qsl, seqs, bt)
    md = NS(**{**vars(md), "slot_mapping": slots.to(device), "block_tables": bt.to(device)})
    impl = make_impl(hq, hk, sink=bs, recent=48, staging=8192 if window else 0)
    layer = NS(layer_name="model.layers.1.self_attn.attn", _oscar_rots=(Rk.to(device), Rv.to(device)))
    caches = [torch.zeros(sum(pages), bs, hk, D, dtype=torch.int8, device=device) for _ in range(2)]
    impl.do_kv_cache_update(layer, hk_.to(device), hv_.to(device), caches, hslots.to(device))
    impl._read = None                       # the one-call step must not need it
    out = impl.forward(layer, q.to(device), k.to(device), v.to(device), caches, md,
                       output=torch.full((N, hq, D), 7.0, dtype=torch.bfloat16, device=device))
    torch.cuda.synchronize()
    arena = tuple(t.cpu() for t in (layer._oscar_stage_k, layer._oscar_stage_v, layer._oscar_slot_owner)) \
        if window else None
    return NS(out=out.cpu().float(), q=q.float() @ Rk, k=k.float() @ Rk, v=v.float() @ Rv,
              caches=[c.cpu() for c in caches], arena=arena, bt=bt, qsl=qsl, seqs=seqs, scale=impl.scale, Rv=Rv)


def _check_short(r, reqs):
    for i, (n, _) in enumerate(reqs):
        if not 0 < n <= 16:
            continue
        a, b = r.qsl[i], r.qsl[i + 1]
        rot = oatt.paged_attention_ref(r.q[a:b], r.k[a:b], r.v[a:b], *r.caches, r.bt[i:i + 1], [0, n], [r.seqs[i]],
                                       r.scale, r.arena)
        want = rot @ r.Rv.t()
        err = (r.out[a:b] - want).norm(dim=-1)
        bar = D ** 0.5 * 1e-3 * rot.abs().max() + 2.0 ** -8 * want.norm(dim=-1)
        assert (err <= bar).all(), (i, err.max().item(), bar.min().item())


# new@history.  Several runs of short requests between long ones, histories
# of many splits, a request without history, one without tokens; two and four
# kv heads, whose reads carry 64 and 32 requests a chunk (40 and 70 short
# ones); a write of at most 2048 vectors (fp32 rotation) and ones that share
# their launch with the operand rotation.
@pytest.mark.parametrize("spec,hq,hk,bs", [
    ("3@4000,40@64,1@2500,16@700,600@33,2@5000,5@0,0@70", 8, 2, 64),
    ("3@4000,40@64,1@2500,16@700,33@33,2@5000,5@0,0@70", 8, 2, 64),
    ("9@6100,300@9,1@300", 8, 4, 128),
    (",".join(["2@70,17@9"] * 40), 8, 4, 32),
    (",".join(["1@40,1@90"] * 35 + ["530@3"]), 2, 2, 32)])
@pytest.mark.parametrize("window", [True, False])
def test_short_rows_against_the_oracle(device, spec, hq, hk, bs, window):
    reqs = [tuple(int(x) for x in r.split("@")) for r in spec.split(",")]
    _check_short(_run(device, reqs, hq, hk, bs, window), reqs)


def test_short_requests_far_apart_in_the_batch(device):
    # more table rows between two short requests than a chunk's 16-bit row tells
    reqs = [(2, 90)] + [(0, 0)] * 33000 + [(17, 5), (3, 200)]
    _check_short(_run(device, reqs, 6, 1, 32, True), reqs)
