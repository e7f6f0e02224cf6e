"""The bulk write's fp16 window images against images built from the fp32
arena it wrote: every slot, bit-exact (seats nothing was kept in stay zero in
both).  The V image is written in whole chunks of eight tokens where a wave's
tokens fill one, else token by token.
"""
import pytest
import torch

from oscar_amd import synthetic
from oscar_amd.kernels import quant, staging

pytestmark = pytest.mark.gpu
D = 256


def _slots(kind, n, bs, pages, g):
    if kind == "scattered":
        return torch.randperm(pages * bs, generator=g)[:n]
    if kind == "reversed":
        return torch.arange(n - 1, -1, -1) + 8
    if kind == "collisions":                       # seats (page mod rows) written by several tokens
        return torch.randint(0, pages * bs, (n,), generator=g)
    if kind == "fours":                            # runs of four tokens in pages of their own, then one run
        short = torch.cat([torch.arange(4) + bs * p + 3 * p for p in range(7)])
        return torch.cat([short, torch.arange(n - 28) + 8 * bs])
    return torch.arange(n) + int(kind)             # consecutive from an offset


@pytest.mark.parametrize("kind", ["0", "5", "8", "31", "reversed", "scattered", "collisions", "fours"])
@pytest.mark.parametrize("bs,hk,skipped", [(32, 1, False), (128, 2, True)])
def test_images_follow_the_arena(device, kind, bs, hk, skipped):
    n, recent, sink = 1061, 300, 64                # above 2048 vectors for one head too; no multiple of 32
    g = torch.Generator().manual_seed(n + bs)
    pages = 2048 // bs
    rows = pages - 5 if kind == "collisions" else pages
    slots = _slots(kind, n, bs, pages, g).to(torch.int64)
    if skipped:
        slots[torch.randperm(n, generator=g)[:50]] = -1
    k, v = (t.to(torch.bfloat16).to(device) for t in synthetic.kv(n, hk, D, seed=3))
    ops = [quant.rotation_operand(r.to(device)) for r in synthetic.rotations(D, seed=2)]
    caches = [torch.zeros(pages, bs, hk, D, dtype=torch.int8, device=device) for _ in range(2)]
    sk = torch.zeros(rows, bs, hk, D, device=device)
    sv, owner = torch.zeros_like(sk), torch.full((rows, bs), -7, dtype=torch.int64, device=device)
    kimg = torch.zeros(staging.k_image_shape(rows, bs, hk), dtype=torch.float16, device=device)
    vimg = torch.zeros(staging.image_shape(rows, bs, hk), dtype=torch.float16, device=device)
    qsl, seqs = [0, 28, n], [28, n - 28]           # the first request's tokens are all recent
    layout = [torch.tensor(x, dtype=torch.int32, device=device) for x in (qsl, seqs)]
    quant.quant_write(k, v, *ops, *caches, slots.to(device), 245, 235, hk, D,
                      window=(*layout, 2, sink, recent, sk, sv, owner,
                              staging.winner_buffer(rows, bs, torch.device(device)), kimg, vimg))
    torch.cuda.synchronize()
    want_k, want_v = staging.stage_images(sk.cpu(), sv.cpu())
    assert torch.equal(kimg.cpu(), want_k) and torch.equal(vimg.cpu(), want_v)
    # the tokens the arena has to hold: the last of each seat, if kept
    winner = {}
    for t, s in enumerate(slots.tolist()):
        if s >= 0:
            winner[((s // bs) % rows, s % bs)] = t
    kept = torch.zeros(rows, bs, dtype=torch.bool)
    for (r, c), t in winner.items():
        i = 0 if t < 28 else 1
        pos = seqs[i] - qsl[i + 1] + t
        kept[r, c] = pos >= seqs[i] - recent or pos < sink
    assert torch.equal((sv != 0).any(-1).any(-1).cpu(), kept)
