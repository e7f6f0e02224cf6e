"""A short window write through oscar_quant_write_window reads its request
layout on the stream: arrays that earlier work of the stream fills give the
same bytes as arrays that were complete before the call.  (Whole numbers and
copies of the same fp32 rotation: bit-exact.)
"""
import pytest
import torch

from oscar_amd import synthetic
from oscar_amd.kernels import quant, staging

pytestmark = pytest.mark.gpu
D = 256


# One request; one of no tokens between others; more than one and more than
# two rounds of 64 starts; a last request that ends before the tokens do.
@pytest.mark.parametrize("lengths,hk,uncovered", [([5], 1, 0), ([3, 0, 40], 2, 0), ([1] * 64, 1, 0), ([2] * 130, 1, 0),
                                                  ([7, 9], 1, 4)])
def test_layout_filled_on_the_stream(device, lengths, hk, uncovered):
    bs, rows, pages, sink, recent = 32, 24, 40, 32, 4
    B, N = len(lengths), sum(lengths) + uncovered
    qsl = torch.tensor([0] + lengths).cumsum(0).to(torch.int32)
    seqs = torch.tensor([n + 40 * (i % 2) for i, n in enumerate(lengths)], dtype=torch.int32)
    meta = torch.cat([qsl, seqs]).to(device)
    k, v = (t.to(torch.bfloat16).to(device) for t in synthetic.kv(N, hk, D, seed=N))
    ops = [quant.rotation_operand(r.to(device)) for r in synthetic.rotations(D, seed=2)]
    slots = torch.randperm(pages * bs, generator=torch.Generator().manual_seed(N))[:N].to(device)
    busy = torch.randn(4096, 4096, device=device)

    def write(late):
        caches = [torch.zeros(pages, bs, hk, D, dtype=torch.int8, device=device) for _ in range(2)]
        sk = torch.zeros(rows, bs, hk, D, device=device)
        arena = [sk, torch.zeros_like(sk), torch.full((rows, bs), -7, dtype=torch.int64, device=device),
                 staging.winner_buffer(rows, bs, torch.device(device)),
                 torch.zeros(staging.k_image_shape(rows, bs, hk), dtype=torch.float16, device=device),
                 torch.zeros(staging.image_shape(rows, bs, hk), dtype=torch.float16, device=device)]
        layout = torch.zeros_like(meta) if late else meta
        torch.cuda.synchronize()
        if late:
            for _ in range(20):
                busy @ busy
            layout.copy_(meta)
        quant.quant_write(k, v, *ops, *caches, slots, 245, 235, hk, D,
                          window=(layout[:B + 1], layout[B + 1:], B, sink, recent, *arena))
        torch.cuda.synchronize()
        return caches + arena[:3] + arena[4:]

    early, late = write(False), write(True)
    for a, b in zip(early, late):
        assert torch.equal(a, b)
    # the keep rule itself: the sink, and the last `recent` positions
    owner = early[4].cpu()
    last = {}
    for t in range(N):
        page, col = divmod(int(slots[t]), bs)
        last[(page % rows, col)] = (t, page)
    for (row, col), (t, page) in last.items():
        i = max((j for j in range(B) if qsl[j] <= t < qsl[j + 1]), default=None)
        pos = None if i is None else int(seqs[i] - qsl[i + 1]) + t
        kept = pos is not None and (pos < sink or pos >= int(seqs[i]) - recent)
        assert owner[row, col] == (page if kept else -1)
