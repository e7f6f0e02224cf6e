"""A large cache write and the same tokens in parts of 5000 (which another
kernel writes, from the same products in the same order): every byte equal.

Sizes around the 128-token workgroups' rounds of 512, where the kernel changes:
13/16 of a round, a whole round, one workgroup over, two rounds but a sixteenth,
and 2 11/16 rounds, with whole and partial last workgroups."""
import pytest
import torch

from oscar_amd import synthetic
from oscar_amd.kernels import quant

pytestmark = pytest.mark.gpu
D = 256


@pytest.mark.parametrize("N,hk", [(26496, 1), (26497, 1), (6656, 4), (30720, 1), (32768, 1), (32769, 1), (16384, 2),
                                  (16400, 2), (63488, 1), (63489, 1), (87936, 1), (87937, 1), (102401, 1), (26000, 4)])
@pytest.mark.parametrize("clip", [(245, 235), (-1, -1)])
def test_bytes_equal_the_parts(device, N, hk, clip):
    bs = 128
    g = torch.Generator(device=device).manual_seed(N)
    k, v = ((torch.randn(N, hk, D, generator=g, device=device)).to(torch.bfloat16) for _ in range(2))
    ops = [quant.rotation_operand(r.to(device)) for r in synthetic.rotations(D, 3)]
    pages = N // bs + 2
    slots = torch.randperm(pages * bs, generator=g, device=device)[:N]
    slots[::17] = -1

    def write(part):
        caches = [torch.zeros(pages, bs, hk, D, dtype=torch.int8, device=device) for _ in range(2)]
        for a in range(0, N, part):
            a = min(a, max(N - part, 0))        # (a short last part would be rotated in fp32)
            quant.quant_write(k[a:a + part], v[a:a + part], *ops, *caches, slots[a:a + part], *clip, hk, D)
        torch.cuda.synchronize()
        return caches

    for got, want in zip(write(N), write(5000)):
        assert torch.equal(got, want)
