"""The fused write's clip threshold and packing where they can go wrong, byte
for byte: with R = I the MFMA rotation is exact (bf16 inputs, products by 1
and 0), so the cache bytes have to be the oracle's (the sign of a zero meta
aside, which torch leaves open).
"""
import pytest
import torch

from oscar_amd.kernels import quant
from tests.test_gpu_quant_write import make_caches, oracle_store, zero_sign_free

pytestmark = pytest.mark.gpu
D = 256


def _vectors(kind, n, hk, g):
    x = torch.randn(n, hk, D, generator=g)
    if kind == "ties":                       # buckets of more values than a candidate list holds
        x = torch.randint(-3, 4, (n, hk, D), generator=g).float()
    elif kind == "constant":
        x = torch.full((n, hk, D), 0.75) * (torch.arange(n) % 3 - 1).float()[:, None, None]
    elif kind == "range":                    # answers far below the histogram's two octaves
        x = x * torch.exp2(torch.rand(n, hk, D, generator=g) * 40 - 30)
    elif kind == "outlier":                  # one value far above the others
        x[..., 17] = 1e4
        x[::2, ..., 200] = -3e4
    return x.to(torch.bfloat16)


# One more token than the short write takes, with a remainder below 32, a
# multiple of 32, and strided inputs with two heads; ratios that pick the
# smallest, middle and largest value, and no clip.
@pytest.mark.parametrize("kind", ["normal", "ties", "constant", "range", "outlier"])
@pytest.mark.parametrize("ratios", [(0.96, 0.92), (0.0, 0.5), (1.0, 0.004), (0.84, 0.85)])
@pytest.mark.parametrize("n,hk", [(1027, 1), (544, 2)])
def test_bytes_with_an_exact_rotation(device, kind, ratios, n, hk):
    _check(device, kind, ratios, n, hk)


# The kernel of 128-token workgroups: exactly one round of them with a remainder
# in the last, most of a round, the fewest that take it, and one less (the kernel
# above).
@pytest.mark.parametrize("n,hk", [(32765, 1), (30721, 1), (30720, 1), (16300, 2), (26497, 1), (26496, 1)])
def test_bytes_of_whole_rounds(device, n, hk):
    _check(device, "ties" if n % 2 else "range", (0.96, 0.5), n, hk)


def _check(device, kind, ratios, n, hk):
    g = torch.Generator().manual_seed(n)
    k, v = _vectors(kind, n, hk, g), _vectors(kind, n, hk, g)
    bs, pages = 32, n // 32 + 7
    caches = make_caches(pages, bs, hk, torch.int8, seed=4)
    slots = torch.randperm(pages * bs, generator=g)[:n]
    slots[::17] = -1
    want = oracle_store(k.float(), v.float(), caches, slots, *ratios)
    op = quant.rotation_operand(torch.eye(D, device=device))
    dev = [c.to(device) for c in caches]
    wide = [torch.zeros(n, hk * D + 8, dtype=torch.bfloat16, device=device) for _ in range(2)]
    for w, x in zip(wide, (k, v)):
        w[:, :hk * D] = x.reshape(n, -1).to(device)
    quant.quant_write(wide[0][:, :hk * D], wide[1][:, :hk * D], op, op, *dev, slots.to(device),
                      quant.clip_index(ratios[0], D), quant.clip_index(ratios[1], D), hk, D)
    torch.cuda.synchronize()
    assert torch.equal(zero_sign_free(dev[0].cpu().view(torch.uint8)), zero_sign_free(want[0].view(torch.uint8)))
    assert torch.equal(dev[1].cpu(), want[1])
