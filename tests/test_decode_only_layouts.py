"""Rows of any stride through the one-call DecodeOnly forward: what the general
route's products and copies (oscar_ascend/backend.py:321-358) take is not refused.

Without a GPU a launch fails with OSCAR_ERR_LAUNCH, so a call whose arguments
are all accepted comes back with that.  (Not run where there is a GPU: the
addresses are host memory.)
"""
import pytest
import torch

from oscar_amd.kernels import _lib, step

pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="the addresses are host memory")
D, HQ = 256, 2
W = HQ * D


def _call(query, out, B):
    R = torch.eye(D)
    caches = [torch.zeros(4, 32, 1, D, dtype=torch.int8) for _ in range(2)]
    ml = step.MtpLayer(R, R, R, *caches, HQ, 1, 245, 235, D ** -0.5)
    return step.decode_only_forward(ml, query, torch.zeros(B, 2, dtype=torch.int32), [40] * B, out, 0)


def _bf16(*shape):
    return torch.zeros(*shape, dtype=torch.bfloat16)


@pytest.mark.parametrize("query,B", [
    (_bf16(1, W), 1), (_bf16(W, 1).t(), 1), (_bf16(1, 1, D).expand(1, HQ, D), 1), (_bf16(1, W).expand(3, W), 3),
    (_bf16(1, HQ, D).expand(3, HQ, D), 3), (_bf16(W, 3).t(), 3), (_bf16(HQ, 3, D).transpose(0, 1), 3),
    (_bf16(4 * W).as_strided((3, W), (5, 1)), 3), (_bf16(3, W + 3)[:, :W], 3)])
def test_query_rows(query, B):
    with pytest.raises(_lib.OscarKernelError, match="launch"):
        _call(query, _bf16(B, W), B)


def test_output_rows():
    # one row: its stride means nothing
    with pytest.raises(_lib.OscarKernelError, match="launch"):
        _call(_bf16(1, W), _bf16(W, 1).t(), 1)
    # rows that overlap or have no contiguous features: the general route's
    assert _call(_bf16(3, W), _bf16(1, W).expand(3, W), 3) is False
    assert _call(_bf16(3, W), _bf16(W, 3).t(), 3) is False
