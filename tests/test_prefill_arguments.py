"""What the two prefill entries over fp32 rows accept and refuse, without a GPU:
where all checks pass the launch fails with OSCAR_ERR_LAUNCH.  (Not run where
there is a GPU: the addresses are host memory.)"""
import ctypes

import pytest
import torch

from oscar_amd.kernels import _lib

pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="the addresses are host memory")
D = 256
OK, INVALID, SMALL, LAUNCH, GEOMETRY = 0, -1, -3, -4, -5


@pytest.mark.parametrize("split", [False, True])
def test_accepted_and_refused(split):
    lib = _lib.load()
    buf = torch.zeros(256, dtype=torch.uint8)
    at = (buf.data_ptr() + 15) & ~15

    def call(new, cached=64, hq=2, hk=1, bs=32, cache=at, kst=(8192, 256, 256), vst=(8192, 256, 256), cols=4, ws=at,
             size=1 << 40):
        args = (at, at, at, new, hq, hk, D, cache, cache, bs, 64, *kst, *vst, at, cols, cached, None, None, None, 0,
                ctypes.c_float(0.1), at)
        if split:
            return lib.oscar_prefill_continuation_split(*args, ws, size, None)
        return lib.oscar_prefill_continuation(*args, None)

    assert call(20) == LAUNCH
    # V slots and strides of any alignment; K strides are multiples of 8
    assert call(20, vst=(32 * 67, 67, 64)) == LAUNCH
    assert call(20, kst=(8192, 252, 256)) == GEOMETRY
    assert call(20, bs=48) == GEOMETRY
    assert call(20, cached=64, cols=1) == INVALID
    assert call(20, cache=None) == INVALID
    # nothing to do: only the counts are looked at
    assert call(0) == OK and call(0, cache=None) == OK and call(0, bs=16) == OK and call(0, cols=0) == OK
    assert call(0, cached=-1) == INVALID and call(0, hq=3, hk=2) == INVALID and call(-1) == INVALID
    if split:
        assert call(20, ws=at + 8) == INVALID
        # as much scratch as is asked for: next to none where whole row blocks
        # are read, partials and operands where shares are
        for new, cached, most in ((20, 64, 256), (2000, 64, 1 << 28)):
            need = lib.oscar_prefill_workspace_bytes(new, 2, 1, cached)
            assert 0 < need <= most and call(new, cached, size=need) == LAUNCH and call(new, cached, size=need - 1) == SMALL
        assert need > 1 << 20
