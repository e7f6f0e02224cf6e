"""oscar_step_forward refuses a step before it enqueues anything.

Without a GPU a launch fails with OSCAR_ERR_LAUNCH, so a refusal that comes
back as what it is came before the first launch.  (Not run where there is a
GPU: the addresses are host memory.)
"""
import ctypes

import pytest
import torch

from oscar_amd.kernels import _lib, step

pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="the addresses are host memory")
D = 256
INVALID, LAUNCH = "invalid argument", "kernel launch failed"


def _call(reqs, cols, window, hq=2, hk=1, bs=32, max_short=16):
    """The status of a step of new@history requests over a table of `cols` pages a request."""
    lib = _lib.load()
    N, B = sum(n for n, _ in reqs), len(reqs)
    buf = torch.zeros(4096, dtype=torch.uint8)
    at = (buf.data_ptr() + 15) & ~15
    args = step.MtpLayerArgs(at, at, at, at, at, 64, bs * hk * 256, hk * 256, 256, bs * hk * 256, hk * 256, 256, bs,
                             hq, hk, D, 245, 235, D ** -0.5, 8 if window else 0, *([at] * 5), bs, 48)
    qsl = [0]
    for n, _ in reqs:
        qsl.append(qsl[-1] + n)
    qs, ss = (ctypes.c_int32 * (B + 1))(*qsl), (ctypes.c_int32 * B)(*[n + h for n, h in reqs])
    need = lib.oscar_step_forward_workspace_bytes(B, ctypes.addressof(qs), ctypes.addressof(ss), hq, hk, max_short)
    assert need > 0
    status = lib.oscar_step_forward(ctypes.addressof(args), at, at, at, at, at, hq * D, at, at, hk * D, at, at, cols,
                                    cols, ctypes.addressof(qs), ctypes.addressof(ss), B, max_short, at, at, need, None)
    return _lib.STATUS.get(status, status)


# A write of at most 2048 vectors (a launch of its own) and of more (with a
# window its seat-winner pass is; without, it shares one with the operands).
@pytest.mark.parametrize("new", [20, 1100])
@pytest.mark.parametrize("window", [True, False])
def test_refused_before_the_first_launch(new, window):
    # a long request's history needs 4 pages
    assert _call([(2, 10), (new, 100)], 4, window) == LAUNCH
    assert _call([(2, 10), (new, 100)], 3, window) == INVALID
    # ... of the second prefill launch of the step
    assert _call([(17, 0)] * 48 + [(new, 100)], 3, window) == INVALID
    # a short request's history beyond what a read can split
    assert _call([(new, 0), (2, 9 << 20)], 1 << 20, window) == INVALID
