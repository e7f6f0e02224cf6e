"""The memory plan sets the scratch of a step with long requests aside: no step
within the engine's limits asks the library for more."""
import ctypes
import random
from types import SimpleNamespace as NS

import pytest

from oscar_amd import integration
from oscar_amd.kernels import _lib
from tests.fake_engine import Engine


def _library(reqs, hq, hk, max_short=16):
    """oscar_step_forward_workspace_bytes of (new, history) requests."""
    qsl = [0]
    for n, _ in reqs:
        qsl.append(qsl[-1] + n)
    qs, ss = (ctypes.c_int32 * len(qsl))(*qsl), (ctypes.c_int32 * len(reqs))(*[n + h for n, h in reqs])
    return _lib.load().oscar_step_forward_workspace_bytes(len(reqs), ctypes.addressof(qs), ctypes.addressof(ss), hq,
                                                          hk, max_short)


@pytest.mark.parametrize("hq,hk", [(6, 1), (1, 1), (12, 2), (8, 8), (64, 4)])
def test_bound_covers_every_step(hq, hk):
    rng = random.Random(hq * 31 + hk)
    for _ in range(200):
        limit, most = rng.randint(17, 20000), rng.randint(1, 300)
        longest = int(2 ** rng.uniform(5, 18))
        short = rng.choice([0, 4, 16])
        reqs, left = [], limit
        for _ in range(rng.randint(1, most)):
            n = min(left, longest, rng.choice([0, 1, 4, 16, 17, 33, int(2 ** rng.uniform(0, 15))]))
            reqs.append((n, rng.randint(0, longest - n)))
            left -= n
        got = _library(reqs, hq, hk, short)
        assert 0 < got <= integration.step_workspace_bytes(limit, most, hk, hq, longest, short), reqs
    # and it is close to what one long request takes, where a long token's
    # scratch (1540 hq + 1024 hk bytes) is more than a short one's (1024 hq + 2048 hk)
    if hq >= 2 * hk:
        assert integration.step_workspace_bytes(8192, 1, hk, hq, 108192) <= 1.05 * _library([(8192, 100000)], hq, hk)


def test_engine_budget_includes_it(monkeypatch):
    engine = Engine("cpu")
    engine.install(monkeypatch)
    integration.install_runner_hooks()
    runner = engine.Worker().model_runner
    targets = {n: m for n, m in engine.layers.items()}
    bare = integration.oscar_fixed_bytes(runner, engine.specs, targets)
    cfg = NS(**vars(runner.vllm_config))
    cfg.scheduler_config = NS(**vars(cfg.scheduler_config), max_num_batched_tokens=2048)
    impl = next(iter(targets.values())).impl
    want = integration.step_workspace_bytes(2048, 4, impl.num_kv_heads, impl.num_heads, 4096,
                                            impl._oscar.paged_max_q_len)
    assert want > 2 * 256 * 264 * 1000
    got = integration.oscar_fixed_bytes(NS(vllm_config=cfg), engine.specs, targets)
    assert got == bare + want
    a = integration.plan_capacity(200 * 10 ** 9, 16)
    b = integration.plan_capacity(200 * 10 ** 9, 16, max_step_tokens=8192)
    assert b["fixed"] - a["fixed"] == integration.step_workspace_bytes(8192, 256, 1, 6, 262144)
