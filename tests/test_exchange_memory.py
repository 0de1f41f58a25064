"""Memory of a replica-exchange set: a region of the largest beta's operators
for every replica only where one workgroup sweeps each."""

import ctypes
import gc
import math

import pytest

pytestmark = pytest.mark.gpu


def _taken(make):
    hip = ctypes.CDLL("/opt/rocm/lib/libamdhip64.so.7")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def now():
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    gc.collect()  # (handles that earlier tests left)
    before = now()
    x = make()
    after = now()
    return x, before - after


def test_no_regions_for_a_set_on_the_flat_kernels(loopgpu):
    lg, n, L = loopgpu, 32, 64
    betas = [0.5 * 128.0 ** (i / (n - 1)) for i in range(n)]
    model = dict(jxy=1.0, jz=1.0, seed=1)
    b, batch = _taken(lambda: lg.Batch([lg.params(lg.SQUARE, L, be, chain_id=i, **model) for i, be in enumerate(betas)]))
    x, exchange = _taken(lambda: lg.Exchange(lg.params(lg.SQUARE, L, 1.0, **model), betas, seed=2))
    # every replica has the candidate slots (9 bytes) of the largest beta
    cap = [math.ceil(0.5 * be + 12 * math.sqrt(0.5 * be) + 16) for be in betas]
    slots = 9 * 2 * L * L * sum(max(cap) - c for c in cap)
    print("batch", batch, "exchange", exchange, "slots", slots, flush=True)
    assert x.profile(1)["chain_sweep"] == 0
    assert exchange < batch + slots + (32 << 20)


def test_a_small_set_takes_the_form_that_needs_them(loopgpu):
    lg = loopgpu
    x = lg.Exchange(lg.params(lg.SQUARE, 16, 1.0, 1.0, 1.0, seed=1), [0.5 * 20.0 ** (i / 31) for i in range(32)], seed=2)
    x.run(3)
    assert x.profile(2)["chain_sweep"] > 0
