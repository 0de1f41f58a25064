"""A sweep whose operators exceed the handle's capacity: an error from this
call and from every later one that sweeps, on the flat kernels and with one
workgroup per chain."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CAPACITY = -3


def _full(loopgpu, c, L):
    """the largest configuration the handle takes: off-diagonal operators on
    one bond of an antiparallel line, all kept by the next sweep, which adds
    diagonal ones on the others"""
    spins = (np.arange(L) & 1).astype(np.int32)
    lo, hi = 0, 1 << 16
    while hi - lo > 2:
        n = (lo + hi) // 4 * 2
        bo = np.full(L + 1, n, np.int32)
        bo[0] = 0
        try:
            c.set_config(spins, bo, (np.arange(n) + 0.5) / n, np.ones(n, np.int32), 7)
            lo = n
        except loopgpu.LoopGPUError as e:
            assert e.code == CAPACITY
            hi = n
    bo = np.full(L + 1, lo, np.int32)
    bo[0] = 0
    c.set_config(spins, bo, (np.arange(lo) + 0.5) / lo, np.ones(lo, np.int32), 7)
    return lo


def _overflow(loopgpu, flat, sweeps, L=16):
    c = loopgpu.Chain(loopgpu.params(loopgpu.CHAIN, L, 4.0, 1.0, 1.0, seed=3))
    assert c.profile(1)["chain_sweep"] > 0
    if flat:
        c.set_launch(group=8)
    n = _full(loopgpu, c, L)
    print("overflow", flat, sweeps, n, flush=True)
    for _ in range(2):
        with pytest.raises(loopgpu.LoopGPUError) as e:
            c.sweep(sweeps)
        assert e.value.code == CAPACITY and "operators" in str(e.value)
    return c


@pytest.mark.parametrize("flat", [False, True])
@pytest.mark.parametrize("sweeps", [1, 2, 5])
def test_error_and_the_handles_after_it(loopgpu, flat, sweeps):
    c = _overflow(loopgpu, flat, sweeps)
    c.close()
    p = loopgpu.params(loopgpu.CHAIN, 16, 4.0, 1.0, 1.0, seed=3)
    a, b = loopgpu.Chain(p), loopgpu.Chain(p)
    b.set_launch(group=8)
    assert np.array_equal(a.sweep(3)[:, :2], b.sweep(3)[:, :2])


@pytest.mark.parametrize("flat", [False, True])
@pytest.mark.parametrize("sweeps", [1, 2, 5])
def test_no_configuration_is_given_out(loopgpu, flat, sweeps):
    """neither state's arrays hold a whole configuration then; one that is set
    comes back as it was"""
    c = _overflow(loopgpu, flat, sweeps)
    for call in (c.info, c.get_config, c.save, lambda: c.set_schedule([1, 9], [0.1, 0.25])):
        with pytest.raises(loopgpu.LoopGPUError) as e:
            call()
        assert e.value.code == CAPACITY
    d = loopgpu.Chain(loopgpu.params(loopgpu.CHAIN, 16, 4.0, 1.0, 1.0, seed=4))
    d.sweep(9)
    ref = d.get_config()
    c.set_config(*ref, 9)
    for x, y in zip(c.get_config(), ref):
        assert np.array_equal(x, y)
    assert c.info() == d.info()
    with pytest.raises(loopgpu.LoopGPUError) as e:
        c.sweep(1)
    assert e.value.code == CAPACITY
