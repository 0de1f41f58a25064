"""Sweeps by one workgroup per chain (csrc/lg_block.hip) against the flat
kernels, which explicit launch settings select: the same trajectories, at the
sizes where the workgroup changes its data layout."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _same(a, b):
    assert np.array_equal(a[..., :2], b[..., :2])  # operators, clusters
    np.testing.assert_allclose(a, b, rtol=1e-9, atol=1e-9)


@pytest.mark.parametrize("kind,L,beta,kw,sweeps", [
    (0, 2, 0.5, {}, 20),                          # one word of every bit set, often no operator at all
    (0, 2, 40.0, {}, 20),
    (1, 2, 9.0, {"jz": 0.6}, 20),
    (0, 32, 4.0, {}, 30),                         # around 64 operators, 128 segments
    (0, 64, 10.0, {"jxy": 1.0, "jz": -0.5}, 30),
    (0, 256, 1.0, {}, 20),                        # as many bonds as threads, few operators
    (1, 16, 10.0, {}, 20),
    (1, 64, 0.3, {}, 10),                         # more sites and bonds than threads, event-free sites
    (1, 14, 6.0, {"h": 0.4}, 20),
    (0, 12, 20.0, {"two_s": 2}, 20),
    (1, 4, 3.0, {"two_s": 3, "d": -0.3}, 20),
    (1, 10, 4.0, {"jxy": 0.0, "jz": -1.0, "hx": 0.8}, 20),
    (0, 10, 6.0, {"hx": -0.5}, 20),               # signed
])
def test_equals_flat_kernels(loopgpu, kind, L, beta, kw, sweeps):
    kw = dict(kw)
    p = loopgpu.params(kind, L, beta, kw.pop("jxy", 1.0), kw.pop("jz", 1.0), seed=31, **kw)
    a, b = loopgpu.Chain(p), loopgpu.Chain(p)
    b.set_launch(group=8)
    print("chain", kind, L, beta, kw, flush=True)
    for n in (1, 2, sweeps):
        _same(a.sweep(n), b.sweep(n))
        for x, y in zip(a.get_config(), b.get_config()):
            assert np.array_equal(x, y)


def test_batches_cold_chains_and_changes_of_form(loopgpu):
    """300 chains (more than the CUs) up to 24000 operators, whose segments
    need the 16-bit parents and accumulators in several passes; then chains
    join (the batch continues from the packed form, several sweeps a launch)
    and flat launches take over."""
    ps = [loopgpu.params(loopgpu.SQUARE, 32, 0.5 * 40.0 ** (i / 299), seed=5, chain_id=i) for i in range(300)]
    a, b = loopgpu.Batch(ps[:290]), loopgpu.Batch(ps[:290])
    b.set_launch(group=8)
    for n in (1, 12, 3):
        print("batch", n, flush=True)
        _same(a.run(n), b.run(n))
    a.add(ps[290:])
    b.add(ps[290:])
    b.set_launch(group=8)
    print("batch of 300", flush=True)
    _same(a.run(5), b.run(5))
    assert [a.chain_info(c) for c in (0, 150, 299)] == [b.chain_info(c) for c in (0, 150, 299)]
    a.set_launch(group=16)
    print("flat", flush=True)
    _same(a.run(2), b.run(2))


@pytest.mark.parametrize("kind,L,beta", [(0, 16, 4.0), (1, 32, 6.0), (1, 48, 12.0)])  # below and above the export's 256 KB
def test_configuration_by_either_way_out(loopgpu, kind, L, beta):
    """operator counts known from the last records, or asked from the device;
    spins alone; after a configuration was set"""
    c = loopgpu.Chain(loopgpu.params(kind, L, beta, seed=3))
    print("config", kind, L, beta, flush=True)
    c.sweep(7)
    a = c.get_config()
    spins = np.zeros(c.n_sites, np.int32)
    assert loopgpu.lib.lg_chain_get_config(c.h, spins.ctypes.data, None, None, None) == 0
    assert np.array_equal(spins, a[0])
    d = loopgpu.Chain(loopgpu.params(kind, L, beta, seed=3))
    d.sweep(7, records=False)
    for x, y in zip(a, d.get_config()):
        assert np.array_equal(x, y)
    d.sweep(3)
    d.set_config(*a, 7)
    assert d.info() == c.info()
    for x, y in zip(a, d.get_config()):
        assert np.array_equal(x, y)
    assert np.array_equal(c.sweep(2)[:, :2], d.sweep(2)[:, :2])
