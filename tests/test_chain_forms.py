"""Which form of the sweep a batch takes, and the one-workgroup form
(csrc/lg_block.hip) where its tables outgrow LDS: parents in memory, event
times cut to 15 bits or read in full, accumulators in windows.  Every case
first shows that the form runs, then compares with the flat kernels: whole
numbers equal, sums to the order of their terms (1e-9 of 2e5 terms each
rounded at 1e-16 leaves a factor of fifty)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _same(a, b):
    assert np.array_equal(a[..., :2], b[..., :2])  # operators, clusters
    np.testing.assert_allclose(a, b, rtol=1e-9, atol=1e-9)


def _one_workgroup(x):
    return x.profile(1)["chain_sweep"] > 0


@pytest.mark.parametrize("kind,L,beta,kw", [
    (0, 2, 0.5, {}),
    (0, 16, 4.0, {}),
    (0, 64, 10.0, {}),
    (0, 256, 1.0, {}),                            # as many bonds as threads
    (1, 16, 8.0, {}),                             # 1024 threads
    (1, 36, 0.3, {}),                             # more sites and bonds than threads, event-free sites
    (1, 14, 6.0, {"h": 0.4}),
    (0, 12, 20.0, {"two_s": 2}),
    (1, 4, 3.0, {"two_s": 3, "d": -0.3}),
    (1, 10, 4.0, {"jxy": 0.0, "jz": -1.0, "hx": 0.8}),
])
@pytest.mark.parametrize("tune", [0, 1, 4])
def test_small_chains_take_it(loopgpu, kind, L, beta, kw, tune):
    """also after a tuning of one sweep a trial, which leaves the rule's choice"""
    kw = dict(kw)
    p = loopgpu.params(kind, L, beta, kw.pop("jxy", 1.0), kw.pop("jz", 1.0), seed=31, **kw)
    a, b = loopgpu.Batch([p]), loopgpu.Batch([p])
    print("form", kind, L, beta, kw, tune, flush=True)
    if tune:
        a.tune(tune)
    if tune != 4:
        assert _one_workgroup(a)
    b.set_launch(group=8)
    b.run(a.chain_info(0)[1], records=False)
    for n in (1, 2, 20):
        _same(a.run(n), b.run(n))


def _betas(lo, hi, n):
    return [lo * (hi / lo) ** (i / (n - 1)) for i in range(n)]


@pytest.mark.parametrize("chains,kind,L,lo,hi,least,kw", [
    # segments beyond 65536: parents in memory, full event times
    (320, 1, 32, 0.5, 40.0, 33000, {}),
    # flips by the clusters' magnetization over windows of accumulators
    (300, 1, 32, 0.5, 20.0, 9000, {"h": 0.01}),
    # virtual sites, site operators
    (300, 0, 96, 0.5, 60.0, 8000, {"two_s": 2}),
    (300, 1, 16, 0.5, 30.0, 8000, {"jxy": 0.0, "jz": -1.0, "hx": 0.8}),
])
def test_cold_batches(loopgpu, chains, kind, L, lo, hi, least, kw):
    kw = dict(kw)
    jxy, jz = kw.pop("jxy", 1.0), kw.pop("jz", 1.0)
    ps = [loopgpu.params(kind, L, be, jxy, jz, seed=5, chain_id=i, **kw) for i, be in enumerate(_betas(lo, hi, chains))]
    a, b = loopgpu.Batch(ps), loopgpu.Batch(ps)
    b.set_launch(group=8)
    assert _one_workgroup(a)
    b.run(1, records=False)
    most = 0
    for n in (1, 10, 3, 2):
        print("batch", kind, L, hi, kw, n, flush=True)
        x = a.run(n)
        _same(x, b.run(n))
        most = max(most, x[..., 0].max())
    assert most > least
    a.set_launch(group=8)
    _same(a.run(1), b.run(1))


def test_pairs_of_many_chains_in_a_chunk(loopgpu):
    """the flat estimator's chunk of 1024 to 4096 segments over chains of two
    segments each up to a few hundred: more of them than it has slots, and
    chunks that begin inside a chain"""
    ps = [loopgpu.params(0, 2 + 2 * (i % 5), be, 1.0, 1.0, seed=5, chain_id=i) for i, be in enumerate(_betas(0.1, 20.0, 400))]
    a, b, c = loopgpu.Batch(ps), loopgpu.Batch(ps), loopgpu.Batch(ps)
    b.set_launch(group=8, link=0)
    c.set_launch(group=8, link=512, compress=1)
    assert _one_workgroup(a)
    b.run(1, records=False)
    c.run(1, records=False)
    for n in (1, 30):
        print("chains", n, flush=True)
        x = a.run(n)
        _same(x, b.run(n))
        _same(x, c.run(n))
