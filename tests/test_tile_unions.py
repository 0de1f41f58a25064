"""Unions by tiles of sites, and pairs of segments apart (csrc/lg_kernels.hip):
labels against the union-find on the whole configuration, sweeps against the
kernel that unites operator by operator."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def _crowded(nb):
    """diagonal operators on three neighbouring bonds, more than a tile's LDS
    takes, and a few elsewhere"""
    rng = np.random.default_rng(9)
    n = np.zeros(nb, int)
    n[10:13], n[300], n[nb - 1] = 20000, 40, 40
    t = np.concatenate([np.sort(rng.random(k)) for k in n if k])
    return (np.zeros(nb, np.int32), np.concatenate([[0], np.cumsum(n)]).astype(np.int32), t,
            (rng.integers(0, 3, len(t)) << 2).astype(np.int32))


@pytest.mark.parametrize("kind,L,beta,nops,graphs", [
    (O.CHAIN, 1024, 700.0, 30000, (0, 1, 2, 3)),
    (O.CHAIN, 1022, 800.0, 60000, (0,)),           # horizontal graphs alone: many pairs
    (O.CHAIN, 40, 20000.0, 3000, (0, 1)),          # one site a tile
    (O.SQUARE, 90, 80.0, 100000, (0, 1, 2, 3)),    # tiles that do not divide the lattice
    (O.SQUARE, 2, 150000.0, 2000, (0, 1, 2, 3)),
    (O.SQUARE, 4, 30000.0, 5000, (0,)),
    (O.CHAIN, 1024, 700.0, None, None),            # a tile beyond its LDS
])
def test_labels(loopgpu, kind, L, beta, nops, graphs):
    print("labels", kind, L, beta, nops, flush=True)
    cfg = _crowded(L) if nops is None else O.random_config(kind, L, nops, np.random.default_rng(L), graphs, False)
    p = loopgpu.params(kind, L, beta, 1.0, 1.0, seed=77)
    labels, spo, tyo, nc = loopgpu.cluster_config(p, *cfg, 5)
    ref = O.looper_labels(kind, L, cfg[1], cfg[2], cfg[3])
    np.testing.assert_array_equal(labels, ref)
    exp_sp, exp_ty, exp_nc = O.expected_flip(kind, L, 77, 0, 5, *cfg, ref)
    np.testing.assert_array_equal(spo, exp_sp)
    np.testing.assert_array_equal(tyo, exp_ty)
    assert nc == exp_nc


@pytest.mark.parametrize("kind,L,beta,kw", [
    (0, 2, 200.0, {}),
    (0, 64, 60.0, {"jz": 0.9}),
    (0, 64, 60.0, {"h": 0.3}),
    (1, 6, 40.0, {}),
    (0, 1000, 800.0, {}),                          # tiles from here on
    (1, 90, 60.0, {"jz": 0.8}),
    (1, 64, 110.0, {"h": 0.2}),
])
def test_sweeps(loopgpu, kind, L, beta, kw):
    """integers the same, sums to the order of their terms; from a warm
    configuration without field (the all-up start stays as it is in one)"""
    warm = loopgpu.Chain(loopgpu.params(kind, L, beta, 1.0, 1.0, seed=13))
    warm.sweep(20)
    p = loopgpu.params(kind, L, beta, 1.0, kw.get("jz", 1.0), seed=13, h=kw.get("h", 0.0))
    chains = []
    for link, compress in ((0, 0), (128, 0), (512, 0), (1536, 0), (1, 0), (512, 1)):
        c = loopgpu.Chain(p)
        c.set_launch(link=link, compress=compress)
        c.set_config(*warm.get_config(), 20)
        chains.append(c)
    ref = chains[0].sweep(10)
    assert ref[-1, 0] > 0
    for i, c in enumerate(chains[1:]):
        print("sweeps", kind, L, beta, kw, i, flush=True)
        r = c.sweep(10)
        assert np.array_equal(r[:, :2], ref[:, :2])
        np.testing.assert_allclose(r, ref, rtol=1e-9, atol=1e-9)
        for x, y in zip(c.get_config(), chains[0].get_config()):
            assert np.array_equal(x, y)


def test_batch_of_chains_in_tiles(loopgpu):
    ps = [loopgpu.params(k, L, b, 1.0, 1.0, seed=3, chain_id=i)
          for i, (k, L, b) in enumerate([(0, 64, 40.0), (1, 48, 60.0), (0, 2, 30.0), (1, 40, 80.0), (1, 32, 40.0), (0, 256, 300.0)])]
    a, b = loopgpu.Batch(ps), loopgpu.Batch(ps)
    b.set_launch(link=0)
    print("batch", flush=True)
    x, y = a.run(20), b.run(20)
    assert np.array_equal(x[..., :2], y[..., :2])
    np.testing.assert_allclose(x, y, rtol=1e-9, atol=1e-9)
