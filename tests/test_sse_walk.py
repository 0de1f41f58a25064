"""The run-wise series walk (csrc/lg_sse.hip) against the oracle's step-by-step
one: strings of no operator, of less and more than 64, of many 64s; every
diagonal operator removed (n above beta W) or most of them kept (hot); all
three classes of locations; the largest lattice the worker takes."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,L,beta,sweeps,kw", [
    (O.CHAIN, 2, 0.02, 60, {}),                                  # empty strings
    (O.CHAIN, 8, 0.5, 60, {"jxy": 1.0, "jz": 0.3}),              # hot: regraphed diagonal operators
    (O.CHAIN, 64, 3.0, 40, {"jxy": -1.0, "jz": 0.5}),            # runs across 64 steps and 64 operators
    (O.SQUARE, 32, 8.0, 6, {}),                                  # thousands of operators
    (O.CHAIN, 4096, 0.5, 6, {}),                                 # 4096 sites and bonds
    (O.CHAIN, 12, 2.0, 40, {"two_s": 2, "d": 0.4, "jxy": -1.0, "jz": 1.0, "hx": 0.6}),
    (O.SQUARE, 6, 3.0, 30, {"jxy": 0.0, "jz": -1.0, "hx": 1.5}),
])
def test_walk_bit_exact_with_oracle(loopgpu, kind, L, beta, sweeps, kw):
    kw = dict(kw)
    jxy, jz = kw.pop("jxy", 1.0), kw.pop("jz", 1.0)
    c = O.PhiloxChain(kind, L, beta, jxy, jz, seed=9, chain_id=4, **kw)
    g = loopgpu.Chain(loopgpu.params(kind, L, beta, jxy, jz, seed=9, chain_id=4, algorithm=loopgpu.SSE, **kw))
    print("walk", kind, L, beta, kw, flush=True)
    rc, rg = c.sweep_sse(sweeps), g.sweep(sweeps)
    assert np.array_equal(rg[:, :2], rc[:, :2])
    np.testing.assert_allclose(rg[:, 2:18], rc[:, 2:18], rtol=1e-9, atol=1e-9)
    for a, b in zip(g.get_config(), c.state()):
        assert np.array_equal(a, b)
