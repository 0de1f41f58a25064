"""A HIP error that an earlier call of the thread left behind (here an
allocation of 2^50 bytes, refused) is not taken for a later call's own."""

import ctypes

import numpy as np
import pytest

from test_zz_no_alloc import noalloc

pytestmark = pytest.mark.gpu


def _leave_an_error(lg):
    gbs = ctypes.c_double()
    assert lg.lib.lg_copy_bandwidth(1 << 50, 1, ctypes.byref(gbs)) == -2  # LG_ERR_DEVICE


@pytest.mark.parametrize("flat", [False, True])
@pytest.mark.parametrize("graph", [False, True])
def test_calls_after_it(loopgpu, flat, graph):
    lg = loopgpu
    ps = [lg.params(lg.CHAIN, 16, 4.0, 1.0, 1.0, seed=1, chain_id=i) for i in range(3)]
    c, b = lg.Chain(ps[0]), lg.Batch(ps)
    if flat:
        c.set_launch(group=8)
        b.set_launch(group=8)
    b.set_graph(graph)
    c.sweep(2)
    b.run(2)
    config = c.get_config()
    for call in (c.get_config, lambda: c.sweep(1), lambda: b.run(2), lambda: c.profile(1), lambda: b.add([ps[0]]),
                 lambda: lg.cluster_config(ps[0], *config, 5), lambda: noalloc(lg, ps[0], *config, 5)):
        _leave_an_error(lg)
        call()
    assert np.array_equal(b.run(1)[0, 0, :2], c.sweep(1)[0, :2])
