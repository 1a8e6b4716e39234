"""Batches in persistent launches whose segments are windows apart: a network of next to no
work beside busy ones, two simulators side by side, runs of every remainder."""
import numpy as np
import pytest

from mgbrain_amd import native as N
from mgbrain_amd import workloads as W

pytestmark = pytest.mark.gpu


def _nets():
    """The first network (whose workgroups are the launch's first) has almost nothing to do."""
    quiet = dict(pops=[dict(num=40, type=N.POISSON, rate=0.01), dict(num=60, type=N.LIFB)],
                 projs=[dict(src=0, tar=1, kind=N.CONN_BERNOULLI, p=0.2, w=1e-4, d=1e-3, index=0, seed=1)],
                 lifconst=W.lifb_consts(), seed=1)
    return [quiet] + [W.brunel_sweep_net(n, 4.0, nu, s) for n, nu, s in ((3000, 400.0, 5), (2000, 300.0, 6), (4000, 500.0, 7))]


@pytest.mark.parametrize("mode", [N.PERSIST_AUTO, N.PERSIST_REGIONS, N.PERSIST_LISTS])
def test_batches_side_by_side(mode):
    print(f"case: two batches of four networks side by side, persistent={mode}", flush=True)

    def make(m):
        return N.Simulator.batch_generated(_nets(), propagation=N.PROP_TILED, persistent=m)

    lengths = (1, 10, 23, 60, 7, 400, 35, 250)
    ref = make(N.PERSIST_OFF)
    for n in lengths:
        ref.run(n)
    c, v, e = ref.fire_counts(), ref.state(N.F_V).view(np.uint32), ref.info()["syn_events"]
    ref.close()
    a, b = make(mode), make(mode)
    assert a.info()["persistent"] and a.info()["segments"] == 4
    for n in lengths:
        a.run(n)
        b.run(n)
    for s in (a, b):
        assert np.array_equal(s.fire_counts(), c) and np.array_equal(s.state(N.F_V).view(np.uint32), v)
        assert s.info()["syn_events"] == e
        s.close()
    assert c.sum() > 10000
