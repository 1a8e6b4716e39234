"""The STDP tables' copy in LDS, whose length each tile takes from its own width: narrow
tiles beside a wide Poisson tile, and intervals on both sides of the copy's end."""
import pytest

from mgbrain_amd import native as N
from tests import harness as H
from tests import netmodels as M
from tests.test_gpu_stdp import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wf", [N.WF_F32, N.WF_BF16])
@pytest.mark.parametrize("tile,tau", [(300, 200.0), (40, 200.0), (700, 900.0)])
def test_intervals_past_the_copy(wf, tile, tau):
    print(f"case: 600 Poisson + 400 LIFB, E->E STDP, tau {tau} steps, tile {tile}, weight_format={wf}", flush=True)
    net = M.config2(scale=0.004, K=60, poisson_rate=0.02, stdp=True)
    net.pops[0] = (600, M.POISSON, 1)              # a Poisson tile wider than the others
    for p in net.projs:                            # about 3 Hz: intervals of thousands of steps
        if p["src"] == 0:
            p.update(k=40, wmin=1.3e-4, wmax=1.3e-4)
    syn = H.host_synapses(net, seed=5)
    sc = M.stdp_consts_config4(J=1e-4)
    sc[2] = sc[3] = tau
    changed, n = _run(net, syn, sc, 12000, 5, wf, prop=N.PROP_TILED, window=10, tile_size=tile)
    print(changed, n)
    assert changed > 100
