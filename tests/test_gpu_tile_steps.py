"""The fused kernel's neuron steps against the oracle, bit for bit, where their batches
(4, 2 and 1 steps) and lanes run out: windows of every remainder, tiles wider than the
workgroup, counts past the cached class sums, tiles of more classes than are cached,
tiles without synapses, each neuron type in each ring form, one launch per window and
persistent."""
import numpy as np
import pytest

from mgbrain_amd import native as N
from mgbrain_amd import workloads as W
from oracle import pyoracle as po
from tests import harness as H
from tests import netmodels as M
from tests.test_gpu_parity import _compare_run, _say

pytestmark = pytest.mark.gpu


def _net(kind):
    if kind == "lifb":
        net = M.config1(scale=0.2, poisson_rate=0.2)
    elif kind == "dense":                 # about 45 excitatory arrivals per neuron and step
        net = M.config1(scale=0.1, p=0.9, poisson_rate=0.5)
    elif kind == "life":
        net = M.config3(scale=0.02, p=0.1, g_exc=0.4, g_inh=5.1)
    else:
        net = M.lif_net()
    syn = H.host_synapses(net, seed=6)
    if kind == "classes":                 # five weights per sign over neighbouring targets
        syn.weight = (syn.weight * (1.0 + 0.1 * (syn.tar % 5))).astype(np.float32)
    return net, syn


@pytest.mark.parametrize("persist", [N.PERSIST_AUTO, N.PERSIST_REGIONS, N.PERSIST_OFF])
@pytest.mark.parametrize("kind,wf,window,tile,block", [
    ("lifb", 1, 1, 100, 512), ("lifb", 1, 5, 333, 64), ("lifb", 2, 7, 333, 128), ("dense", 1, 0, 256, 256),
    ("dense", 1, 3, 400, 64), ("dense", 2, 0, 256, 1024), ("life", 1, 0, 200, 512), ("life", 2, 6, 300, 128),
    ("lif", 1, 3, 256, 64), ("lif", 2, 11, 300, 512), ("classes", 1, 10, 256, 512), ("classes", 1, 9, 500, 128)])
def test_steps_of_a_window(kind, wf, window, tile, block, persist):
    _say(f"case: {kind}, weight_format={wf}, window={window}, tile={tile}, block={block}, persistent={persist}")
    net, syn = _net(kind)
    n = _compare_run(net, syn, 300, seed=6, acc=po.ACC_F32 if wf == 1 else po.ACC_FIXED,
                     gpu_kw=dict(weight_format=wf, window=window, tile_size=tile, prop_block=block, propagation=2,
                                 persistent=persist))
    assert n > 100


def test_regions_with_tiles_a_window_ahead():
    """List regions where some tiles have next to nothing to do (three Poisson neurons)
    beside tiles of many synapses: the light tiles publish the next window's count while
    others still wait for this one's."""
    _say("case: 3-neuron Poisson tiles beside LIFB tiles, 30000 steps, list regions")
    pops = [dict(num=3, type=N.POISSON, rate=0.3), dict(num=900, type=N.POISSON, rate=0.05),
            dict(num=6000, type=N.LIFB)]
    projs = [dict(src=s, tar=2, kind=N.CONN_FIXED_INDEGREE, k=k, w=w, dmin=1e-3, dmax=2e-3, index=i, seed=9)
             for i, (s, k, w) in enumerate(((0, 3, 1e-5), (1, 300, 1e-5), (2, 400, -1e-5)))]
    out = []
    for mode in (N.PERSIST_REGIONS, N.PERSIST_OFF):
        g = N.Simulator.generated(pops, projs, W.lifb_consts(), seed=9, propagation=2, tile_size=60, prop_block=512,
                                  persistent=mode)
        assert g.info()["persistent"] == (2 if mode == N.PERSIST_REGIONS else 0)
        g.run(30000)
        out.append((g.fire_counts(), g.state(N.F_V).view(np.uint32), g.info()["spikes"]))
        g.close()
    (ca, va, na), (cb, vb, nb) = out
    assert na == nb and na > 100000
    assert np.array_equal(ca, cb) and np.array_equal(va, vb)
