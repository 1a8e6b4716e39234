"""Persistent launches whose windows pass their spikes with the wait's flags, against one
launch per window, bit for bit: no spikes, as many as a flag holds (14 a tile) and more
(the rest through the tile's part of the list), past the 1,024 a tile's list holds in LDS,
steps up to 31, tiles of 2,048, more flags than a workgroup reads at once."""
import numpy as np
import pytest

from mgbrain_amd import native as N
from mgbrain_amd import workloads as W
from tests.test_gpu_persistent import _compare, _say

pytestmark = pytest.mark.gpu


def _make(n, wf, tile, block, delay, g, records=2_000_000):
    pops, projs, _, _ = W.vogels_abbott(scale=n / 80000.0, p=0.05, seed=4, g_exc=g, g_inh=8 * g)
    for p in projs:
        p["d"] = float(np.float32(delay))
    return lambda mode: N.Simulator.generated(pops, projs, W.life_const1(), seed=4, weight_format=wf, tile_size=tile,
                                              prop_block=block, propagation=N.PROP_TILED, persistent=mode,
                                              record_capacity=records)


@pytest.mark.parametrize("mode", [N.PERSIST_AUTO, N.PERSIST_REGIONS, N.PERSIST_LISTS])
@pytest.mark.parametrize("n,wf,tile,block,delay,g", [
    (4000, N.WF_CLASS, 60, 128, 0.0008, 0.1), (4000, N.WF_BF16, 60, 128, 0.0008, 0.1),
    (4000, N.WF_CLASS, 300, 512, 0.0032, 0.1), (4000, N.WF_F32, 300, 512, 0.0032, 0.1),
    (4000, N.WF_FP8, 250, 64, 0.0001, 0.1), (4000, N.WF_CLASS, 1000, 64, 0.0032, 0.4),
    (6000, N.WF_BF16, 2048, 1024, 0.0016, 0.4), (300, N.WF_CLASS, 7, 64, 0.0008, 0.4)])
def test_spikes_with_the_flags(n, wf, tile, block, delay, g, mode):
    _say(f"case: {n} neurons, weight_format={wf}, tile={tile}, block={block}, delay={delay}, g={g}, persistent={mode}")
    _compare(_make(n, wf, tile, block, delay, g), mode)


def test_spikes_with_the_flags_without_records():
    _say("case: 4000 neurons, no records, 20000 steps")
    out = []
    for mode in (N.PERSIST_AUTO, N.PERSIST_OFF):
        g = _make(4000, N.WF_CLASS, 60, 512, 0.0008, 0.1, records=0)(mode)
        g.run(20000)
        out.append((g.fire_counts(), g.state(N.F_V).view(np.uint32), g.info()["spikes"], g.info()["syn_events"]))
        g.close()
    (ca, va, na, ea), (cb, vb, nb, eb) = out
    assert na == nb > 200 and ea == eb
    assert np.array_equal(ca, cb) and np.array_equal(va, vb)


def test_default_block_keeps_two_launches_on_the_device():
    """256 tiles of 700: two persistent launches with workgroups of 512 fit on the device at
    once, one with wider ones.  Two simulators side by side run as one by itself."""
    _say("case: 179,200 neurons in 256 tiles, two simulators side by side")
    pops = [dict(num=179200, type=N.LIFB, v_min=0.0, v_max=0.019)]
    projs = [dict(src=0, tar=0, kind=N.CONN_FIXED_INDEGREE, k=20, w=2e-4, dmin=8e-4, dmax=8e-4, index=0, seed=3)]

    def sim():
        return N.Simulator.generated(pops, projs, W.lifb_consts(0.012), seed=3, propagation=N.PROP_TILED, tile_size=700)

    alone, a, b = sim(), sim(), sim()
    i = a.info()
    assert i["persistent"] and 129 <= i["tiles"] <= 256 and i["tile_size"] > 512 and i["block"] == 512
    alone.run(400)
    v = alone.state(N.F_V).view(np.uint32)
    for _ in range(4):
        a.run(100)
        b.run(100)
    assert alone.info()["spikes"] > 1000
    assert np.array_equal(a.state(N.F_V).view(np.uint32), v) and np.array_equal(b.state(N.F_V).view(np.uint32), v)
