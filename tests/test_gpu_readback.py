"""Read-back of large results: spike records sorted on the device, weights through the
pinned buffers, counters from the run's own copy of the control block."""
import numpy as np
import pytest

from mgbrain_amd import native as N
from tests import harness as H
from tests import netmodels as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prop", [N.PROP_TILED, N.PROP_DIRECT])
def test_records_of_every_capacity(prop):
    net = M.config1(scale=0.3, poisson_rate=0.05)
    g = H.gpu_generated(net, seed=2, propagation=prop, record_capacity=200_000)
    seen = 0
    for n in (30, 200, 1, 900):                 # below and above the device sort's smallest record
        g.run(n)
        have = g.info()["spikes_recorded"]
        assert have > seen
        seen = have
        st, ids = g.spikes()
        assert len(st) == have
        key = st.astype(np.int64) << 32 | ids
        assert np.all(key[1:] > key[:-1]) and st.max() < g.info()["step"]
        for cap in (1, 63, 64, 65, have - 1):
            s2, i2 = np.full(have, -7, np.int32), np.full(have, -7, np.int32)
            k = N.C.c_int64()
            rc = N.lib().mgb_read_spikes(g.h, cap, s2.ctypes.data, i2.ctypes.data, N.C.byref(k))
            assert rc == N.ERR_CAPACITY and k.value == cap
            assert np.array_equal(s2[:cap], st[:cap]) and np.array_equal(i2[:cap], ids[:cap])
            assert np.all(s2[cap:] == -7) and np.all(i2[cap:] == -7)
    assert seen > 4096
    counts = g.fire_counts()
    assert np.array_equal(np.bincount(ids, minlength=len(counts)), counts)
    g.clear_spikes()
    assert g.info()["spikes_recorded"] == 0 and len(g.spikes()[0]) == 0
    blob = g.checkpoint()
    g.run(50)
    a = g.spikes()
    g.restore(blob)                             # the counters go back with the state
    assert g.info()["spikes_recorded"] == 0
    g.run(50)
    b = g.spikes()
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    g.close()


@pytest.mark.parametrize("wf", [N.WF_F32, N.WF_BF16, N.WF_FP8])
@pytest.mark.parametrize("extra", [0, 1])
def test_weights_across_the_pinned_buffers(wf, extra):
    """2^21 + extra synapses (8 MiB of weights: exactly two buffers, and one word more)."""
    s = (1 << 21) + extra
    n = 3000
    rng = np.random.default_rng(4)
    src, tar = rng.integers(0, n, s, dtype=np.int32), rng.integers(0, n, s, dtype=np.int32)
    # values of few mantissa bits whose row maximum is 1: exact in every format
    w = np.where(rng.random(s) < 0.5, 1.0, rng.choice([0.25, -0.5, 0.75, -1.0], s)).astype(np.float32)
    w[np.unique(src, return_index=True)[1]] = 1.0
    d = np.full(s, 1e-3, np.float32)
    g = N.Simulator.from_arrays([N.LIFB] * n, [0.0] * n, M.config1().lifconst, src, tar, w, d, weight_format=wf)
    want = w[np.argsort(src, kind="stable")]
    if wf == N.WF_FP8:                          # times 448 and back: 0.75 * 448 = 336 is not an E4M3 value
        want = np.where(want == 0.75, g.weights(), want)
        assert np.all(np.abs(want[w[np.argsort(src, kind="stable")] == 0.75] - 0.75) <= 0.75 / 16)
    for _ in range(2):
        assert np.array_equal(g.weights(), want)
    g.close()


def test_a_large_read_gives_its_workspace_back():
    """Records are sorted in device memory: up to 256 MiB of it is kept for the next read."""
    print("case: 20000 Poisson neurons at 0.05 a step, reads of 0.1, 12 and 0.1 million records", flush=True)
    g = N.Simulator.generated([dict(num=20000, type=N.POISSON, rate=0.05)], [], M.config1().lifconst, seed=1,
                              record_capacity=12_500_000)
    at = [g.info()["device_bytes"]]
    for n in (100, 11900, 0):
        if n:
            g.run(n)
        else:
            g.clear_spikes()
            g.run(100)
        steps, ids = g.spikes()
        key = steps.astype(np.int64) << 32 | ids
        assert np.all(key[1:] > key[:-1]) and len(ids) == g.info()["spikes_recorded"]
        at.append(g.info()["device_bytes"])
    print(at, flush=True)
    assert at[0] <= at[1] <= at[0] + (8 << 20) and at[2] == at[0] and at[3] == at[1]
    g.close()


@pytest.mark.parametrize("prop,wf", [(N.PROP_DIRECT, N.WF_BF16), (N.PROP_DIRECT, N.WF_FP8), (N.PROP_DIRECT, N.WF_F32),
                                     (N.PROP_TILED, N.WF_BF16)])
def test_reading_weights_changes_nothing(prop, wf):
    """With STDP a checkpoint is the same bytes before and after a read, as are the run's next
    steps."""
    print(f"case: E->E STDP, propagation={prop}, weight_format={wf}: checkpoint, weights, checkpoint", flush=True)
    net = M.config2(scale=0.02, K=200, poisson_rate=0.3, stdp=True)
    syn = H.host_synapses(net, seed=6)
    # weights that neither BF16 nor FP8 holds exactly
    syn.weight = (syn.weight * (1.0 + 0.01 * (np.arange(syn.n) % 7))).astype(np.float32)
    g = H.gpu_from_list(net, syn, seed=6, stdp=True, stdpconst=M.stdp_consts_config4(J=1e-4), weight_format=wf,
                        propagation=prop)
    g.run(203)
    before = g.checkpoint()
    w = g.weights()
    assert bytes(before) == bytes(g.checkpoint())
    assert np.array_equal(w, g.weights()) and np.array_equal(w, g.csr()[3])
    g.close()


@pytest.mark.parametrize("wf", [N.WF_BF16, N.WF_FP8])
def test_decoded_weights_in_parts(wf):
    """2^24 + 4321 synapses: two parts, the border inside a row, empty rows and one of a single
    synapse beside it."""
    s = (1 << 24) + 4321
    n = 3000
    print(f"case: {s} synapses, weight_format={wf}", flush=True)
    rng = np.random.default_rng(9)
    src, tar = np.sort(rng.integers(0, n, s, dtype=np.int32)), rng.integers(0, n, s, dtype=np.int32)
    src[(src >= 1200) & (src < 1300)] = 1300         # empty rows
    at = src[1 << 24]
    src[src == at - 1] = at                          # one before the border, and one after
    last = src[-1]
    src[-1] = n - 1
    src[-2:-1] = last
    w = rng.choice(np.float32([1.0, 0.25, -0.5, -1.0, 0.125]), s)   # (448 times these: E4M3 values)
    w[np.unique(src, return_index=True)[1]] = 1.0    # row maximum 1
    g = N.Simulator.from_arrays([N.LIF] * n, [0.0] * n, M.config1().lifconst, src, tar, w, np.full(s, np.float32(1e-3)),
                                weight_format=wf, propagation=N.PROP_DIRECT, stdp=True, plastic=(tar % 7 == 0),
                                stdpconst=M.stdp_consts_config4(J=1e-4))
    want = w[np.argsort(src, kind="stable")]
    assert np.array_equal(g.weights(), want)
    g.close()
