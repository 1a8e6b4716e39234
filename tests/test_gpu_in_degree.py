"""What rests on the in-degree, for lists in any order.  Where 64 consecutive synapses have
one target and sign (target-major lists, fixed in-degree generators) the statistics count
them by wave."""
import numpy as np
import pytest

from mgbrain_amd import native as N
from mgbrain_amd import workloads as W
from tests import harness as H
from tests import netmodels as M
from tests.test_gpu_parity import _compare_run

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


def _two_targets(k, order, **opts):
    """k inputs of one sign on each of two neurons, from a pool that fires in every step."""
    tar = np.repeat([0, 1], k) if order == "target" else np.tile([0, 1], k)
    src = np.tile(np.arange(k), 2) if order == "target" else np.repeat(np.arange(k), 2)
    w, d = np.full(2 * k, np.float32(1e-7)), np.full(2 * k, np.float32(1e-3))
    return N.Simulator.from_arrays([N.POISSON] * k + [N.LIFB] * 2, [1.0] * k + [0.0] * 2, W.lifb_consts(), src, tar + k,
                                   w, d, **opts)


@pytest.mark.parametrize("order", ["target", "source"])
def test_class_words_up_to_65535_inputs(order):
    """A ring word counts 16 bits of each sign: more inputs of one sign are refused as CLASS
    words, and AUTO takes another format."""
    for k, ok in ((65535, True), (65536, False), (70000, False)):
        _say(f"case: {k} inputs of one sign, listed by {order}")
        s = _two_targets(k, order)
        assert (s.info()["weight_format"] == N.WF_CLASS) == ok
        s.close()
        if ok:
            _two_targets(k, order, weight_format=N.WF_CLASS).close()
        else:
            with pytest.raises(N.MGBError) as e:
                _two_targets(k, order, weight_format=N.WF_CLASS)
            assert e.value.status == N.ERR_UNSUPPORTED and "65535" in str(e.value)


@pytest.mark.parametrize("persist", [N.PERSIST_AUTO, N.PERSIST_REGIONS, N.PERSIST_OFF])
@pytest.mark.parametrize("k", [130, 600, 1500])
def test_many_arrivals_in_one_step_of_a_target_major_list(k, persist):
    """Half of a neuron's k inputs arrive in every step: the class sums of hundreds of
    arrivals, for synapses listed target by target (fixed in-degree), against the oracle."""
    _say(f"case: fixed in-degree {k} from a pool firing every other step, persistent={persist}")
    w, lo, hi = float(np.float32(3.2e-4 / k)), float(np.float32(1e-3)), float(np.float32(2e-3))
    net = M.Net([(2000, M.POISSON, 1), (300, M.LIFB, 0)],
                [dict(src=0, tar=1, wmin=w, wmax=w, dmin=lo, dmax=hi, kind=M.FIXK, k=k)], M.config2().lifconst)
    net.rates = [0.5, 0.0]
    syn = H.host_synapses(net, seed=3)
    n = _compare_run(net, syn, 600, seed=3, generated=True,
                     gpu_kw=dict(weight_format=N.WF_CLASS, propagation=N.PROP_TILED, persistent=persist))
    assert n > 600 * 900


@pytest.mark.parametrize("prop", [N.PROP_TILED, N.PROP_DIRECT])
def test_the_most_arrivals_of_a_class_word(prop):
    """65535 arrivals in every step, listed by target and by source: one sum of 65535 equal
    terms, the table's last entry."""
    _say(f"case: 65535 inputs, all arriving in every step, propagation={prop}")
    w, v, acc = np.float32(1e-7), np.float32(0.0), np.float32(0.0)
    for _ in range(65535):
        acc = np.float32(acc + w)
    out = []
    for order in ("target", "source"):
        s = _two_targets(65535, order, propagation=prop)
        s.run(14)
        out.append(s.state(N.F_V)[-2:])
        s.close()
    for _ in range(4):                     # steps 10 to 13: v + (i - 0.005 v), with the sum fused
        v = np.float32(v + np.float32(np.float64(acc) + np.float64(np.float32(-0.005)) * np.float64(v)))
    for o in out:
        assert np.array_equal(o.view(np.uint32), np.array([v, v]).view(np.uint32)), (o, v)
