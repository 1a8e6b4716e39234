"""What rests on the in-degree, for lists in any order.  Where 64 consecutive synapses have
one target and sign (target-major lists, fixed in-degree generators) the statistics count
them by wave."""
import numpy as np
import pytest

from mgbrain_amd import native as N
from mgbrain_amd import workloads as W

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
