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


def _driven(k, w, d=1e-3, n=300, seed=3, plastic=0, g=None):
    """n LIFB neurons with k inputs of weight w each (fixed in-degree: listed target by
    target) from a pool that fires in every step, and with g as many of weight g."""
    pops = [dict(num=700, type=N.POISSON, rate=1.0), dict(num=n, type=N.LIFB, v_min=0.0, v_max=0.0)]
    projs = [dict(src=0, tar=1, kind=N.CONN_FIXED_INDEGREE, k=k, w=x, dmin=d, dmax=d, index=j, seed=seed, plastic=plastic)
             for j, x in enumerate((w,) if g is None else (w, g))]
    return dict(pops=pops, projs=projs, lifconst=W.lifb_consts(), seed=seed)


def _v_after(total, steps):
    v = 0.0
    for _ in range(steps):
        v += total - 0.005 * v
    return v


FORMATS = [N.WF_F32, N.WF_BF16, N.WF_FP8]


@pytest.mark.parametrize("prop", [N.PROP_TILED, N.PROP_DIRECT])
@pytest.mark.parametrize("wf", FORMATS)
@pytest.mark.parametrize("k", [63, 130, 1000, 6400])
def test_all_inputs_of_a_step_fit_the_fixed_point_sum(k, wf, prop):
    """Every input of a neuron arrives in every step.  The sum's error is at most half a
    fixed-point unit an input; the potential rounds once a step (2^-24 relative, 4 steps)."""
    w = float(np.float32(1e-3 / k))
    _say(f"case: {k} inputs arriving in every step, weight_format={wf}, propagation={prop}")
    s = N.Simulator.generated(**_driven(k, w), weight_format=wf, propagation=prop)
    scale = s.info()["fix_scale_exc"]
    assert k * round(w * scale) <= 2**31 - 1
    s.run(14)                                     # arrivals in steps 10 to 13
    want = _v_after(k * w, 4)
    tol = 4 * (0.5 * k / scale + 4 * 2.0**-24 * want)
    assert np.abs(s.state(N.F_V)[700:].astype(np.float64) - want).max() <= tol
    blob = s.checkpoint()                         # the pending inputs with the scale they have
    s.run(3)
    t = N.Simulator.generated(**_driven(k, w), weight_format=wf, propagation=prop)
    t.restore(blob)
    t.run(3)
    assert np.array_equal(s.state(N.F_V), t.state(N.F_V))
    s.close()
    t.close()


@pytest.mark.parametrize("wf", FORMATS)
def test_sums_of_a_batch_and_of_both_signs(wf):
    """Each network of a batch has its own scale; excitatory and inhibitory inputs of a
    neuron have sums of their own until it reads them."""
    _say(f"case: batch of networks of 100, 3000 and 640 + 640 inputs, weight_format={wf}")
    nets = [_driven(100, float(np.float32(1e-5))), _driven(3000, float(np.float32(4e-7)), seed=4),
            _driven(640, float(np.float32(3e-6)), seed=5, g=float(np.float32(-1.5e-6)))]
    want = [_v_after(x, 4) for x in (1e-3, 1.2e-3, 0.96e-3)]
    for prop in (N.PROP_TILED, N.PROP_DIRECT):
        s = N.Simulator.batch_generated(nets, weight_format=wf, propagation=prop)
        s.run(14)
        v = s.state(N.F_V).astype(np.float64)
        for b, x in enumerate(want):
            # (the codes of the third network's weights: 2^-9 for BF16, 2^-4 for FP8)
            rel = {N.WF_F32: 1e-5, N.WF_BF16: 2.0**-8, N.WF_FP8: 2.0**-3}[wf] if b == 2 else 1e-5
            assert np.abs(v[1000 * b + 700:1000 * (b + 1)] - x).max() <= 4 * rel * x, (prop, b)
        s.close()


@pytest.mark.parametrize("prop,wf", [(N.PROP_TILED, N.WF_F32), (N.PROP_TILED, N.WF_BF16), (N.PROP_DIRECT, N.WF_F32)])
def test_plastic_inputs_at_their_largest(prop, wf):
    """Plastic weights count with the largest value that plasticity can give them."""
    w = 1e-6
    sc = np.array(W.stdp_consts(w), dtype=np.float32)
    s = N.Simulator.generated(**_driven(1000, w, plastic=1), weight_format=wf, propagation=prop, stdp=True, stdpconst=sc)
    top = max(abs(float(sc[4])), abs(float(sc[5])), w)
    assert 1000 * round(top * s.info()["fix_scale_exc"]) <= 2**31 - 1
    s.close()


def test_scales_that_held_stay():
    """Where no sum can leave int32 the scale is the one of in-degree * max |w|, for lists in
    source order (every synapse counted) as before."""
    rng = np.random.default_rng(2)
    n, m = 500, 40000
    src, tar = np.sort(rng.integers(0, n, m)), rng.integers(0, n, m)
    w = rng.choice(np.float32([1e-5, 2e-5, -3e-5]), m)
    s = N.Simulator.from_arrays([N.LIFB] * n, [0.0] * n, W.lifb_consts(), src, tar, w, np.full(m, np.float32(1e-3)),
                                weight_format=N.WF_F32)
    deg = np.bincount(tar, minlength=n).max()
    assert s.info()["fix_scale_exc"] == 2.0**np.floor(np.log2(2147483520.0 / (deg * float(np.float32(3e-5)))))
    s.close()


@pytest.mark.parametrize("wf", [N.WF_F32, N.WF_BF16])
def test_a_volley_of_plastic_inputs(wf):
    """All inputs plastic, delays of 1 to 2 ms in 11 steps: what arrives at once when every
    source fires in one step fits, at the largest weights, for every target and delay."""
    w, k, n = 1e-6, 640, 300
    net = _driven(k, w, n=n, plastic=1)
    net["projs"][0]["dmax"] = 2e-3
    sc = np.array(W.stdp_consts(w), dtype=np.float32)
    s = N.Simulator.generated(**net, weight_format=wf, propagation=N.PROP_TILED, stdp=True, stdpconst=sc)
    _, col, dl, _ = s.csr()
    most = np.bincount((col.astype(np.int64) - 700) * 32 + dl, minlength=32 * n).max()
    assert 60 < most < 150
    assert most * round(float(sc[4]) * s.info()["fix_scale_exc"]) <= 2**31 - 1
    s.close()


@pytest.mark.parametrize("prop", [N.PROP_TILED, N.PROP_DIRECT])
def test_checkpoint_from_before_the_scale_was_lowered(prop):
    """A checkpoint whose pending inputs are in the units of in_bal * max |w| (in_bal: 10 for
    the 10 waves of 640 synapses) loads, its ring words brought to the units of now."""
    k, w = 640, float(np.float32(1.7e-6))
    net = _driven(k, w)
    net["pops"][0]["rate"] = 0.002                             # few enough for the old units
    make = lambda: N.Simulator.generated(**net, weight_format=N.WF_F32, propagation=prop)
    a, b, c = make(), make(), make()
    drop = int(np.floor(np.log2(2147483520.0 / (10 * w)))) - int(np.log2(a.info()["fix_scale_exc"]))
    _say(f"case: propagation={prop}, scale lowered by {drop} bits")
    assert drop >= 5
    a.run(133)
    blob = np.frombuffer(bytes(a.checkpoint()), np.uint8).copy()
    head = blob[8:60].view(np.int32)
    n, npad, D, window, tiled, G = (int(head[i]) for i in (1, 2, 3, 4, 5, 8))
    assert n == 1000 and tiled == (prop == N.PROP_TILED)
    at = 96 + 24 * npad + 72 + 4 * (3 if tiled else 2) * npad * window
    if tiled:
        slab = (D * int(head[7]) + 3) // 4 * 4                  # (LIFB neurons: one ring)
        words = G * slab
        h = 1469598103934665603
        for v in a.tiles():
            h = (h ^ int(v)) * 1099511628211 % 2**64
    else:
        words, h = 2 * D * npad, 0
    ring = blob[at:at + 4 * words].view(np.int32)
    assert np.count_nonzero(ring) > 1000 and np.abs(ring.astype(np.int64)).max() < 2**31 >> drop
    ring <<= drop
    old = blob[88:96].view(np.uint64)
    assert int(old[0]) != h
    old[0] = h
    b.restore(blob.tobytes())
    with pytest.raises(N.MGBError):                             # (neither tiling)
        old[0] = h ^ 1
        c.restore(blob.tobytes())
    a.run(200)
    b.run(200)
    assert a.state(N.F_V)[700:].min() > 1e-4
    assert np.array_equal(a.state(N.F_V).view(np.uint32), b.state(N.F_V).view(np.uint32))
    assert np.array_equal(a.fire_counts(), b.fire_counts())
    for s in (a, b, c):
        s.close()


@pytest.mark.parametrize("prop", [N.PROP_TILED, N.PROP_DIRECT])
def test_fp8_scales_whose_codes_round_up(prop):
    """A caller's FP8 scale of w / 0.00110: the code is 2^-9, 1.78 times the weight.  The scale
    of in-degree * max |w| holds 1.06 times it; w is such that little is left of int32."""
    _say(f"case: 1000 inputs in every step, codes above the weights, propagation={prop}")
    k, d = 1000, np.float32(1e-3)
    w = np.float32(0.98 * 2.0**31 / 1.0625 / k / 2.0**40)
    scale = np.float32(w / np.float32(0.0011))
    src, tar = np.repeat(np.arange(k), 2), np.tile([k, k + 1], k)       # (in source order)
    s = N.Simulator.from_arrays([N.POISSON] * k + [N.LIFB] * 2, [1.0] * k + [0.0] * 2, W.lifb_consts(), src, tar,
                                np.full(2 * k, w), np.full(2 * k, d), weight_format=N.WF_FP8, propagation=prop,
                                fp8_scale=np.full(k + 2, scale))
    code = float(np.float32(2.0**-9) * scale)
    assert np.all(s.weights() == np.float32(code)) and code > 1.7 * float(w)
    at = s.info()["fix_scale_exc"]
    assert at == 2.0**39 and k * round(code * at) <= 2**31 - 1
    s.run(14)
    want = _v_after(k * code, 4)
    assert np.abs(s.state(N.F_V)[k:] - want).max() <= 4 * (0.5 * k / at + 4 * 2.0**-24 * want)
    s.close()
