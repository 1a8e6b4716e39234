"""The work that is timed: simulations as a program asks the library for them.

Every case builds (or is handed) a network, advances it and reads results back through
mgbrain_amd.native.Simulator, whose calls are the C ABI's one to one.  Launch shapes and
kernels are left to the library, as in a program that has not been tuned.

Families (the "family" of a case) and what they stand for:

  loop     closed-loop use: a small network advanced by a few steps, then read; the call's
           latency is the cost (a robot or an experiment in the loop)
  oneshot  a whole experiment: a synapse list in host memory becomes a simulator, is run
           for some milliseconds and read (parameter scans over small networks)
  brunel   a balanced network of equal weights per projection, one second at a time, with
           its raster read back (spikes recorded on the device)
  coba     a conductance-based network (Vogels-Abbott), with its weight formats
  hetero   current-based neurons with a weight of their own per synapse and delays from
           one step on, so that every step depends on the one before
  long     delays of up to several milliseconds, beyond the fused kernel's ring
  stdp     plastic excitatory synapses; the weights are part of the result
  batch    independent networks of a parameter sweep in one simulator
"""
from __future__ import annotations

import numpy as np

from mgbrain_amd import native as N
from mgbrain_amd import workloads as W

STEP = 1e-4            # 0.1 ms, the step of every workload here
FORMATS = {"auto": N.WF_AUTO, "f32": N.WF_F32, "bf16": N.WF_BF16, "fp8": N.WF_FP8}

# Spikes per neuron and second that each family's networks settle at, for the estimate of
# the work (measured on these networks; Poisson inputs fire at the case's own rate).
HZ = {"loop": 30.0, "oneshot": 28.0, "brunel": 28.0, "coba": 1.3, "hetero": 42.0, "long": 42.0, "stdp": 26.0,
      "batch": 60.0}


def listed():
    return [
        # the smallest call: one millisecond of a thousand neurons, read after each call
        dict(name="loop_1k", family="loop", n=1000, k=50, steps=10),
        # a network of a cortical column's order in the loop, two milliseconds a call
        dict(name="loop_5k", family="loop", n=5003, k=400, steps=20),
        # list to rates: 2500 neurons, a million synapses, 30 ms
        dict(name="oneshot_1m", family="oneshot", n=2500, k=400, steps=300),
        # the benchmark's smaller balanced network with its raster, one second
        dict(name="brunel_11k", family="brunel", n=10000, k=1000, steps=10000),
        # the benchmark's large balanced network (1e9 synapses) with its raster, one second
        dict(name="brunel_110k", family="brunel", n=100000, k=10000, steps=10000),
        # the conductance benchmark at full size, exact and in reduced weight formats
        dict(name="coba_80k", family="coba", n=80000, p=0.02, wf="auto", steps=10000),
        dict(name="coba_20k_bf16", family="coba", n=20000, p=0.02, wf="bf16", steps=5000),
        # weights from a distribution, delays from one step on
        dict(name="hetero_12k", family="hetero", n=10007, k=500, dmax=20, steps=5000),
        # slow axons: delays of 1 to 6 ms
        dict(name="long_12k", family="long", n=10007, k=500, dmax=60, steps=5000),
        # two seconds of plasticity on a fifth of the benchmark's network, weights read back
        dict(name="stdp_22k", family="stdp", n=20000, k=2000, wf="bf16", steps=20000),
        # a parameter sweep in one simulator, exact and with BF16 weights
        dict(name="batch_16", family="batch", nets=16, lo=2000, hi=20000, wf="auto", steps=2000),
        dict(name="batch_6_bf16", family="batch", nets=6, lo=2000, hi=8000, wf="bf16", steps=2000),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    family = rng.choice(sorted(HZ))
    if family == "loop":
        return dict(family=family, n=_log(rng, 300, 6000), k=_log(rng, 20, 500), steps=_log(rng, 5, 60))
    if family == "oneshot":
        return dict(family=family, n=_log(rng, 500, 6000), k=_log(rng, 50, 500), steps=_log(rng, 100, 300))
    if family == "brunel":
        n = _log(rng, 2000, 100000)
        return dict(family=family, n=n, k=_log(rng, 300, max(400, n // 10)), steps=_log(rng, 1000, 10000))
    if family == "coba":
        n = _log(rng, 4000, 80000)
        return dict(family=family, n=n, p=round(min(0.2, 1600.0 / n), 4), wf=rng.choice(["auto", "f32", "bf16", "fp8"]),
                    steps=_log(rng, 1000, 10000))
    if family in ("hetero", "long"):
        lo, hi = (12, 32) if family == "hetero" else (40, 100)
        return dict(family=family, n=_log(rng, 1000, 15000), k=_log(rng, 100, 500), dmax=rng.randint(lo, hi),
                    steps=_log(rng, 500, 5000))
    if family == "stdp":
        n = _log(rng, 4000, 30000)
        return dict(family=family, n=n, k=_log(rng, 300, 2000), wf=rng.choice(["f32", "bf16"]),
                    steps=_log(rng, 1000, 10000))
    return dict(family=family, nets=rng.randint(3, 16), lo=2000, hi=_log(rng, 4000, 20000),
                wf=rng.choice(["auto", "bf16"]), steps=_log(rng, 500, 2000))


# ---- networks -------------------------------------------------------------------------


def _sizes(case):
    """(Poisson, excitatory, inhibitory) neurons: a Poisson pool of a tenth beside n neurons
    of which a fifth are inhibitory."""
    n_e = case["n"] * 4 // 5
    return max(1, case["n"] // 10), n_e, case["n"] - n_e


def _inputs(case):
    """Synapses of one neuron from (the pool, excitatory, inhibitory neurons)."""
    k = case["k"]
    return max(1, k // 5), max(1, k * 16 // 25), max(1, k * 4 // 25)


RATE = 0.01           # the pool's probability of firing in a step (100 Hz)


def _weight(case):
    """Drive of 1.4 thresholds (20 mV, membrane time constant 20 ms) from the pool alone."""
    return 0.020 * 1.4 * 0.005 / (_inputs(case)[0] * RATE)


def _lists(case, seed):
    """A network as a program holds it before the call: per neuron types, rates and initial
    potentials, per synapse source, target, weight and delay (seconds), every neuron with a
    fixed number of inputs of each kind from random sources."""
    rng = np.random.default_rng([seed, case["n"], case["k"]])
    n_p, n_e, n_i = _sizes(case)
    n = n_p + n_e + n_i
    current = case["family"] in ("hetero", "long")
    types = np.full(n, N.LIF if current else N.LIFB, dtype=np.int32)
    types[:n_p] = N.POISSON
    rate = np.zeros(n, dtype=np.float32)
    rate[:n_p] = RATE
    v = np.zeros(n, dtype=np.float32)
    v[n_p:] = rng.random(n_e + n_i, dtype=np.float32) * np.float32(0.019)
    # current-based neurons: 8 mV-equivalent units over 240 inputs at 200 Hz of input
    j = 0.008 * 240.0 / case["k"] if current else _weight(case)
    if current:
        rate[:n_p] = 2 * RATE
    lo = 1 if case["family"] == "hetero" else 10
    hi = case.get("dmax", 20)
    srcs, tars, ws = [], [], []
    target = np.arange(n_p, n, dtype=np.int32)
    for first, count, k, w in zip((0, n_p, n_p + n_e), (n_p, n_e, n_i), _inputs(case), (j, j, -5.0 * j)):
        tar = np.repeat(target, k)
        srcs.append(rng.integers(first, first + count, tar.size, dtype=np.int32))
        tars.append(tar)
        ww = np.full(tar.size, w, dtype=np.float32)
        if current:           # a log-normal spread of the weights
            ww *= np.exp(np.float32(0.5) * rng.standard_normal(tar.size, dtype=np.float32) - np.float32(0.125))
        ws.append(ww)
    src, tar, w = np.concatenate(srcs), np.concatenate(tars), np.concatenate(ws)
    delay = rng.integers(lo, hi + 1, src.size, dtype=np.int32).astype(np.float32) * np.float32(STEP)
    return dict(types=types, rate=rate, v=v, src=src, tar=tar, w=w, delay=delay)


def _lif_const():
    return W.gen_life_const(0.0, 0.0, 0.010, 0.25, 0.020, 0.002, 0.005, 0.005, 0.020, 0.0)


def _from_lists(case, net, seed, **opts):
    const = _lif_const() if case["family"] in ("hetero", "long") else W.lifb_consts()
    return N.Simulator.from_arrays(net["types"], net["rate"], const, net["src"], net["tar"], net["w"], net["delay"],
                                   step=STEP, v_init=net["v"], seed=seed, **opts)


def _balanced(case, seed):
    """The balanced network in generator form (delays of 1 to 2 ms; a fixed number of inputs
    of each kind), which the library expands on the device."""
    n_p, n_e, n_i = _sizes(case)
    j = float(np.float32(_weight(case)))
    g = float(np.float32(-5.0 * _weight(case)))
    lo, hi = float(np.float32(0.001)), float(np.float32(0.002))
    pops = [dict(num=n_p, type=N.POISSON, rate=RATE), dict(num=n_e, type=N.LIFB, v_min=0.0, v_max=0.019),
            dict(num=n_i, type=N.LIFB, v_min=0.0, v_max=0.019)]
    projs = []
    for tar in (1, 2):
        for src, k, w in zip((0, 1, 2), _inputs(case), (j, j, g)):
            projs.append(dict(src=src, tar=tar, kind=N.CONN_FIXED_INDEGREE, k=k, w=w, dmin=lo, dmax=hi,
                              index=len(projs), seed=seed,
                              plastic=1 if case["family"] == "stdp" and src == 1 and tar == 1 else 0))
    return pops, projs


def _sweep(case, seed):
    """Networks of a sweep over inhibition and input rate, their sizes log-spaced."""
    m = case["nets"]
    out = []
    for b in range(m):
        n = int(round(case["lo"] * (case["hi"] / case["lo"]) ** (b / max(1, m - 1))))
        out.append(W.brunel_sweep_net(n, W.SWEEP_G[b % 4], W.SWEEP_NU_HZ[(b // 4) % 4], 1000 * seed + b))
    return out


def _spikes_expected(case):
    return (case["n"] * HZ[case["family"]] * STEP + _sizes(case)[0] * RATE) * case["steps"]


SETTLE = {"loop": 200, "brunel": 2000, "coba": 1000, "hetero": 1000, "long": 1000, "stdp": 1000, "batch": 500}


def prepare(case, seed):
    family = case["family"]
    if family == "oneshot":
        return dict(case=case, seed=seed, net=_lists(case, seed))
    state = dict(case=case)
    wf = FORMATS[case.get("wf", "auto")]
    if family in ("loop", "hetero", "long"):
        sim = _from_lists(case, _lists(case, seed), seed)
    elif family == "brunel":
        cap = int(2 * _spikes_expected(case)) + 20000
        pops, projs = _balanced(case, seed)
        sim = N.Simulator.generated(pops, projs, W.lifb_consts(), seed=seed, record_capacity=cap)
        state["steps"], state["ids"] = np.zeros(cap, dtype=np.int32), np.zeros(cap, dtype=np.int32)
    elif family == "coba":
        pops, projs, _, _ = W.vogels_abbott(scale=case["n"] / 80000.0, p=case["p"], seed=seed)
        if case["n"] != 80000:        # the conductances keep the drive of 1600 inputs
            by = 1600.0 / (case["n"] * case["p"])
            for q in projs:
                q["w"] = float(np.float32(q["w"] * by))
        sim = N.Simulator.generated(pops, projs, W.life_const1(), seed=seed, weight_format=wf)
    elif family == "stdp":
        pops, projs = _balanced(case, seed)
        sim = N.Simulator.generated(pops, projs, W.lifb_consts(), seed=seed, weight_format=wf, stdp=True,
                                    stdpconst=W.stdp_consts(_weight(case)))
    else:
        sim = N.Simulator.batch_generated(_sweep(case, seed), weight_format=wf)
    # past the transient of the initial potentials
    sim.run(SETTLE[family])
    sim.sync()
    if family == "brunel":
        sim.clear_spikes()
    state["sim"] = sim
    return state


def run(state):
    case = state["case"]
    if case["family"] == "oneshot":
        sim = _from_lists(case, state["net"], state["seed"])
        sim.run(case["steps"])
        out = dict(counts=sim.fire_counts(), V=sim.state(N.F_V))
        sim.close()
        return out
    sim = state["sim"]
    sim.run(case["steps"])
    out = dict(counts=sim.fire_counts(), V=sim.state(N.F_V))
    if case["family"] == "brunel":
        steps, ids = sim.spikes()
        sim.clear_spikes()
        # a raster of fixed size, as a program's own buffer holds it: -1 past its end
        a, b = state["steps"], state["ids"]
        a[:len(steps)], a[len(steps):] = steps, -1
        b[:len(ids)], b[len(ids):] = ids, -1
        out.update(steps=a, ids=b)
    elif case["family"] == "stdp":
        out["weights"] = sim.weights()
    elif case["family"] == "coba":
        out.update(g_exc=sim.state(N.F_IEXC), g_inh=sim.state(N.F_IINH))
    return out


def work(case):
    """Bytes: each neuron's state in and out once, the result, and two bytes of target and delay
    and the weight (none where all of a projection share it) of every synapse that carries a spike,
    from the rates in HZ; an experiment from a list reads the list once.  Operations: five per
    neuron and step and one per synapse that carries a spike."""
    family, steps = case["family"], case["steps"]
    seconds = steps * STEP
    if family == "batch":
        sizes = [sum(p["num"] for p in net["pops"]) for net in _sweep(case, 0)]
        n = float(sum(sizes))
        events = sum(m * min(0.1 * m, 5000.0) * HZ["batch"] * seconds for m in sizes)
    elif family == "coba":
        n = float(case["n"])
        events = n * n * case["p"] * HZ["coba"] * seconds
    else:
        ks = _inputs(case)
        n = float(sum(_sizes(case)))
        pool = (2 if family in ("hetero", "long") else 1) * RATE / STEP
        events = case["n"] * (ks[0] * pool + (ks[1] + ks[2]) * HZ[family]) * seconds
    word = {"hetero": 6.0, "long": 6.0, "stdp": 8.0}.get(family, 2.0)
    if family in ("coba", "batch"):
        word += {"auto": 0.0, "f32": 4.0, "bf16": 2.0, "fp8": 1.0}[case["wf"]]
    total = n * 40.0 + events * word
    if family == "oneshot":
        total += 16.0 * case["n"] * case["k"]
    if family == "stdp":
        total += 8.0 * case["n"] * case["k"]
    return dict(bytes=total, flops=5.0 * n * steps + events)


# ---- what the small networks give in 64 bits ---------------------------------------------


def _philox(c0, c1, tag, k0, k1):
    """Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11) of the counters (c0[i], c1, 0, tag)."""
    m32 = np.uint64(0xFFFFFFFF)
    x0 = c0.astype(np.uint64)
    x1, x2, x3 = (np.full_like(x0, c) for c in (c1, 0, tag))
    for r in range(10):
        a, b = np.uint64((k0 + r * 0x9E3779B9) & 0xFFFFFFFF), np.uint64((k1 + r * 0xBB67AE85) & 0xFFFFFFFF)
        p, q = np.uint64(0xD2511F53) * x0, np.uint64(0xCD9E8D57) * x2
        x0, x1, x2, x3 = (q >> np.uint64(32)) ^ x1 ^ a, q & m32, (p >> np.uint64(32)) ^ x3 ^ b, p & m32
    return x0, x1, x2, x3


def exact(case, seed):
    """The small networks step by step in 64 bits.  The others run until rounding has decided
    single spikes, after which no two precisions agree."""
    if case["family"] not in ("loop", "oneshot"):
        return None
    net = _lists(case, seed)
    n = len(net["types"])
    n_p = _sizes(case)[0]
    order = np.argsort(net["src"], kind="stable")
    ptr = np.searchsorted(net["src"][order], np.arange(n + 1))
    tar, w = net["tar"][order], net["w"][order].astype(np.float64)
    lag = np.rint(net["delay"][order] / np.float32(STEP)).astype(np.int64)
    d = int(lag.max()) + 1
    ring = np.zeros((d, n))
    v, refr, counts = net["v"].astype(np.float64), np.zeros(n, dtype=np.int64), np.zeros(n, dtype=np.int32)
    live = np.arange(n) >= n_p
    rate = net["rate"][:n_p]
    ids = np.arange(n_p)
    for s in range(case["steps"] + SETTLE.get(case["family"], 0)):
        u = _philox(ids, s >> 2, 0x504F4953, seed & 0xFFFFFFFF, seed >> 32)[s & 3]
        u = ((u >> np.uint64(8)) + np.uint64(1)).astype(np.float64) * 2.0 ** -24
        arrived = ring[s % d].copy()
        ring[s % d] = 0.0
        resting = live & (refr > 0)
        fired = live & ~resting & (v >= float(np.float32(0.020)))
        move = live & ~resting & ~fired
        v[move] += arrived[move] - float(np.float32(0.005)) * v[move]
        v[fired] = float(np.float32(0.010))
        refr[resting] -= 1
        refr[fired] = 19              # 2 ms less the step of the spike
        fired[:n_p] = rate > u
        counts[fired] += 1
        for i in np.flatnonzero(fired):
            k = slice(ptr[i], ptr[i + 1])
            np.add.at(ring, ((s + lag[k]) % d, tar[k]), w[k])
    return dict(counts=None, V=v)
