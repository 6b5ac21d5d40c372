"""Performance cases: what programs built on brian_amd spend their time on.

Each case is one pass of such a program's loop through the public entry
points: a ``Network.run`` and the monitors read after it, a batched engine's
run and its results, one evaluation of a fitting loop, one gradient or one
training epoch of the learned proposal, one spike-train distance matrix.

``listed`` gives the cases, ``draw`` further ones of the same ranges;
``prepare`` builds what a program holds before the pass, ``run`` is the pass,
``work`` the bytes and operations it cannot do without, ``tolerance`` how far
a correct implementation's outputs may lie apart and ``exact`` the outputs in
64 bits from numpy alone.

A network's pass reads the whole raster and returns what a program makes of it
whatever its length: the spikes of every neuron (``spikes``) and of every step
(``rate``).  Networks whose deliveries are whole counts do not depend on the
order of the additions, so these and the state are compared exactly; networks
with weights of their own per synapse sum them by floating atomics in any order.
"""
from __future__ import annotations

import math

import numpy as np

import brian_amd as B
from brian_amd import _lib, batch
from brian_amd import workloads as W
from brian_amd.core import sp as sparse     # the matrices its connections take
from brian_amd.equations import Equations
from brian_amd.learned import MLP
from brian_amd.modelfitting import FitEngine, OUInput, spike_steps

ms, mV, nS = 1e-3, 1e-3, 1e-9
DT = 1e-4


# ------------------------------------------------------------------- cases
def listed():
    return [
        # examples/misc/CUBA.py as it is written: 4000 neurons, no delays,
        # the default FP64, run 20 ms at a time.  The smallest step there is.
        {"name": "cuba_4k_fp64", "kind": "cuba", "n": 4000, "indegree": 80, "delay": 0, "refractory": 0,
         "precision": 64, "steps": 200},
        # the reference's C++ benchmark network (32,000 neurons, 80 synapses
        # each, 5 ms refractoriness, no delays) on the FP32 path
        {"name": "cuba_32k_refractory_fp32", "kind": "cuba", "n": 32000, "indegree": 80, "delay": 0,
         "refractory": 5, "precision": 32, "steps": 1000},
        # the headline: 2^20 neurons, in-degree 80, 1 ms delays, 0.2 s, with
        # the raster and the state read back
        {"name": "cuba_1m_fp32", "kind": "cuba", "n": 1 << 20, "indegree": 80, "delay": 10, "refractory": 0,
         "precision": 32, "steps": 2000},
        # many independent networks of 500 to 20,000 neurons with delays of
        # their own per synapse, one persistent launch
        {"name": "uneven_256_fp32", "kind": "uneven", "nnet": 256, "precision": 32, "steps": 1000},
        # conductance-based Hodgkin-Huxley neurons, exponential Euler (the
        # reference's COBAHH), default FP64
        {"name": "cobahh_4k_fp64", "kind": "cobahh", "n": 4000, "precision": 64, "steps": 200},
        # examples/plasticity/STDP1.py: 1000 Poisson inputs onto one neuron
        {"name": "stdp_1000x1_fp64", "kind": "stdpnet", "nin": 1000, "nout": 1, "precision": 64, "steps": 1000},
        # Poisson inputs onto a layer through weights and delays of their own
        {"name": "poisson_layer_fp32", "kind": "layer", "nin": 4000, "n": 4000, "indegree": 80, "precision": 32,
         "steps": 500},
        # 1024 plastic neurons with 1000 inputs each, in one batch
        {"name": "stdp_batch_1024x1000_fp32", "kind": "stdpbatch", "ninst": 1024, "nin": 1000, "precision": 32,
         "steps": 10000},
        # one swarm evaluation of a fitting loop: new candidates in, the run
        # of all of them against their targets' input, the counts out
        {"name": "fit_512k_fp32", "kind": "fit", "ntarget": 256, "pop": 2000, "precision": 32, "steps": 10000},
        # forward, loss and backward of the learned proposal, host to host
        {"name": "mlp_grad_1024", "kind": "mlpgrad", "nin": 64, "nh": 256, "nu": 4, "rows": 1024},
        # one epoch of its training in mini-batches of 1024
        {"name": "mlp_train_65k", "kind": "mlptrain", "nin": 64, "nh": 256, "nu": 4, "rows": 65536, "batch": 1024},
        # the distance matrix of 500 filtered spike trains of 1 s
        {"name": "van_rossum_500", "kind": "distance", "n": 500, "t": 10000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cuba", "cuba", "uneven", "cobahh", "stdpnet", "layer", "stdpbatch", "fit", "mlpgrad",
                       "mlptrain", "distance"])
    prec = rng.choice([32, 32, 64])
    if kind == "cuba":
        return {"kind": kind, "n": _log(rng, 1000, 500000), "indegree": rng.choice([20, 57, 80]),
                "delay": rng.choice([0, 1, 3, 10, 20]), "refractory": rng.choice([0, 0, 5]), "precision": prec,
                "steps": _log(rng, 100, 1000)}
    if kind == "uneven":
        return {"kind": kind, "nnet": _log(rng, 8, 256), "precision": 32, "steps": _log(rng, 100, 1000)}
    if kind == "cobahh":
        return {"kind": kind, "n": _log(rng, 500, 5000), "precision": prec, "steps": _log(rng, 100, 300)}
    if kind == "stdpnet":
        return {"kind": kind, "nin": _log(rng, 100, 2000), "nout": _log(rng, 1, 64), "precision": prec,
                "steps": _log(rng, 100, 1000)}
    if kind == "layer":
        return {"kind": kind, "nin": _log(rng, 500, 5000), "n": _log(rng, 500, 5000),
                "indegree": rng.choice([31, 80]), "precision": prec, "steps": _log(rng, 100, 500)}
    if kind == "stdpbatch":
        return {"kind": kind, "ninst": _log(rng, 8, 1024), "nin": _log(rng, 100, 1024), "precision": prec,
                "steps": _log(rng, 500, 8000)}
    if kind == "fit":
        return {"kind": kind, "ntarget": _log(rng, 1, 256), "pop": _log(rng, 100, 2000), "precision": prec,
                "steps": _log(rng, 500, 8000)}
    if kind == "mlpgrad":
        return {"kind": kind, "nin": rng.choice([17, 40, 64, 90]), "nh": rng.choice([64, 128, 256]),
                "nu": rng.choice([2, 3, 4, 8]), "rows": 256 * rng.randint(1, 16)}
    if kind == "mlptrain":
        return {"kind": kind, "nin": rng.choice([17, 40, 64, 90]), "nh": rng.choice([64, 128, 256]),
                "nu": rng.choice([2, 3, 4, 8]), "rows": _log(rng, 4096, 60000), "batch": rng.choice([256, 512, 1024])}
    return {"kind": "distance", "n": _log(rng, 5, 500), "t": _log(rng, 100, 10000)}


# ------------------------------------------------------- networks: the parts
CUBA = {"taum": 20 * ms, "taue": 5 * ms, "taui": 10 * ms, "Vt": -50 * mV, "Vr": -60 * mV, "El": -49 * mV}
CUBA_EQS = """
dv/dt  = (ge+gi-(v-El))/taum : volt
dge/dt = -ge/taue : volt
dgi/dt = -gi/taui : volt
"""


def _weights_cuba(indegree):
    # the benchmark's weights at 80 synapses, kept at the same total drive
    return 1.62 * mV * 80 / indegree, -9 * mV * 80 / indegree


def _cuba_inputs(case, seed):
    """Initial potentials and, per target, its distinct presynaptic neurons."""
    rng = np.random.default_rng([seed, 1])
    n, k = case["n"], min(case["indegree"], case["n"])
    v0 = CUBA["Vr"] + rng.random(n) * (CUBA["Vt"] - CUBA["Vr"])
    return v0, _csr(rng, n, n, k)


def _csr(rng, nsrc, ntgt, k):
    """k distinct sources per target: rows by source, ascending targets."""
    pre = rng.integers(0, nsrc, size=(ntgt, k))
    key = np.unique(pre * ntgt + np.arange(ntgt)[:, None])   # repeats of a pair drop out
    rows = np.bincount(key // ntgt, minlength=nsrc)
    return np.concatenate([[0], np.cumsum(rows)]).astype(np.int64), (key % ntgt).astype(np.int32)


def _rows(csr, lo, hi):
    ptr, col = csr
    return ptr[lo:hi + 1] - ptr[lo], col[ptr[lo]:ptr[hi]]


def _prepare_cuba(case, seed):
    n, prec = case["n"], case["precision"]
    capacity = max(1 << 20, int(n * case["steps"] * DT * 60))
    if case["delay"] > 0 and not case["refractory"] and case["indegree"] == 80:
        # the large networks' builder: connectivity sampled on the device
        S0 = np.zeros((3, n))
        S0[0] = CUBA["Vr"] + np.random.default_rng([seed, 1]).random(n) * (CUBA["Vt"] - CUBA["Vr"])
        h, g, _, _ = batch.build_cuba_fixed_indegree(n, 80, seed=seed, delay_steps=case["delay"], precision=prec,
                                                     capacity=capacity, S0=S0)
        return {"h": h, "g": g}
    v0, csr = _cuba_inputs(case, seed)
    ne = int(0.8 * n)
    we, wi = _weights_cuba(case["indegree"])
    eqs = Equations(CUBA_EQS, **{k: CUBA[k] for k in ("taum", "taue", "taui", "El")})
    h = _lib.NetHandle(DT, prec)
    S0 = np.zeros((3, n))
    S0[0] = v0
    g = h.add_group(S0)
    h.set_linear(g, *eqs.linear_propagator(DT))
    h.set_threshold(g, 0, CUBA["Vt"])
    h.add_reset_op(g, 0, 0, CUBA["Vr"])
    if case["refractory"]:
        period = case["refractory"] * ms
        h.set_refractory(g, int(period / DT) + 1, period - 0.5 * DT)
    for lo, m, var, w in ((0, ne, 1, we), (ne, n - ne, 2, wi)):
        ptr, col = _rows(csr, lo, lo + m)
        h.add_connection(g, lo, m, g, 0, n, var, ptr, col, np.full(len(col), w), delay_steps=case["delay"])
    h.record(g, capacity)
    h.prepare()
    return {"h": h, "g": g}


def _facade_cuba(case, seed):
    """The example script's objects."""
    clock = B.Clock(dt=DT)
    v0, csr = _cuba_inputs(case, seed)
    n = case["n"]
    ne = int(0.8 * n)
    we, wi = _weights_cuba(case["indegree"])
    eqs = Equations(CUBA_EQS, **{k: CUBA[k] for k in ("taum", "taue", "taui", "El")})
    P = B.NeuronGroup(n, model=eqs, threshold=CUBA["Vt"], reset=CUBA["Vr"], clock=clock)
    P.v = v0
    Pe, Pi = P.subgroup(ne), P.subgroup(n - ne)
    Ce = B.Connection(Pe, P, "ge", weight=_matrix(_rows(csr, 0, ne), we, (ne, n)))
    Ci = B.Connection(Pi, P, "gi", weight=_matrix(_rows(csr, ne, n), wi, (n - ne, n)))
    M = B.SpikeMonitor(P)
    net = B.Network(P, Ce, Ci, M, precision=case["precision"])
    net.run(0 * ms)     # builds the device network, as the first run of a script does
    return {"net": net, "P": P, "M": M, "vars": ("v", "ge", "gi")}


def _matrix(csr, w, shape):
    ptr, col = csr
    return sparse.csr_matrix((np.broadcast_to(np.asarray(w, float), (len(col),)).copy(), col, ptr), shape=shape)


HH = {"area": 20000e-12, "VT": -63 * mV, "El": -60 * mV, "EK": -90 * mV, "ENa": 50 * mV, "taue": 5 * ms,
      "taui": 10 * ms, "Ee": 0.0, "Ei": -80 * mV}
HH.update(Cm=1e-6 * 1e4 * HH["area"], gl=5e-5 * 1e4 * HH["area"], g_na=100e-3 * 1e4 * HH["area"],
          g_kd=30e-3 * 1e4 * HH["area"])
HH_EQS = """
dv/dt = (gl*(El-v)+ge*(Ee-v)+gi*(Ei-v)-g_na*(m*m*m)*h*(v-ENa)-g_kd*(n*n*n*n)*(v-EK))/Cm : volt
dm/dt = alpham*(1-m)-betam*m : 1
dn/dt = alphan*(1-n)-betan*n : 1
dh/dt = alphah*(1-h)-betah*h : 1
dge/dt = -ge*(1./taue) : siemens
dgi/dt = -gi*(1./taui) : siemens
alpham = 0.32*(mV**-1)*(13*mV-v+VT)/(exp((13*mV-v+VT)/(4*mV))-1.)/ms : Hz
betam = 0.28*(mV**-1)*(v-VT-40*mV)/(exp((v-VT-40*mV)/(5*mV))-1)/ms : Hz
alphah = 0.128*exp((17*mV-v+VT)/(18*mV))/ms : Hz
betah = 4./(1+exp((40*mV-v+VT)/(5*mV)))/ms : Hz
alphan = 0.032*(mV**-1)*(15*mV-v+VT)/(exp((15*mV-v+VT)/(5*mV))-1.)/ms : Hz
betan = .5*exp((10*mV-v+VT)/(40*mV))/ms : Hz
"""


def _hh_inputs(case, seed):
    rng = np.random.default_rng([seed, 2])
    n = case["n"]
    v0 = HH["El"] + (rng.standard_normal(n) * 5 - 5) * mV
    ge0 = (rng.standard_normal(n) * 1.5 + 4).clip(0) * 10 * nS
    gi0 = (rng.standard_normal(n) * 12 + 20).clip(0) * 10 * nS
    return v0, ge0, gi0, _csr(rng, n, n, min(80, n))


def _prepare_cobahh(case, seed):
    clock = B.Clock(dt=DT)
    v0, ge0, gi0, csr = _hh_inputs(case, seed)
    n = case["n"]
    ne = int(0.8 * n)
    eqs = Equations(HH_EQS, **HH)
    P = B.NeuronGroup(n, model=eqs, threshold=B.EmpiricalThreshold(threshold=-20 * mV, refractory=3 * ms, clock=clock),
                      implicit=True, freeze=True, clock=clock)
    P.v, P.ge, P.gi = v0, ge0, gi0
    Pe, Pi = P.subgroup(ne), P.subgroup(n - ne)
    Ce = B.Connection(Pe, P, "ge", weight=_matrix(_rows(csr, 0, ne), 6 * nS, (ne, n)))
    Ci = B.Connection(Pi, P, "gi", weight=_matrix(_rows(csr, ne, n), 67 * nS, (n - ne, n)))
    M = B.SpikeMonitor(P)
    net = B.Network(P, Ce, Ci, M, precision=case["precision"])
    net.run(0 * ms)
    return {"net": net, "P": P, "M": M, "vars": ("v", "m", "n", "h", "ge", "gi")}


STDP = {"taum": 10 * ms, "taue": 5 * ms, "taupre": 20 * ms, "taupost": 20 * ms, "Ee": 0.0, "vt": -54 * mV,
        "vr": -60 * mV, "El": -74 * mV, "gmax": 0.01, "rate": 15.0}
STDP_EQS = """
dv/dt = (ge*(Ee-vr) + El - v)/taum : volt
dge/dt = -ge/taue : 1
"""


def _stdp_amplitudes():
    Ap = 0.01
    return Ap, -Ap * STDP["taupre"] / STDP["taupost"] * 1.05


def _stdpnet_weights(case, seed):
    # the example's weights at its 1000 inputs, the same drive at other counts
    rng = np.random.default_rng([seed, 3])
    return rng.random((case["nin"], case["nout"])) * _stdpnet_gmax(case)


def _stdpnet_gmax(case):
    return STDP["gmax"] * 1000.0 / case["nin"]


def _prepare_stdpnet(case, seed):
    clock = B.Clock(dt=DT)
    gmax = _stdpnet_gmax(case)
    G = B.PoissonGroup(case["nin"], rates=STDP["rate"], clock=clock, seed=seed & 0x7FFFFFFF)
    eqs = Equations(STDP_EQS, **{k: STDP[k] for k in ("Ee", "vr", "El", "taum", "taue")})
    P = B.NeuronGroup(case["nout"], model=eqs, threshold=STDP["vt"], reset=STDP["vr"], clock=clock)
    P.v = STDP["vr"]
    C = B.Connection(G, P, "ge", weight=_stdpnet_weights(case, seed), structure="dense")
    Ap, Am = _stdp_amplitudes()
    S = B.ExponentialSTDP(C, STDP["taupre"], STDP["taupost"], Ap, Am, wmax=gmax)
    M = B.SpikeMonitor(P)
    net = B.Network(G, P, C, S, M, precision=case["precision"])
    net.run(0 * ms)
    return {"net": net, "P": P, "M": M, "C": C, "vars": ("v", "ge")}


LAYER_RATE = 20.0


def _layer_inputs(case, seed):
    rng = np.random.default_rng([seed, 4])
    csr = _csr(rng, case["nin"], case["n"], min(case["indegree"], case["nin"]))
    nnz = len(csr[1])
    w = 1.5 * mV * 80 / case["indegree"] * (0.5 + rng.random(nnz))
    d = (0.5 + 4.4 * rng.random(nnz)) * ms
    v0 = CUBA["Vr"] + rng.random(case["n"]) * (CUBA["Vt"] - CUBA["Vr"])
    return csr, w, d, v0


def _prepare_layer(case, seed):
    clock = B.Clock(dt=DT)
    csr, w, d, v0 = _layer_inputs(case, seed)
    shape = (case["nin"], case["n"])
    G = B.PoissonGroup(case["nin"], rates=LAYER_RATE, clock=clock, seed=seed & 0x7FFFFFFF)
    eqs = Equations(CUBA_EQS, **{k: CUBA[k] for k in ("taum", "taue", "taui")}, El=-60 * mV)
    P = B.NeuronGroup(case["n"], model=eqs, threshold=CUBA["Vt"], reset=CUBA["Vr"], clock=clock)
    P.v = v0
    C = B.DelayConnection(G, P, "ge", max_delay=5 * ms)
    C.connect_from_sparse(_matrix(csr, w, shape), delay=_matrix(csr, d, shape))
    M = B.SpikeMonitor(P)
    net = B.Network(G, P, C, M, precision=case["precision"])
    net.run(0 * ms)
    return {"net": net, "P": P, "M": M, "vars": ("v", "ge")}


# ---------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "cuba":
        # a script's size goes through the Brian objects, larger ones through the handle
        facade = case["n"] <= 5000 and not case["refractory"] and not case["delay"]
        st.update(_facade_cuba(case, seed) if facade else _prepare_cuba(case, seed))
    elif kind == "uneven":
        # sizes at the quantiles of the log-uniform law between 500 and 20,000
        q = (np.arange(case["nnet"]) + 0.5) / case["nnet"]
        d = W.uneven_batch(case["nnet"], seed=seed & 0xFFFFFFF, sizes=np.rint(500 * 40.0 ** q))
        h, g, _, _ = batch.build_uneven(d, precision=case["precision"], tuning={"persist": 1},
                                        capacity=max(1 << 20, int(d["N"] * case["steps"] * DT * 60)))
        st.update(h=h, g=g, n=d["N"])
    elif kind == "cobahh":
        st.update(_prepare_cobahh(case, seed))
    elif kind == "stdpnet":
        st.update(_prepare_stdpnet(case, seed))
    elif kind == "layer":
        st.update(_prepare_layer(case, seed))
    elif kind == "stdpbatch":
        d = W.stdp_batch(case["ninst"], case["nin"], wseed=seed)
        scale = 1000.0 / case["nin"]
        st["h"] = _lib.StdpBatchHandle(case["precision"], DT, d["ninst"], d["nin"], d["A"], d["C"], d["S0"], 0,
                                       d["vt"], 0, d["vr"], 1, d["w0"] * scale, d["rate"], seed, d["decay_pre"],
                                       d["decay_post"], d["Ap"] * scale, d["Am"] * scale, 0.0, d["gmax"] * scale)
    elif kind == "fit":
        st.update(_prepare_fit(case, seed))
    elif kind in ("mlpgrad", "mlptrain"):
        rng = np.random.default_rng([seed, 6])
        nin, nu, rows = case["nin"], case["nu"], case["rows"]
        st["X"] = rng.standard_normal((rows, nin)).astype(np.float32)
        st["U"] = rng.random((rows, nu)).astype(np.float32)
        st["mlp"] = MLP(nin, case["nh"], nu, params=_mlp_params(case, seed))
        st["seed"] = seed & 0x7FFFFFFF
    else:
        st["X"] = _traces(case, seed)
    return st


def _traces(case, seed):
    """Spike trains at 5 to 50 Hz through an exponential filter of 10 ms."""
    rng = np.random.default_rng([seed, 7])
    n, t = case["n"], case["t"]
    spikes = rng.random((t, n)) < (5 + 45 * rng.random(n)) * DT
    a, x, out = math.exp(-DT / (10 * ms)), np.zeros(n), np.empty((t, n))
    for k in range(t):
        x = x * a + spikes[k]
        out[k] = x
    return np.ascontiguousarray(out.T)


def _prepare_fit(case, seed):
    rng = np.random.default_rng([seed, 5])
    nt, steps = case["ntarget"], case["steps"]
    trains = []
    for _ in range(nt):        # target trains at 20 to 80 Hz with a refractory gap
        rate = 20 + 60 * rng.random()
        isi = 30 + rng.exponential(1 / (rate * DT), size=int(steps * DT * 160) + 8)
        t = np.cumsum(isi)
        trains.append(t[t < steps].astype(np.int32))
    cand = np.repeat(np.arange(nt), case["pop"])
    m = len(cand)
    values = {k: W.log_uniform(rng, lo, hi, m) for k, (lo, hi) in W.FIT_BOUNDS.items()}
    refr = spike_steps(values.pop("refractory"), DT)
    eng = FitEngine(Equations(W.FIT_EQS, tau_t=W.FIT_TAU_T), W.FIT_THRESHOLD, W.FIT_RESET,
                    OUInput(nt, steps, 0.5e-9, 0.2e-9, 5e-3, seed=seed), trains, cand, DT, 40,
                    precision=case["precision"])
    return {"eng": eng, "values": values, "refr": refr}


def _mlp_params(case, seed):
    rng = np.random.default_rng([seed, 8])
    nin, nh, nu = case["nin"], case["nh"], case["nu"]
    w3 = np.zeros((nh, 32))
    w3[:, :2 * nu] = rng.standard_normal((nh, 2 * nu)) * 0.3 / math.sqrt(nh)
    b3 = np.zeros(32)
    b3[:nu] = 0.5
    parts = [rng.standard_normal((nin, nh)) * math.sqrt(2 / nin), 0.1 * rng.standard_normal(nh),
             rng.standard_normal((nh, nh)) * math.sqrt(2 / nh), 0.1 * rng.standard_normal(nh), w3, b3]
    return np.concatenate([p.ravel() for p in parts]).astype(np.float32)


# -------------------------------------------------------------------- run
def _counts(st, idx, steps, n):
    """Spikes per neuron and per step of the pass just run (the values of a
    SpikeCounter and a PopulationRateMonitor)."""
    first = st.get("done", 0)
    st["done"] = first + st["case"]["steps"]
    return {"spikes": np.bincount(idx, minlength=n),
            "rate": np.bincount(steps - first, minlength=st["case"]["steps"])}


def run(st):
    case = st["case"]
    kind = case["kind"]
    if "net" in st:
        net, M, P = st["net"], st["M"], st["P"]
        net.run(case["steps"] * DT)
        i, t = M.it
        M.reinit()
        out = {v: P.state_(v) for v in st["vars"]}
        out.update(_counts(st, i, np.rint(t / DT).astype(np.int64), len(P)))
        if "C" in st:
            out["w"] = np.asarray(st["C"].W.todense())
        return out
    if kind in ("cuba", "uneven"):
        h, g = st["h"], st["g"]
        h.run(case["steps"])
        steps, idx = h.get_spikes(g)
        h.clear_spikes(g)
        n = st.get("n", case.get("n"))
        return {"v": h.get_state(g, 0, n), "ge": h.get_state(g, 1, n), "gi": h.get_state(g, 2, n),
                **_counts(st, idx, steps, n)}
    if kind == "stdpbatch":
        h = st["h"]
        h.run(case["steps"])
        return {"w": h.weights(), "a_pre": h.a_pre(), "a_post": h.a_post(), "state": h.state()}
    if kind == "fit":
        eng = st["eng"]
        eng.set_candidates(st["values"], init_state={"V": 0.0, "Vt": 0.0}, refractory_steps=st["refr"])
        eng.run()
        nc, ns = eng.results()
        return {"coincidences": nc, "spikes": ns}
    if kind == "mlpgrad":
        loss, g = st["mlp"].grad(st["X"], st["U"])
        return {"loss": loss, "grad": g}
    if kind == "mlptrain":
        loss = st["mlp"].train(st["X"], st["U"], epochs=1, batch=case["batch"], lr=1e-3, seed=st["seed"])
        return {"loss": loss, "params": st["mlp"].params()}
    return {"d": _lib.pairwise_sq_distance(st["X"], DT / (10 * ms))}


# ------------------------------------------------------------------- work
def work(case):
    kind = case["kind"]
    s = case.get("precision", 64) // 8
    if kind in ("cuba", "cobahh"):
        # state in and out, the raster, and per spike (about 6 Hz, 20 Hz for
        # the conductance-based network) its row's columns; 12 operations of
        # the linear update per neuron and step, 300 of the nonlinear one
        n, steps = case["n"], case["steps"]
        spikes = n * steps * DT * (6 if kind == "cuba" else 20)
        k = case.get("indegree", 80)
        m, ops = (3, 12) if kind == "cuba" else (6, 300)
        return {"bytes": 2 * m * s * n + spikes * (16 + 4 * k), "flops": n * steps * ops + spikes * k}
    if kind == "uneven":
        n = case["nnet"] * 5286              # the mean of the log-uniform sizes
        spikes = n * case["steps"] * DT * 4.4
        events = spikes * 151                # 2 % of a spike's own network
        return {"bytes": 2 * 3 * s * n + spikes * 16 + events * 5, "flops": n * case["steps"] * 12 + events}
    if kind == "stdpnet":
        syn = case["nin"] * case["nout"]
        ev = case["steps"] * DT * (STDP["rate"] + 20) * syn
        return {"bytes": 2 * s * syn, "flops": ev * 4 + case["steps"] * (case["nin"] * 12 + case["nout"] * 14)}
    if kind == "layer":
        ev = case["nin"] * LAYER_RATE * case["steps"] * DT * case["n"] * case["indegree"] / case["nin"]
        return {"bytes": 2 * 3 * s * case["n"] + ev * (4 + 1 + s),
                "flops": ev + case["steps"] * (case["n"] * 12 + case["nin"] * 12)}
    if kind == "stdpbatch":
        syn = case["ninst"] * case["nin"]
        return {"bytes": 2 * (3 if s == 4 else 2) * s * syn, "flops": syn * case["steps"] * 10}
    if kind == "fit":
        m = case["ntarget"] * case["pop"]
        return {"bytes": m * (8 * 5 + 4 + 8) + case["ntarget"] * case["steps"] * s, "flops": m * case["steps"] * 20}
    if kind in ("mlpgrad", "mlptrain"):
        nin, nh, nu, rows = case["nin"], case["nh"], case["nu"], case["rows"]
        p = nin * nh + nh * nh + nh * 32 + 2 * nh + 32
        fl = 2 * rows * (2 * nin * nh + 3 * nh * nh + 3 * nh * 2 * nu)
        steps = 1 if kind == "mlpgrad" else max(1, rows // case["batch"])
        return {"bytes": 4 * rows * (nin + nu) + 4 * p * (2 if kind == "mlpgrad" else 6 * steps), "flops": fl}
    n, t = case["n"], case["t"]
    return {"bytes": 8 * (n * t + n * n), "flops": 1.5 * n * n * t}


def tolerance(case):
    kind = case["kind"]
    if kind in ("cuba", "uneven", "fit"):
        return "exact"
    if kind == "cobahh":
        # exp and division to the last place or so, over a few hundred steps of
        # a spiking (expanding) system
        return {"rel": 1e-10, "max": 1e-6, "differ": 0.0} if case["precision"] == 64 else \
            {"rel": 1e-3, "max": 0.2, "differ": 0.005}
    if kind in ("stdpnet", "layer"):
        # weights summed by atomics in any order
        return {"rel": 1e-12, "max": 1e-9, "differ": 0.0} if case["precision"] == 64 else \
            {"rel": 1e-2, "max": 0.8, "differ": 0.01}   # one spike a step apart moves a neuron by its reset
    if kind == "stdpbatch":
        return {"rel": 1e-12, "max": 1e-9} if case["precision"] == 64 else {"rel": 2e-3, "max": 0.5}
    if kind == "mlpgrad":
        return {"rel": 5e-3, "max": 0.2}        # BF16 operands: 1.4e-3 from the 64-bit gradient
    if kind == "mlptrain":
        # partial sums of the gradient in another order: 1.2e-3 to 5.8e-3 after an epoch
        return {"rel": 2e-2, "max": 0.4}
    return {"rel": 1e-13, "max": 1e-11}


# ------------------------------------------------------------------ exact
def exact(case, seed):
    kind = case["kind"]
    if kind == "cuba":
        # in 32 bits a spiking recurrent network leaves the 64-bit trajectory
        # within milliseconds; the device-sampled connectivity has no other source
        if case["precision"] == 32 or case["n"] * case["steps"] > 3e8 or (
                case["delay"] > 0 and not case["refractory"] and case["indegree"] == 80):
            return None
        S = _exact_cuba(case, seed)
        return {"v": S[0], "ge": S[1], "gi": S[2], "spikes": None, "rate": None}
    if kind == "cobahh":
        return _exact_cobahh(case, seed)
    if kind == "stdpnet":
        return _exact_stdpnet(case, seed) if case["nin"] * case["nout"] * case["steps"] <= 1e9 else None
    if kind == "layer":
        return _exact_layer(case, seed)
    if kind == "stdpbatch":
        return _exact_stdpbatch(case, seed) if case["ninst"] * case["nin"] * case["steps"] <= 2e8 else None
    if kind == "mlpgrad":
        return _exact_mlpgrad(case, seed)
    if kind == "distance":
        X = _traces(case, seed)
        D = np.zeros((len(X), len(X)))
        for i in range(len(X)):
            d = X[i] - X[i + 1:]
            D[i, i + 1:] = D[i + 1:, i] = (d * d).sum(axis=1) * (DT / (10 * ms))
        return {"d": D}
    # uneven: connectivity sampled on the device; fit: whole numbers;
    # mlptrain: the order of the shuffled batches is the library's own
    return None


def _propagator(rates, feeds, const):
    """One step of dv/dt = rates[0] (v_inf - v) + sum feeds[j] x_j, dx_j/dt =
    -rates[j] x_j in closed form: (A, C) with v_inf * rates[0] = const."""
    m = len(rates)
    e = np.exp(-DT * np.asarray(rates))
    A, C = np.diag(e), np.zeros(m)
    for j in range(1, m):
        A[0, j] = feeds[j] / (rates[0] - rates[j]) * (e[j] - e[0])
    C[0] = const / rates[0] * (1 - e[0])
    return A, C


def _cuba_propagator(El):
    r = [1 / CUBA["taum"], 1 / CUBA["taue"], 1 / CUBA["taui"]]
    return _propagator(r, [0, r[0], r[0]], El * r[0])


def _exact_cuba(case, seed):
    n, delay = case["n"], case["delay"]
    ne = int(0.8 * n)
    v0, (ptr, col) = _cuba_inputs(case, seed)
    we, wi = _weights_cuba(case["indegree"])
    A, C = _cuba_propagator(CUBA["El"])
    S = np.zeros((3, n))
    S[0] = v0
    last = np.full(n, -10 ** 9)
    period, gap = int(case["refractory"] * ms / DT) + 1, case["refractory"] * ms - 0.5 * DT
    spikes = {}
    for k in range(case["steps"]):
        S = A @ S + C[:, None]
        s = S[0] > CUBA["Vt"]
        if case["refractory"]:
            s &= (last < 0) | (last * DT + gap <= k * DT)
        last[s] = k
        spikes[k] = np.nonzero(s)[0]
        for i in spikes.pop(k - delay, ()):
            if i < ne:
                S[1, col[ptr[i]:ptr[i + 1]]] += we
            else:
                S[2, col[ptr[i]:ptr[i + 1]]] += wi
        S[0][(k - last < period) if case["refractory"] else s] = CUBA["Vr"]
    return S


def _hh_rhs(j, v, m, n, h, ge, gi):
    p = HH
    if j == 0:
        return (p["gl"] * (p["El"] - v) + ge * (p["Ee"] - v) + gi * (p["Ei"] - v)
                - p["g_na"] * (m * m * m) * h * (v - p["ENa"]) - p["g_kd"] * (n * n * n * n) * (v - p["EK"])) / p["Cm"]
    VT = p["VT"]
    if j == 1:
        a = 0.32 / mV * (13 * mV - v + VT) / (np.exp((13 * mV - v + VT) / (4 * mV)) - 1.) / ms
        b = 0.28 / mV * (v - VT - 40 * mV) / (np.exp((v - VT - 40 * mV) / (5 * mV)) - 1) / ms
        return a * (1 - m) - b * m
    if j == 2:
        a = 0.032 / mV * (15 * mV - v + VT) / (np.exp((15 * mV - v + VT) / (5 * mV)) - 1.) / ms
        b = .5 * np.exp((10 * mV - v + VT) / (40 * mV)) / ms
        return a * (1 - n) - b * n
    if j == 3:
        a = 0.128 * np.exp((17 * mV - v + VT) / (18 * mV)) / ms
        b = 4. / (1 + np.exp((40 * mV - v + VT) / (5 * mV))) / ms
        return a * (1 - h) - b * h
    return -ge / p["taue"] if j == 4 else -gi / p["taui"]


def _exact_cobahh(case, seed):
    n = case["n"]
    ne = int(0.8 * n)
    v0, ge0, gi0, (ptr, col) = _hh_inputs(case, seed)
    z = np.zeros(n)
    S = [v0, z, z.copy(), z.copy(), ge0, gi0]
    last, count = np.full(n, -10 ** 9), np.zeros(n, np.int64)
    for k in range(case["steps"]):
        new = []
        for j in range(6):
            b = _hh_rhs(j, *[z if q == j else S[q] for q in range(6)])
            a = _hh_rhs(j, *[z + 1 if q == j else S[q] for q in range(6)]) - b
            new.append((S[j] + b / a) * np.exp(a * DT) - b / a)
        S = new
        s = (S[0] > -20 * mV) & (k - last > 29)      # one less than 3 ms, a whole number of steps
        last[s] = k
        count += s
        for i in np.nonzero(s)[0]:
            if i < ne:
                S[4][col[ptr[i]:ptr[i + 1]]] += 6 * nS
            else:
                S[5][col[ptr[i]:ptr[i + 1]]] += 67 * nS
    return dict(zip(("v", "m", "n", "h", "ge", "gi"), S), spikes=None, rate=None)


def _mix(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


_GOLD = np.uint64(0x9E3779B97F4A7C15)


def _keys(seed, n):
    with np.errstate(over="ignore"):
        return _mix(np.uint64(seed) * _GOLD + np.arange(n, dtype=np.uint64))


def _poisson(keys, step, rate):
    """The documented counter stream of Poisson groups: the upper 32 bits
    below floor(rate dt 2^32)."""
    with np.errstate(over="ignore"):
        u = _mix(keys + np.uint64(step) * _GOLD) >> np.uint64(32)
    return u < np.uint64(math.floor(rate * DT * 2 ** 32))


def _stdp_propagator():
    r = [1 / STDP["taum"], 1 / STDP["taue"]]
    return _propagator(r, [0, (STDP["Ee"] - STDP["vr"]) * r[0]], STDP["El"] * r[0])


def _exact_stdpnet(case, seed):
    gmax, w = _stdpnet_gmax(case), _stdpnet_weights(case, seed)
    keys = _keys(seed & 0x7FFFFFFF, case["nin"])
    A, C = _stdp_propagator()
    Ap, Am = (a * gmax for a in _stdp_amplitudes())
    dp, dm = math.exp(-DT / STDP["taupre"]), math.exp(-DT / STDP["taupost"])
    S = np.zeros((2, case["nout"]))
    S[0] = STDP["vr"]
    apre, apost = np.zeros(case["nin"]), np.zeros(case["nout"])
    for k in range(case["steps"]):
        pre = np.nonzero(_poisson(keys, k, STDP["rate"]))[0]
        S = A @ S + C[:, None]
        post = S[0] > STDP["vt"]
        apre *= dp
        apost *= dm
        S[1] += w[pre].sum(axis=0)
        apre[pre] += Ap
        w[pre] = np.clip(w[pre] + apost, 0, gmax)
        apost[post] += Am
        w[:, post] = np.clip(w[:, post] + apre[:, None], 0, gmax)
        S[0][post] = STDP["vr"]
    return {"v": S[0], "ge": S[1], "w": w, "spikes": None, "rate": None}


def _exact_layer(case, seed):
    (ptr, col), w, d, v0 = _layer_inputs(case, seed)
    d = (1 / DT * d).astype(np.int64)
    keys = _keys(seed & 0x7FFFFFFF, case["nin"])
    A, C = _cuba_propagator(-60 * mV)
    S = np.zeros((3, case["n"]))
    S[0] = v0
    ring = np.zeros((64, case["n"]))
    for k in range(case["steps"]):
        S = A @ S + C[:, None]
        s = S[0] > CUBA["Vt"]
        for i in np.nonzero(_poisson(keys, k, LAYER_RATE))[0]:
            q = slice(ptr[i], ptr[i + 1])
            np.add.at(ring, ((k + d[q]) % 64, col[q]), w[q])
        S[1] += ring[k % 64]
        ring[k % 64] = 0
        S[0][s] = CUBA["Vr"]
    return {"v": S[0], "ge": S[1], "spikes": None, "rate": None}


def _exact_stdpbatch(case, seed):
    ninst, nin = case["ninst"], case["nin"]
    scale = 1000.0 / nin
    gmax = STDP["gmax"] * scale
    # the same weights and initial state as the workload's
    w = np.random.default_rng(seed).random((ninst, nin)) * STDP["gmax"] * scale
    A, C = _stdp_propagator()
    Ap, Am = (a * gmax for a in _stdp_amplitudes())
    dp, dm = math.exp(-DT / STDP["taupre"]), math.exp(-DT / STDP["taupost"])
    key = (_keys(seed, ninst * nin) >> np.uint64(32)).astype(np.uint32).reshape(ninst, nin)
    thr = np.uint64(math.floor(STDP["rate"] * DT * 2 ** 32))
    S = np.zeros((2, ninst))
    S[0] = STDP["vr"]
    apre, apost = np.zeros((ninst, nin)), np.zeros(ninst)
    for k in range(case["steps"]):
        h = key + np.uint32((k * 0x9E3779B9) & 0xFFFFFFFF)      # the documented 32-bit stream
        for shift, mul in ((16, 0x85EBCA6B), (13, 0xC2B2AE35)):
            h = (h ^ (h >> np.uint32(shift))) * np.uint32(mul)
        pre = (h ^ (h >> np.uint32(16))) < thr
        S = A @ S + C[:, None]
        post = S[0] > STDP["vt"]
        apre *= dp
        apost *= dm
        S[1] += (w * pre).sum(axis=1)
        apre[pre] += Ap
        w = np.where(pre, np.clip(w + apost[:, None], 0, gmax), w)
        apost[post] += Am
        w[post] = np.clip(w[post] + apre[post], 0, gmax)
        S[0][post] = STDP["vr"]
    return {"w": w, "a_pre": apre, "a_post": apost, "state": S.T.copy()}


def _exact_mlpgrad(case, seed):
    nin, nh, nu, rows = case["nin"], case["nh"], case["nu"], case["rows"]
    rng = np.random.default_rng([seed, 6])
    X = rng.standard_normal((rows, nin)).astype(np.float32).astype(np.float64)
    U = rng.random((rows, nu)).astype(np.float32).astype(np.float64)
    p, at, parts = _mlp_params(case, seed).astype(np.float64), 0, []
    for shape in ((nin, nh), (nh,), (nh, nh), (nh,), (nh, 32), (32,)):
        parts.append(p[at:at + math.prod(shape)].reshape(shape))
        at += math.prod(shape)
    W1, b1, W2, b2, W3, b3 = parts
    a1 = np.maximum(X @ W1 + b1, 0)
    a2 = np.maximum(a1 @ W2 + b2, 0)
    o = a2 @ W3 + b3
    mu, raw = o[:, :nu], o[:, nu:2 * nu]
    s = np.clip(raw, -7, 3)
    e, iv = U - mu, np.exp(-2 * s)
    dO = np.zeros_like(o)
    dO[:, :nu] = -e * iv / rows
    dO[:, nu:2 * nu] = np.where((raw > -7) & (raw < 3), 1 - e * e * iv, 0) / rows
    d2 = (dO @ W3.T) * (a2 > 0)
    d1 = (d2 @ W2.T) * (a1 > 0)
    g = [X.T @ d1, d1.sum(0), a1.T @ d2, d2.sum(0), a2.T @ dO, dO.sum(0)]
    return {"loss": float((0.5 * e * e * iv + s).sum() / rows), "grad": np.concatenate([x.ravel() for x in g])}
