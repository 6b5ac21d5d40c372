"""Small networks in one workgroup (net_small.hpp; BM_TUNE_SMALL 2) against
the windowed kernels (BM_TUNE_SMALL 0), each arm's route checked.  Deliveries
that are counts: rasters and state equal bit for bit; weights per synapse: equal
up to the order of the floating additions (a handful of values per target and
step, so 1e-12 relative in FP64).  Then where the one or the other is taken."""
import numpy as np
import pytest

from brian_amd import workloads as W
from brian_amd._lib import NetHandle
from brian_amd.equations import Equations
from tests.netbuild import cuba_propagator

pytestmark = pytest.mark.gpu
DT = 1e-4


def _csr(rng, nsrc, ntgt, p):
    m = rng.random((nsrc, ntgt)) < p
    ptr = np.concatenate([[0], np.cumsum(m.sum(1))])
    return ptr, np.nonzero(m)[1]


WINDOWS, ONE_WORKGROUP = 1, 2


def _advance(h, stretches, small, fits=True, shortest=1):
    h.set_tuning("small", 2 if small else 0)
    for s in stretches:
        h.run(s)
        assert h.get_tuning("route") == (ONE_WORKGROUP if small and fits and s >= shortest else WINDOWS)


def _both(build, stretches, exact=True, rtol=1e-12, fits=True, shortest=1):
    out = []
    for small in (True, False):
        h, read = build()
        _advance(h, stretches, small, fits, shortest)
        out.append(read(h))
        h.close()
    assert len(out[0]) == len(out[1])
    for a, b in zip(*out):
        if exact or np.issubdtype(np.asarray(a).dtype, np.integer):
            np.testing.assert_array_equal(a, b)
        else:
            np.testing.assert_allclose(a, b, rtol=rtol, atol=rtol * 1e-2)
    return out[0]


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n,kind", [
    (1, "plain"), (63, "plain"), (1025, "plain"), (4000, "plain"), (8192, "plain"), (8193, "plain"), (14900, "plain"), (1000, "refractory"),
    (1000, "refractory_array"), (2049, "vt"), (700, "delays"), (300, "dense_raster")])
def test_count_network(n, kind, precision):
    A, C = cuba_propagator()

    def build():
        rng = np.random.default_rng(n)
        ne = max(1, int(0.8 * n))
        p = min(1.0, 80 / n)
        S0 = np.zeros((4, n))
        S0[0] = W.Vr + rng.random(n) * (W.Vt - W.Vr) * (1.0 if kind != "dense_raster" else 3.0)
        S0[3] = W.Vt + 1e-3 * rng.random(n)
        AA, CC = np.eye(4), np.zeros(4)
        AA[:3, :3], CC[:3] = A, C
        h = NetHandle(DT, precision)
        g = h.add_group(S0)
        h.set_linear(g, AA, CC)
        if kind == "vt":
            h.set_threshold(g, 0, 0.0, 3)
            h.add_reset_op(g, 0, 0, W.Vr)
            h.add_reset_op(g, 3, 1, 1e-3)
        else:
            h.set_threshold(g, 0, -0.058 if kind == "dense_raster" else W.Vt)
            h.add_reset_op(g, 0, 0, W.Vr if kind != "dense_raster" else -0.0579)
        if kind == "refractory":
            h.set_refractory(g, 51, 5e-3 - 0.5 * DT)
        if kind == "refractory_array":
            r = (1 + 7 * rng.random(n)) * 1e-3
            h.set_refractory(g, int(r.max() / DT) + 1, r.max() - 0.5 * DT, per_neuron=r)
        for lo, m, var, w in ((0, ne, 1, W.we), (ne, n - ne, 2, W.wi)):
            if m == 0:
                continue
            ptr, col = _csr(rng, m, n, p)
            kw = {}
            if kind == "delays" and var == 1:
                kw = {"syn_delay": rng.integers(0, 20, len(col)), "max_delay_steps": 20}
            h.add_connection(g, lo, m, g, 0, n, var, ptr, col, np.full(len(col), w), **kw)
        h.record(g, 1 << 17)
        h.prepare()
        return h, lambda h: [*h.get_spikes(g), *[h.get_state(g, v, n) for v in range(4)]]

    # 8192 neurons in FP64 and 16,384 in FP32, as far as the rings fit the LDS
    out = _both(build, (2, 300, 1, 4, 250), fits=precision == 32 or n <= 8192, shortest=1 if n <= 4096 else 4)
    if n > 1:
        assert len(out[0]) > 5


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("nin,nout,inter,update", [
    (1000, 1, 0, 0), (200, 64, 1, 0), (333, 17, 2, 1), (64, 65, 3, 0), (1, 3, 0, 1)])
def test_poisson_stdp_network(nin, nout, inter, update, precision):
    """Poisson inputs through plastic weights onto a group, and back from it
    through fixed weights of their own onto a second group."""
    d = W.stdp_batch(1, nin)

    def build():
        rng = np.random.default_rng(nin + nout)
        h = NetHandle(DT, precision)
        p = h.add_poisson(nin, 15.0 * (1 + 3 * rng.random(nin)), 7)
        g = h.add_group(np.vstack([np.full(nout, -0.055), np.zeros(nout)]))
        h.set_linear(g, d["A"], d["C"])
        h.set_threshold(g, 0, d["vt"])
        h.add_reset_op(g, 0, 0, d["vr"])
        gmax = 10.0 / nin
        c = h.add_connection(p, 0, nin, g, 0, nout, 1, np.arange(nin + 1) * nout, np.tile(np.arange(nout), nin),
                             rng.random(nin * nout) * gmax)
        sid = h.add_stdp(c, d["decay_pre"], d["decay_post"], 0.01 * (gmax if update == 0 else 1),
                         -0.0105 * (gmax if update == 0 else 1), 0.0, gmax, update, inter)
        g2 = h.add_group(np.zeros((1, 5)))
        h.set_linear(g2, np.array([[0.99]]), np.array([0.0]))
        ptr, col = _csr(rng, nout, 5, 0.5)
        h.add_connection(g, 0, nout, g2, 0, 5, 0, ptr, col, rng.random(len(col)), delay_steps=2)
        h.record(g, 1 << 16)
        h.record(p, 1 << 17)
        h.set_poisson_rates(p, 100, 200.0 + 0.0 * np.arange(150), False)
        h.prepare()

        def read(h):
            return [*h.get_spikes(p), *h.get_spikes(g), h.get_weights(c, nin * nout),
                    *h.get_stdp_traces(sid, nin, nout), h.get_state(g, 0, nout), h.get_state(g, 1, nout),
                    h.get_state(g2, 0, 5)]
        return h, read

    # FP32: the additions of a step in another order, an ulp of 6e-8 each
    out = _both(build, (3, 400, 7, 500), exact=False, rtol=1e-11 if precision == 64 else 2e-4)
    assert len(out[0]) > (5 if nin > 1 else 0)
    if nin >= 64:
        assert len(out[2]) > 5


def test_long_run_and_rate_changes():
    """A run of more steps than one launch takes, and new rates between
    runs."""
    def build():
        h = NetHandle(DT, 64)
        p = h.add_poisson(3, np.array([20.0, 30.0, 5.0]), 1)
        g = h.add_group(np.zeros((1, 2)))
        h.set_linear(g, np.array([[0.999]]), np.array([0.0]))
        h.set_threshold(g, 0, 2.0)
        h.add_reset_op(g, 0, 0, 0.0)
        h.add_connection(p, 0, 3, g, 0, 2, 0, [0, 2, 4, 6], [0, 1, 0, 1, 0, 1], np.full(6, 0.75))
        h.record(g, 1 << 14)
        h.prepare()
        return h, lambda h: [*h.get_spikes(g), h.get_state(g, 0, 2)]
    out = []
    for small in (True, False):
        h, read = build()
        _advance(h, (20011,), small)
        h.set_poisson_base_rates(0, np.array([100.0, 200.0, 0.0]))
        _advance(h, (2000,), small)
        out.append(read(h))
        h.close()
    assert len(out[0][0]) > 20
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("vt", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("small", [0, 2])      # windowed kernels, one workgroup
@pytest.mark.parametrize("kind", ["counts", "weights", "program"])
def test_constants_without_a_literal(kind, small, vt):
    """Thresholds and reset values that are infinite or NaN, against the kernels
    that read them from tables (specialize 0)."""
    out = []
    for specialize in (1, 0):
        n = 70
        h = NetHandle(DT, 64)
        g = h.add_group(np.random.default_rng(3).random((2, n)))
        if kind == "program":
            code, consts, nregs = Equations("dv/dt = (b - v)/(10*ms) : 1\ndw/dt = -w*w/(20*ms) : 1",
                                            b=vt).compile_program()
            h.set_program(g, 1, nregs, code, consts)
            h.set_threshold(g, 1, 0.5)
            h.add_reset_op(g, 1, 0, 0.9)
        else:
            h.set_linear(g, np.diag([0.99, 0.98]), np.zeros(2))
            h.set_threshold(g, 0, vt)
            h.add_reset_op(g, 1, 0, -vt)
        w = np.full(n, 0.01) if kind == "counts" else 0.01 * np.arange(n)
        h.add_connection(g, 0, n, g, 0, n, 0, np.arange(n + 1), np.arange(n), w)
        h.record(g, 1 << 14)
        h.prepare()
        h.set_tuning("small", small)
        h.set_tuning("specialize", specialize)
        h.run(40)
        assert h.get_tuning("route") == (ONE_WORKGROUP if small and specialize and kind != "program" else WINDOWS)
        out.append([*h.get_spikes(g), h.get_state(g, 0, n), h.get_state(g, 1, n)])
        h.close()
    assert len(out[0][0]) == (0 if kind != "program" and not vt < 0 else len(out[1][0]))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


def test_raster_regions_fill_evenly():
    """Runs of as many steps as there are append regions: the raster still
    holds the capacity asked for."""
    n, runs = 3000, 64

    def build():
        h = NetHandle(DT, 64)
        g = h.add_group(np.random.default_rng(1).random((1, n)))
        h.set_linear(g, np.eye(1), np.array([1 / 150]))
        h.set_threshold(g, 0, 1.0)
        h.add_reset_op(g, 0, 0, 0.0)
        h.add_connection(g, 0, 1, g, 0, n, 0, np.array([0, 1]), np.array([0]), np.array([1e-3]))
        h.record(g, n * 32 * runs // 140)
        h.prepare()
        return h, lambda h: [*h.get_spikes(g), h.get_state(g, 0, n)]

    out = _both(build, [32] * runs)
    assert len(out[0]) > n * 32 * runs // 160


def _deliveries(n, row, precision=64, exact_weights=True, poisson=None, stdp=False):
    """n neurons (or Poisson sources at a rate, and n neurons) with `row`
    synapses each and no delay."""
    rng = np.random.default_rng(n + row)
    h = NetHandle(DT, precision)
    src = None if poisson is None else h.add_poisson(n, np.full(n, float(poisson)), 5)
    S0 = np.zeros((2, n))
    S0[0] = rng.random(n)
    g = h.add_group(S0)
    h.set_linear(g, np.diag([1.0, 0.9]), np.array([0.01 if poisson is None else 0.0, 0.0]))
    h.set_threshold(g, 0, 1.0)
    h.add_reset_op(g, 0, 0, 0.0)
    col = np.sort(rng.integers(0, n, (n, row)), axis=1).ravel()
    w = np.full(n * row, 1e-3) if exact_weights else 1e-3 * rng.random(n * row)
    c = h.add_connection(g if src is None else src, 0, n, g, 0, n, 1, np.arange(n + 1) * row, col, w)
    if stdp:
        h.add_stdp(c, 0.99, 0.99, 1e-5, -1e-5, 0.0, 1e-3, 0, 0)
    h.record(g, n * 64)
    h.prepare()
    return h, src, g


@pytest.mark.parametrize("n,row,precision,exact_weights,stdp,route", [
    # at 100 Hz: 10,000 deliveries a step of 1000 neurons, 3200 and 20,000 of 4000,
    # 6400 of 8000
    (1000, 1000, 64, True, False, ONE_WORKGROUP), (4000, 80, 64, True, False, ONE_WORKGROUP),
    (4000, 500, 64, True, False, WINDOWS), (8000, 80, 64, True, False, WINDOWS),
    (8000, 20, 64, True, False, ONE_WORKGROUP), (8000, 2000, 64, True, False, WINDOWS),
    (2000, 100, 32, False, False, ONE_WORKGROUP), (4000, 80, 32, False, False, WINDOWS),
    (4000, 80, 64, False, False, ONE_WORKGROUP)])
def test_dense_networks_keep_the_windows(n, row, precision, exact_weights, stdp, route):
    h, _, g = _deliveries(n, row, precision, exact_weights, stdp=stdp)
    assert h.get_tuning("small") == 1
    h.run(8)
    assert h.get_tuning("route") == route
    a = h.get_spikes(g)
    h.close()
    h, _, g = _deliveries(n, row, precision, exact_weights, stdp=stdp)
    h.set_tuning("small", 2 if route == WINDOWS else 0)
    h.run(8)
    assert h.get_tuning("route") == (ONE_WORKGROUP if route == WINDOWS else WINDOWS)
    for x, y in zip(a, h.get_spikes(g)):        # the potentials do not see the deliveries
        np.testing.assert_array_equal(x, y)
    h.close()


@pytest.mark.parametrize("n", [4096, 4097])
def test_short_runs_compile_nothing(n):
    """Runs of 1 to 3 steps, as of scripts that go on step by step, find their
    kernel compiled at prepare."""
    A = 0.9 + 0.05 * np.random.default_rng().random()
    h = NetHandle(DT, 64)
    g = h.add_group(np.random.default_rng(0).random((1, n)))
    h.set_linear(g, np.array([[A]]), np.array([0.2]))
    h.set_threshold(g, 0, 1.0)
    h.add_reset_op(g, 0, 0, 0.0)
    h.add_connection(g, 0, 1, g, 0, n, 0, np.array([0, 1]), np.array([0]), np.array([1e-3]))
    h.prepare()
    compiled = h.get_tuning("compiled")
    for steps in (1, 3, 8, 2):
        h.run(steps)
        assert h.get_tuning("route") == (WINDOWS if n > 4096 and steps < 4 else ONE_WORKGROUP)
    assert h.get_tuning("compiled") == compiled
    h.close()


def _scan(kind, value):
    """A network of the kind with its constants set by value."""
    h = NetHandle(DT, 64)
    n = 40
    src = h.add_poisson(n, np.full(n, 100.0), 5)
    g = h.add_group(np.full((2, n), 0.5))
    h.set_linear(g, np.array([[0.99, 0.1 * value], [0.0, 0.95 - 0.01 * value]]), np.array([0.01 * value, 0.001]))
    if kind == "empirical":
        h.set_empirical_threshold(g, 0, 0.9 + 0.01 * value, 10 + int(10 * value))
    else:
        h.set_threshold(g, 0, 0.9 + 0.01 * value)
    h.add_reset_op(g, 0, 0, 0.1 * value)
    w = np.full(n, 0.1 * value) if kind == "empirical" else 0.1 * value * np.arange(n)
    c = h.add_connection(src, 0, n, g, 0, n, 1, np.arange(n + 1), np.arange(n), w,
                         delay_steps=0 if kind == "stdp" else 3)
    if kind == "stdp":
        h.add_stdp(c, 0.99, 0.99, 1e-3 * value, -1e-3 * value, 0.0, 5.0, 0, 0)
    h.record(g, 1 << 14)
    h.prepare()
    return h, g


@pytest.mark.parametrize("kind", ["stdp", "layer", "empirical"])
def test_scanned_constants_share_kernels(kind):
    """Networks that differ in constants alone compile once, and each runs with
    its own (against the kernels that read tables)."""
    values = np.random.default_rng(0).random(4) + 0.5
    h, _ = _scan(kind, 0.25)
    compiled = h.get_tuning("compiled")
    h.close()
    spikes = set()
    for v in values:
        out = []
        for specialize in (1, 0):
            h, g = _scan(kind, v)
            h.set_tuning("specialize", specialize)
            h.run(300)
            out.append([*h.get_spikes(g), h.get_state(g, 0, 40), h.get_state(g, 1, 40)])
            assert h.get_tuning("compiled") == compiled
            h.close()
        for a, b in zip(*out):
            np.testing.assert_array_equal(a, b)
        spikes.add(len(out[0][0]))
    assert len(spikes) > 1 and min(spikes) > 0


def test_idle_kernels_are_dropped():
    """Beyond 32 kernels that no network uses, those used longest ago are
    unloaded; a network's own stay."""
    def build(value):
        h = NetHandle(DT, 64)
        g = h.add_group(np.linspace(0, 1, 50)[None, :])
        h.set_linear(g, np.array([[1.0]]), np.array([value]))
        h.set_threshold(g, 0, 1.0)
        h.add_reset_op(g, 0, 0, 0.0)
        h.record(g, 1 << 12)
        h.prepare()
        return h, g

    def run(h, g):
        h.run(150)
        return h.get_spikes(g)

    values = 0.01 + 0.01 * np.random.default_rng().random(40)
    held, g = build(values[0])
    want = run(held, g)
    for v in values[1:]:
        h, q = build(v)
        run(h, q)
        h.close()
    compiled = held.get_tuning("compiled")
    h, _ = build(values[-1])                  # still there
    assert h.get_tuning("compiled") == compiled
    h.close()
    h, _ = build(values[1])                   # dropped
    assert h.get_tuning("compiled") == compiled + 1
    h.close()
    first = len(want[0])
    s, i = run(held, g)
    assert len(s) > first > 0
    h, q = build(values[0])                   # the held network's own
    assert h.get_tuning("compiled") == compiled + 1
    np.testing.assert_array_equal(run(h, q), want)
    # another shape: the kernel that the captured launches hold falls idle, as the
    # one used longest ago
    for net, gid in ((held, g), (h, q)):
        net.set_tuning("neurons_per_thread", 2)
        net.run(150)
    plain, p = build(values[0])
    plain.run(450)
    for x, y in zip(held.get_spikes(g), plain.get_spikes(p)):
        np.testing.assert_array_equal(x, y)
    plain.close()
    h.close()
    held.close()


@pytest.mark.parametrize("stdp", [False, True])
def test_poisson_rates_choose_the_kernel(stdp):
    """Sources at 20 Hz leave a step little to deliver, at 4000 Hz much; base
    rates and tables set between runs count, and switching changes nothing but
    the kernel."""
    out = []
    for small in (1, 0):
        h, p, g = _deliveries(2000, 500 if stdp else 100, 64, False, poisson=20, stdp=stdp)
        h.set_tuning("small", small)
        routes = []
        for rates, table in ((None, None), (4000.0, None), (20.0, None), (None, 4000.0)):
            if rates is not None:
                h.set_poisson_base_rates(p, np.full(2000, rates))
            if table is not None:
                h.set_poisson_rates(p, 0, np.full(40, table), False)
            h.run(8)
            routes.append(h.get_tuning("route"))
        assert routes == ([ONE_WORKGROUP, WINDOWS, ONE_WORKGROUP, WINDOWS] if small else [WINDOWS] * 4)
        out.append(h.get_state(g, 1, 2000))
        h.close()
    np.testing.assert_allclose(out[0], out[1], rtol=1e-12)


def test_small_refuses_other_values():
    h, _, _ = _deliveries(100, 5)
    for v in (-1, 3):
        with pytest.raises(Exception, match="small must be"):
            h.set_tuning("small", v)
    h.close()
