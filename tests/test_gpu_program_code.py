"""Nonlinear models compiled as C (k_lean and the general sweep) against the
bytecode interpreter (BM_TUNE_SPECIALIZE 0), which the oracle tests hold to
the reference's schemes: the same operations in the same order, so models of
sums, products, quotients and square roots give equal bits.  Transcendental
functions come from the run-time compiler's device library, which need not be
the build's (a process that loaded torch uses torch's): there a step differs by
a few units in the last place of dt/tau times the function, under 1e-13
relative over 337 steps in FP64."""
import numpy as np
import pytest

from brian_amd._lib import NetHandle
from brian_amd.equations import Equations

pytestmark = pytest.mark.gpu
DT = 1e-4
# every kind of instruction: functions, powers, comparisons, time, a parameter
EQS = """
dv/dt = (sin(v) + w*cos(w) - tanh(v*w) + 0.3*abs(w)**1.5 + clip(v, -1.0, 0.5) - p*t)/(10*ms) + 40.0/second : 1
dw/dt = (exp(-v*v) - w + sqrt(1.0 + v*v) - log(2.0 + w*w) + v**2/(3.0 + w*w))/(20*ms) : 1
p : 1
"""
PLAIN = """
dv/dt = (1.5/(1.0 + w*w) - v + 0.1*sqrt(abs(w)) - clip(p*t, 0.0, 0.5))/(10*ms) : 1
dw/dt = (v*v - w)/(20*ms) : 1
p : 1
"""


def _run(precision, scheme, n, delay, specialize, timed=False, refr=None, empirical=None, eqs=EQS):
    rng = np.random.default_rng(n)
    e = Equations(eqs)
    code, consts, nregs = e.compile_program()
    h = NetHandle(DT, precision)
    S0 = rng.random((3, n))
    g = h.add_group(S0)
    h.set_program(g, scheme, nregs, code, consts)
    if empirical is None:
        h.set_threshold(g, 0, 0.9)
        h.add_reset_op(g, 0, 0, 0.1)
    else:
        h.set_empirical_threshold(g, 0, 0.9, empirical)
    if refr:
        h.set_refractory(g, int(refr / DT) + 1, refr - 0.5 * DT)
    if timed:
        h.set_timed_input(g, 2, rng.random((50, n)), True)
    # three targets per neuron onto w; the weight is a power of two, so that
    # k_lean's fused count * w + x and the general kernel's two roundings agree
    ptr = np.arange(n + 1) * 3
    col = np.sort(np.array([rng.integers(0, n, 3) for _ in range(n)]), axis=1).ravel()
    h.add_connection(g, 0, n, g, 0, n, 1, ptr, col, np.full(3 * n, 0.0625), delay_steps=delay)
    h.record(g, 1 << 18)
    h.prepare()
    h.set_tuning("specialize", specialize)
    h.run(37)
    h.run(300)
    out = [h.get_state(g, j, n) for j in range(3)] + list(h.get_spikes(g))
    h.close()
    return out


@pytest.mark.parametrize("precision,eqs", [(64, PLAIN), (32, PLAIN), (64, EQS)])
@pytest.mark.parametrize("scheme,n,delay,kw", [
    (1, 1, 0, {}), (1, 257, 0, {}), (2, 1000, 0, {}), (2, 255, 7, {}), (1, 300, 1, {}),
    (1, 300, 0, {"refr": 2e-3}), (2, 300, 0, {"empirical": 15}), (1, 300, 3, {"empirical": 15}),
    (1, 300, 2, {"timed": True}), (3, 300, 0, {}), (3, 300, 4, {"refr": 1e-3})])
def test_compiled_program_equals_interpreter(precision, eqs, scheme, n, delay, kw):
    if scheme == 3 and eqs is EQS:
        pytest.skip("exponential Euler needs an affine model")
    a = _run(precision, scheme, n, delay, 1, eqs=eqs, **kw)
    b = _run(precision, scheme, n, delay, 0, eqs=eqs, **kw)
    if n > 1:
        assert len(b[3]) > 50
    assert all(np.isfinite(x).all() for x in b)
    for x, y in zip(a, b):
        if eqs is EQS and x.dtype == np.float64:
            np.testing.assert_allclose(x, y, rtol=1e-13, atol=1e-14)
        else:
            np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("m,n", [(5, 1), (6, 300), (8, 513)])
def test_wide_linear_model_on_lean_kernel(m, n):
    """Linear models of 5 to 8 variables on k_lean against the general
    kernel, FP64, bit for bit."""
    out = []
    for spec in (1, 0):
        rng = np.random.default_rng(m)
        h = NetHandle(DT, 64)
        g = h.add_group(rng.random((m, n)))
        h.set_linear(g, np.eye(m) * 0.97 + 0.01 * rng.random((m, m)), 0.02 * rng.random(m))
        h.set_threshold(g, 0, 1.0)
        h.add_reset_op(g, 0, 0, 0.0)
        h.add_reset_op(g, 1, 1, 0.25)
        ptr = np.arange(n + 1)
        h.add_connection(g, 0, n, g, 0, n, m - 1, ptr, rng.permutation(n), np.full(n, 0.03), delay_steps=5)
        h.record(g, 1 << 16)
        h.prepare()
        h.set_tuning("specialize", spec)
        h.run(200)
        out.append([h.get_state(g, j, n) for j in range(m)] + list(h.get_spikes(g)))
        h.close()
    assert len(out[0][-1]) > 0
    for x, y in zip(*out):
        np.testing.assert_array_equal(x, y)
