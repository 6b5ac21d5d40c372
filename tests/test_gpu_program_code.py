"""Nonlinear models compiled as C (k_lean and the general sweep) against the
bytecode interpreter (BM_TUNE_SPECIALIZE 0), which the oracle tests hold to
the reference's schemes: the same operations in the same order, so models of
sums, products, quotients and square roots give equal bits.  Transcendental
functions come from the run-time compiler's device library, which need not be
the build's (a process that loaded torch uses torch's).  With the versions that
test_functions_in_any_process knows they have the same bits too; another's may
differ by a few units in the last place of dt/tau times the function, under 1e-13
relative over 337 steps in FP64."""
import os
import subprocess
import sys

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


# affine in each variable of its own, coefficients by functions of the others
AFFINE = """
dv/dt = (0.4 + m*exp(-0.5*m) - v + h*sin(m))/(10*ms) : 1
dm/dt = am*(1 - m) - bm*m : Hz
dh/dt = (tanh(v) + 0.2*sqrt(1.0 + v*v) + cos(v)*log(2.0 + v*v)/3.0 + abs(v)**1.5 - h)/(15*ms) : 1
am = 0.3*exp((v - 0.5)/0.4)/ms : Hz
bm = 0.4/(1 + exp((0.5 - v)/0.3))/ms : Hz
"""


def _run(precision, scheme, n, delay, specialize, timed=False, refr=None, empirical=None, eqs=EQS, quiet=False):
    rng = np.random.default_rng(n)
    e = Equations(eqs)
    code, consts, nregs = e.compile_program()
    h = NetHandle(DT, precision)
    S0 = rng.random((3, n))
    g = h.add_group(S0)
    h.set_program(g, scheme, nregs, code, consts)
    if quiet:
        h.set_threshold(g, 0, np.inf)
    elif empirical is None:
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
    if not quiet:
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


FUNCTIONS = ["exp(v)", "log(2.0 + v)", "sqrt(1.5 + v)", "abs(v)**1.7", "sin(3.0*v)", "cos(3.0*v)", "tanh(v)",
             "1.0/(1.3 + v*v)", "v**3"]


def function_bits():
    """One step of dv/dt = f(v) - v, compiled and interpreted, equal bit for bit."""
    for f in FUNCTIONS:
        code, consts, nregs = Equations(f"dv/dt = ({f} - v)/(10*ms) : 1").compile_program()
        for precision in (64, 32):
            out = []
            for specialize in (1, 0):
                h = NetHandle(DT, precision)
                g = h.add_group(np.linspace(-1.4, 2, 20000)[None, :])
                h.set_program(g, 1, nregs, code, consts)
                h.prepare()
                h.set_tuning("specialize", specialize)
                h.run(1)
                out.append(h.get_state(g, 0, 20000))
                h.close()
            assert np.isfinite(out[1]).all()
            np.testing.assert_array_equal(out[0], out[1], err_msg=f"{f} in FP{precision}")


@pytest.mark.parametrize("first", ["", "import torch"])
def test_functions_in_any_process(first):
    """A process that loaded torch, and with it torch's run-time compiler, gives
    the results of one that did not: both those of the interpreter, which is
    compiled with the library."""
    p = subprocess.run([sys.executable, "-c", f"{first}\nfrom tests.test_gpu_program_code import function_bits\n"
                        "function_bits()\nprint('equal')"], capture_output=True, text=True, timeout=100,
                       cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert p.returncode == 0 and "equal" in p.stdout, p.stdout + p.stderr


@pytest.mark.parametrize("scheme,delay,eqs", [(1, 0, EQS), (2, 0, EQS), (2, 5, EQS), (1, 0, AFFINE), (3, 0, AFFINE),
                                               (3, 1, AFFINE), (3, 6, AFFINE)])
def test_compiled_functions_fp32(scheme, delay, eqs):
    """FP32 with functions, on k_lean and the general kernel, without spikes: a
    function apart by 2 units in the last place (2^-22 of its value) changes a
    step by dt/tau of that, under 1e-8 for values and slopes of order 1, and
    the sum after it may round the other way (2^-24): 7e-8 a step, which slopes
    of up to 4/(10 ms) let grow by e^1.5 in 37 steps: 1.2e-5."""
    a = _run(32, scheme, 300, delay, 1, eqs=eqs, quiet=True)
    b = _run(32, scheme, 300, delay, 0, eqs=eqs, quiet=True)
    assert len(a[3]) == len(b[3]) == 0
    for x, y in zip(a[:3], b[:3]):
        assert np.isfinite(y).all() and np.abs(y).max() < 20
        np.testing.assert_allclose(x, y, rtol=1.2e-5, atol=1.2e-5)


@pytest.mark.parametrize("delay,kw", [(0, {}), (1, {}), (5, {}), (0, {"refr": 2e-3}), (4, {"empirical": 15})])
def test_exponential_euler_with_functions(delay, kw):
    """Exponential Euler of a model with functions in its coefficients (as
    Hodgkin-Huxley gates), FP64: a step is apart by a few units in the last
    place of S + B and of B, 1e-15, and a difference lasts for tau, 150 steps:
    1.5e-13."""
    a = _run(64, 3, 300, delay, 1, eqs=AFFINE, **kw)
    b = _run(64, 3, 300, delay, 0, eqs=AFFINE, **kw)
    assert len(b[3]) > 50
    for x, y in zip(a, b):
        if x.dtype == np.float64:
            assert np.isfinite(y).all()
            np.testing.assert_allclose(x, y, rtol=1.5e-13, atol=1.5e-13)
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
