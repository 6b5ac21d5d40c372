"""Reading a raster sorts it on the device (raster.hip): entries by (step,
index), repeats kept, at the sizes where the path changes (one workgroup's
LDS, one tile of the radix sort, several tiles, 64-bit keys), against numpy's
sort of the generator's table."""
import ctypes as C
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from brian_amd._lib import NetHandle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,N,steps", [
    (0, 10, 50), (1, 1, 1), (2, 1, 3), (3, 300, 4), (63, 20, 40), (1024, 70000, 2), (4095, 1000, 100),
    (4096, 1000, 100), (4097, 1000, 100), (4097, 40, 4096), (8192, 1 << 20, 700), (50000, 257, 300),
    (300001, 1 << 20, 2000), (100000, 1 << 20, 5000), (5000, 1 << 22, 40000)])
def test_raster_is_sorted(n, N, steps):
    rng = np.random.default_rng(n)
    s, i = np.sort(rng.integers(0, steps, n)), rng.integers(0, N, n)
    order = np.lexsort((i, s))
    s, i = s[order], i[order]
    h = NetHandle(1e-4, 32)
    g = h.add_generator(N, s, i)
    h.record(g, max(n * 64, 1))            # every region may receive all of a window's spikes
    h.prepare()
    half = steps // 2
    h.run(half)
    a = h.get_spikes(g)
    np.testing.assert_array_equal(a[0], s[s < half])
    np.testing.assert_array_equal(a[1], i[s < half])
    if n % 2:
        h.clear_spikes(g)                  # later entries only: the keys start at this step
        s, i = s[s >= half], i[s >= half]
    h.run(steps - half)
    b = h.get_spikes(g)
    np.testing.assert_array_equal(b[0], s)
    np.testing.assert_array_equal(b[1], i)
    h.close()


def test_rasters_read_by_several_threads():
    rng = np.random.default_rng(5)
    h = NetHandle(1e-4, 32)
    want = {}
    for n in (500, 20000, 60000):
        s, i = np.sort(rng.integers(0, 200, n)), rng.integers(0, 3000, n)
        order = np.lexsort((i, s))
        g = h.add_generator(3000, s[order], i[order])
        h.record(g, n * 64)
        want[g] = (s[order], i[order])
    h.prepare()
    h.run(200)
    with ThreadPoolExecutor(6) as pool:
        reads = [(g, pool.submit(h.get_spikes, g)) for _ in range(8) for g in want]
        for g, r in reads:
            np.testing.assert_array_equal(r.result()[0], want[g][0])
            np.testing.assert_array_equal(r.result()[1], want[g][1])
    h.close()


@pytest.mark.parametrize("regions", [1, 2, 3])
@pytest.mark.parametrize("n", [1, 30, 4095, 4200, 8190, 8195, 12000])
def test_few_regions(regions, n):
    """A workgroup of 256 neurons appends to a region: up to 2 of them and 8192
    entries are sorted on the host, others on the device."""
    rng = np.random.default_rng(n)
    N = 256 * regions
    per = min(n, 30 * regions)                # neurons that spike at every step
    who = np.sort(rng.permutation(N)[:per])
    S0 = np.zeros((1, N))
    S0[0, who] = 2
    h = NetHandle(1e-4, 32)
    g = h.add_group(S0)
    h.set_linear(g, np.eye(1), np.zeros(1))
    h.set_threshold(g, 0, 1.0)
    h.record(g, 2 * n + 64)
    h.prepare()
    steps = max(1, n // per)
    h.run(steps)
    s, i = h.get_spikes(g)
    np.testing.assert_array_equal(s, np.repeat(np.arange(steps), per))
    np.testing.assert_array_equal(i, np.tile(who, steps))
    h.close()


def _free_bytes():
    hip = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_large_raster_gives_its_buffers_back():
    """8 million spikes need 128 MB to sort; the handle does not keep them."""
    n, steps = 1 << 20, 8
    h = NetHandle(1e-4, 32)
    g = h.add_group(np.ones((1, n)))
    h.set_linear(g, np.eye(1), np.zeros(1))
    h.set_threshold(g, 0, 0.5)
    h.record(g, n * steps)
    h.prepare()
    h.run(steps)
    h.sync()
    before = _free_bytes()
    s, i = h.get_spikes(g)
    assert abs(before - _free_bytes()) < 64 << 20
    np.testing.assert_array_equal(s, np.repeat(np.arange(steps), n))
    np.testing.assert_array_equal(i, np.tile(np.arange(n), steps))
    h.close()
