"""Copies between host and device arrive whole at every size, alignment and
list length, also when the pinned ring they go through is used up many times
over, by one thread or several."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [0, 1, 15, 16, 17, 255, 257, 4095, 4096, 4097, 16383, 16384, 16385, 40000, 65535, 65536, 65537, 300001]


def _bytes(n, seed):
    return np.random.default_rng(seed).integers(0, 256, n, dtype=np.uint8)


@pytest.mark.parametrize("shift", [0, 1, 8])
def test_one_piece(shift):
    from ktir_cpu_amd import runtime as rt
    buf = rt.DeviceBuffer(1 << 19)
    for k, n in enumerate(SIZES):
        a = _bytes(n, k)
        buf.memset(0x5a)
        (buf.upload if k % 2 else lambda x, o: buf.put([(x, o)]))(a, shift)
        got = np.empty(n + 2 * shift, np.uint8)
        buf.download_into(got, 0)
        np.testing.assert_array_equal(got[shift:shift + n], a)
        assert (got[:shift] == 0x5a).all() and (got[shift + n:] == 0x5a).all()
    buf.free()


@pytest.mark.parametrize("count,size", [(1, 100), (9, 4000), (25, 70), (5, 65536), (3, 65537), (17, 20000)])
def test_lists(count, size):
    from ktir_cpu_amd import runtime as rt
    step = (size + 128) // 128 * 128
    buf = rt.DeviceBuffer(step * count)
    a = [_bytes(size - i, i) for i in range(count)]
    buf.put([(x, i * step) for i, x in enumerate(a)])
    out = [np.empty_like(x) for x in a]
    buf.fetch([(x, i * step) for i, x in enumerate(out)])
    for x, y in zip(a, out):
        np.testing.assert_array_equal(x, y)
    buf.free()


def _many(seed, errors):
    """2.4 MB of 48 KB uploads queued one after another from one host array that changes at once."""
    from ktir_cpu_amd import runtime as rt
    try:
        n, size = 50, 48 << 10
        buf = rt.DeviceBuffer(n * size)
        want, host = _bytes(n * size, seed), np.empty(size, np.uint8)
        for i in range(n):
            host[:] = want[i * size:(i + 1) * size]
            buf.put([(host, i * size)])
            host[:] = 0
        got = np.empty(size, np.uint8)
        for i in range(n):
            buf.fetch([(got, i * size)])
            np.testing.assert_array_equal(got, want[i * size:(i + 1) * size])
        buf.free()
    except BaseException as e:      # reported by the test's own thread
        errors.append(e)


@pytest.mark.parametrize("threads", [1, 4])
def test_ring_used_many_times_over(threads):
    errors = []
    ts = [threading.Thread(target=_many, args=(7 + t, errors)) for t in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors[0]


def test_ring_without_coherent_default():
    """The same where the runtime's own default for pinned memory is not
    coherent: the same parts of the ring, read by kernel after kernel, hold other
    bytes each time."""
    import os
    import subprocess
    import sys
    code = ("from tests import test_gpu_small_copies as t\ne = []\nfor s in range(4): t._many(s, e)\n"
            "assert not e, e[0]\nprint('whole')")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", code], cwd=root, env=dict(os.environ, HIP_HOST_COHERENT="0"),
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "whole" in r.stdout, r.stdout + r.stderr
