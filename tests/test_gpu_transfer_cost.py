"""What a state transfer costs beside a plain copy of the same bytes."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from mose_amd import abi, cases

pytestmark = pytest.mark.gpu


def _hip():
    """The HIP runtime that the library is linked with (a second one in the process would see no GPU)."""
    from mose_amd.lib import load
    load()
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64.so" in line)
    return C.CDLL(path)


def _least(fns, n=40):
    """Least seconds of each of fns over n turns taken one after the other."""
    out = [1e9] * len(fns)
    for _ in range(n):
        for q, f in enumerate(fns):
            t0 = time.perf_counter()
            f()
            out[q] = min(out[q], time.perf_counter() - t0)
    return out


def test_mid_size_uploads_cost_a_plain_copy():
    """Uploads of 1.3 to 12 MiB: the plain copy and the conversion kernel.  Through helper threads they took 1.4 times
    as long in sum (764, 1188 us); half of that excess is allowed."""
    from mose_amd.lib import GpuSolver
    H, dst = _hip(), C.c_void_p()
    plain = put = 0.0
    for n in (28, 32, 40, 50, 64):
        g = GpuSolver(cases.vortex(dims=(n, n, n)))
        P = np.random.default_rng(n).random(abi.padded_shape((n, n, n))) + 0.5
        size = C.c_size_t(P.nbytes)
        assert H.hipMalloc(C.byref(dst), size) == 0

        def copy():
            assert H.hipMemcpy(dst, C.c_void_p(P.ctypes.data), size, 1) == 0      # to the device
            assert H.hipDeviceSynchronize() == 0

        a, b = _least([copy, lambda: g.put_state(1, P)])
        print("%d^3: copy %.1f us, put_state %.1f us" % (n, a * 1e6, b * 1e6))
        plain, put = plain + a, put + b
        assert H.hipFree(dst) == 0
        g.close()
    assert put < 1.2 * (plain + 5 * 15e-6), (plain, put)


def test_pinned_arrays_are_copied_at_the_rate_of_the_link():
    """States of 32 MiB: from and to pinned memory in 0.67 of the time that pageable memory takes (613 us up, 622 us
    down; 940 and 948 us); through the chunk buffers they took as long."""
    from mose_amd.lib import GpuSolver, _dp, load
    L, H = load(), _hip()
    n = 90
    g = GpuSolver(cases.vortex(dims=(n, n, n)))
    P = np.random.default_rng(n).random(abi.padded_shape((n, n, n))) + 0.5
    Q = np.empty_like(P)
    mem = C.c_void_p()
    assert H.hipHostMalloc(C.byref(mem), C.c_size_t(P.nbytes), 0) == 0
    pp = C.cast(mem, C.POINTER(C.c_double))
    pin = np.ctypeslib.as_array(pp, shape=P.shape)
    pin[...] = P
    put, put_pin = _least([lambda: L.mose_put_state(g.h, 1, _dp(P)), lambda: L.mose_put_state(g.h, 1, pp)], 15)
    get, get_pin = _least([lambda: L.mose_get_state(g.h, 1, _dp(Q)), lambda: L.mose_get_state(g.h, 1, pp)], 15)
    print("put %.1f us, pinned %.1f us; get %.1f us, pinned %.1f us" % (put * 1e6, put_pin * 1e6, get * 1e6, get_pin * 1e6))
    assert np.array_equal(pin, Q) and np.max(np.abs(Q - P)) < 1e-13
    assert put_pin < 0.85 * put and get_pin < 0.85 * get
    g.close()
    del pin
    assert H.hipHostFree(mem) == 0


@pytest.mark.parametrize("n", [32, 50])
def test_a_small_transfer_does_not_wait_for_a_large_one(n):
    """A context's fetches (2 and 6 MiB) beside another's 88 MiB fetches on a second thread: they share the link
    (0.13 to 0.4 and 0.6 to 0.9 ms).  Taking turns, each waited 2.2 ms."""
    from mose_amd.lib import GpuSolver, _dp, load
    L = load()
    small, large = GpuSolver(cases.vortex(dims=(n, n, n))), GpuSolver(cases.vortex(dims=(128, 128, 128)))
    S, B = small.get_state(1), large.get_state(1)
    ref = S.copy()

    def median():
        t = []
        for _ in range(40):
            S[...] = 0.0
            t0 = time.perf_counter()
            L.mose_get_state(small.h, 1, _dp(S))
            t.append(time.perf_counter() - t0)
            assert np.array_equal(S, ref)
        return sorted(t)[len(t) // 2]

    alone = median()
    whole = _least([lambda: L.mose_get_state(large.h, 1, _dp(B))], 10)[0]
    stop = threading.Event()

    def loop():
        while not stop.is_set():
            L.mose_get_state(large.h, 1, _dp(B))

    other = threading.Thread(target=loop)
    other.start()
    try:
        beside = median()
    finally:
        stop.set()
        other.join()
    print("%d^3: alone %.1f us, beside %.1f us" % (n, alone * 1e6, beside * 1e6))
    assert beside < alone + 0.5 * whole      # (a transfer that takes turns waits for a whole one)
    small.close()
    large.close()
