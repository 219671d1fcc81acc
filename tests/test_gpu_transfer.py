"""State transfers through the pinned chunk buffers: sizes around the plain-copy limit (1 MiB) and
the 4 MiB chunk, against the transfer that stages through a fixed device array."""
import threading

import numpy as np
import pytest

from mose_amd import abi, cases

pytestmark = pytest.mark.gpu


def _random_state(dims, seed):
    rng = np.random.default_rng(seed)
    P = rng.standard_normal(abi.padded_shape(dims))
    P[..., 0] = 0.5 + rng.random(P.shape[:-1])
    P[..., 4] = 0.5 + rng.random(P.shape[:-1])
    return P


# bytes: 26^3 cells with ghosts are below 1 MiB, 27 x 27 x 36 just above it; 64^3 is 10 MiB, 47 x 47 x 47
# just below one chunk of 4 MiB and 48 x 48 x 47 above it
@pytest.mark.parametrize("dims", [(2, 2, 2), (22, 22, 22), (23, 23, 32), (43, 43, 43), (44, 44, 43), (61, 59, 57), (90, 90, 90)])
def test_round_trip_and_fixed_staging_agree(dims):
    from mose_amd.lib import GpuSolver
    g = GpuSolver(cases.vortex(dims=dims))
    for seed in (1, 2):
        P = _random_state(dims, seed)
        g.put_state(1, P)
        Q = g.get_state(1)
        # primitive -> conserved -> primitive: a few roundings of O(1) values
        assert np.max(np.abs(Q - P)) < 1e-13
        assert np.array_equal(Q, g.get_state_noalloc(1))


def test_contexts_on_two_threads():
    from mose_amd.lib import GpuSolver
    out = {}

    def run(key, dims):
        g = GpuSolver(cases.vortex(dims=dims))
        ok = True
        for seed in range(4):
            P = _random_state(dims, seed)
            g.put_state(1, P)
            ok = ok and np.max(np.abs(g.get_state(1) - P)) < 1e-13
        g.close()
        out[key] = ok

    threads = [threading.Thread(target=run, args=(k, d)) for k, d in enumerate([(61, 59, 57), (50, 40, 30)])]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert out == {0: True, 1: True}
