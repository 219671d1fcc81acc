"""Steady adjoint iterations where the transposed ghost fill runs in the stage kernel and the primitives
are formed once a solve (k faces of type 0) against those where neither can be (k faces of type 400: the
fill extrapolates from its own ghost cells); the k faces' fluxes cancel in a block one cell thick."""
import numpy as np
import pytest

from mose_amd import abi, cases

pytestmark = pytest.mark.gpu


def _solve(kface, ni, nj, iters, every):
    from mose_amd.lib import GpuSolver
    case = cases.bump_channel(ni=ni, nj=nj, ncontrol=4, limiter="minmod", alpha=0.01)
    for r in case.bc:
        if r["f"] >= 5:
            r["type"] = kface
    rng = np.random.default_rng(3)
    blk = case.blocks[0]
    prim = np.ascontiguousarray(abi.interior(blk.P))
    prim[..., 0] *= 1.0 + 0.01 * rng.random(prim.shape[:-1])
    blk.P = cases.padded_state(blk.dims, prim)
    bar = np.zeros(abi.padded_shape(blk.dims))
    abi.interior(bar)[:, 0, :, 4] = 0.01
    g = GpuSolver(case)
    out = g.adjoint_solve([bar], max_iter=iters, rtol=0.0, check_every=every)
    again = g.adjoint_solve([bar], max_iter=iters, rtol=0.0, check_every=iters)
    g.close()
    assert np.array_equal(out[0][0], again[0][0]) and out[3] == again[3]
    return abi.interior(out[0][0]), out[2], out[3]


@pytest.mark.parametrize("ni,nj,iters,every", [(40, 20, 12, 5), (17, 9, 7, 1), (65, 33, 10, 10)])
def test_folded_fill_equals_separate_fill(ni, nj, iters, every):
    a, b = _solve(0, ni, nj, iters, every), _solve(400, ni, nj, iters, every)
    for v in (0, 1, 2, 4):
        assert np.linalg.norm(a[0][..., v] - b[0][..., v]) <= 1e-11 * np.linalg.norm(b[0][..., v])
    assert abs(a[1] - b[1]) <= 1e-11 * b[1]
