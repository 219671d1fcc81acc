"""Residual smoothing of a residual that overflows: infinities as the oracle's divisions give them, no NaN."""
import numpy as np
import pytest

from mose_amd import abi, cases

pytestmark = pytest.mark.gpu


def test_an_infinite_residual_stays_infinite():
    """A wide cell of 1.2 times the density and pressure beside narrow ones, all near 1e307: the energy flux of their
    face, times dt over the narrow cell's volume, overflows; the smoothing carries it to four cells."""
    from mose_amd.lib import GpuSolver
    from oracle.oracle import OracleSolver
    n = 12
    dims = (n, 3, 1)
    nodes = cases.cartesian_nodes(dims, (0, 0, 0), (1.0, 1.0, 1.0))
    nodes[..., 0] = np.concatenate([[0.0, 10.0], 10.0 + np.arange(1, n)])
    prim = np.zeros(dims[::-1] + (5,))
    prim[..., 0] = prim[..., 4] = 1e307
    prim[:, :, 0, (0, 4)] *= 1.2
    cfg = abi.make_cfg(1.4, 1.0 / 1.4, 300.0, "first-order", "HLLE", 1, True, irs_beta=0.5)
    bc = cases.bc_records([{"dims": dims, "faces": [300, 300, 300, 300, 0, 0]}])
    case = cases.Case("overflow", cfg, [cases.Block(dims, nodes, cases.padded_state(dims, prim))], bc)
    g, o = GpuSolver(case), OracleSolver(case)
    g.step()
    o.step()
    Pg, Po = abi.interior(g.get_state(1)), abi.interior(o.get_state(1))
    inf = np.isinf(Po)
    assert inf[..., 4].sum() == 4 * 3 and not np.isnan(Po).any()
    assert np.array_equal(np.where(inf, Pg, 0.0), np.where(inf, Po, 0.0))
    np.testing.assert_allclose(np.where(inf, 0.0, Pg), np.where(inf, 0.0, Po), rtol=1e-12, atol=1e-12)
    g.close()
