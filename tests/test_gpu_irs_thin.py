"""Residual smoothing at blocks a few cells thick, with and without 101 connections, against the oracle."""
import numpy as np
import pytest

from mose_amd import abi, cases

from helpers import perturb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 3, 4), (33, 2, 3), (5, 17, 2), (8, 4, 65)])
@pytest.mark.parametrize("parts", [1, 2])
@pytest.mark.parametrize("beta", [0.5, 0.3])
def test_smoothed_steps_match_the_oracle(dims, parts, beta):
    from mose_amd.lib import GpuSolver
    from oracle.oracle import OracleSolver
    if parts > 1 and dims[0] < 5:
        pytest.skip("nothing to split")
    case = perturb(cases.vortex(dims=dims, cfl=0.4), amp=0.01, seed=6)
    c = case.cfg
    case.cfg = abi.make_cfg(c.gamma, c.Rgas, c.cfl, "vanleer", "HLLC", 3, True, irs_beta=beta)
    if parts > 1:
        case = cases.split_block_case(case, axis=0, parts=parts)
    g, o = GpuSolver(case), OracleSolver(case)
    for _ in range(3):
        g.step()
        o.step()
    for b in range(1, len(case.blocks) + 1):
        Pg, Po = abi.interior(g.get_state(b)), abi.interior(o.get_state(b))
        assert np.linalg.norm(Pg - Po) <= 1e-12 * np.linalg.norm(Po)
    g.close()
