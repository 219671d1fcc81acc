"""The default tiling (shape and k chunk by the cost rule of mose_finalize) against the fixed
32x8 patch in 32-plane chunks and against the oracle, at sizes around the patch and chunk edges."""
import numpy as np
import pytest

from mose_amd import abi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 2, 2), (32, 16, 3), (33, 17, 2), (31, 15, 65), (65, 9, 33), (5, 70, 12)])
@pytest.mark.parametrize("local", [False, True])
def test_default_tiling_matches_fixed_tiling_and_oracle(dims, local, monkeypatch):
    from mose_amd.lib import GpuSolver
    from oracle.oracle import OracleSolver
    case = cases.vortex(dims=dims, cfl=0.4)
    c = case.cfg
    case.cfg = abi.make_cfg(c.gamma, c.Rgas, c.cfl, "vanleer", "HLLC", 3, not local)
    g = GpuSolver(case)
    monkeypatch.setenv("MOSE_TILE_SHAPE", "0")
    monkeypatch.setenv("MOSE_KCHUNK", "32")
    f = GpuSolver(case)
    assert f.tiling()["tile"] == (32, 8) and f.tiling()["kchunk"] == 32
    o = OracleSolver(case)
    for _ in range(3):
        ng, nf, no = g.step()[2], f.step()[2], o.step()[2]
    Pg, Pf, Po = (abi.interior(s.get_state(1)) for s in (g, f, o))
    assert np.linalg.norm(Pg - Pf) <= 1e-13 * np.linalg.norm(Pf)
    assert np.linalg.norm(Pg - Po) <= 1e-12 * np.linalg.norm(Po)
    # norms: sums over the tiles in another order
    assert np.allclose(ng, nf, rtol=1e-12, atol=1e-15) and np.allclose(ng, no, rtol=1e-9, atol=1e-13)
