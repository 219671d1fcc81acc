"""Every limiter with every Riemann solver: a march in one call, whose steps before the last run the stage kernel
without norms, against the same steps in calls of one, bit for bit."""
import numpy as np
import pytest

from mose_amd import abi, cases

from helpers import perturb, skewed_nodes

pytestmark = pytest.mark.gpu

LIMS = ["minmod", "vanleer", "vanalbada", "first-order", "mc", "superbee"]
SOLVERS = ["HLLC", "AUSM+", "HLLE", "SLAU", "SLAU2", "HLLE++", "HLLC+"]


def _box(cfg):
    case = perturb(cases.vortex(dims=(21, 10, 6)), amp=0.01, seed=3)
    case.cfg = cfg
    return case


def _curved(cfg):
    dims = (14, 9, 6)
    prim = np.zeros(dims[::-1] + (5,))
    prim[..., 0], prim[..., 1], prim[..., 2], prim[..., 4] = 1.0, 0.5, 0.1, 1.0 / 1.4
    blk = cases.Block(dims, skewed_nodes(dims, amp=0.02), cases.padded_state(dims, prim))
    bc = cases.bc_records([{"dims": dims, "faces": [400, 400, 300, 300, 400, 400]}])
    return perturb(cases.Case("curved", cfg, [blk], bc), amp=0.01, seed=4)


def _viscous(cfg):
    case = perturb(cases.taylor_green(n=16, nbox=1), amp=0.005, seed=5)
    cfg.gamma, cfg.Rgas = case.cfg.gamma, case.cfg.Rgas
    case.cfg = cfg
    return case


@pytest.mark.parametrize("rs", SOLVERS)
@pytest.mark.parametrize("lim", LIMS)
def test_every_scheme_in_one_call_and_in_single_steps(lim, rs):
    from mose_amd.lib import GpuSolver
    forms = [(m, kw) for m in (_box, _curved, _viscous)
             for kw in ({}, {"precision": abi.PREC_FP32_FLUX}, {"time_accurate": False}, {"muscl_sd": True})]
    for make, kw in forms:
        if kw.get("muscl_sd") and (make is _viscous or lim == "first-order"):      # refused
            continue
        kw = dict({"time_accurate": True}, **kw)
        a, b = (GpuSolver(make(abi.make_cfg(1.4, 1.0 / 1.4, 0.3, lim, rs, 3, kw["time_accurate"],
                                            **{k: v for k, v in kw.items() if k != "time_accurate"}))) for _ in range(2))
        ta, na = a.advance(4)
        for _ in range(4):
            tb, nb = b.advance(1)
        assert ta == tb and np.array_equal(na, nb), (make, kw)
        assert np.array_equal(a.get_state(1), b.get_state(1), equal_nan=True), (make, kw)
        a.close()
        b.close()
