"""A march in one call against the same steps in calls of one: the steps before a call's last one leave
out the norms and the ghost layers that only a caller can see, and change no bit of the rest."""
import numpy as np
import pytest

from mose_amd import abi, cases

from helpers import perturb

pytestmark = pytest.mark.gpu


def _plane(dims, kfaces, riemann="HLLC", viscous=False, precision=abi.PREC_FP64, sd=False):
    nodes = cases.cartesian_nodes(dims, (0, 0, 0), (1.0, 0.7, 0.1))
    xc = cases.cell_centres(nodes)
    prim = np.zeros(dims[::-1] + (5,))
    prim[..., 0] = 1.0 + 0.1 * np.sin(2 * np.pi * xc[..., 0])
    prim[..., 1] = 0.3 * np.cos(2 * np.pi * xc[..., 1] / 0.7)
    prim[..., 2] = 0.2 * np.sin(2 * np.pi * xc[..., 0])
    prim[..., 4] = 1.0
    iper = [{"type": 201, "bs": 1, "fs": 2}, {"type": 201, "bs": 1, "fs": 1}]      # viscous blocks: no open faces
    faces = (iper if viscous else [400, 0]) + [{"type": 201, "bs": 1, "fs": 4}, {"type": 201, "bs": 1, "fs": 3}] + kfaces
    bc = cases.bc_records([{"dims": dims, "faces": faces}])
    cfg = abi.make_cfg(1.4, 1.0 / 1.4, 0.4, "vanleer", riemann, 3, True, precision=precision, muscl_sd=sd)
    case = cases.Case("plane", cfg, [cases.Block(dims, nodes, cases.padded_state(dims, prim))], bc)
    if viscous:
        case.meta["viscous"] = [(0, [0.02, 1.0, 0.4, 0.71, 0.3])]
    return case


CASES = {
    "box_fp64": lambda: perturb(cases.vortex(dims=(33, 9, 7), cfl=0.4), seed=1),
    "box_fp32": lambda: perturb(cases.vortex(dims=(20, 17, 12), cfl=0.4, precision=abi.PREC_FP32_FLUX), seed=2),
    "viscous_fp64": lambda: perturb(cases.taylor_green(n=20, nbox=2), amp=0.01, seed=3),
    "viscous_fp32": lambda: perturb(cases.taylor_green(n=18, nbox=1, precision=abi.PREC_FP32_FLUX), amp=0.01, seed=4),
    "viscous_fp32_hllc": lambda: perturb(cases.taylor_green(n=24, nbox=1, riemann="HLLC", precision=abi.PREC_FP32_FLUX),
                                         amp=0.01, seed=5),
    "tube": lambda: cases.sod(n=70),
    "channel": lambda: cases.bump_channel(ni=40, nj=20, ncontrol=4, limiter="minmod"),
    "plane_0": lambda: _plane((37, 18, 1), [0, 0]),
    "plane_0_fp32": lambda: _plane((37, 18, 1), [0, 0], precision=abi.PREC_FP32_FLUX),
    "plane_0_400": lambda: _plane((37, 18, 1), [0, 400]),
    "plane_detector": lambda: _plane((37, 18, 1), [0, 0], riemann="HLLC+"),
    "plane_muscl_sd": lambda: _plane((37, 18, 1), [0, 0], sd=True),
    "plane_viscous": lambda: _plane((37, 18, 1), [0, 0], viscous=True),
}


# (the viscous plane's flow leaves the scheme's range at its twelfth step)
@pytest.mark.parametrize("name,nsteps", [(c, n) for c in sorted(CASES) for n in (1, 2, 9, 18) if c != "plane_viscous" or n < 12])
def test_one_call_equals_single_steps(name, nsteps):
    from mose_amd.lib import GpuSolver
    a, b = GpuSolver(CASES[name]()), GpuSolver(CASES[name]())
    ta, na = a.advance(nsteps)
    for _ in range(nsteps):
        tb, nb = b.advance(1)
    assert ta == tb and np.array_equal(na, nb)
    for q in range(1, len(a.dims) + 1):
        assert np.array_equal(a.get_state(q), b.get_state(q), equal_nan=True)      # ghost layers included
    a.close()
    b.close()
