"""FP32-flux layouts: the k chunk of the tiles (the default one or a forced divisor of 32) changes
no bit of the state against 32-plane chunks; sizes around the chunk's and the patch's edges."""
import numpy as np
import pytest

from mose_amd import abi, cases

from helpers import perturb, skewed_nodes

pytestmark = pytest.mark.gpu


def _box(dims, limiter, riemann, viscous=False):
    case = perturb(cases.vortex(dims=dims, limiter=limiter, riemann=riemann, precision=abi.PREC_FP32_FLUX), seed=5)
    if viscous:
        case.meta["viscous"] = [(0, [0.02, 1.0, 0.4, 0.71, 0.3])]
    return case


def _skewed(dims, limiter, riemann):
    prim = np.zeros(tuple(dims[::-1]) + (5,))
    prim[..., 0], prim[..., 1], prim[..., 2], prim[..., 4] = 1.0, 1.5, 0.2, 1.0 / 1.4
    blk = cases.Block(tuple(dims), skewed_nodes(dims), cases.padded_state(dims, prim))
    inflow = {"type": 405, "mach": 1.8, "T": 1.05, "p": 0.7, "alpha": 0.1, "beta": -0.05, "rel_fac": 0.8}
    bc = cases.bc_records([{"dims": tuple(dims), "faces": [inflow, 400, 300, 300, 400, 400]}])
    cfg = abi.make_cfg(1.4, 1.0 / 1.4, 0.4, limiter, riemann, 3, True, precision=abi.PREC_FP32_FLUX)
    return perturb(cases.Case("skewed", cfg, [blk], bc), amp=0.03, seed=3)


def _states(case, monkeypatch, kchunk):
    from mose_amd.lib import GpuSolver
    if kchunk:
        monkeypatch.setenv("MOSE_TILE_SHAPE", "0")
        monkeypatch.setenv("MOSE_KCHUNK", str(kchunk))
    g = GpuSolver(case)
    monkeypatch.delenv("MOSE_KCHUNK", raising=False)
    monkeypatch.delenv("MOSE_TILE_SHAPE", raising=False)
    if kchunk:
        assert g.tiling()["kchunk"] == kchunk
    g.advance(3)
    out = [abi.interior(g.get_state(b)).copy() for b in range(1, len(case.blocks) + 1)]
    g.close()
    return out


def _same(case, monkeypatch):
    ref = _states(case, monkeypatch, 32)
    for kc in (0, 1, 2, 8, 16):
        for a, b in zip(ref, _states(case, monkeypatch, kc)):
            assert np.array_equal(a, b), (kc, np.max(np.abs(a - b)))


@pytest.mark.parametrize("limiter", ["minmod", "vanleer", "vanalbada", "mc", "superbee"])
@pytest.mark.parametrize("riemann", ["HLLC", "AUSM+", "HLLE", "SLAU", "SLAU2", "HLLE++", "HLLC+"])
def test_chunk_keeps_the_bits(limiter, riemann, monkeypatch):
    _same(_box((33, 9, 70), limiter, riemann), monkeypatch)


@pytest.mark.parametrize("dims", [(20, 17, 31), (33, 8, 33), (31, 10, 65), (5, 4, 32)])
@pytest.mark.parametrize("riemann", ["HLLC", "AUSM+"])
def test_chunk_keeps_the_bits_viscous(dims, riemann, monkeypatch):
    _same(_box(dims, "vanleer", riemann, viscous=True), monkeypatch)


@pytest.mark.parametrize("limiter", ["minmod", "vanleer", "mc"])
def test_chunk_keeps_the_bits_general_metrics(limiter, monkeypatch):
    _same(_skewed((14, 11, 40), limiter, "HLLC"), monkeypatch)
