"""The persistent stage launch with more tiles than workgroups (claims from the own queue, tiles of other queues, the
counters' reset): the bits of the launch with one workgroup per tile, which makes no claims."""
import numpy as np
import pytest

from mose_amd import abi, cases

from helpers import perturb

pytestmark = pytest.mark.gpu

PRECS = [abi.PREC_FP64, abi.PREC_FP32_FLUX]


def _tiles(case, tile, kchunk):
    up = lambda a, b: -(-a // b)
    return sum(up(b.dims[0], tile[0]) * up(b.dims[1], tile[1]) * up(b.dims[2], kchunk) for b in case.blocks)


def _march(case, mode, nsteps):
    from mose_amd.lib import GpuSolver
    import os
    os.environ["MOSE_TILE_XCD"] = str(mode)
    g = GpuSolver(case)
    t = g.tiling()
    assert t["kchunk"] == 1 and t["persistent"] == (mode < 2)
    norms = [g.step()[2] for _ in range(nsteps)] + [g.advance(nsteps)[1]]
    states = [g.get_state(b) for b in range(1, len(case.blocks) + 1)]
    g.close()
    return t, states, norms


def _compare(monkeypatch, case, least_tiles):
    monkeypatch.setenv("MOSE_TILE_SHAPE", "0")
    monkeypatch.setenv("MOSE_KCHUNK", "1")
    monkeypatch.setenv("MOSE_TILE_XCD", "0")      # restored after the test
    for xcd in (0, 1):
        t, a, na = _march(case, xcd, 2)
        n = _tiles(case, t["tile"], 1)
        assert n >= least_tiles, n
        _, b, nb = _march(case, xcd + 2, 2)
        for x, y in zip(a, b):
            assert np.array_equal(x.view(np.uint64), y.view(np.uint64))
        assert np.array_equal(na, nb)


@pytest.mark.parametrize("prec", PRECS)
def test_many_more_tiles_than_workgroups(monkeypatch, prec):
    """Uneven blocks; more tiles than any occupancy of 256 threads a workgroup allows (2048 threads on each of 256
    CUs)."""
    case = perturb(cases.multiblock_chain(nblocks=12, seed=21, lo=30, hi=70, precision=prec), amp=0.01, seed=1)
    _compare(monkeypatch, case, 8 * 256 + 1)


# one j tile a plane and block: 32 x 8 m x nk cells are m nk tiles of 32 x 8 x 1
@pytest.mark.parametrize("m,nk", [(8, 65), (7, 75), (8, 97), (7, 111), (8, 129), (9, 115)])
@pytest.mark.parametrize("prec", PRECS)
def test_just_more_tiles_than_workgroups(monkeypatch, prec, m, nk):
    """520 to 1035 tiles, some no multiple of the eight queues: a few above two, three or four workgroups on each of
    256 CUs."""
    case = perturb(cases.vortex(dims=(32, 8 * m, nk), cfl=0.4, precision=prec), amp=0.01, seed=2)
    _compare(monkeypatch, case, m * nk)
