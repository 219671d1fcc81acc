"""The autotuner never leaves a layout with a slower tiling than it had."""
import pytest

from mose_amd import abi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [
    lambda: cases.vortex(dims=(33, 25, 17), cfl=0.4),
    lambda: cases.vortex(dims=(33, 25, 17), cfl=0.4, precision=abi.PREC_FP32_FLUX),
    lambda: cases.multiblock_chain(nblocks=4, seed=3, lo=12, hi=40, precision=abi.PREC_FP64),
], ids=["box_fp64", "box_fp32", "chain_fp64"])
def test_a_faster_tiling_in_use_stays(case):
    """Layouts whose default of one or two planes a chunk takes less than half the time of the tuner's shortest chunks
    (a plane is a serial step of some 6 us: 17-plane boxes take three such chains of 8)."""
    from mose_amd.lib import GpuSolver
    g = GpuSolver(case())
    before = g.tiling()
    assert before["kchunk"] < 8
    choice, ms = g.autotune(3)
    assert choice["kchunk"] in (8, 16, 32, 64) and ms > 0
    assert g.tiling() == before
    g.advance(2)
    g.close()
