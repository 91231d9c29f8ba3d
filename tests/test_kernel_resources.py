"""Registers and scratch of the built kernels whose speed on large grids hangs
on the wavefronts that fit a SIMD: 512 vector registers in units of eight, 800
scalar registers in units of sixteen, 160 KB of LDS per four SIMDs in units of
1280 bytes."""
import pytest

from mbsolve_amd import capi, isa_check


@pytest.fixture(scope="module")
def kernels():
    return isa_check.resources(capi.LIB_PATH)


def _tile(algo, cells, storage="d", red=0):
    return "_ZN3mbh11tile_kernelINS_%sELi%dE%sLb%dEEEvNS_5KArgsE" % (
        algo, cells, storage, red)


NOOP, CAYLEY, BLOCH = "9algo_noop", "11algo_cayleyILi%dEE", \
    "13algo_bloch2_tILi0EE"


@pytest.mark.parametrize("name,waves,scratch", [
    (_tile(NOOP, 1), 8, 0), (_tile(NOOP, 1, red=1), 8, 0),
    (_tile("14algo_noop_fast", 1, "f"), 8, 0), (_tile("13algo_noop_hz0", 1, "f"),
                                            8, 0),
    (_tile("13algo_noop_hz0", 2, "f"), 8, 0),
    (_tile(NOOP, 2), 8, 0), (_tile(NOOP, 4), 5, 0), (_tile(NOOP, 8), 3, 0),
    (_tile(NOOP, 4, red=1), 5, 0),
    (_tile(CAYLEY % 2, 1), 4, 0), (_tile(CAYLEY % 2, 4), 2, 48),
    (_tile(CAYLEY % 2, 1, red=1), 4, 0),
    (_tile(CAYLEY % 3, 1), 2, 0), (_tile(CAYLEY % 3, 1, "f"), 2, 0),
    (_tile(BLOCH, 4), 3, 36), (_tile(BLOCH, 4, "f"), 3, 36),
])
def test_wavefronts_fit(kernels, name, waves, scratch):
    k = kernels[name]
    assert 512 // (-(-k["vgpr"] // 8) * 8) >= waves, k
    assert 800 // (-(-k["sgpr"] // 16) * 16) >= waves, k
    # one wavefront per workgroup
    assert 163840 // (-(-k["lds"] // 1280) * 1280) >= 4 * waves, k
    assert k["scratch"] <= scratch, k
