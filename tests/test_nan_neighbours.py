"""Faces beside a cell whose state is not finite: the biased slope there is NaN or infinite, and the limiter
gives what the oracle's gives.  Where a run has diverged in one cell the others keep the oracle's values."""
import numpy as np
import pytest

import pyemu
import pyoracle as po
from test_hostemu_parity import _ogrid


@pytest.fixture(autouse=True)
def restore():
    yield
    pyemu.set_fused(0)
    pyemu.set_tile_config(0)


def _case(flux, limiter, bad, amplitude=0.02):
    cs, nodes, q, bref = _ogrid(9, 20, 1, flux, limiter, perturb=amplitude)
    q[4, 7, 0] = bad
    return cs, nodes, q, bref


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf], ids=str)
@pytest.mark.parametrize("limiter", range(10))
@pytest.mark.parametrize("flux", [po.FLUX_ROE, po.FLUX_SLAU])
def test_ordered_tiles_give_the_oracles_bits(flux, limiter, bad):
    case = _case(flux, limiter, bad)
    ro = po.residual(*case)
    for shape in range(3):
        pyemu.set_tile_config(shape)
        assert np.array_equal(pyemu.residual(*case)[0], ro, equal_nan=True), shape


@pytest.mark.parametrize("limiter", [po.LIM_MINMOD2, po.LIM_VANALBADA2, po.LIM_SUPERBEE2, po.LIM_MC2, po.LIM_CADA3,
                                     po.LIM_SMOOTHVANALBADA])
@pytest.mark.parametrize("flux", [0, 1, 4, 5, 6])
def test_fused_tiles_beside_a_nan_cell(flux, limiter):
    """The residuals that are finite in the oracle, to rounding (1e-12 of the largest, as in
    test_fused_tile.py), and no others."""
    case = _case(flux, limiter, np.nan)
    ro = po.residual(*case)[..., :4]
    finite = np.isfinite(ro)
    assert not finite.all()
    pyemu.set_fused(1)
    for shape in range(3):
        pyemu.set_tile_config(shape)
        r = pyemu.residual(*case)[0][..., :4]
        assert np.array_equal(np.isfinite(r), finite)
        assert np.max(np.abs(r - ro)[finite]) <= 1e-12 * np.max(np.abs(ro[finite]))
