"""The fused Euler tile on the host, beside test_fused_tile.py: folded and chained updates for every table on
periodic boxes (one smaller than a tile and ragged, one of uniform geometry), and the states of the limiter
that is unstable at the amplitudes used there."""
import numpy as np
import pytest

import pyemu
import pyoracle as po
from conftest import rel_err
from test_fused_tile import TOL, _box
from test_hostemu_parity import _ogrid


@pytest.fixture(autouse=True)
def restore():
    yield
    pyemu.set_fused(0)
    pyemu.set_fold(0)
    pyemu.set_tile_config(0)
    pyemu.set_uniform_geometry(0)


def _with_table(args, rk):
    from hyperboliconvergence_amd import cases
    n, a, b = cases.rk_table({11: "ssp11", 33: "ssp33", 34: "ssp34", 44: "rk4"}[rk])
    cs = args[0]
    cs.nstages, cs.dt_mode, cs.cfl = n, po.DT_GLOBAL, 0.4
    for s in range(6):
        cs.beta[s] = b[s]
        for k in range(6):
            cs.alpha[s][k] = a[s, k]
    return args


@pytest.mark.parametrize("rk", [11, 33, 34, 44])
@pytest.mark.parametrize("mode", [0, 1], ids=["ordered", "fused"])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("size,uniform", [((5, 21), 0), ((32, 64), 1)], ids=["ragged", "uniform"])
def test_folded_and_chained_updates_on_boxes(rk, mode, precision, size, uniform):
    args = _with_table(_box(*size, po.FLUX_AUSMPUP, False), rk)
    assert args[0].nstages == {11: 1, 33: 3, 34: 4, 44: 4}[rk]
    out = []
    for fold in (0, 1):
        pyemu.set_fused(mode)
        pyemu.set_fold(fold)
        pyemu.set_uniform_geometry(uniform)
        out.append(pyemu.integrate(*args, 4, precision))
        assert pyemu.set_uniform_geometry(uniform) == bool(uniform)
    assert out[0][2] == out[1][2] == 0
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]


@pytest.mark.parametrize("shape", range(3))
def test_states_of_the_unlimited_slopes(shape):
    cs, nodes, q, bref = _ogrid(9, 20, 1, po.FLUX_ROE_FACEFRAME, po.LIM_NOLIMIT2, perturb=1e-3)
    cs.cfl = 0.1
    qo, to, _ = po.integrate(cs, nodes, q, 3, bref)
    assert np.isfinite(qo).all()
    pyemu.set_fused(1)
    pyemu.set_tile_config(shape)
    qe, te, st = pyemu.integrate(cs, nodes, q, bref, 3)
    assert st == 0 and rel_err(qe, qo) <= TOL and te == to
