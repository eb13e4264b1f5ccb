"""The fused Euler tile and the folded and chained updates (host execution of the kernels' phases) under
AddressSanitizer and UndefinedBehaviorSanitizer: the smallest mesh, ragged ones, every boundary kind, both
offset widths, uniform geometry, chained one-stage and folded longer tables.  Every access stays inside its
buffer, and the sanitized build gives the ordinary one's bits."""
import numpy as np
import pytest

import pyemu
import pyoracle as po
from test_fused_tile import FLUXES, _box
from test_hostemu_parity import _ogrid
from test_hostemu_sanitized import _run, driver  # noqa: F401  (the fixture that builds the program)


def _check(driver, tmp_path, case, fused=(1, 2), uniform=0, fold=0, nsteps=3, precision=0):
    cs, nodes, q, bref = case
    for tiles in range(3):
        for mode in fused:
            res, qs, tail = _run(driver, tmp_path, cs, nodes, q, bref, precision, nsteps,
                                 tiles + 16 * uniform + 32 * mode + 128 * fold)
            pyemu.set_tile_config(tiles)
            pyemu.set_uniform_geometry(uniform)
            pyemu.set_fused(mode)
            pyemu.set_fold(fold)
            try:
                r_ref, _ = pyemu.residual(cs, nodes, q, bref, precision)
                q_ref, t_ref, st_ref = pyemu.integrate(cs, nodes, q, bref, nsteps, precision)
                assert pyemu.set_uniform_geometry(0) == bool(uniform)
            finally:
                pyemu.set_tile_config(0)
                pyemu.set_uniform_geometry(0)
                pyemu.set_fused(0)
                pyemu.set_fold(0)
            assert np.array_equal(res, r_ref.ravel()) and np.array_equal(qs, q_ref.ravel())
            assert tail[0] == t_ref and tail[1] == st_ref == 0


@pytest.mark.parametrize("flux", FLUXES)
@pytest.mark.parametrize("shape", [(3, 3), (8, 17), (16, 33)], ids=str)
def test_periodic_ring(driver, tmp_path, flux, shape):   # noqa: F811
    _check(driver, tmp_path, _ogrid(*shape, 1, flux, po.LIM_MINMOD2))


@pytest.mark.parametrize("walls", [False, True], ids=["periodic", "walls"])
@pytest.mark.parametrize("size", [(3, 3), (19, 23)], ids=str)
def test_boxes(driver, tmp_path, walls, size):   # noqa: F811
    _check(driver, tmp_path, _box(*size, po.FLUX_AUSMPUP, walls))


@pytest.mark.parametrize("bc", [(po.BC_FIXED, po.BC_ENTROPY, 0, 0), (po.BC_RIEMANN, po.BC_WALL, 0, 0)], ids=str)
@pytest.mark.parametrize("basis", [0, 1])
def test_boundary_kinds(driver, tmp_path, bc, basis):   # noqa: F811
    _check(driver, tmp_path, _ogrid(10, 18, basis, po.FLUX_ROE_FACEFRAME, po.LIM_VANALBADA2, bc=bc))


def test_uniform_geometry(driver, tmp_path):   # noqa: F811
    _check(driver, tmp_path, _box(32, 64, po.FLUX_AUSMPUP, False), fused=(1,), uniform=1)
    _check(driver, tmp_path, _box(32, 64, po.FLUX_AUSMPUP, False), fused=(1,), uniform=1, fold=1)


@pytest.mark.parametrize("rk", [11, 33, 44])
@pytest.mark.parametrize("mode,precision", [(0, 0), (0, 1), (1, 0), (2, 0)], ids=["ordered", "mixed", "fused", "wide"])
def test_folded_and_chained_updates(driver, tmp_path, rk, mode, precision):   # noqa: F811
    _check(driver, tmp_path, _ogrid(10, 18, 1, po.FLUX_AUSMPUP, po.LIM_MINMOD2, dt=po.DT_GLOBAL, rk=rk), fused=(mode,),
           fold=1, precision=precision)
