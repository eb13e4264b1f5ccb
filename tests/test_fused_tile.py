"""The fused Euler tile (hc_fused.hpp, hc_fused_flux.hpp) executed on the host against the oracle.

It evaluates the same scheme in other operations, so results agree to rounding and not bit for bit:
the residual within 1e-12 of its largest value (a face flux is some 10^2 operations of 1.1e-16 on
terms up to 10^2 times their sum), a few steps' state within 1e-12.  Every tile shape, offset width and
the uniform-geometry variant give the same bits, since every fused operation is explicit.
"""
import numpy as np
import pytest

import pyemu
import pyoracle as po
from conftest import rel_err
from test_hostemu_parity import _ogrid

TOL = 1e-12
FLUXES = (0, 1, 4, 5, 6)   # Roe and SLAU keep the reference's order on the GPU (fused_euler)


@pytest.fixture(autouse=True)
def fused():
    pyemu.set_fused(1)
    yield
    pyemu.set_fused(0)
    pyemu.set_tile_config(0)
    pyemu.set_uniform_geometry(0)


def _check(cs, nodes, q, bref, nsteps=3):
    ro = po.residual(cs, nodes, q, bref)
    qo, to, _ = po.integrate(cs, nodes, q, nsteps, bref)
    first = None
    for shape in range(3):
        for width in (1, 2):
            pyemu.set_tile_config(shape)
            pyemu.set_fused(width)
            r, _ = pyemu.residual(cs, nodes, q, bref)
            qe, te, st = pyemu.integrate(cs, nodes, q, bref, nsteps)
            for v in range(5):
                assert np.max(np.abs(r[..., v] - ro[..., v])) <= TOL * np.max(np.abs(ro[..., :4] if v < 4 else ro[..., v]))
            if not np.isfinite(qo).all():   # an unstable limiter on this noise: only the residual compares
                qe = te = None
            else:
                assert st == 0 and rel_err(qe, qo) <= TOL and abs(te - to) <= 1e-13 * abs(to)
            if first is None:
                first = r, qe, te
            assert np.array_equal(r, first[0]) and np.array_equal(qe, first[1]) and te == first[2], (shape, width)


@pytest.mark.parametrize("flux", FLUXES)
@pytest.mark.parametrize("basis", [0, 1])
@pytest.mark.parametrize("shape", [(3, 5), (7, 16), (13, 37), (16, 17), (31, 33)], ids=str)
def test_fluxes_and_tile_edges(flux, basis, shape):
    _check(*_ogrid(*shape, basis, flux, po.LIM_MINMOD2))


# van Leer's bare ratio is not homogeneous in the slopes: contexts with it keep the ordered kernels
@pytest.mark.parametrize("limiter", [k for k in range(10) if k != po.LIM_VANLEER2])
def test_limiters(limiter):
    _check(*_ogrid(9, 20, 1, po.FLUX_ROE_FACEFRAME, limiter))


@pytest.mark.parametrize("bc,dt,rk", [((po.BC_FIXED, po.BC_ENTROPY, 0, 0), po.DT_GLOBAL, 11),
                                      ((po.BC_RIEMANN, po.BC_WALL, 0, 0), po.DT_GLOBAL, 33),
                                      ((po.BC_WALL, po.BC_FIXED, 0, 0), po.DT_LOCAL, 22),
                                      ((po.BC_ENTROPY, po.BC_RIEMANN, 0, 0), po.DT_GLOBAL, 44),
                                      ((po.BC_FIXED, po.BC_WALL, 0, 0), po.DT_LOCAL, 34)], ids=str)
def test_boundaries_time_steps_and_tables(bc, dt, rk):
    _check(*_ogrid(10, 18, 1, po.FLUX_AUSMPUP, po.LIM_SMOOTHVANALBADA, bc=bc, dt=dt, rk=rk))


def _box(ni, nj, flux, walls):
    from hyperboliconvergence_amd import cases
    import hyperboliconvergence_amd as hca
    cfg = cases.config_isentropic_vortex(ni, flux=flux)
    nodes = cases.mesh_linspace(ni, nj, -10.0, 10.0, -10.0, 10.0)
    c = cases.cell_centres(nodes)
    cs = cfg["case"]
    if walls:
        for k in range(4):
            cs.bc[k] = hca.BC_WALL
    return cs, nodes, cases.isentropic_vortex(c[..., 0], c[..., 1], beta=3.0), np.ones((2 * ni + 2 * nj, 4))


@pytest.mark.parametrize("flux", [po.FLUX_RUSANOV, po.FLUX_AUSMPUP])
@pytest.mark.parametrize("walls", [False, True], ids=["periodic", "walls"])
@pytest.mark.parametrize("size", [(3, 3), (4, 33), (19, 23)], ids=str)
def test_boxes(flux, walls, size):
    """Periodic in both directions, smaller than the halo of a tile and ragged; walls on all four sides."""
    _check(*_box(*size, flux, walls))


@pytest.mark.parametrize("flux", FLUXES)
def test_uniform_geometry_gives_the_general_tiles_bits(flux):
    cs, nodes, q, bref = _box(32, 64, flux, False)   # spacings exact in binary
    general = pyemu.residual(cs, nodes, q, bref)[0]
    steps = pyemu.integrate(cs, nodes, q, bref, 2)
    for shape in range(3):
        pyemu.set_tile_config(shape)
        pyemu.set_uniform_geometry(1)
        assert np.array_equal(pyemu.residual(cs, nodes, q, bref)[0], general)
        assert pyemu.set_uniform_geometry(1)
        assert np.array_equal(pyemu.integrate(cs, nodes, q, bref, 2)[0], steps[0])


@pytest.mark.parametrize("rk", [11, 33, 34, 44])
@pytest.mark.parametrize("mode", [0, 1], ids=["ordered", "fused"])
@pytest.mark.parametrize("precision", [0, 1])
def test_folded_updates_give_the_update_kernels_bits(rk, mode, precision):
    for flux, box in ((po.FLUX_AUSMPUP, True), (po.FLUX_ROE_FACEFRAME, False)):
        args = _box(5, 21, flux, False) if box else _ogrid(10, 18, 1, flux, po.LIM_MINMOD2, dt=po.DT_GLOBAL, rk=rk)
        out = []
        for fold in (0, 1):
            pyemu.set_fused(mode)
            pyemu.set_fold(fold)
            out.append(pyemu.integrate(*args, 4, precision))
        pyemu.set_fold(0)
        assert out[0][2] == out[1][2] == 0
        assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("flux", [po.FLUX_ROE_FACEFRAME, po.FLUX_SLAU])
def test_ordered_tiles_inside_the_mesh(flux, precision):
    """Tiles away from every side take their metric without the side tests, in the same order: the oracle's
    bits in FP64, and in both precisions the bits of shapes whose tiles lie elsewhere."""
    cs, nodes, q, bref = _ogrid(26, 70, 1, flux, po.LIM_MINMOD2)
    pyemu.set_fused(0)
    out = []
    for shape in range(3):
        pyemu.set_tile_config(shape)
        out.append(pyemu.residual(cs, nodes, q, bref, precision)[0])
        assert np.array_equal(out[-1], out[0])
    if precision == 0:
        assert np.array_equal(out[0], po.residual(cs, nodes, q, bref))
