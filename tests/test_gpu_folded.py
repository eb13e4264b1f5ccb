"""GPU: the updates that a stage kernel forms while it loads its tiles (the stage-0 update of tables of three
and more stages, the chained steps of one-stage tables) against the update kernel, where both can be run.

A two-stage table runs the update kernel.  The three-stage table that repeats its second row and adds nothing
of the third stage ends in the same state, operation for operation (the accumulator receives 1/2 R0, then
1/2 R1, then 0 R2), but folds its stage-0 update, so the two states compare the two updates.  Chained steps
compare with single ones on boxes whose spacing is exact in binary: the uniform-geometry variant.  (Mixed
one-stage contexts do not chain; their rows of test_gpu_chained.py compare unchained runs.)"""
import numpy as np
import pytest

import pyoracle as po
from conftest import rel_err
from test_gpu_batch import _batch, _cyl, _single
from test_gpu_chained import _table

pytestmark = pytest.mark.gpu


def _box(ni, nj, flux, limiter=None):
    from hyperboliconvergence_amd import cases
    cfg = cases.config_isentropic_vortex(ni, flux=flux)
    if limiter is not None:
        cfg["case"].limiter = limiter
    nodes = cases.mesh_linspace(ni, nj, -10.0, 10.0, -10.0, 10.0)
    c = cases.cell_centres(nodes)
    cfg.update(nodes=nodes, q=cases.isentropic_vortex(c[..., 0], c[..., 1], beta=3.0),
               bref=np.ones((2 * ni + 2 * nj, 4)))
    return cfg


def _two_or_three(cfg, stages):
    import hyperboliconvergence_amd as hca
    cs = cfg["case"]
    cs.nstages, cs.dt_mode, cs.cfl = stages, hca.DT_GLOBAL, 0.4
    rows = [[1.0], [0.5, 0.5], [0.5, 0.5, 0.0]][:stages]
    for s in range(6):
        cs.beta[s] = 1.0 if s < stages else 0.0
        for k in range(6):
            cs.alpha[s][k] = rows[s][k] if s < stages and k < len(rows[s]) else 0.0
    return cfg


@pytest.mark.parametrize("flux", ["FLUX_ROE_FACEFRAME", "FLUX_SLAU", "FLUX_AUSMPUP"])
@pytest.mark.parametrize("grid", ["cylinder", "uniform"])
def test_folded_update_gives_the_update_kernels_bits_in_fp64(flux, grid):
    import hyperboliconvergence_amd as hca
    flux = getattr(hca, flux)
    for tiles in range(hca.NTILECFG):
        out = []
        for stages in (2, 3):
            cfg = _cyl(40, 21, 0.3, 2.0, flux=flux, perturb=0.005) if grid == "cylinder" else _box(32, 64, flux)
            with _single(_two_or_three(cfg, stages), tiles=tiles) as ctx:
                assert ctx.uniform_geometry() == (grid == "uniform")
                ctx.step(4)
                assert ctx.status() == 0
                out.append((ctx.get_state(), ctx.time()))
        assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1], tiles


@pytest.mark.parametrize("flux", ["FLUX_ROE_FACEFRAME", "FLUX_SLAU", "FLUX_AUSMPUP"])
def test_folded_update_of_mixed_contexts(flux):
    """Mixed objects are compiled with contraction, so the two updates may round differently in FP64; a
    difference of an FP64 rounding can flip the rounding of a face state to FP32, 2^-24 of it.  Over one step
    the states differ by at most (CFL 0.4) x (some 10 terms) x 2^-24 = 2.4e-7 of the largest."""
    import hyperboliconvergence_amd as hca
    for tiles in range(hca.NTILECFG):
        out = []
        for stages in (2, 3):
            cfg = _two_or_three(_cyl(40, 21, 0.3, 2.0, flux=getattr(hca, flux), perturb=0.005), stages)
            with _single(cfg, precision=1, tiles=tiles) as ctx:
                ctx.step(1)
                assert ctx.status() == 0
                out.append((ctx.get_state(), ctx.time()))
        d = rel_err(out[0][0], out[1][0])
        print(f"mixed folded against update kernel: {d:.2e}")
        assert d <= 2.4e-7 and out[0][1] == out[1][1], tiles


@pytest.mark.parametrize("flux", ["FLUX_RUSANOV", "FLUX_AUSMPUP", "FLUX_SLAU"])
def test_chained_steps_on_uniform_geometry(flux):
    import hyperboliconvergence_amd as hca
    cfgs = [_table(_box(n, m, getattr(hca, flux)), "ssp11") for n, m in ((16, 16), (32, 64))]
    out = {}
    for tiles in range(hca.NTILECFG):
        for uniform in (1, 0):
            for chunks, graph in (([1] * 9, 0), ([9], 0), ([2, 7], 4)):
                with _batch(cfgs) as b:
                    b.set_tiles(tiles)
                    b.set_graph_steps(graph)
                    b.set_uniform_geometry(uniform)
                    assert b.uniform_geometry() == bool(uniform)
                    for n in chunks:
                        b.step(n)
                    assert b.status() == 0
                    out[tiles, uniform, graph, len(chunks)] = [b.get_case_state(k) for k in range(2)] + [
                        b.case_time(k) for k in range(2)]
    first = next(iter(out.values()))
    for key, other in out.items():
        assert all(np.array_equal(x, y) for x, y in zip(first, other)), key


@pytest.mark.parametrize("flux", range(7))
def test_van_leer_runs_the_ordered_tile(flux):
    """Contexts with van Leer's ratio keep the reference's order in every flux: the oracle's bits on a periodic
    box (no pow), whose spacing is not exact, in every tile shape."""
    cfg = _box(24, 33, flux, po.LIM_VANLEER2)
    ro = po.residual(cfg["case"], cfg["nodes"], cfg["q"], cfg["bref"])
    qo, _, _ = po.integrate(cfg["case"], cfg["nodes"], cfg["q"], 2, cfg["bref"])
    for tiles in range(3):
        with _single(cfg, tiles=tiles) as ctx:
            assert np.array_equal(ctx.residual(), ro, equal_nan=True)
            ctx.step(2)
            assert np.array_equal(ctx.get_state(), qo, equal_nan=True)
