"""GPU: chained one-stage steps (each residual kernel forms the update of the step before it) against the
kernels of single steps, bit for bit: general and uniform geometry, every tile shape, a batch of meshes of
which one is smaller than a tile, graphs of an even number of steps and remainders.  And the folded
stage-0 update of longer tables: the same bits in every tile shape."""
import numpy as np
import pytest

from test_gpu_batch import _batch, _cyl

pytestmark = pytest.mark.gpu


def _table(cfg, rk):
    from hyperboliconvergence_amd import cases
    import hyperboliconvergence_amd as hca
    n, a, b = cases.rk_table(rk)
    cs = cfg["case"]
    cs.nstages, cs.dt_mode, cs.cfl = n, hca.DT_GLOBAL, 0.4
    for s in range(6):
        cs.beta[s] = b[s]
        for k in range(6):
            cs.alpha[s][k] = a[s, k]
    return cfg


def _boxes(flux):
    from hyperboliconvergence_amd import cases
    out = []
    for ni, nj in ((6, 5), (48, 40)):
        cfg = cases.config_isentropic_vortex(ni, flux=flux)
        nodes = cases.mesh_linspace(ni, nj, -10.0, 10.0, -10.0, 10.0)
        c = cases.cell_centres(nodes)
        cfg.update(nodes=nodes, q=cases.isentropic_vortex(c[..., 0], c[..., 1], beta=3.0),
                   bref=np.ones((2 * ni + 2 * nj, 4)))
        out.append(cfg)
    return out


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind", ["cylinder", "boxes", "ordered"])
def test_chained_steps_give_the_bits_of_single_steps(kind, precision):
    import hyperboliconvergence_amd as hca
    if kind == "boxes":
        cfgs = _boxes(hca.FLUX_AUSMPUP)
    else:
        flux = hca.FLUX_SLAU if kind == "ordered" else hca.FLUX_AUSMPUP
        cfgs = [_cyl(n, m, 0.3, 2.0, flux=flux, perturb=0.005, seed=n) for n, m in ((40, 21), (64, 32))]
    cfgs = [_table(c, "ssp11") for c in cfgs]
    for tiles in range(hca.NTILECFG):
        out = []
        for chunks, graph in (([1] * 9, 0), ([9], 0), ([2, 7], 4)):
            with _batch(cfgs, precision) as b:
                b.set_tiles(tiles)
                b.set_graph_steps(graph)
                for n in chunks:
                    b.step(n)
                assert b.status() == 0
                out.append([b.get_case_state(k) for k in range(len(cfgs))] + [b.case_time(k) for k in range(len(cfgs))])
        for other in out[1:]:
            assert all(np.array_equal(x, y) for x, y in zip(out[0], other)), tiles


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("rk", ["ssp33", "rk4"])
def test_folded_updates_give_the_same_bits_in_every_tile_shape(rk, precision):
    import hyperboliconvergence_amd as hca
    for flux in (hca.FLUX_ROE_FACEFRAME, hca.FLUX_AUSMPUP, hca.FLUX_SLAU):
        cfgs = [_table(_cyl(n, m, 0.3, 2.0, flux=flux, perturb=0.005, seed=n), rk) for n, m in ((40, 21), (64, 32))]
        out = []
        for tiles in range(hca.NTILECFG):
            with _batch(cfgs, precision) as b:
                b.set_tiles(tiles)
                b.step(5)
                assert b.status() == 0
                out.append([b.get_case_state(k) for k in range(len(cfgs))])
        for other in out[1:]:
            assert all(np.array_equal(x, y) for x, y in zip(out[0], other)), flux
