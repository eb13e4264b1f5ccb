"""GPU: the fused Euler tile with 64-bit offsets, which a mesh of 2^24 cells along one side takes (32-bit
contexts multiply rows by widths in 24 bits): a strip of unit cells whose flow repeats, against a short box
with one period of it, bit for bit (the spacing is exact), whatever tile configuration is asked for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NI, PERIOD, LONG = 3, 4096, 1 << 24


def _run(nj, q):
    import hyperboliconvergence_amd as hca
    from hyperboliconvergence_amd import cases
    cs = cases.config_isentropic_vortex(16, hca.FLUX_AUSMPUP)["case"]
    cs.period_i[0], cs.period_i[1], cs.period_j[0], cs.period_j[1] = float(NI), 0.0, 0.0, float(nj)
    with hca.Context(0) as ctx:
        ctx.set_mesh(np.stack(np.meshgrid(np.arange(NI + 1.0), np.arange(nj + 1.0), indexing="ij"), -1))
        ctx.set_case(cs)
        ctx.set_uniform_geometry(0)
        ctx.set_boundary_refs(np.ones((2 * NI + 2 * nj, 4)))
        ctx.set_state(np.tile(q, (1, nj // PERIOD, 1)))
        for tiles in range(hca.NTILECFG):
            ctx.set_tiles(tiles)
            ctx.step(1)
        assert ctx.status() == 0
        return ctx.get_state(), ctx.time()


def test_strip_repeats_the_short_box():
    rng = np.random.default_rng(1)
    q = np.array([0.3, 0.1, 1.0, 1.0 / 1.4]) * (1.0 + 0.01 * rng.standard_normal((NI, PERIOD, 4)))
    short, t0 = _run(PERIOD, q)
    long, t1 = _run(LONG, q)
    assert t0 == t1
    assert all(np.array_equal(short, long[:, k:k + PERIOD]) for k in range(0, LONG, PERIOD))
