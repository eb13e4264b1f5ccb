"""GPU: the device memory of a context, per cell, is that of the arrays its precision reads (a context of
2048x1024 cells against the sum of its arrays), and a context whose precision is switched holds and gives
what one built in that precision does."""
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NI, NJ = 2048, 1024
SLOTS = 2 * 14 * 8          # FP64 face slots, both directions
FP32 = 2 * 14 * 4           # their FP32 copies: mixed contexts
WEIGHTS = 2 * 5 * 8         # weight planes of the fused tile: FP64 contexts that run it
# cell volume and centre, three states, one accumulator of classical RK4, deferred residual, spectral
# radius, stored residual
REST = 8 * (3 + 3 * 4 + 4 + 4 + 1 + 5)


def _free():
    import torch
    gc.collect()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return torch.cuda.mem_get_info(0)[0]


def _cfg(flux, ni, nj, box=False):
    from hyperboliconvergence_amd import cases
    cfg = cases.config_cylinder_ogrid(nth=64, nr=40) if box else cases.config_cylinder_ogrid(nth=nj, nr=ni)
    cfg["case"].flux = flux
    if box:   # the same case on a box, periodic along j
        cfg["nodes"] = cases.mesh_linspace(ni, nj, 0.0, 1.0, 0.0, 3.0)
        cfg["case"].period_j[0], cfg["case"].period_j[1] = 0.0, 3.0
        cfg["bref"] = np.broadcast_to(cfg["bref"][0], (2 * ni + 2 * nj, 4)).copy()
    return cfg


def _context(cfg, precision):
    import hyperboliconvergence_amd as hca
    ctx = hca.Context(0)
    ctx.set_precision(precision)
    ctx.set_mesh(cfg["nodes"])
    ctx.set_case(cfg["case"])
    ctx.set_boundary_refs(cfg["bref"])
    return ctx


def test_bytes_per_cell():
    import hyperboliconvergence_amd as hca
    N = NI * NJ
    fused, ordered = _cfg(hca.FLUX_ROE_FACEFRAME, NI, NJ, True), _cfg(hca.FLUX_ROE, NI, NJ, True)
    FP64, MIXED = hca.PRECISION_FP64, hca.PRECISION_MIXED
    with _context(_cfg(hca.FLUX_ROE, 8, 16), FP64):   # the library and its kernels are loaded
        pass
    for cfg, first, then, slots in ((fused, FP64, FP64, WEIGHTS), (fused, MIXED, MIXED, FP32), (ordered, FP64, FP64, 0),
                                    (fused, FP64, MIXED, FP32), (fused, MIXED, FP64, WEIGHTS), (ordered, MIXED, FP64, 0)):
        before = _free()
        with _context(cfg, first) as ctx:
            if then != first:
                ctx.set_precision(then)
            used = (before - _free()) / N
        # beside the arrays: a row of faces more than cells, the tables of tiles and chunks, and each of some
        # 30 allocations rounded up to 2 MiB, 1 B a cell; the precisions' slots differ by 80 and 112 B
        assert 0 <= used - (SLOTS + slots + REST) <= 30, (first, then, used, SLOTS + slots + REST)


@pytest.mark.parametrize("first,then", [(0, 1), (1, 0)], ids=["to-mixed", "to-fp64"])
def test_switched_precision_gives_the_bits_of_a_new_context(first, then):
    import hyperboliconvergence_amd as hca
    cfg = _cfg(hca.FLUX_ROE_FACEFRAME, 40, 64)
    rng = np.random.default_rng(5)
    q = cfg["q"] * (1.0 + 0.01 * rng.standard_normal(cfg["q"].shape))
    out = []
    for switch in (True, False):
        with _context(cfg, first if switch else then) as ctx:
            ctx.set_state(q)
            if switch:
                ctx.step(2)
                for p in (then, first, then):
                    ctx.set_precision(p)
                ctx.set_state(q)
            ctx.set_tiles(0)
            out.append((ctx.residual(), ctx.step(5), ctx.get_state()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][2], out[1][2])


def test_second_residual_buffer_of_chained_steps():
    """One-stage tables with a global step: FP64 contexts hold a second deferred residual, mixed ones do not."""
    import hyperboliconvergence_amd as hca
    from test_gpu_chained import _table
    N, rest = NI * NJ, REST - 8 * 4   # no accumulator
    cfg = _table(_cfg(hca.FLUX_ROE_FACEFRAME, NI, NJ, True), "ssp11")
    FP64, MIXED = hca.PRECISION_FP64, hca.PRECISION_MIXED
    with _context(_cfg(hca.FLUX_ROE, 8, 16), FP64):
        pass
    for first, then, extra in ((FP64, FP64, WEIGHTS + 8 * 4), (MIXED, MIXED, FP32), (FP64, MIXED, FP32),
                               (MIXED, FP64, WEIGHTS + 8 * 4)):
        before = _free()
        with _context(cfg, first) as ctx:
            if then != first:
                ctx.set_precision(then)
            used = (before - _free()) / N
        assert 0 <= used - (SLOTS + extra + rest) <= 30, (first, then, used, SLOTS + extra + rest)


@pytest.mark.parametrize("first,then", [(0, 1), (1, 0)], ids=["to-mixed", "to-fp64"])
def test_no_room_for_the_other_precision(first, then):
    """The device is filled but for some 200 MB, less than either precision's slots of 2048x2048 cells: the switch is
    refused, and the context steps on as one that never tried."""
    import torch
    import hyperboliconvergence_amd as hca
    cfg = _cfg(hca.FLUX_ROE_FACEFRAME, 2 * NJ, NI, True)
    q = np.broadcast_to(cfg["bref"][0], (2 * NJ, NI, 4))
    q = q * (1.0 + 0.01 * np.random.default_rng(7).standard_normal(q.shape))
    out = []
    for refused in (True, False):
        with _context(cfg, first) as ctx:
            ctx.set_tiles(0)
            ctx.set_state(q)
            ctx.step(1)
            if refused:
                # the free memory that is reported is not all there is: block by block to the end
                filler = [torch.empty(_free() - 2**30, dtype=torch.uint8, device="cuda")]
                try:
                    for _ in range(100):
                        filler.append(torch.empty(64 * 2**20, dtype=torch.uint8, device="cuda"))
                except torch.OutOfMemoryError:
                    pass
                del filler[-3:]
                _free()
                with pytest.raises(hca.HCError):
                    ctx.set_precision(then)
                del filler
                _free()
            ctx.step(2)
            assert ctx.status() == 0
            out.append((ctx.get_state(), ctx.residual()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
