"""Time marching launches the levels that step together at once; the substep entry points launch
one level at a time in the reference's order.  Both give the same bits."""
import numpy as np
import pytest

from zllbm_amd import grid as g
from zllbm_amd import hip
from tests import scenarios as sc

pytestmark = pytest.mark.gpu


def _nested(levels):
    """2D box with `levels` nested levels around its middle (16 cells of each level's spacing)."""
    boxes, c = [], 13
    for _ in range(levels - 1):
        boxes.append(((c - 4, c - 4), (c + 4, c + 4)))
        c *= 2
    return g.refined_box_grid(2, (24, 24), boxes)


def _reference_order(s, top):
    count = [0] * (top + 1)

    def step(l):
        count[l] += 1
        s.step_level(l, count[l])
        if l > 0 and count[l] % 2 == 0:
            s.transfer_levels(l)
        if l < top:
            step(l + 1)
            step(l + 1)
    step(0)


# 8 levels: more than one launch takes
@pytest.mark.parametrize("levels,graphs", [(2, True), (3, True), (4, True), (8, False)])
@pytest.mark.parametrize("precision,collision", [(hip.FP64, (hip.MRT,)), (hip.FP32_SHIFTED, (hip.SRT, hip.SRT, hip.MRT)),
                                                 (hip.BF16_SHIFTED, (hip.MRT, hip.SRT))])
@pytest.mark.parametrize("scheme", [sc.PER, sc.BB, sc.NEE])
def test_marching_equals_substeps(levels, graphs, precision, collision, scheme):
    grid = _nested(levels)
    kw = dict(nu0=2e-3, bc=sc.all_bc(2, scheme), collision=collision, precision=precision)
    a, b = hip.Solver(grid, **kw).build(), hip.Solver(grid, **kw).build()
    a.graphs_enable(graphs)
    for l in range(levels):
        rho, u = sc.level_fields(grid, l, u0=0.02)
        for s in (a, b):
            s.init_macro(l, rho, u)
    a.time_marching(3)
    for _ in range(3):
        _reference_order(b, levels - 1)
    for l in range(levels):
        np.testing.assert_array_equal(a.f(l), b.f(l))
    a.time_marching(2)
    for _ in range(2):
        _reference_order(b, levels - 1)
    for l in range(levels):
        np.testing.assert_array_equal(a.f(l), b.f(l))


@pytest.mark.parametrize("les,precision", [(hip.LES_SMAGORINSKY, hip.FP32_SHIFTED), (hip.LES_MLP, hip.FP32_SHIFTED)])
def test_marching_equals_substeps_3d_forced(les, precision):
    """The learned closure's kernel with a resolved and an unresolved level in one launch, and
    immersed-boundary markers on the finer one."""
    import os
    from zllbm_amd import closure, geometry
    from tests.test_gpu_mlp import ROOT
    grid, kw = sc.amr3d()
    kw.update(collision=(hip.MRT,), les=les, cs=0.1, precision=precision, has_force=True)
    xyz, area = geometry.fibonacci_sphere_markers((8.5, 8.5, 8.5), 1.5, 0.5)
    runs = []
    for _ in range(2):
        s = hip.Solver(grid, **kw)
        s.set_ib(1, xyz, area, np.zeros_like(xyz))
        s.build()
        if les == hip.LES_MLP:
            s.mlp_set(closure.ClosureModel.load(os.path.join(ROOT, "zllbm_amd", "data", "closure_turbulence.npz")))
        for l in range(2):
            s.init_macro(l, *sc.level_fields(grid, l, u0=0.03))
        runs.append(s)
    runs[0].time_marching(4)
    for _ in range(4):
        _reference_order(runs[1], 1)
    for l in range(2):
        np.testing.assert_array_equal(runs[0].f(l), runs[1].f(l))
    np.testing.assert_array_equal(runs[0].ib_force(1), runs[1].ib_force(1))


@pytest.mark.parametrize("levels", [1, 2])
@pytest.mark.parametrize("graphs", [True, False])
def test_no_steps_without_a_closure(levels, graphs):
    """Marching no step asks for nothing: it succeeds before the learned closure is set, on one
    level and on several, and any step before that is refused."""
    grid = g.uniform_grid(3, (6, 6, 6)) if levels == 1 else sc.amr3d()[0]
    s = hip.Solver(grid, nu0=0.01, bc=sc.all_bc(3, sc.PER), collision=(hip.MRT,), les=hip.LES_MLP,
                   precision=hip.FP32_SHIFTED).build()
    s.graphs_enable(graphs)
    s.time_marching(0)
    with pytest.raises(RuntimeError, match="learned closure not set"):
        s.time_marching(1)
    s.time_marching(0)


# a single level with launches per face: replayed graphs below 32 MiB of populations, launches above
# (512 x 511 nodes of 9 FP64 values are 18 MiB, 705 x 706 are 35 with the padding of their bricks)
@pytest.mark.parametrize("cells", [(7, 9), (511, 510), (704, 705)])
def test_single_level_channel_as_graphs_and_launches(cells):
    grid = g.uniform_grid(2, cells)
    bc = {g.XMIN: (sc.NEE, (0.03, 0.)), g.XMAX: (sc.NEE, (0.03, 0.)), g.YMIN: (sc.BB, (0., 0.)), g.YMAX: (sc.BB, (0.02, 0.))}
    runs = []
    for graphs in (True, False):
        s = hip.Solver(grid, nu0=0.02, bc=bc, collision=(hip.MRT,)).build()
        s.graphs_enable(graphs)
        s.init_macro(0, *sc.level_fields(grid, 0, u0=0.02))
        runs.append(s)
    for n in (1, 2, 5, 4, 1, 3, 2):
        for s in runs:
            s.time_marching(n)
        np.testing.assert_array_equal(runs[0].f(0), runs[1].f(0))


def _every_substep_order(s, top):
    """The reference's order with time interpolation: an exchange after every substep."""
    count = [0] * (top + 1)

    def step(l):
        count[l] += 1
        s.step_level(l, count[l])
        if l > 0:
            s.transfer_levels(l)
        if l < top:
            step(l + 1)
            step(l + 1)
    step(0)


# the finest region keeps only the 3 cells to level 1's edge that it needs, so the exchange with level 2
# touches level-1 nodes that the exchange with level 1 touches
def _overlapping():
    return g.refined_mask_grid(2, (24, 24), 3, lambda k, c: np.ones(len(c), bool), margin=3, buffer=0)


@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("precision", [hip.FP64, hip.FP32_SHIFTED, hip.BF16_SHIFTED])
@pytest.mark.parametrize("time_interp", [False, True])
@pytest.mark.parametrize("scheme", [sc.BB, sc.PER])
@pytest.mark.parametrize("overlap", [True, False])
def test_exchanges_keep_the_reference_order(overlap, scheme, time_interp, precision, graphs):
    """Exchanges that share nodes, and (with time interpolation) several exchanges after one batch of
    steps, against one launch per level in the reference's order."""
    grid = _overlapping() if overlap else _nested(4)
    top = grid.max_level
    kw = dict(nu0=0.02, bc=sc.all_bc(2, scheme), collision=(hip.MRT,), precision=precision, time_interp=time_interp)
    a, b = hip.Solver(grid, **kw).build(), hip.Solver(grid, **kw).build()
    assert a.transfer_info(1)["overlaps_finer_transfer"] == overlap
    a.graphs_enable(graphs)
    for l in range(top + 1):
        rho, u = sc.level_fields(grid, l, 0.05, noise=1e-3)
        for s in (a, b):
            s.init_macro(l, rho, u)
    for n in (1, 3, 2):
        a.time_marching(n)
        for _ in range(n):
            (_every_substep_order if time_interp else _reference_order)(b, top)
        for l in range(top + 1):
            np.testing.assert_array_equal(a.f(l), b.f(l))
