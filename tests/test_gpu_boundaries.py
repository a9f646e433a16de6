"""Bounce-back and periodic faces resolved in the pull, in every combination of faces, against the
oracle's face-by-face conditions; and the levels that stay with the launches per face (a
non-equilibrium-extrapolation face, a periodic twin whose own source is absent)."""
import itertools

import numpy as np
import pytest

from oracle.zlbm_oracle import Oracle
from zllbm_amd import grid as g
from zllbm_amd import hip
from tests import scenarios as sc
from tests.test_gpu_parity import assert_close

pytestmark = pytest.mark.gpu

PER, BB, NEE = g.BC_PERIODIC, g.BC_BOUNCE_BACK, g.BC_NEE
REST, LID = (0., 0., 0.), (0.03, 0.02, -0.01)
# the two faces of an axis
AXES = {"periodic": ((PER, REST), (PER, REST)), "walls": ((BB, REST), (BB, REST)), "lid": ((BB, REST), (BB, LID)),
        "lids": ((BB, LID), (BB, (-0.02, 0.01, 0.03))), "channel": ((NEE, (0.02, 0., 0.)), (NEE, (0.02, 0., 0.)))}


def _bc(names):
    return {1 + 2 * a + side: AXES[n][side] for a, n in enumerate(names) for side in (0, 1)}


def _random_state(n, dims, seed):
    rng = np.random.default_rng(seed)
    return 1.0 + 0.01 * rng.random(n), 0.02 * (rng.random((n, dims)) - 0.5)


def _compare(grid, names, steps, precision=hip.FP64, **kw):
    bc = _bc(names)
    o = Oracle(grid, nu0=0.05, bc=bc, **kw)
    s = hip.Solver(grid, nu0=0.05, bc=bc, precision=precision, **kw).build()
    for l, lev in enumerate(grid.levels):
        rho, u = _random_state(lev.n, grid.dims, l)
        o.init_macro(l, rho, u)
        s.init_macro(l, rho, u)
    for n in (1, steps - 1):          # a download in between takes the resolved pull too
        o.time_marching(n)
        s.time_marching(n)
        for l in range(len(grid.levels)):
            if precision == hip.FP64:
                assert_close(s.f(l), o.f(l))
            else:
                assert np.max(np.abs(s.f(l) - o.f(l))) < 2e-7
    return s


@pytest.mark.parametrize("names", list(itertools.product(["periodic", "walls", "lid", "lids", "channel"], repeat=2)))
def test_faces_2d(names):
    s = _compare(g.uniform_grid(2, (17, 9)), names, 30, collision=(hip.MRT,))
    boundary = "channel" in names
    assert (s.info(0)[1] > 0) == boundary      # resolved boundary nodes are bulk nodes


@pytest.mark.parametrize("names", list(itertools.product(["periodic", "walls", "lids"], repeat=3)))
def test_faces_3d(names):
    s = _compare(g.uniform_grid(3, (5, 8, 6)), names, 12, collision=(hip.SRT,))
    assert s.info(0)[1] == 0


@pytest.mark.parametrize("cells", [(1, 1), (1, 30), (7, 8), (8, 7), (16, 15)])
@pytest.mark.parametrize("names", [("periodic", "periodic"), ("lid", "periodic"), ("walls", "lid")])
def test_small_and_ragged_2d(cells, names):
    _compare(g.uniform_grid(2, cells), names, 10)


@pytest.mark.parametrize("cells", [62, 63, 64, 127, 128])
@pytest.mark.parametrize("names", [("channel", "walls"), ("walls", "channel"), ("channel", "periodic")])
def test_face_kernel_workgroups(cells, names):
    """Faces of one node less, as many and one more than one and two workgroups of 64 (a face of
    `cells` cells has cells + 1 nodes), in the launches per face."""
    _compare(g.uniform_grid(2, (cells, cells)), names, 10, collision=(hip.MRT,))


@pytest.mark.parametrize("precision", [hip.FP64, hip.FP32_SHIFTED])
@pytest.mark.parametrize("names", [("periodic", "periodic", "periodic"), ("walls", "periodic", "walls"),
                                   ("periodic", "lid", "walls")])
def test_les_3d(names, precision):
    _compare(g.uniform_grid(3, (4, 9, 3)), names, 10, precision=precision, collision=(hip.MRT,),
             les=hip.LES_SMAGORINSKY, cs=0.1)


@pytest.mark.parametrize("names", [("periodic", "periodic"), ("walls", "periodic"), ("lid", "walls"), ("channel", "walls")])
def test_holes_keep_their_values(names):
    """Nodes taken out at random: absent sources keep their populations, and periodic twins with
    an absent source of their own leave the level to the launches per face."""
    grid = g.uniform_grid(2, (21, 14))
    keep = np.random.default_rng(7).random(grid.levels[0].n) > 0.1
    lev = grid.levels[0]
    grid.levels[0] = g.Level(lev.keys[keep], lev.flags[keep])
    _compare(grid, names, 10)


@pytest.mark.parametrize("names", [("periodic", "periodic", "periodic"), ("walls", "walls", "walls"),
                                   ("channel", "walls", "walls")])
def test_refined_box_3d(names):
    """A refined level in the middle of a level with boundaries."""
    grid, _ = sc.amr3d()
    _compare(grid, names, 4, collision=(hip.MRT,), les=hip.LES_SMAGORINSKY, cs=0.1)


@pytest.mark.parametrize("axis", [0, 1])
def test_immersed_boundary_across_a_periodic_face(axis):
    """Supports of markers on a periodic plane are deferred nodes whose pull is resolved."""
    grid = g.uniform_grid(2, (20, 20))
    bc = _bc(("periodic", "periodic"))
    t = np.linspace(0, 2 * np.pi, 24, endpoint=False)
    c = np.array([11.3, 11.1])
    c[axis] = 1.2
    xy = c + 3.0 * np.stack([np.cos(t), np.sin(t)], 1)
    xy = 1.0 + (xy - 1.0) % 20.0
    area = np.full(24, 2 * np.pi * 3.0 / 24)
    kw = dict(nu0=0.05, bc=bc, has_force=True, collision=(hip.MRT,))
    o, s = Oracle(grid, **kw), hip.Solver(grid, **kw)
    o.set_ib(0, xy, area, np.zeros_like(xy))
    s.set_ib(0, xy, area, np.zeros_like(xy))
    s.build()
    rho, u = _random_state(grid.levels[0].n, 2, 5)
    o.init_macro(0, rho, u)
    s.init_macro(0, rho, u)
    o.time_marching(8)
    s.time_marching(8)
    assert_close(s.f(0), o.f(0), rtol=1e-8)


def test_learned_closure_walls():
    """The FP32 learned closure takes resting and periodic faces from the table and leaves moving
    walls to the launches per face: both against the FP64 solver of the same closure."""
    from tests.test_gpu_mlp import ROOT
    import os
    from zllbm_amd import closure
    model = closure.ClosureModel.load(os.path.join(ROOT, "zllbm_amd", "data", "closure_turbulence.npz"))
    grid = g.uniform_grid(3, (9, 10, 7))
    for names in (("periodic", "walls", "periodic"), ("walls", "walls", "walls"), ("periodic", "lid", "walls")):
        out = []
        for precision in (hip.FP32_SHIFTED, hip.FP64):
            s = hip.Solver(grid, nu0=0.01, bc=_bc(names), precision=precision, collision=(hip.MRT,), les=hip.LES_MLP,
                           cs=0.1, mlp_operands=hip.MLP_OPERANDS_FP16).build()
            s.mlp_set(model)
            rho, u = _random_state(grid.levels[0].n, 3, 2)
            s.init_macro(0, rho, u)
            s.time_marching(11)
            out.append(s.macros(0)[1])
            assert (s.info(0)[1] > 0) == (precision == hip.FP32_SHIFTED and "lid" in names)
        assert np.linalg.norm(out[0] - out[1]) < 1e-4 * np.linalg.norm(out[1])


@pytest.mark.parametrize("names", [("periodic", "walls"), ("walls", "walls"), ("periodic", "lid"), ("channel", "walls")])
def test_learned_closure_walls_2d(names):
    """As above in 2D (its own kernels, with and without the table)."""
    from tests.test_gpu_mlp import ROOT
    import os
    from zllbm_amd import closure
    model = closure.ClosureModel.load(os.path.join(ROOT, "zllbm_amd", "data", "closure_turbulence.npz"))
    grid = g.uniform_grid(2, (21, 18))
    out = []
    for precision in (hip.FP32_SHIFTED, hip.FP64):
        s = hip.Solver(grid, nu0=0.01, bc=_bc(names), precision=precision, collision=(hip.MRT,), les=hip.LES_MLP,
                       cs=0.1, mlp_operands=hip.MLP_OPERANDS_FP16).build()
        s.mlp_set(model)
        rho, u = _random_state(grid.levels[0].n, 2, 2)
        s.init_macro(0, rho, u)
        s.time_marching(11)
        out.append(s.macros(0)[1])
        assert (s.info(0)[1] > 0) == ("channel" in names or (precision == hip.FP32_SHIFTED and "lid" in names))
    assert np.linalg.norm(out[0] - out[1]) < 1e-4 * np.linalg.norm(out[1])


@pytest.mark.parametrize("precision", [hip.FP64, hip.FP32_SHIFTED, hip.BF16_SHIFTED])
@pytest.mark.parametrize("names", [("lid", "periodic"), ("walls", "lids"), ("lids", "periodic", "walls")])
def test_conservation_sums_the_populations(names, precision):
    """The sums on the device take the resolved pull as the downloads do: FP64 sums in another order,
    some 500 values of at most 1/2."""
    grid = g.uniform_grid(len(names), (17, 19) if len(names) == 2 else (6, 5, 9))
    s = hip.Solver(grid, nu0=0.05, bc=_bc(names), precision=precision, collision=(hip.MRT,)).build()
    s.init_macro(0, *_random_state(grid.levels[0].n, len(names), 3))
    s.time_marching(5)
    rho, u = s.macros(0)
    want = np.zeros(4)
    want[0] = rho.sum()
    want[1:1 + len(names)] = (rho[:, None] * u).sum(0)
    np.testing.assert_allclose(s.conservation(0), want, rtol=0, atol=1e-11)
