"""Downloads of populations and macroscopic variables at sizes from one node row to many staging
chunks (1 MiB of output: 6,898 nodes of D3Q19 populations, 43,690 nodes of 2D macros), against the
uploaded values and the oracle."""
import numpy as np
import pytest

from oracle.zlbm_oracle import Oracle, lattice
from zllbm_amd import grid as g
from zllbm_amd import hip
from tests import scenarios as sc
from tests.test_gpu_parity import assert_close

pytestmark = pytest.mark.gpu

C2 = np.array([(0, 0), (1, 0), (0, 1), (-1, 0), (0, -1), (1, 1), (-1, 1), (-1, -1), (1, -1)])


def _macros(f, c):
    """Sums in direction order, as the device forms them (c is -1, 0 or 1: exact products)."""
    rho, j = f[:, 0].copy(), np.zeros((len(f), c.shape[1]))
    for q in range(1, f.shape[1]):
        rho += f[:, q]
        j += c[q] * f[:, q:q + 1]
    return rho, j / rho[:, None]


@pytest.mark.parametrize("dims,cells", [(2, (1, 1)), (2, (130, 7)), (2, (419, 415)), (2, (600, 601)),
                                        (3, (2, 3, 1)), (3, (29, 30, 28)), (3, (31, 41, 60))])
def test_downloads_return_what_was_uploaded(dims, cells):
    grid = g.uniform_grid(dims, cells)
    n, q = grid.levels[0].n, 9 if dims == 2 else 19
    f = 0.05 + 0.01 * np.random.default_rng(n).random((n, q))
    s = hip.Solver(grid, nu0=0.1, bc=sc.all_bc(dims, sc.BB)).build()
    s.set_f(0, f)
    np.testing.assert_array_equal(s.f(0), f)
    if dims == 2:
        rho, u = s.macros(0)
        rho_h, u_h = _macros(f, C2)
        np.testing.assert_array_equal(rho, rho_h)
        np.testing.assert_array_equal(u, u_h)
    # a smaller download after a larger one, and again
    np.testing.assert_array_equal(s.f(0), f)


@pytest.mark.parametrize("precision", [hip.FP64, hip.FP32_SHIFTED, hip.BF16_SHIFTED])
def test_downloads_after_steps(precision):
    grid, kw = sc.cavity(n=200)
    o, s = Oracle(grid, **kw), hip.Solver(grid, precision=precision, **kw).build()
    rng = np.random.default_rng(3)
    rho, u = 1.0 + 1e-3 * rng.random(grid.levels[0].n), 1e-2 * rng.random((grid.levels[0].n, 2))
    o.init_macro(0, rho, u)
    s.init_macro(0, rho, u)
    o.time_marching(3)
    s.time_marching(3)
    f = s.f(0)
    if precision == hip.FP64:
        assert_close(f, o.f(0))
    rho_s, u_s = s.macros(0)
    rho_h, u_h = _macros(f, C2)
    np.testing.assert_array_equal(rho_s, rho_h)
    np.testing.assert_array_equal(u_s, u_h)


# 2D: 231 x 225 nodes are 2 chunks of macros; 3D: 41 x 43 x 40 are 11 of populations and 3 of macros
# (32,768 nodes), each with nodes whose pull the boundary conditions resolve in every chunk
@pytest.mark.parametrize("precision", [hip.FP64, hip.FP32_SHIFTED, hip.BF16_SHIFTED])
@pytest.mark.parametrize("cells", [(230, 224), (40, 42, 39)])
def test_macros_of_many_chunks_after_steps(cells, precision):
    """Macros are the sums of the populations, which (FP64) are the oracle's."""
    dims = len(cells)
    grid = g.uniform_grid(dims, cells)
    bc = sc.all_bc(dims, sc.BB)
    bc[g.XMIN] = bc[g.XMAX] = (sc.PER, (0., 0., 0.))
    bc[g.YMAX] = (sc.BB, (0.03, 0., 0.))
    kw = dict(nu0=0.02, bc=bc, collision=(hip.MRT,))
    s = hip.Solver(grid, precision=precision, **kw).build()
    rho, u = sc.level_fields(grid, 0, 0.05, noise=1e-3)
    s.init_macro(0, rho, u)
    s.time_marching(3)
    f = s.f(0)
    if precision == hip.FP64:
        o = Oracle(grid, **kw)
        o.init_macro(0, rho, u)
        o.time_marching(3)
        assert_close(f, o.f(0))
    c = np.stack(lattice(dims)[:dims], 1)
    rho_s, u_s = s.macros(0)
    rho_h, u_h = _macros(f, c)
    np.testing.assert_array_equal(rho_s, rho_h)
    np.testing.assert_array_equal(u_s, u_h)
