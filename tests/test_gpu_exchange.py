"""The coarse/fine exchange, which stages and rescales aux rows itself, at boxes whose interfaces
start at odd and even nodes of a brick, with thin and wide boxes and both interpolations, against
the oracle; and the closure's workspace over calls of growing and shrinking size."""
import threading

import numpy as np
import pytest

from oracle.zlbm_oracle import Oracle
from zllbm_amd import closure, grid as g
from zllbm_amd import hip
from tests import scenarios as sc
from tests.test_gpu_mlp import _ctx, _data
from tests.test_gpu_parity import assert_close

pytestmark = pytest.mark.gpu

BOXES = {
    "2d even": (2, (24, 20), [((8, 6), (16, 14))]),
    "2d odd": (2, (27, 23), [((5, 5), (16, 15)), ((15, 14), (23, 25))]),
    "3d even": (3, (16, 16, 16), [((6, 6, 6), (12, 12, 12))]),
    "3d odd": (3, (17, 19, 16), [((5, 5, 5), (12, 13, 12)), ((14, 15, 14), (20, 21, 20))]),
}


# FP64: rounding of sums in another order than the oracle's, 1e-12 of the largest population as the
# other substep tests.  FP32 shifted: a few 2^-24 of |f - w| < 0.05 a step over 6 steps of collision
# and exchange, far below 2e-6; populations are up to 1/3.
@pytest.mark.parametrize("precision,tol", [(hip.FP64, 1e-12), (hip.FP32_SHIFTED, 2e-6)])
@pytest.mark.parametrize("interp", [hip.INTERP_LAGRANGIAN, hip.INTERP_LINEAR])
@pytest.mark.parametrize("box", sorted(BOXES))
def test_exchange_against_oracle(box, interp, precision, tol):
    dims, cells, boxes = BOXES[box]
    grid = g.refined_box_grid(dims, cells, boxes)
    kw = dict(nu0=0.01, bc=sc.all_bc(dims, sc.PER), collision=(hip.MRT,), interp_method=interp)
    o, s = Oracle(grid, **kw), hip.Solver(grid, precision=precision, **kw).build()
    for l in range(grid.max_level + 1):
        rho, u = sc.level_fields(grid, l, 0.05, noise=1e-3)
        o.init_macro(l, rho, u)
        s.init_macro(l, rho, u)
    o.time_marching(6)
    s.time_marching(6)
    for l in range(grid.max_level + 1):
        assert_close(s.f(l), o.f(l), rtol=0 if tol > 1e-10 else tol, atol=tol)


def test_closure_workspace_sizes():
    """Each call's result is that of a new solver, whatever the sizes before it: the sizes grow,
    shrink and pass the largest workspace that is kept (64 MiB, 1.67M samples)."""
    s = _ctx()
    p = closure.init_params(3)
    X, T = _data(1_700_000, seed=9)
    for n in (100, 5000, 33, 1_700_000, 70000, 1):
        loss, grad = s.mlp_gradient(p, X[:n], T[:n])
        lref, gref = _ctx().mlp_gradient(p, X[:n], T[:n])
        assert loss == lref
        np.testing.assert_array_equal(grad, gref)
        q, h = s.mlp_train(p, X[:n], T[:n], 2, 64, 1e-3, seed=5)
        qr, hr = _ctx().mlp_train(p, X[:n], T[:n], 2, 64, 1e-3, seed=5)
        np.testing.assert_array_equal(h, hr)
        np.testing.assert_array_equal(q, qr)


def test_calls_from_two_threads():
    """Gradients and downloads of one solver from two threads at once take turns."""
    s = _ctx()
    p = closure.init_params(3)
    X, T = _data(6000, seed=4)
    want = {n: s.mlp_gradient(p, X[:n], T[:n]) for n in (500, 6000)}
    bad = []

    def run(n):
        for _ in range(20):
            loss, grad = s.mlp_gradient(p, X[:n], T[:n])
            if loss != want[n][0] or not np.array_equal(grad, want[n][1]):
                bad.append(n)

    threads = [threading.Thread(target=run, args=(n,)) for n in want]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


# rows of more than 32,768 nodes: FP64 in 3D forms them as a table in a launch of its own (k_c2f_sources),
# in 2D the gather stages them itself, as every smaller exchange does
LARGE = {
    "3d": lambda: g.refined_box_grid(3, (62, 62, 62), [((5, 5, 5), (57, 57, 57))]),
    "2d": lambda: g.refined_mask_grid(2, (400, 400), 2, lambda k, c: np.floor(c / 14).sum(1) % 2 == 0, buffer=0),
}


@pytest.mark.parametrize("name", sorted(LARGE))
def test_large_fp64_exchange(name):
    """Against the oracle; then time interpolation on and off again (its second table is made at the
    switch), each against a solver that was built so and starts from the same populations."""
    grid = LARGE[name]()
    kw = dict(nu0=0.01, bc=sc.all_bc(grid.dims, sc.PER), collision=(hip.MRT,))
    o, s = Oracle(grid, **kw), hip.Solver(grid, **kw).build()
    assert s.transfer_info(1)["source_rows"] > 32768
    for l in range(2):
        rho, u = sc.level_fields(grid, l, 0.05, noise=1e-3)
        o.init_macro(l, rho, u)
        s.init_macro(l, rho, u)
    o.time_marching(3)
    s.time_marching(3)
    for l in range(2):
        assert_close(s.f(l), o.f(l))
    for on in (True, False):
        s.set_time_interpolation(on)
        r = hip.Solver(grid, time_interp=on, **kw).build()
        for l in range(2):
            r.set_f(l, s.f(l))
        s.time_marching(2)
        r.time_marching(2)
        for l in range(2):
            np.testing.assert_array_equal(r.f(l), s.f(l))


# BF16 rows are staged in units of 8 bytes.  A store rounds f - w by up to 2^-9 of itself; the bounds
# are those of the refined BF16 runs of 10 and 12 steps
@pytest.mark.parametrize("interp", [hip.INTERP_LAGRANGIAN, hip.INTERP_LINEAR])
@pytest.mark.parametrize("box", sorted(BOXES))
def test_exchange_bf16_tracks_fp64(box, interp):
    dims, cells, boxes = BOXES[box]
    grid = g.refined_box_grid(dims, cells, boxes)
    kw = dict(nu0=0.01, bc=sc.all_bc(dims, sc.PER), collision=(hip.MRT,), interp_method=interp)
    runs = [hip.Solver(grid, precision=p, **kw).build() for p in (hip.FP64, hip.BF16_SHIFTED)]
    for s in runs:
        for l in range(grid.max_level + 1):
            s.init_macro(l, *sc.level_fields(grid, l, 0.05, noise=1e-3))
        s.time_marching(6)
    for l in range(grid.max_level + 1):
        (rho, u), (rho_b, u_b) = (s.macros(l) for s in runs)
        assert np.linalg.norm(u_b - u) < 6e-3 * np.linalg.norm(u)
        assert np.sqrt(np.mean((rho_b - rho) ** 2)) < 2.5e-4


def test_downloads_beside_gradients():
    """Populations (7 staging chunks) and macros (2) from two threads while a third takes gradients:
    the calls that share the staging buffer and the workspace take turns."""
    grid = g.uniform_grid(3, (34, 35, 36))
    s = hip.Solver(grid, nu0=0.02, bc=sc.all_bc(3, sc.PER), collision=(hip.MRT,)).build()
    s.init_macro(0, *sc.level_fields(grid, 0, 0.05, noise=1e-3))
    s.time_marching(3)
    p = closure.init_params(3)
    X, T = _data(6000, seed=4)
    f, (rho, u), (loss, grad) = s.f(0), s.macros(0), s.mlp_gradient(p, X, T)
    bad = []

    def run(same):
        for _ in range(15):
            if not same():
                bad.append(same)

    def macros_same():
        r, v = s.macros(0)
        return np.array_equal(r, rho) and np.array_equal(v, u)

    def gradient_same():
        l, d = s.mlp_gradient(p, X, T)
        return l == loss and np.array_equal(d, grad)

    threads = [threading.Thread(target=run, args=(c,))
               for c in (lambda: np.array_equal(s.f(0), f), macros_same, gradient_same)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
