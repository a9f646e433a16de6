"""The FP32 gradient kernel at the edges of its tiles (32 samples a wavefront, 128 a workgroup, at
most 256 workgroups) against the FP64 oracle, and minibatches drawn from the sample set."""
import numpy as np
import pytest

from oracle import mlp_oracle as mo
from zllbm_amd import closure, hip
from tests.test_gpu_mlp import _ctx, _data

pytestmark = pytest.mark.gpu


# a sum of n terms in FP32 is off by at most a few 2^-24 of the sum of their magnitudes; 2e-5 of the
# largest gradient component, as the other gradient tests
@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 127, 128, 129, 1000, 32767, 32768, 32769, 70001])
def test_gradient_at_tile_edges(n):
    s = _ctx()
    X, T = _data(n, seed=n)
    p = closure.init_params(n)
    loss, gd = s.mlp_gradient(p, X, T)
    lref, gref = mo.loss_and_grad(p.astype(np.float64), X.astype(np.float64), T.astype(np.float64))
    assert abs(loss - lref) <= 1e-5 * lref
    assert np.max(np.abs(gd - gref)) <= 2e-5 * np.max(np.abs(gref))
    again = s.mlp_gradient(p, X, T)
    assert again[0] == loss
    np.testing.assert_array_equal(again[1], gd)
    if n <= hip.MLP_NOALLOC_MAX_SAMPLES:
        noalloc = s.mlp_gradient_noalloc(p, X, T)
        assert noalloc[0] == loss
        np.testing.assert_array_equal(noalloc[1], gd)


@pytest.mark.parametrize("n,batch", [(50, 7), (5000, 129), (300, 300)])
def test_minibatch_loss(n, batch):
    """The first recorded loss is the batch's: samples hash(seed, k) mod n, or all in order."""
    s = _ctx()
    X, T = _data(n, seed=batch)
    p = closure.init_params(1)
    _, hist = s.mlp_train(p, X, T, 1, batch, 1e-3, seed=77)
    u = np.uint32
    with np.errstate(over="ignore"):
        x = u((77 * 1000003 + 1) & 0xFFFFFFFF) * u(2654435761) + np.arange(batch, dtype=u)
        x ^= x >> u(16)
        x *= u(0x7feb352d)
        x ^= x >> u(15)
        x *= u(0x846ca68b)
        x ^= x >> u(16)
    at = np.arange(n) if batch >= n else (x % u(n)).astype(np.int64)
    lref, _ = mo.loss_and_grad(p.astype(np.float64), X[at].astype(np.float64), T[at].astype(np.float64))
    assert abs(hist[0] - lref) <= 1e-5 * lref


# BF16 operands: 64 samples a wavefront, 256 a workgroup, at most 256 workgroups.  A difference in
# the order of an FP32 sum moves an operand to the next BF16 value in about one case of 2^16 per
# last bit: the bound of the emulation test, 5e-4 of the largest gradient component, for sets large
# enough that single roundings average out, ten times that below.
@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 257, 65536, 65537])
def test_gradient_bf16_at_tile_edges(n):
    s = _ctx()
    X, T = _data(n, seed=n + 7)
    p = closure.init_params(3)
    loss, gd = s.mlp_gradient(p, X, T, form=hip.MLP_BF16_MFMA)
    lemu, gemu = mo.loss_and_grad_lowp(p.astype(np.float64), X.astype(np.float64), T.astype(np.float64), mo.bf16_round)
    assert abs(loss - lemu) <= 1e-3 * lemu + 1e-6
    assert np.max(np.abs(gd - gemu)) <= (5e-4 if n > 1000 else 5e-3) * np.max(np.abs(gemu))
