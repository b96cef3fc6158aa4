"""The warm-start network's kernels at the row counts where their tiles end: 16 rows per
wave, 64 per training workgroup, 256 training workgroups, and 1,024 waves' rows, above which
the forward kernels take sixteen waves per workgroup."""
import numpy as np
import pytest

from cardiomechanics_amd import materials as MT
from cardiomechanics_amd import mesh as M
from cardiomechanics_amd.context import MechanicsContext
from cardiomechanics_amd.hip import DeviceArray
from cardiomechanics_amd.warmstart import WarmStartNet
from oracle import mlp as OM
from test_gpu_warmstart import bf16_forward

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def net():
    with MechanicsContext(M.cube_mesh(1), [MT.cube_guccione()]) as ctx:
        net = WarmStartNet(ctx, seed=9)
        w = np.random.default_rng(3).normal(0, 0.15, net.n_weights).astype(np.float32)
        net.set_weights(w)
        yield net, w.astype(np.float64)
        net.close()


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 63, 65, 64 * 256, 16 * 1024, 16 * 1024 + 1, 16 * 4096 + 17])
def test_forward_and_gradient_at_the_edges_of_the_tiles(net, rows):
    """FP32 sums of at most 128 products of values below one: 128 * 2^-24 of the sum of their
    magnitudes, 1e-5 of the largest output; gradients sum over the rows as well, in 256 partial
    sums of at most 64 * 2^6 rows, 4e-5.  bfloat16: tests/test_gpu_warmstart.py's bound for the
    emulated roundings."""
    net, w = net
    rng = np.random.default_rng(rows)
    X = rng.normal(size=(rows, 8)).astype(np.float32)
    T = rng.normal(size=(rows, 3)).astype(np.float32)
    guard = np.full((rows + 4, 3), 7.0, np.float32)   # rows past the end stay as they are
    Xd, Td, Yd = DeviceArray(X), DeviceArray(T), DeviceArray(guard)
    Yo, _, _ = OM.forward(w, X.astype(np.float64))
    net.forward(Xd, Yd, rows)
    net.sync()
    Y = Yd.download().reshape(-1, 3)
    assert np.abs(Y[:rows] - Yo).max() <= 1e-5 * np.abs(Yo).max() and (Y[rows:] == 7.0).all()
    net.forward(Xd, Yd, rows, bf16=True)
    net.sync()
    Y, Ye = Yd.download().reshape(-1, 3), bf16_forward(w, X)
    assert np.abs(Y[:rows] - Ye).max() <= 2e-3 * max(np.abs(Ye).max(), 1.0) and (Y[rows:] == 7.0).all()
    loss, g = net.loss_grad(Xd, Td, rows, want_grad=True)
    again, g2 = net.loss_grad(Xd, Td, rows, want_grad=True)
    assert loss == again and g.tobytes() == g2.tobytes()
    lo, go = OM.loss_grad(w, X.astype(np.float64), T.astype(np.float64))
    assert abs(loss - lo) <= 4e-5 * abs(lo)
    for a, b in [(0, 1024), (1024, 1152), (1152, 17536), (17536, 17664), (17664, 18048), (18048, 18051)]:
        assert np.linalg.norm(g[a:b] - go[a:b]) <= 4e-5 * np.linalg.norm(go[a:b])


def test_bf16_small_and_saturated_activations(net):
    """Pre-activations from 1e-6 to far past saturation, and infinite inputs, pass through the
    bfloat16 kernel's tanh as through numpy's."""
    net, _ = net
    w = np.zeros(net.n_weights, np.float32)
    w[0:128] = 1.0                                    # hidden 1: input 0 in every unit
    w[1152:17536:129] = 1.0                           # hidden 2: identity
    w[17664:18048:3] = 1.0 / 128                      # output 0: mean of the units
    saved = net.weights()
    net.set_weights(w)
    v = np.concatenate([10.0 ** np.arange(-6.0, 3.0), [0.0, 0.24, 0.26, np.inf]])
    X = np.zeros((2 * len(v), 8), np.float32)
    X[:, 0] = np.concatenate([v, -v])
    Y = DeviceArray(np.zeros((len(X), 3), np.float32))
    net.forward(DeviceArray(X), Y, len(X), bf16=True)
    net.sync()
    got = Y.download().reshape(-1, 3)[:, 0]
    want = bf16_forward(w.astype(np.float64), np.nan_to_num(X, posinf=1e4, neginf=-1e4))[:, 0]
    net.set_weights(saved)
    # one bfloat16 rounding that falls the other way: 2^-8 of the value
    assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(want))
