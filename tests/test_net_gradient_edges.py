"""The network's gradients where the weight- and bias-gradient kernels' splits
change: a single position, fewer row segments than one workgroup takes, rows of
one position more than a segment of 16, enough positions for every workgroup,
and several sizes after one another on one network (its workspaces only grow).
The bounds are those of bfloat16 weights and activations: 1e-3 for the loss, 3e-2
per layer for the gradients."""
import numpy as np
import pytest

from oracle import net as on

pytestmark = pytest.mark.gpu


def test_gradients_at_the_splits():
    from robtop_amd.learned import WarmStartNet
    theta = on.random_params(12).astype(np.float32)
    net = WarmStartNet(0)
    net.set_params(theta)
    for shape in [(1, 1, 1), (25, 33, 49), (3, 5, 17), (1, 33, 1), (9, 8, 16), (25, 33, 49)]:
        print(f"[learned] gradient {shape}", flush=True)
        rng = np.random.default_rng(3 + sum(shape))
        x = rng.standard_normal(shape + (4,)).astype(np.float32)
        t = rng.standard_normal(shape + (3,)).astype(np.float32)
        loss, g = net.gradient(x, t)
        lo, go = on.loss_and_grad(theta.astype(np.float64), x.astype(np.float64), t.astype(np.float64), emulate=True)
        assert abs(loss - lo) / lo < 1e-3, (shape, loss, lo)
        pg, po = on.unpack(g), on.unpack(go)
        for name in on.LAYERS:
            for k in (0, 1):
                e = np.linalg.norm(pg[name][k] - po[name][k]) / max(np.linalg.norm(po[name][k]), 1e-300)
                assert e < 3e-2 or np.linalg.norm(po[name][k]) == 0 == np.linalg.norm(pg[name][k]), (shape, name, k, e)
    net.close()


@pytest.mark.parametrize("nx", [17, 20, 31, 32])
def test_infinity_in_a_rows_last_position(nx):
    """An input of infinity at the end of a row, which the first layer's negative weights and its ReLU turn into 0:
    the weight gradients of the taps that would pair it with a position past the row stay finite."""
    from robtop_amd.learned import WarmStartNet
    print(f"[learned] infinity at x = {nx - 1}", flush=True)
    theta = on.random_params(21).astype(np.float32)
    w = theta[:27 * 16 * 16].reshape(27, 16, 16)
    w[:, :, 0] = -np.abs(w[:, :, 0]) - 0.01
    net = WarmStartNet(0)
    net.set_params(theta)
    rng = np.random.default_rng(nx)
    shape = (5, 6, nx)
    x = rng.standard_normal(shape + (4,)).astype(np.float32)
    x[2, 3, nx - 1, 0] = np.inf
    t = rng.standard_normal(shape + (3,)).astype(np.float32)
    loss, g = net.gradient(x, t)
    with np.errstate(invalid="ignore"):
        lo, go = on.loss_and_grad(theta.astype(np.float64), x.astype(np.float64), t.astype(np.float64), emulate=True)
    assert np.isfinite(lo) and abs(loss - lo) / lo < 1e-3, (loss, lo)
    pg, po = on.unpack(g), on.unpack(go)
    for name in on.LAYERS:
        wg, wo = pg[name][0], po[name][0]
        if name == "E0A":
            assert np.isfinite(wo[0::3]).all() and np.isnan(wo[1::3, :, 0]).any()
            wg, wo = wg[0::3], wo[0::3]     # the taps at dx = -1
        assert np.isfinite(wg).all(), name
        assert np.linalg.norm(wg - wo) < 3e-2 * np.linalg.norm(wo), name
    net.close()
