"""The backward convolutions of the learned stage's network (k_conv_bwd_data,
k_conv_bwd_w) at the edges of their splits, against the float64 oracle: grids
of 1 to 15 nodes per axis, even and odd (the parity classes of the stride-2
layers are empty, single or uneven), and more positions than one chunk of the
weight gradient.  Tolerance relative to max|g|: 1e-4, the bar of the network's
gradient (FP32 sums of at most a few thousand terms against float64)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh", [(8, 8, 8), (16, 8, 8), (8, 24, 16), (32, 16, 24), (40, 56, 16), (48, 32, 40)])
def test_network_gradient_vs_oracle(gputo, mesh):
    import learn_oracle

    print("case", mesh, flush=True)
    s = gputo.Solver(*mesh, 4, precision=1, learned=True)
    n0, n1, n2 = s.learn_info()["grid"]
    rng = np.random.default_rng(91)
    p = rng.normal(0.0, 0.05, learn_oracle.nparams()).astype(np.float32).astype(np.float64)
    s.learn_params(p)
    x = rng.normal(size=(4, n0, n1, n2)).astype(np.float32).astype(np.float64)
    gy = rng.normal(size=(3, n0, n1, n2)).astype(np.float32).astype(np.float64)
    g = s.learn_grad(x, gy)
    _, go = learn_oracle.run(p, x, gy)
    assert np.abs(g - go).max() < 1e-4 * np.abs(go).max()
    assert np.array_equal(g, s.learn_grad(x, gy))  # deterministic, nothing left over from the first call
    s.close()


@pytest.mark.parametrize("mesh", [(16, 8, 8), (48, 32, 40)])
def test_network_gradient_with_an_input_that_is_nan(gputo, mesh):
    """A NaN in the input is cut off by the first ReLU, and no gradient passes
    there: the weight gradient leaves those positions out.  Tolerance as above."""
    import learn_oracle

    print("case", mesh, flush=True)
    s = gputo.Solver(*mesh, 4, precision=1, learned=True)
    n0, n1, n2 = s.learn_info()["grid"]
    rng = np.random.default_rng(92)
    p = rng.normal(0.0, 0.05, learn_oracle.nparams()).astype(np.float32).astype(np.float64)
    s.learn_params(p)
    x = rng.normal(size=(4, n0, n1, n2)).astype(np.float32).astype(np.float64)
    gy = rng.normal(size=(3, n0, n1, n2)).astype(np.float32).astype(np.float64)
    x[1, n0 // 2, n1 // 2, n2 // 2] = np.nan
    x[3, 0, 0, n2 - 1] = np.nan
    g, y = s.learn_grad(x, gy), s.learn_forward(x)
    s.close()
    yo, go = learn_oracle.run(p, x, gy)
    assert np.abs(y - yo).max() < 1e-4 * np.abs(yo).max()
    assert np.abs(g - go).max() < 1e-4 * np.abs(go).max()
