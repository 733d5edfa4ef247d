"""Gradients of the warm-start network with a NaN or an infinity in the input: a pre-activation that
is NaN passes no gradient (the comparison y > 0 is false), so only what multiplies a NaN activation
becomes NaN."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,B", [(8, 1), (16, 2)])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_no_gradient_through_a_nan(wlc, n, B, value):
    rng = np.random.default_rng(3)
    x = rng.standard_normal((B, n, n, n, 11)).astype(np.float32)
    t = rng.standard_normal((B, n, n, n, 3)).astype(np.float32)
    x[0, 1, 2, 3, 4] = value
    net = wlc.UNet(n, B, seed=3)
    loss = net.gradients(x, t)
    g, layers = net.grads(), net.layers()
    net.close()
    assert np.isnan(loss)
    for l in layers:
        db = g[l["boff"]:l["boff"] + l["cout_real"]]
        # the output layer has no ReLU; the others' gradients are stopped at their NaN outputs
        assert np.isnan(db).all() if not l["relu"] else np.isfinite(db).all()
    w0 = g[layers[0]["woff"]:layers[0]["boff"]].reshape(layers[0]["cout"], 27, layers[0]["cin"])
    bad = np.isnan(w0).any(axis=(0, 1))
    assert bad[4] and bad.sum() == 1
