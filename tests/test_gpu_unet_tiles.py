"""The warm-start network's convolution tiles and packed weights: every tile the dispatch
can pick gives the same bits as the smallest (16 voxels x 16 channels per wave), which
test_conv_and_gradients_match_oracle pins to the oracle, as test_network_gradients_match_oracle does
the weight gradients of all layers in grouped launches; and the packed weights stay current."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# a 12^3 sample alone takes the smallest tile; the batch has the waves for the one named, with a
# ragged last workgroup
@pytest.mark.parametrize("B,edge,cin,cout", [
    (38, 12, 32, 64),   # 64 voxels x 64 channels; the input gradient 64 x 32
    (20, 12, 16, 32),   # 32 x 32, 16-channel steps
    (38, 12, 48, 16),   # 64 x 16, both directions
    (4, 12, 32, 128),   # 16 x 32
])
def test_tiles_equal_the_smallest(wlc, B, edge, cin, cout):
    rng = np.random.default_rng(B + cin)
    x = rng.standard_normal((B, edge, edge, edge, cin))
    w = rng.standard_normal((cout, 27, cin)) * 0.2
    b = rng.standard_normal(cout)
    dy = rng.standard_normal((B, edge, edge, edge, cout))
    y, dx, dw, db = wlc.test_conv3d(x, w, b, dy)
    dws, dbs = np.zeros_like(dw, dtype=np.float64), np.zeros(cout)
    for k in range(B):
        yk, dxk, dwk, dbk = wlc.test_conv3d(x[k:k + 1], w, b, dy[k:k + 1])
        assert np.array_equal(y[k:k + 1], yk) and np.array_equal(dx[k:k + 1], dxk), k
        dws += dwk
        dbs += dbk
    for got, ref in ((dw, dws), (db, dbs)):
        assert np.abs(got - ref).max() <= 2e-5 * np.abs(ref).max()


def test_packed_weights_follow_every_route(wlc):
    """The packed copies of the weights that the kernels read are rewritten by the optimiser step, by
    set_params and by a resize of the network alike."""
    rng = np.random.default_rng(6)
    x = rng.standard_normal((1, 16, 16, 16, 11)).astype(np.float32)
    t = rng.standard_normal((1, 16, 16, 16, 3)).astype(np.float32)
    net = wlc.UNet(16, 1, seed=5)
    y = net.forward(x)
    net.gradients(x, t)
    net.adam(1e-3)
    q, y2 = net.params(), net.forward(x)
    assert not np.array_equal(y, y2)
    net.resize(8, 2)
    y8 = net.forward(np.ascontiguousarray(np.repeat(x[:, :8, :8, :8], 2, 0)))
    assert np.array_equal(y8[0], y8[1])
    net.close()
    for n, ref in ((16, y2), (8, y8[:1])):
        other = wlc.UNet(n, 1, seed=9)
        other.set_params(q)
        assert np.array_equal(other.forward(np.ascontiguousarray(x[:, :n, :n, :n])), ref)
        other.close()
