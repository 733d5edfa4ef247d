"""The convolution tiles that test_gpu_unet_tiles.py does not launch, among them those of the network's
first and last layers at its usual sizes, against the smallest tile; and the epilogues of the network
(activation, upsampled store, output, gradient mask) in large tiles, on a batch against its samples
alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# a 12^3 sample alone takes the smallest tile (16 x 16)
@pytest.mark.parametrize("B,edge,cin,cout", [
    (38, 12, 32, 16),   # 64 voxels x 16 channels, 32-channel steps; the input gradient 64 x 32, 16-channel steps
    (38, 12, 16, 64),   # 64 x 64, 16-channel steps
    (10, 12, 16, 32),   # 16 x 32, 16-channel steps
    (20, 12, 32, 32),   # 32 x 32, 32-channel steps, both directions
])
def test_tiles_equal_the_smallest(wlc, B, edge, cin, cout):
    rng = np.random.default_rng(B + cin + cout)
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
    # sums of up to 65664 voxels in another order
    for got, ref in ((dw, dws), (db, dbs)):
        assert np.abs(got - ref).max() <= 2e-5 * np.abs(ref).max()


# a sample alone takes the smallest tile on 16^3 and smaller ones than the batch on 32^3; the batch
# fills 64-voxel tiles on the finest level (16^3) or the two finest (32^3)
@pytest.mark.parametrize("n,B", [(16, 32), (32, 16)])
def test_batch_equals_its_samples(wlc, n, B):
    rng = np.random.default_rng(n)
    x = rng.standard_normal((B, n, n, n, 11)).astype(np.float32)
    t = rng.standard_normal((B, n, n, n, 3)).astype(np.float32)
    net = wlc.UNet(n, B, seed=4)
    layers = net.layers()
    p = net.params()
    for l in layers:
        p[l["boff"]:l["boff"] + l["cout_real"]] = 0.1 * rng.standard_normal(l["cout_real"])
    net.set_params(p)
    y = net.forward(x)
    loss, g = net.gradients(x, t), net.grads()
    net.resize(n, 1)
    gs, ls = np.zeros(g.shape), 0.0
    for k in range(B):
        assert np.array_equal(net.forward(x[k:k + 1]), y[k:k + 1]), k
        ls += net.gradients(x[k:k + 1], t[k:k + 1])
        gs += net.grads()
    net.close()
    # the batch's loss is the mean: its gradients are those of the samples over B (a power of two,
    # which no rounding sees), summed over the voxels in another order
    assert loss == pytest.approx(ls / B, rel=1e-5)
    for l in layers:
        for a, n_ in ((l["woff"], l["cout"] * 27 * l["cin"]), (l["boff"], l["cout"])):
            got, ref = g[a:a + n_] * float(B), gs[a:a + n_]
            assert np.abs(got - ref).max() <= 2e-5 * np.abs(ref).max(), l
