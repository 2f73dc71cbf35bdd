"""Sizes at the edges of the convolution's tiles (16 x 4, 8 or 16 pixels, the taller ones for launches of
many workgroups): a batch equals its images one at a time bit for bit, and one image the oracle
within the network's bars (2 % of the output range, 0.2 % on average)."""
import numpy as np
import pytest

from cumulus3d_amd import init_net, pm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,h,w", [
    (130, 8, 8),    # images smaller than a tile
    (48, 40, 56),   # remainders in both directions
    (30, 136, 24),  # two tile columns, the second half empty
])
def test_conv_tile_edges(batch, h, w):
    from oracle import nn_oracle as nno

    rng = np.random.default_rng(7)
    feat = np.zeros((batch, h, w, 64), np.float32)
    feat[..., :33] = rng.uniform(0, 1, (batch, h, w, 33))
    bits = nno.bf16_bits(feat)
    be = pm.HipPatchMatch()
    big, one = (init_net.InitNet(be, n, h, w, seed=11) for n in (batch, 1))
    big.set_features(bits)
    head = big.predict(batch, want_head=True)[3]
    for b in (0, batch - 1):
        one.set_features(bits[b : b + 1])
        assert np.array_equal(one.predict(1, want_head=True)[3][0].view(np.uint32), head[b].view(np.uint32))
    out = nno.Net(one.get_params().astype(np.float64), bf=True).forward(nno.bf16(feat[:1]))["out"][..., :5]
    err = np.abs(head[0] - out[0])
    assert err.max() <= 0.02 * np.abs(out).max() and err.mean() <= 0.002 * np.abs(out).max()
    be.close()


@pytest.mark.parametrize("batch,h,w", [(3, 8, 8), (4, 40, 72), (17, 24, 40)])
def test_weight_gradient_tiles_and_slices(batch, h, w):
    """The gradient reduces tiles of 32 x 16 pixels into slices by the number of tiles; the convolutions
    give an image the same bits in any batch, so a batch's gradients are its images' summed (fp32
    sums: 1e-5 relative)."""
    from oracle import nn_oracle as nno

    rng = np.random.default_rng(9)
    feat = np.zeros((batch, h, w, 64), np.float32)
    feat[..., :33] = rng.uniform(0, 1, (batch, h, w, 33))
    bits = nno.bf16_bits(feat)
    depth = rng.uniform(20, 60, (batch, h, w)).astype(np.float32)
    normal = np.tile(np.float32([0.1, -0.2, -0.97]), (batch, h, w, 1))
    be = pm.HipPatchMatch()
    big, one = (init_net.InitNet(be, n, h, w, seed=11) for n in (batch, 1))
    big.set_features(bits)
    total = np.zeros(big.n)
    for b in range(batch):
        big.set_labels(b, depth[b], normal[b], w - 3, h - 2, 15.0, 120.0)
        one.set_features(bits[b : b + 1])
        one.set_labels(0, depth[b], normal[b], w - 3, h - 2, 15.0, 120.0)
        total += one.train_step(1, init_net.TrainParams(), step=False, want_grads=True)[1]
    got = big.train_step(batch, init_net.TrainParams(), step=False, want_grads=True)[1]
    for name, woff, boff, cin, cout, k, relu in nno.layout()[0]:
        for lo, hi in ((woff, boff), (boff, boff + cout)):
            assert np.linalg.norm(got[lo:hi] - total[lo:hi]) <= 1e-5 * np.linalg.norm(total[lo:hi]), name
    be.close()
