"""The training products of the network at sizes that leave remainders in
their 64 x 64 x 64 blocks, against the FP64 restatement."""
import numpy as np
import pytest

from oracle import mlp_ref
from tests.test_gpu_surrogate import cosine, make_net, ref_arrays, rel

pytestmark = pytest.mark.gpu


# (om, pm, hidden, layers, rows): less than one block everywhere; an output
# width of 60 and an odd number of K tiles; a padded hidden width and split
# rows whose last range is short; several blocks both ways and a short K tile
@pytest.mark.parametrize("shape", [(3, 4, 8, 1, 8), (5, 12, 40, 1, 72), (6, 12, 72, 2, 584),
                                   (9, 20, 200, 3, 1096)])
def test_products_with_remainders(shape):
    # inputs, weights and activations in bfloat16 (2^-9 relative), a few of
    # them in a row per layer: 2 % normwise
    om, pm, hidden, layers, n = shape
    net = make_net(om, pm, hidden, layers, batch=n, chunk=(n + 63) // 64 * 64)
    try:
        rng = np.random.default_rng(11)
        for l in range(layers + 1):
            K, N = net.widths[l], net.widths[l + 1]
            net.set_layer(l, rng.normal(0, 1 / np.sqrt(K), (N, K)), rng.normal(0, 0.1, N))
        x = rng.normal(size=(n, net.nin)).astype(np.float32)
        t = rng.normal(size=(n, net.nout)).astype(np.float32)
        ws, bs = ref_arrays(net)
        xb = mlp_ref.bf16_round(x)
        _, _, y_ref = mlp_ref.forward(ws, bs, xb)
        for rows in (n, n - 3):
            assert rel(net.forward(x[:rows]), y_ref[:rows]) <= 0.02, rows
        loss, gws, gbs = net.gradients(x, t)
        loss_ref, gw_ref, gb_ref = mlp_ref.gradients(ws, bs, xb, t)
        assert abs(loss - loss_ref) <= 0.02 * loss_ref
        for l in range(layers + 1):
            assert rel(gws[l], gw_ref[l]) <= 0.02, (l, rel(gws[l], gw_ref[l]))
            assert cosine(gws[l], gw_ref[l]) >= 0.999, l
            assert rel(gbs[l], gb_ref[l]) <= 0.02, (l, rel(gbs[l], gb_ref[l]))
    finally:
        net.close()


def test_gradients_keep_the_order_of_their_sums():
    """The weight gradient is the sum in turn of partials over 256 rows, the
    bias gradient of eight sums over every 8th row: whatever the products'
    blocks are, so that a training run repeats to the bit.  Row 0 gives 1 and
    the rows from 256 on 2^-31, which vanish one by one beside 1 and count when
    they are summed among themselves first, so the result tells the order."""
    om, pm, hidden, n = 16, 64, 512, 2048
    net = make_net(om, pm, hidden, 1, batch=n, chunk=n)
    try:
        assert n * net.nout == 1 << 21
        net.set_layer(0, np.zeros((hidden, net.nin)), np.full(hidden, 8.0))  # gelu(8) = 8
        net.set_layer(1, np.zeros((net.nout, hidden)), np.zeros(net.nout))   # outputs 0
        dz = np.zeros(n)
        dz[0] = 1.0
        dz[256:] = 2.0 ** -31
        t = np.repeat((-dz * 2.0 ** 20)[:, None], net.nout, axis=1)  # dz = -2 t / 2^21
        _, gws, gbs = net.gradients(np.zeros((n, net.nin)), t)
        f = np.float32
        gw = f(0)
        for part in np.split(dz * 8, n // 256):
            # 16 rows a step; what a step adds is exact
            p = f(0)
            for step in np.split(part, 16):
                p = f(p + f(step.sum()))
            gw = f(gw + p)
        gb = f(0)
        for group in range(8):
            s = f(0)
            for v in dz[group::8]:
                s = f(s + f(v))
            gb = f(gb + s)
        assert gw == 8 + 7 * 2.0 ** -20 and gb == 1 + 7 * 2.0 ** -23
        assert np.all(gws[1] == gw), (gws[1].min(), gws[1].max(), gw)
        assert np.all(gbs[1] == gb), (gbs[1].min(), gbs[1].max(), gb)
    finally:
        net.close()
