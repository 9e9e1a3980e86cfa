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
