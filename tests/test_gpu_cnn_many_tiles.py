"""The closure network's convolutions and weight gradients where a block works through several tiles
(16 x 4 x 8 cells in the convolutions, 16 x 4 x 4 in the weight gradients; blocks number the tiles
or the CUs, whichever is less): the next tile's loads in flight, LDS used again, bias sums carried
from tile to tile, samples that start inside a block's run, runs of unequal length and blocks
without a tile, against the numpy statement with the same BF16 roundings (tests/cnn_ref.py)."""
import numpy as np
import pytest

import cnn_ref as cr

pytestmark = pytest.mark.gpu

# as for single tiles (test_gpu_cnn_shapes.py): an FP32 sum beside a BF16 rounding boundary may fall
# on either side, which moves an operand by 2^-8 of itself, a few per cent of them at most
TOL = 2.0 ** -9


@pytest.mark.parametrize("shape", [(3, 35, 50, 33), (5, 9, 61, 40), (2, 70, 17, 64), (300, 3, 5, 7)])
def test_gradients_of_many_tiles(need_gpu, shape):
    from simpletcsolver_amd import Cnn
    nb, nz, ny, nx = shape
    tiles = nb * -(-nx // 16) * -(-ny // 4) * -(-nz // 8)
    assert tiles > 256
    rng = np.random.default_rng(nx)
    x = rng.standard_normal(shape + (5,)).astype(np.float32)
    y = (0.3 * rng.standard_normal(shape + (4,))).astype(np.float32)
    params = cr.init_params(6)
    net = Cnn(nx, ny, nz, batch=nb, seed=1)
    for l, (w, b) in enumerate(params):
        net.set_layer(l, w, b)
    loss_ref, grads, f = cr.loss_and_grads(params, x, y, bf=True)
    out = net.predict(x)
    want = f["out"][..., :4]
    assert np.linalg.norm(out - want) <= TOL * np.linalg.norm(want)
    # no cell is far off either: an output is a sum of 27 x 32 products of which each may move so
    assert np.abs(out - want).max() <= 16 * TOL * np.abs(want).max()
    loss = net.gradients(x, y)
    assert abs(loss - loss_ref) <= 1e-5 * loss_ref
    for l in range(3):
        _, _, gw, gb = net.layer(l)
        for got, ref in ((gw, grads[l][0]), (gb, grads[l][1])):
            assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref), (l, shape)
    net.close()
