"""The closure network's training kernels at the edges of their tiles (16 x 4 x 4 cells): rows
of one cell, of a tile less and more one, several tiles, and grids thinner than a tile in y and
z (whose periodic images wrap more than once), against the numpy statement with the same BF16
roundings (tests/cnn_ref.py)."""
import numpy as np
import pytest

import cnn_ref as cr

pytestmark = pytest.mark.gpu

# Both sides form the same BF16 operands and sum exact products, in another order.  An FP32 sum
# next to a BF16 rounding boundary may fall on either side, which moves that one operand of the
# next product by 2^-8 of itself; if every operand did, the result would move by less than
# 2^-8, and at most a few per cent of them do: 2^-9 covers both layers behind a gradient.
TOL = 2.0 ** -9


@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (1, 1, 3, 15), (2, 2, 5, 16), (1, 5, 4, 17),
                                   (3, 4, 9, 32), (1, 9, 6, 33), (2, 7, 3, 50)])
def test_gradients_at_tile_edges(need_gpu, shape):
    from simpletcsolver_amd import Cnn
    nb, nz, ny, nx = shape
    rng = np.random.default_rng(nx + 100 * ny)
    x = rng.standard_normal(shape + (5,)).astype(np.float32)
    y = (0.3 * rng.standard_normal(shape + (4,))).astype(np.float32)
    params = cr.init_params(5)
    net = Cnn(nx, ny, nz, batch=nb, seed=1)
    for l, (w, b) in enumerate(params):
        net.set_layer(l, w, b)
    loss_ref, grads, f = cr.loss_and_grads(params, x, y, bf=True)
    out = net.predict(x)
    assert np.linalg.norm(out - f["out"][..., :4]) <= TOL * np.linalg.norm(f["out"][..., :4])
    loss = net.gradients(x, y)
    assert abs(loss - loss_ref) <= 1e-5 * loss_ref
    for l in range(3):
        _, _, gw, gb = net.layer(l)
        for got, want in ((gw, grads[l][0]), (gb, grads[l][1])):
            assert np.linalg.norm(got - want) <= TOL * np.linalg.norm(want), (l, shape)
    net.close()
