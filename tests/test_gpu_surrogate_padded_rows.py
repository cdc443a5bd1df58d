"""The surrogate's gradient where the last rows do not fill a tile: the rows that pad it have all features 0, so their
activations are those of the biases alone.  With a bias that bf16 rounds to infinity, and a weight on the first feature that
brings the given rows back into range, the padding's activations are infinite; the gradient must not see them (infinity
times their gradient, 0, is NaN).  Output weights are 0, so the hidden layers' gradients are exactly 0."""
import numpy as np
import pytest

from oracle import mlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 9, 31])
def test_padding_does_not_enter_the_gradient(rows):
    from sfsim_amd import atmosphere as atm
    blocks = [np.zeros(s, np.float32) for s in mlp.SHAPES]  # W1 b1 W2 b2 W3 b3 W4 b4
    blocks[0][0, :] = -3.38e38
    blocks[1][:] = 3.4e38
    x = np.zeros((rows, 10), np.float32)
    x[:, 0] = 1.0
    T = np.zeros((rows, 16), np.float32)
    T[:, :15] = 0.5
    with atm.Atmosphere(0) as ctx:
        sg = atm.Surrogate(ctx, seed=1, batch=64)
        sg.set_weights(np.concatenate([b.reshape(-1) for b in blocks]), trained=False)
        print("rows", rows, flush=True)
        y, g, loss = sg.eval(x, T)
    assert np.all(y == 0.0)
    assert np.all(np.isfinite(g))
    ends = np.cumsum([b.size for b in blocks])
    assert np.all(g[:ends[6]] == 0.0)  # W1 .. W4
    np.testing.assert_allclose(g[ends[6]:ends[6] + 15], -0.5, rtol=1e-6)
    assert loss == pytest.approx(0.5 * 15 * 0.25, rel=1e-6)
