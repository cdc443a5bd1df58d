"""The surrogate's forward and backward pass at row counts around its tiles (32 rows per workgroup, 16 per loss partial,
8 per step of the weight gradients, splits of at least 64 rows, 256 rows per round of the bias sums), against the FP64
network.  Bounds: the rounding of every product's operands to bf16 (2^-9 relative, at most six in a chain) and of the
outputs' difference to the targets leave at most ~3e-2 in the norm of a gradient; 5e-2 is allowed.  A row's output
does not depend on the other rows."""
import numpy as np
import pytest

from oracle import mlp

pytestmark = pytest.mark.gpu

ROWS = [1, 8, 15, 17, 32, 33, 63, 65, 257, 2047, 2049]


@pytest.fixture(scope="module")
def net():
    from sfsim_amd import atmosphere as atm
    rng = np.random.default_rng(5)
    theta = np.concatenate([rng.uniform(-1, 1, s).reshape(-1) * (np.sqrt(6.0 / sum(s)) if len(s) == 2 else 0.1)
                            for s in mlp.SHAPES]).astype(np.float32)
    x = rng.uniform(0, 1, (max(ROWS), 10)).astype(np.float32)
    T = np.zeros((max(ROWS), 16), np.float32)
    T[:, :15] = rng.normal(0.0, 1.0, (max(ROWS), 15))
    with atm.Atmosphere(0) as ctx:
        sg = atm.Surrogate(ctx, seed=1, batch=2112)
        sg.set_weights(theta, trained=False)
        yield sg, theta.astype(np.float64), x, T, sg.eval(x)[0]


@pytest.mark.parametrize("rows", ROWS)
def test_rows(net, rows):
    sg, theta, x, T, y_all = net
    print("rows", rows, flush=True)
    y, g, loss = sg.eval(x[:rows], T[:rows])
    assert np.array_equal(y, y_all[:rows])
    mask = np.zeros((rows, 16))
    mask[:, :15] = 1.0
    ref_loss, ref = mlp.loss_and_grad(theta, mlp.encode(x[:rows]), T[:rows].astype(np.float64), mask)
    assert loss == pytest.approx(ref_loss, rel=5e-2)
    offsets = np.cumsum([0] + [int(np.prod(s)) for s in mlp.SHAPES])
    for b in range(8):
        a, r = g[offsets[b]:offsets[b + 1]].astype(np.float64), ref[offsets[b]:offsets[b + 1]]
        assert np.linalg.norm(a - r) <= 5e-2 * np.linalg.norm(r), b
