"""Ray scattering at the edges of its kernel's shapes, against the FP64 oracle's stage on the same dJ table: one, two,
four and eight texels per lane (slabs of up to 64, 128, 256 and 512 entries), one and several column groups, the
last grid of the exact sun coordinate and the first of the other, slabs that end inside a wavefront, one and odd
sample counts, and a grid whose every sun direction is clamped (two headings).  Tolerance 1e-3 relative, as for
every scattering table (floor: 1e-6 of the table's channel maximum)."""
import numpy as np
import pytest

from tests.parity import TOL_SCATTER, assert_close, oracle_params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    from sfsim_amd import atmosphere
    ctx = atmosphere.Atmosphere(0)
    yield ctx
    ctx.close()


SHAPES = [((3, 5, 2, 2), 7), ((3, 4, 5, 4), 1), ((4, 9, 15, 4), 16), ((4, 9, 16, 4), 16), ((3, 8, 21, 6), 9),
          ((3, 8, 32, 8), 13), ((3, 5, 23, 11), 10), ((3, 6, 64, 16), 12), ((2, 5, 85, 12), 6), ((2, 5, 128, 2), 8),
          ((2, 5, 300, 2), 5), ((2, 5, 512, 2), 4), ((2, 5, 3, 300), 6), ((2, 5, 2, 512), 4)]


@pytest.mark.parametrize("shape,steps", SHAPES, ids=lambda v: str(v))
def test_ray_scatter_shapes(gpu, oracle, shape, steps):
    from sfsim_amd import atmosphere as atm
    P = atm.make_params(planet={"height": 100000.0}, transmittance_shape=(4, 9), surface_radiance_shape=(4, 9),
                        scatter_shape=shape, ray_steps=steps, sphere_steps=4, iterations=1)
    n = int(np.prod(shape))
    rng = np.random.default_rng(n)
    dJ = rng.uniform(0.5e-6, 1e-6, (n, 3)).astype(np.float32)  # neighbours of like size, as in a smooth table
    print("ray scatter", shape, steps, flush=True)
    got = gpu.ray_scatter_table(P, dJ)
    idx = np.sort(rng.choice(n, size=min(n, 600), replace=False))
    ref = oracle.stage_ray_scatter(oracle_params(oracle, P), dJ.astype(np.float64), idx)
    assert_close(f"dS {shape}", got.reshape(-1, 3)[idx], ref, TOL_SCATTER)


def test_ray_scatter_sample_by_sample_path(gpu, oracle):
    """A grid of several column groups on which rays have more items in one group than its wavefronts look up."""
    from sfsim_amd import atmosphere as atm
    shape = (2, 6, 200, 5)
    P = atm.make_params(planet={"height": 100000.0}, transmittance_shape=(4, 9), surface_radiance_shape=(4, 9),
                        scatter_shape=shape, ray_steps=6, sphere_steps=4, iterations=1)
    n = int(np.prod(shape))
    rng = np.random.default_rng(3)
    dJ = rng.uniform(0.5e-6, 1e-6, (n, 3)).astype(np.float32)
    got = gpu.ray_scatter_table(P, dJ)
    idx = np.sort(rng.choice(n, size=600, replace=False))
    ref = oracle.stage_ray_scatter(oracle_params(oracle, P), dJ.astype(np.float64), idx)
    assert_close("dS", got.reshape(-1, 3)[idx], ref, TOL_SCATTER)
