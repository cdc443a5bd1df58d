"""Point scattering with the most directions and the longest surface-radiance tables together, against the FP64 oracle's
stage on the same tables: the weights of the directions do not all fit a workgroup's LDS and are made for some latitude
rings at a time, with the surface-radiance table in LDS or, next to a wide slab, in memory; one and two entries per lane,
with and without the Mie strength.  Tolerance 1e-3 relative, as for every scattering table (floor: 1e-6 of the table's
channel maximum)."""
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


SHAPES = [((3, 6, 16, 4), 50, 1024), ((3, 6, 16, 4), 55, 512), ((3, 7, 8, 8), 55, 1024), ((16, 128, 32, 8), 55, 768),
          ((3, 6, 32, 8), 55, 1024), ((3, 5, 16, 16), 52, 1024), ((2, 5, 2, 512), 51, 1024), ((2, 3, 3, 129), 55, 1025)]


@pytest.mark.parametrize("mie", [False, True])
@pytest.mark.parametrize("shape,sphere_steps,columns", SHAPES, ids=lambda v: str(v))
def test_many_directions_and_columns(gpu, oracle, shape, sphere_steps, columns, mie):
    from sfsim_amd import atmosphere as atm
    P = atm.make_params(planet={"height": 100000.0}, transmittance_shape=(4, 9), surface_radiance_shape=(2, columns),
                        scatter_shape=shape, ray_steps=4, sphere_steps=sphere_steps, iterations=1)
    n = int(np.prod(shape))
    rng = np.random.default_rng(n)
    dS = rng.uniform(0.05, 0.1, (n, 3)).astype(np.float32)
    M = rng.uniform(0.005, 0.01, (n, 3)).astype(np.float32) if mie else None
    dE = rng.uniform(0.5, 1.0, (2 * columns, 3)).astype(np.float32)
    print("point scatter", shape, sphere_steps, columns, mie, flush=True)
    got = gpu.point_scatter_table(P, dS, dE, mie_strength=M)
    idx = np.sort(rng.choice(n, size=min(n, 200), replace=False))
    f64 = lambda a: a.astype(np.float64)  # noqa: E731
    ref = oracle.stage_point_scatter(oracle_params(oracle, P), 1 if mie else 0, f64(dS), f64(M) if mie else None, f64(dE), idx)
    assert_close(f"dJ {shape}", got.reshape(-1, 3)[idx], ref, TOL_SCATTER)
