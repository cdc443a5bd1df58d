"""Point scattering at the edges of its kernel's shapes, against the FP64 oracle's stage on the same tables, with and
without the Mie strength: slabs of one wavefront and of several, one and two entries per lane, one and several
blocks of sun elevations (the last one shorter), heights whose rays do not fill a workgroup, one latitude ring, a
surface-radiance table too long for LDS, and the most headings.  Tolerance 1e-3 relative, as for every scattering
table (floor: 1e-6 of the table's channel maximum)."""
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


SHAPES = [((3, 5, 2, 2), 2, (3, 2)), ((3, 7, 5, 4), 6, (4, 9)), ((4, 9, 16, 4), 8, (3, 1024)), ((3, 8, 23, 7), 9, (3, 1025)),
          ((3, 6, 33, 8), 14, (4, 17)), ((32, 64, 32, 8), 4, (4, 17)), ((3, 6, 64, 16), 10, (4, 17)),
          ((2, 5, 300, 3), 8, (4, 9)), ((2, 5, 3, 300), 8, (4, 9)), ((2, 5, 2, 512), 8, (4, 9)), ((3, 4, 6, 5), 55, (4, 9))]


@pytest.mark.parametrize("mie", [False, True])
@pytest.mark.parametrize("shape,sphere_steps,surface", SHAPES, ids=lambda v: str(v))
def test_point_scatter_shapes(gpu, oracle, shape, sphere_steps, surface, mie):
    from sfsim_amd import atmosphere as atm
    P = atm.make_params(planet={"height": 100000.0}, transmittance_shape=(4, 9), surface_radiance_shape=surface,
                        scatter_shape=shape, ray_steps=4, sphere_steps=sphere_steps, iterations=1)
    n = int(np.prod(shape))
    rng = np.random.default_rng(n)
    dS = rng.uniform(0.05, 0.1, (n, 3)).astype(np.float32)
    M = rng.uniform(0.005, 0.01, (n, 3)).astype(np.float32) if mie else None
    dE = rng.uniform(0.5, 1.0, (surface[0] * surface[1], 3)).astype(np.float32)
    print("point scatter", shape, sphere_steps, surface, mie, flush=True)
    got = gpu.point_scatter_table(P, dS, dE, mie_strength=M)
    idx = np.sort(rng.choice(n, size=min(n, 400), replace=False))
    f64 = lambda a: a.astype(np.float64)  # noqa: E731
    ref = oracle.stage_point_scatter(oracle_params(oracle, P), 1 if mie else 0, f64(dS), f64(M) if mie else None, f64(dE), idx)
    assert_close(f"dJ {shape}", got.reshape(-1, 3)[idx], ref, TOL_SCATTER)
