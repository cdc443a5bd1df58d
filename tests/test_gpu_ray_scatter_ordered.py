"""Ray scattering in plain order (the order sums, and the grids whose columns have more items than a wavefront looks up).

Grids of many sun elevations against the FP64 oracle's stage on the same dJ table, with one, two and four texels
per lane, one sample at a time and several, and in a batch.  The order sums' first order against the stage calls on
the same tables, on grids of each form (the exact sun coordinate and the other, slabs that end inside a wavefront,
odd sample counts): at most 256 positive FP32 terms added in two orders, each with a handful of roundings of
6e-8, differ by less than 256 x 6e-8 + 1e-6 = 1.7e-5 of their sum (floor: 1e-6 of the channel maximum)."""
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


def params(shape, steps, iterations=1):
    from sfsim_amd import atmosphere as atm
    return atm.make_params(planet={"height": 100000.0, "brightness": (0.2, 0.2, 0.2)}, transmittance_shape=(4, 9),
                           surface_radiance_shape=(4, 9), scatter_shape=shape, ray_steps=steps, sphere_steps=4,
                           iterations=iterations)


@pytest.mark.parametrize("shape,steps", [((2, 5, 171, 2), 1), ((2, 5, 200, 5), 7), ((3, 6, 256, 4), 9), ((2, 5, 257, 3), 6),
                                         ((2, 4, 512, 2), 5), ((16, 70, 180, 2), 4), ((33, 64, 192, 2), 3),
                                         ((64, 70, 171, 3), 3), ((16, 32, 180, 3), 4), ((33, 64, 150, 6), 3)], ids=lambda v: str(v))
def test_many_sun_elevations(gpu, oracle, shape, steps):
    P = params(shape, steps)
    n = int(np.prod(shape))
    rng = np.random.default_rng(n)
    dJ = rng.uniform(0.5e-6, 1e-6, (n, 3)).astype(np.float32)
    print("ray scatter", shape, steps, flush=True)
    got = gpu.ray_scatter_table(P, dJ)
    idx = np.sort(rng.choice(n, size=400, replace=False))
    ref = oracle.stage_ray_scatter(oracle_params(oracle, P), dJ.astype(np.float64), idx)
    assert_close(f"dS {shape}", got.reshape(-1, 3)[idx], ref, TOL_SCATTER)


def test_many_sun_elevations_in_a_batch(gpu):
    P = params((2, 5, 200, 3), 7, 2)
    Q = params((2, 5, 200, 3), 7, 2)
    Q.mie.scatter_g = 0.7
    print("batch", flush=True)
    gpu.build_batch([P, Q])
    for a, p in enumerate((P, Q)):
        got = [gpu.fetch_batch(p, a, i) for i in range(4)]
        gpu.build(p)
        for i in range(4):
            np.testing.assert_array_equal(got[i].view(np.uint32), gpu.fetch(p, i).view(np.uint32))


@pytest.mark.parametrize("shape,steps", [((3, 5, 2, 2), 4), ((4, 9, 15, 4), 16), ((3, 8, 21, 6), 9), ((2, 5, 64, 16), 13),
                                         ((32, 64, 32, 8), 5), ((48, 96, 24, 6), 4), ((40, 64, 12, 8), 4), ((3, 5, 7, 146), 11),
                                         ((2, 5, 200, 5), 6)], ids=lambda v: str(v))
def test_order_sums(gpu, shape, steps):
    from sfsim_amd import atmosphere as atm
    P = params(shape, steps, 5)
    print("order sums", shape, steps, flush=True)
    first = atm.order_sums(gpu, P)[0].reshape(-1, 3)
    r1, m1 = gpu.single_scatter_tables(P)
    dJ = gpu.point_scatter_table(P, r1, gpu.surface_radiance_base_table(P), mie_strength=m1)
    want = gpu.ray_scatter_table(P, dJ).reshape(-1, 3)
    bound = 1.7e-5 * np.maximum(np.abs(want), 1e-6 * np.abs(want).max(axis=0))
    assert np.all(np.abs(first.astype(np.float64) - want) <= bound)
