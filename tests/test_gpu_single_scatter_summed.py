"""Single scattering with every sun segment summed node by node, at the edges of its kernel's shapes, against the
FP64 oracle's stage: entry groups of fewer than 64, exactly 64 and 65 entries, sample counts around the chunk of 16 and
its quarters, the smallest and the largest.  Tolerance 1e-3 relative, as for every scattering table."""
import numpy as np
import pytest

from tests.parity import TOL_SCATTER, assert_close, oracle_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,steps", [((3, 6, 2, 2), 1), ((3, 6, 9, 7), 15), ((3, 6, 8, 8), 16), ((3, 6, 13, 5), 17),
                                         ((2, 5, 43, 3), 63), ((2, 4, 5, 4), 256)], ids=lambda v: str(v))
def test_single_scatter_summed_shapes(oracle, shape, steps):
    from sfsim_amd import atmosphere as atm
    P = atm.make_params(planet={"height": 100000.0}, transmittance_shape=(4, 9), surface_radiance_shape=(4, 9),
                        scatter_shape=shape, ray_steps=steps, sphere_steps=4, iterations=0)
    OP = oracle_params(oracle, P)
    with atm.Atmosphere(0) as ctx:
        ctx.sun_table = (0, 0)
        print("summed single scatter", shape, steps, flush=True)
        R1, M1 = ctx.single_scatter_tables(P)
        again = ctx.single_scatter_tables(P)
    np.testing.assert_array_equal(R1, again[0])  # the items' order among the wavefronts does not enter the sums
    np.testing.assert_array_equal(M1, again[1])
    assert_close("R1", R1, oracle.stage_single_scatter(OP, 0), TOL_SCATTER)
    assert_close("M1", M1, oracle.stage_single_scatter(OP, 1), TOL_SCATTER)
