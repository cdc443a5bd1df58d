"""Single scattering with every sun segment summed node by node on a grid of more rays than one dimension of a launch holds
workgroups of 256 threads (2^32 threads), one sample per ray: entries across the grid against the FP64 oracle's stage."""
import ctypes

import numpy as np
import pytest

from tests.parity import TOL_SCATTER, assert_close, oracle_params

pytestmark = pytest.mark.gpu


def test_more_rays_than_a_launch_dimension_holds(oracle):
    from sfsim_amd import atmosphere as atm
    shape = (4100, 4100, 2, 2)
    P = atm.make_params(planet={"height": 100000.0}, transmittance_shape=(4, 9), surface_radiance_shape=(4, 9),
                        scatter_shape=shape, ray_steps=1, sphere_steps=4, iterations=0)
    n = int(np.prod(shape))
    out = np.full((n, 3), np.nan, np.float32)
    with atm.Atmosphere(0) as ctx:
        ctx.sun_table = (0, 0)
        print("summed single scatter", shape, flush=True)
        ctx._check(atm.lib().sfsim_atmo_single_scatter_tables(ctx._ctx, ctypes.byref(P), atm._fp(out), None))
    idx = np.unique(np.concatenate([np.random.default_rng(1).integers(0, n, 300), [0, n - 1, n // 2]]))
    ref = oracle.stage_single_scatter(oracle_params(oracle, P), 0, idx)
    assert_close("R1", out[idx], ref, TOL_SCATTER)
    assert np.isfinite(out).all()
