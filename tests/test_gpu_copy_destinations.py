"""Copies to the host by several threads of one context at once (fetches of tables of one chunk, several, and several rings of
the pinned ring, and of a batch), each equal byte for byte to the same table fetched alone, and into pinned memory
of the caller's, which takes no detour."""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def built():
    from sfsim_amd import atmosphere as atm
    P = atm.make_params(planet={"height": 100000.0, "brightness": (0.2, 0.2, 0.2)}, transmittance_shape=(64, 64),
                        surface_radiance_shape=(16, 33), scatter_shape=(48, 16, 32, 16), ray_steps=8, sphere_steps=6,
                        iterations=1)
    with atm.Atmosphere(0) as ctx:
        ctx.build(P)
        ctx.build_batch([P, P, P])
        yield atm, ctx, P, [ctx.fetch(P, i) for i in range(4)]


def test_fetches_from_several_threads(built):
    _, ctx, P, want = built
    jobs = [(k, i) for _ in range(6) for i in range(4) for k in range(4)]
    print("threads", flush=True)
    with ThreadPoolExecutor(8) as pool:
        got = list(pool.map(lambda j: ctx.fetch(P, j[1]) if j[0] == 3 else ctx.fetch_batch(P, j[0], j[1]), jobs))
    for (_, i), g in zip(jobs, got):
        np.testing.assert_array_equal(g.view(np.uint32), want[i].view(np.uint32))


@pytest.mark.parametrize("rows", [682, 683, 1365, 1366, 2048, 5462])
def test_sizes_around_one_copy_and_chunks(rows):
    """768 bytes a row: 511.5 and 512.25 KiB, 1023.75 and 1024.5 KiB, exactly 3 chunks, 8 chunks and a little (one ring)."""
    from sfsim_amd import atmosphere as atm
    P = atm.make_params(planet={"height": 100000.0}, transmittance_shape=(rows, 64), surface_radiance_shape=(4, 9),
                        scatter_shape=(2, 3, 2, 2), ray_steps=4, sphere_steps=4, iterations=0)
    hip = ctypes.CDLL("libamdhip64.so.7")
    hip.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
    hip.hipHostFree.argtypes = [ctypes.c_void_p]
    p, n = ctypes.c_void_p(), rows * 64 * 3
    assert hip.hipHostMalloc(ctypes.byref(p), 4 * n, 0) == 0
    try:
        want = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_float)), (n,))
        print("rows", rows, flush=True)
        with atm.Atmosphere(0) as ctx:
            ctx.build(P)
            got = ctx.fetch(P, 0)
            assert atm.lib().sfsim_atmo_fetch(ctx._ctx, 0, atm._fp(want), n) == 0
            np.testing.assert_array_equal(got.ravel().view(np.uint32), want.view(np.uint32))
            np.testing.assert_array_equal(ctx.generate_atmosphere_luts(P)["transmittance"].ravel().view(np.uint32),
                                          want.view(np.uint32))
    finally:
        hip.hipHostFree(p)


@pytest.mark.parametrize("which", range(4))
def test_pinned_destination(built, which):
    atm, ctx, P, want = built
    hip = ctypes.CDLL("libamdhip64.so.7")
    hip.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
    hip.hipHostFree.argtypes = [ctypes.c_void_p]
    n = want[which].size
    p = ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(p), 4 * n, 0) == 0
    try:
        got = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_float)), (n,))
        got[:] = np.nan
        print("pinned", which, flush=True)
        assert atm.lib().sfsim_atmo_fetch(ctx._ctx, which, atm._fp(got), n) == 0
        np.testing.assert_array_equal(got.view(np.uint32), want[which].ravel().view(np.uint32))
        got[:] = np.nan
        if which == 0:
            assert atm.lib().sfsim_atmo_transmittance_table(ctx._ctx, ctypes.byref(P), atm._fp(got)) == 0
            np.testing.assert_array_equal(got.view(np.uint32), ctx.transmittance_table(P).ravel().view(np.uint32))
    finally:
        hip.hipHostFree(p)
