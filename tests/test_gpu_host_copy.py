"""GPU test of the copies to host memory, which pass through a ring of 8 pinned chunks of 512 KiB emptied by
several threads: tables of one chunk or less, a chunk and a remainder, about one ring and several rings, by each
entry point that copies tables out, equal byte for byte to the same tables written to device memory."""
import numpy as np
import pytest

from test_zz_no_alloc import TABLES, DeviceBuffers

pytestmark = pytest.mark.gpu


# bytes of a scatter table: 192 KiB; 528 KiB (a chunk and a remainder); exactly 3 chunks; 3.5 MiB (7); 4.5 MiB
# (9, one past the ring); 14.9 MiB with an odd tail (nearly four rings)
@pytest.mark.parametrize("shape", [(16, 16, 8, 8), (16, 16, 11, 16), (32, 16, 16, 16), (16, 32, 28, 21),
                                   (48, 16, 32, 16), (53, 41, 25, 24)])
def test_host_tables_equal_device_tables(shape):
    from sfsim_amd import atmosphere as atm
    P = atm.make_params(planet={"height": 100000.0, "brightness": (0.2, 0.2, 0.2)}, transmittance_shape=(64, 64),
                        surface_radiance_shape=(16, 33), scatter_shape=shape, ray_steps=16, sphere_steps=10,
                        iterations=1)
    with atm.Atmosphere(0) as ctx:
        print("host copies", shape, flush=True)
        host = [ctx.generate_atmosphere_luts(P) for _ in range(2)]
        bufs = DeviceBuffers([host[0][k].size for k in TABLES])
        try:
            ctx.generate_luts_noalloc(P, bufs.ptrs)
            dev = [bufs.read(i) for i in range(len(TABLES))]
        finally:
            bufs.free()
        ctx.build(P)
        ctx.build_batch([P, P])
        for i, k in enumerate(TABLES):
            for h in host:
                np.testing.assert_array_equal(h[k].ravel().view(np.uint32), dev[i].view(np.uint32))
            for h in (ctx.fetch(P, i), ctx.fetch_batch(P, 0, i), ctx.fetch_batch(P, 1, i)):
                np.testing.assert_array_equal(h.ravel().view(np.uint32), dev[i].view(np.uint32))
