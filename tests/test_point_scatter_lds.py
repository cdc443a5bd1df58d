"""CPU checks of how a point-scatter workgroup lays out its LDS (no launch: the library's own host function), over the
shapes that the entry points accept: sun elevations x headings up to 1024 entries, 1 to 1000 sphere directions,
surface-radiance tables on both sides of the longest that is kept in LDS, with and without the Mie strength, grids of
few rays and of many."""
import ctypes

import pytest

from sfsim_amd import atmosphere as atm


class Lds(ctypes.Structure):
    _fields_ = [(n, ctypes.c_uint) for n in ("bytes", "plane8", "plane16", "pitch", "dirs")] + [
        ("at", ctypes.c_uint * 4), ("size", ctypes.c_uint * 4)]


def lds_of(shape, ne1, steps, mie, batch=0):
    fn = getattr(atm.lib(), "_ZN5sfsim17point_scatter_ldsEPKiiiib")
    fn.restype = Lds
    return fn((ctypes.c_int * 4)(*shape), ne1, steps, batch, ctypes.c_bool(mie))


SLABS = [(nl, na) for nl in range(2, 513) for na in range(2, 1024 // nl + 1)]


@pytest.mark.parametrize("mie", [False, True])
@pytest.mark.parametrize("rays", [(3, 5), (32, 64), (4, 2047)])
def test_texel_behind_the_last_one_is_inside(rays, mie):
    """Lanes read the texel behind their own where a lane of their wavefront needs it: 16 bytes at plane16 and 8 at
    plane8, of two slabs (four with the Mie strength) of `pitch` x (headings + 1) texels."""
    for nl, na in SLABS:
        for ne1, steps in ((2, 2), (17, 14), (64, 28), (1024, 8), (1025, 55)):
            p = lds_of((*rays, nl, na), ne1, steps, mie)
            texels = (4 if mie else 2) * p.pitch * (na + 1) + 1
            where = (rays, nl, na, ne1, steps)
            assert p.plane16 == 2 * p.plane8 and p.plane16 % 16 == 0, where
            assert p.plane8 + 8 * texels <= p.plane16, where
            assert p.plane16 + 16 * texels <= p.bytes, where


LDS_BYTES = 160 * 1024  # of a CU


@pytest.mark.parametrize("mie", [False, True])
@pytest.mark.parametrize("rays,batch", [((3, 5), 0), ((32, 64), 0), ((4, 2047), 16)])
def test_every_accepted_shape_fits(rays, batch, mie):
    """Within a CU's LDS whatever the number of directions and of surface-radiance columns, no array over another,
    and the weights of at least the largest latitude ring (sphere_steps directions at most) at a time."""
    for nl, na in SLABS:
        for ne1 in (2, 512, 768, 1024, 1025):
            for steps in (2, 3, 14, 28, 40, 50, 55):
                p = lds_of((*rays, nl, na), ne1, steps, mie, batch)
                where = (rays, nl, na, ne1, steps)
                assert p.bytes <= LDS_BYTES, where
                assert p.dirs >= min(steps, atm.sphere_directions(False, steps)), where
                texels = (4 if mie else 2) * p.pitch * (na + 1) + 1
                spans = sorted([(p.plane8, p.plane8 + 8 * texels), (p.plane16, p.plane16 + 16 * texels)] +
                               [(a, a + n) for a, n in zip(p.at, p.size) if n])
                assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:])) and spans[-1][1] <= p.bytes, where
                assert all(a % 16 == 0 for a in p.at), where
