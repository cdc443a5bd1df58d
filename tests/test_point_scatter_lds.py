"""CPU checks of how a point-scatter workgroup lays out its LDS (no launch: the library's own host function), over the
shapes that the entry points accept: sun elevations x headings up to 1024 entries, 1 to 1000 sphere directions,
surface-radiance tables on both sides of the longest that is kept in LDS, with and without the Mie strength, grids of
few rays and of many."""
import ctypes

import pytest

from sfsim_amd import atmosphere as atm


class Lds(ctypes.Structure):
    _fields_ = [(n, ctypes.c_uint) for n in ("bytes", "plane8", "plane16", "pitch")]


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
