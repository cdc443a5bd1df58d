"""CPU check of ray scattering's lookups: on no ray does a group of columns have more items (a column and a sun
direction) than its wavefronts look up, counted on the host as the kernel lists them (no launch).  All slabs of up to 1024
entries on a small grid, and finer ones with many items: 103 to 115 sun elevations by 5 or 6 headings among them."""
import ctypes

from sfsim_amd import atmosphere as atm


class Items(ctypes.Structure):
    _fields_ = [("most", ctypes.c_int), ("capacity", ctypes.c_int)]  # capacity 0: the kernel without items


def items(shape, radius=6378000.0, height=100000.0):
    fn = getattr(atm.lib(), "_ZN5sfsim14ray_items_mostEPKidd")
    fn.restype = Items
    return fn((ctypes.c_int * 4)(*shape), ctypes.c_double(radius), ctypes.c_double(height))


def test_every_slab():
    for nl in range(2, 513):
        for na in range(2, 1024 // nl + 1):
            r = items((3, 7, nl, na))
            assert r.most <= r.capacity or r.capacity == 0, (nl, na, r.most, r.capacity)
            assert (r.capacity > 0) == (nl <= 170 or (nl <= 256 and na == 2)), (nl, na)


def test_finer_grids():
    seen = 0
    for nl, na in [(n, a) for n in range(103, 116) for a in (5, 6)] + [(128, 2), (128, 8), (129, 7), (170, 6), (256, 2), (32, 8), (64, 16)]:
        for rays, height in (((8, 32), 100000.0), ((5, 65), 35000.0), ((31, 66), 250000.0)):
            r = items((*rays, nl, na), height=height)
            seen = max(seen, r.most)
            assert r.most <= r.capacity <= 512, (nl, na, rays, r.most, r.capacity)
    assert seen > 384
