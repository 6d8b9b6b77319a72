"""Every tile shape of the multi-tile sort at the sizes where the choice
changes and around one tile, against the oracle's stable radix order."""
import numpy as np
import pytest

import compute_amd as ca
import oracle as O

pytestmark = pytest.mark.gpu

# the last size of each shape, and a ragged one past it
LINES = {("uint32", 0): [16385, 1 << 18, 2500000, 12000000], ("float32", 4): [8193, 1 << 20, 5000000],
         ("uint64", 0): [8193, 1 << 19, 6000000], ("int64", 4): [8193, 1 << 20, 6000000],
         ("float64", 8): [8193, 1 << 20, 6000000], ("int32", 8): [8193, 1 << 20, 6000000]}


def _bits(a):
    return a.view("u%d" % a.dtype.itemsize)


@pytest.mark.parametrize("dt,vb", sorted(LINES))
@pytest.mark.parametrize("off", [0, 1])
def test_sort_shape_lines(queue, dt, vb, off):
    rng = np.random.default_rng(vb + off)
    t = np.dtype(dt)
    for line in LINES[dt, vb]:
        n = line + off * 4099
        if t.kind == "f":
            k = rng.uniform(-1e6, 1e6, n + 1).astype(t)
            k[::50] = 0.0
            k[7::50] = -0.0
        else:
            k = rng.integers(0, 256, (n + 1) * t.itemsize, dtype=np.uint8).view(t)
        desc = bool(off)
        d = ca.DeviceArray.from_host(k, queue)
        v = np.arange(n, dtype="u%d" % vb) if vb else None
        dv = ca.DeviceArray.from_host(v, queue) if vb else None
        ca.sort(queue, d, dv, api=ca.RADIX_SORT, n=n, key_ptr=d.at(off), descending=desc)
        e = O.radix_order_sort(k[off:off + n], v, descending=desc)
        ek, ev = e if vb else (e, None)
        got = d.to_host(queue)
        assert np.array_equal(_bits(got[off:off + n].copy()), _bits(ek)), n
        assert got[0 if off else n].tobytes() == k[0 if off else n].tobytes()  # the element beside the range
        if vb:
            assert np.array_equal(dv.to_host(queue), ev), n


# sizes of every tile shape, the largest ones the tuned, XCD-grouped shapes'
IDLE = [("uint32", 0, [16385, 300007, 3000017, 13000027]), ("uint32", 4, [8193, 1200007, 5200003]),
        ("uint64", 0, [8193, 600011, 6100007]), ("uint64", 4, [8193, 1200007, 6100007]),
        ("int32", 8, [8193, 1200007, 6100007]), ("uint32", 1, [30011]), ("int32", 2, [30011]), ("uint32", 16, [30011]),
        ("uint64", 16, [30011]), ("uint16", 0, [16385, 1000003]), ("int16", 4, [30011]), ("uint8", 4, [30011])]
# byte positions that vary: none; first one at an odd position (the later
# passes read the other array); an odd number of them (one idle pass copies)
MOVING = {1: [(), (0,)], 2: [(), (0,), (1,)], 4: [(), (1, 2), (0, 1, 3), (1,), (3,), (0, 2)],
          8: [(), (1, 2), (0, 3, 5), (1,), (2, 4, 6, 7), (1, 2, 3, 4, 5, 6)]}


def _moving_keys(dt, n, moving, rng):
    w = np.dtype(dt).itemsize
    k = np.full(n, 0x81A5C37E5B9D4F01 & ((1 << 8 * w) - 1), "u%d" % w)
    b = k.view(np.uint8).reshape(n, w)
    for i in moving:
        b[:, i] = rng.integers(0, 256, n, dtype=np.uint8)
    return k.view(dt)


@pytest.mark.parametrize("dt,vb,sizes", IDLE)
def test_sort_with_idle_passes(queue, dt, vb, sizes):
    """Keys with bytes that are the same in all of them: the passes over those
    bytes are left out, in every tile shape and value width."""
    rng = np.random.default_rng(vb)
    for n in sizes:
        for i, moving in enumerate(MOVING[np.dtype(dt).itemsize]):
            if n > 2000000 and i not in (1, 2):
                continue
            k = _moving_keys(dt, n, moving, rng)
            order = np.arange(n, dtype=np.uint32)
            v = rng.integers(0, 256, (n, vb), dtype=np.uint8)
            for desc in (False, True) if n < 100000 else (bool(i & 1),):
                d = ca.DeviceArray.from_host(k, queue)
                dv = ca.DeviceArray.from_host(v.reshape(-1), queue) if vb else None
                ca.check(ca.lib().bcmi_sort(queue.h, ca.RADIX_SORT, ca.DTYPE[k.dtype], d.ptr, dv.ptr if vb else None,
                                            vb, n, int(desc)))
                ek, eo = O.radix_order_sort(k, order, descending=desc)
                assert np.array_equal(d.to_host(queue), ek), (n, moving, desc)
                if vb:
                    assert np.array_equal(dv.to_host(queue).reshape(n, vb), v[eo]), (n, moving, desc)


@pytest.mark.parametrize("dt,vb", [("uint32", 0), ("uint64", 4)])
def test_noalloc_sort_with_idle_passes(queue, dt, vb):
    rng = np.random.default_rng(vb + 1)
    for n in (1000003, 20011):
        for moving in MOVING[np.dtype(dt).itemsize]:
            k = _moving_keys(dt, n, moving, rng)
            v = np.arange(n, dtype=np.uint32)
            d, dv = ca.DeviceArray.from_host(k, queue), ca.DeviceArray.from_host(v, queue)
            ca.check(ca.lib().bcmi_sort_noalloc(queue.h, ca.RADIX_SORT, ca.DTYPE[k.dtype], d.ptr,
                                                dv.ptr if vb else None, vb, n, 0))
            ek, ev = O.radix_order_sort(k, v)
            assert np.array_equal(d.to_host(queue), ek), (n, moving)
            if vb:
                assert np.array_equal(dv.to_host(queue), ev), (n, moving)
