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
