"""The one-workgroup sort (block_sort.hip) at the edges of its shapes, on both
sides of its largest size, against the oracle's stable radix order."""
import numpy as np
import pytest

import compute_amd as ca
import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [33, 63, 1023, 1024, 1025, 2048, 2049, 4096, 4097, 8191, 8192, 8193, 16384, 16385]


def _keys(dt, n, kind, rng):
    dt = np.dtype(dt)
    if kind == "full":
        k = rng.integers(0, 256, n * dt.itemsize, dtype=np.uint8).view(dt)
        if dt.kind == "f":
            k = np.where(np.isfinite(k), k, dt.type(0.5)).astype(dt)
            k[::7] = 0.0
            k[3::11] = -0.0
            k[5::13] = np.inf
            k[6::17] = np.nan
        return k
    if kind == "narrow":  # two bytes of range, away from zero
        return (rng.integers(0, 300 if dt.itemsize > 1 else 100, n) + 11).astype(dt)
    if kind == "clustered":  # long runs of equal leading bits, distinct low bits
        base = rng.integers(0, 4, n).astype(np.uint64) << np.uint64(8 * dt.itemsize - 3)
        k = (base | rng.integers(0, 200, n).astype(np.uint64)).astype("u%d" % dt.itemsize).view(dt)
        return k
    return np.full(n, 7, dt)


def _bits(a):
    return a.view("u%d" % a.dtype.itemsize)


@pytest.mark.parametrize("dt", ["uint8", "int16", "uint32", "int32", "float32", "uint64", "int64", "float64"])
@pytest.mark.parametrize("kind", ["full", "narrow", "clustered", "one value"])
def test_block_sort_shapes(queue, dt, kind):
    rng = np.random.default_rng(len(kind) * 100 + np.dtype(dt).itemsize)
    for n in SIZES:
        k = _keys(dt, n, kind, rng)
        for desc in (False, True):
            d = ca.DeviceArray.from_host(k, queue)
            ca.sort(queue, d, api=ca.RADIX_SORT, descending=desc)
            assert np.array_equal(_bits(d.to_host(queue)), _bits(O.radix_order_sort(k, descending=desc))), (n, desc)
            v = np.arange(n, dtype=np.uint32)
            dk, dv = ca.DeviceArray.from_host(k, queue), ca.DeviceArray.from_host(v, queue)
            ca.sort(queue, dk, dv, api=ca.RADIX_SORT, descending=desc)
            ek, ev = O.radix_order_sort(k, v, descending=desc)
            assert np.array_equal(_bits(dk.to_host(queue)), _bits(ek)), (n, desc)
            assert np.array_equal(dv.to_host(queue), ev), (n, desc)


@pytest.mark.parametrize("vb", [1, 2, 8, 16])
@pytest.mark.parametrize("dt", ["uint16", "float32", "uint64"])
def test_block_sort_value_widths(queue, dt, vb):
    rng = np.random.default_rng(vb)
    for n in (100, 3001, 8192):
        k = _keys(dt, n, "full", rng)
        v = rng.integers(0, 256, (n, vb), dtype=np.uint8)
        # one element into the allocation: nothing is aligned to 16 bytes
        dk = ca.DeviceArray.from_host(np.concatenate([k[:1], k, k[:1]]), queue)
        dv = ca.DeviceArray.from_host(np.concatenate([v[:1], v, v[:1]]).reshape(-1), queue)
        ca.check(ca.lib().bcmi_sort(queue.h, ca.SORT_BY_KEY, ca.DTYPE[k.dtype], dk.at(1), dv.at(vb), vb, n, 0))
        ek, order = O.radix_order_sort(k, np.arange(n, dtype=np.uint32))
        got, gv = dk.to_host(queue), dv.to_host(queue).reshape(n + 2, vb)
        assert np.array_equal(_bits(got[1:-1].copy()), _bits(ek))
        assert np.array_equal(gv[1:-1], v[order])
        for a, b in ((got, k), (gv, v)):  # the elements around the range
            assert a[0].tobytes() == b[0].tobytes() and a[-1].tobytes() == b[0].tobytes()
