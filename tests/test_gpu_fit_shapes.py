"""Size-dependent tile shapes of the scans, by-key reductions, selections,
reductions and transforms: both sides of each line, one tile's edges, ranges
off the 16-byte grid, and the tuned shapes at small sizes (fit_size = 0),
against the oracle or numpy."""
import numpy as np
import pytest

import compute_amd as ca
import oracle as O

pytestmark = pytest.mark.gpu


def _dev(q, a, off=0):
    """a at element `off` of its allocation, with a guard element on each side."""
    pad = np.zeros(off + 1, a.dtype)
    return ca.DeviceArray.from_host(np.concatenate([pad[:off], a, pad[:1]]), q)


@pytest.mark.parametrize("dt", ["int32", "uint64", "int16"])
@pytest.mark.parametrize("off_in,off_out", [(0, 0), (1, 1), (1, 3)])
def test_scan_lines(queue, dt, off_in, off_out):
    rng = np.random.default_rng(off_out)
    for n in (1, 7, 8191, 8192, 8193, 16385, 1500000, 1500001, 2500000, 2500001):
        x = rng.integers(0, 100, n).astype(dt)
        d = _dev(queue, x, off_in)
        o = ca.DeviceArray.from_host(np.full(n + off_out + 1, 77, dt), queue)
        for excl in (False, True):
            init = np.array([5], dt)
            ca.check(ca.lib().bcmi_scan(queue.h, ca.DTYPE[x.dtype], ca.PLUS, d.at(off_in), o.at(off_out), n,
                                        init.ctypes.data, int(excl), ca.COMPENSATED))
            got = o.to_host(queue)
            assert np.array_equal(got[off_out:off_out + n], O.scan(x, excl, 5) if excl else O.scan(x, False)), (n, excl)
            assert (got[:off_out] == 77).all() and got[-1] == 77  # nothing beside the range


@pytest.mark.parametrize("n", [1001, 2500000, 2500001, 6000000, 6000001])
@pytest.mark.parametrize("off", [0, 3])
def test_float_scan_lines(queue, n, off):
    x = (np.random.default_rng(n).standard_normal(n) * 100).astype(np.float32)
    d = _dev(queue, x, off)
    o = ca.DeviceArray(n + off, np.float32, queue)
    ca.check(ca.lib().bcmi_scan(queue.h, ca.F32, ca.PLUS, d.at(off), o.at(off), n, None, 0, ca.COMPENSATED))
    e = np.cumsum(x.astype(np.longdouble))
    # one rounding to float, and FP64 sums on the way (as the scan's bound)
    bound = np.spacing(np.abs(e).astype(np.float32)).astype(np.float64) + 2.0 ** -50 * np.cumsum(np.abs(x.astype(np.float64)))
    assert (np.abs(o.to_host(queue)[off:].astype(np.longdouble) - e) <= bound).all()


@pytest.mark.parametrize("vdt", ["int32", "int64"])
@pytest.mark.parametrize("n", [1, 100000, 100001, 500000, 500001, 1500000, 1500001])
@pytest.mark.parametrize("koff,voff", [(0, 0), (1, 3)])
def test_by_key_lines(queue, vdt, n, koff, voff):
    rng = np.random.default_rng(n)
    k = np.cumsum(rng.integers(0, 20, n) == 0).astype(np.int32)
    v = rng.integers(-100, 100, n).astype(vdt)
    dk, dv = _dev(queue, k, koff), _dev(queue, v, voff)
    ko, vo, cnt = ca.DeviceArray(n, np.int32, queue), ca.DeviceArray(n, vdt, queue), ca.DeviceArray(1, np.uint64, queue)
    ca.check(ca.lib().bcmi_reduce_by_key(queue.h, ca.I32, ca.DTYPE[v.dtype], ca.PLUS, dk.at(koff), dv.at(voff), n,
                                         ko.ptr, vo.ptr, cnt.ptr, ca.COMPENSATED))
    heads = np.flatnonzero(np.concatenate([[True], k[1:] != k[:-1]]))
    assert int(cnt.to_host(queue)[0]) == heads.size
    assert np.array_equal(ko.to_host(queue)[:heads.size], k[heads])
    assert np.array_equal(vo.to_host(queue)[:heads.size], np.add.reduceat(v, heads))
    out = ca.DeviceArray(n + voff, vdt, queue)
    c = np.cumsum(v)
    start = np.repeat(heads, np.diff(np.concatenate([heads, [n]])))
    ca.check(ca.lib().bcmi_segmented_scan(queue.h, ca.I32, ca.DTYPE[v.dtype], dk.at(koff), dv.at(voff), out.at(voff),
                                          n, None, 0, ca.COMPENSATED))
    assert np.array_equal(out.to_host(queue)[voff:], (c - c[start] + v[start]).astype(vdt))


@pytest.mark.parametrize("dt,line", [("int32", 384 * 16384), ("float32", 384 * 16384), ("int64", 192 * 8192),
                                     ("uint8", 384 * 16384), ("uint8", 192 * 16384), ("int16", 192 * 16384)])
@pytest.mark.parametrize("off", [0, 1])
def test_select_lines(queue, dt, line, off):
    rng = np.random.default_rng(off)
    for n in (1, 4095, 4096, 4097, line, line + 1):
        x = rng.integers(0, 100, n).astype(dt)
        pred = ca.predicate(dt, "<", 50)
        keep = x < 50
        d = _dev(queue, x, off)
        out, rest = ca.DeviceArray(n, dt, queue), ca.DeviceArray(n, dt, queue)
        got = ca.copy_if(queue, d, out, pred, n=n, in_ptr=d.at(off))
        assert got == keep.sum() and np.array_equal(out.to_host(queue)[:got], x[keep]), n
        cnt = ca.DeviceArray(1, np.uint64, queue)
        ca.check(ca.lib().bcmi_partition(queue.h, ca.DTYPE[x.dtype], d.at(off), out.ptr, rest.ptr, n,
                                         ca.C.byref(pred), cnt.ptr))
        assert np.array_equal(out.to_host(queue)[:got], x[keep]), n
        assert np.array_equal(rest.to_host(queue)[:n - got], x[~keep]), n
        got = ca.unique(queue, d, out, n=n, in_ptr=d.at(off))
        first = np.concatenate([[True], x[1:] != x[:-1]])
        assert got == first.sum() and np.array_equal(out.to_host(queue)[:got], x[first]), n
        assert ca.count_if(queue, d, pred, n=n, in_ptr=d.at(off)) == keep.sum(), n


@pytest.mark.parametrize("dt", ["int8", "int32", "int64", "float64"])
@pytest.mark.parametrize("aoff,boff", [(0, 0), (1, 1), (1, 3)])
def test_fold_and_transform_edges(queue, dt, aoff, boff):
    rng = np.random.default_rng(boff)
    for n in (1, 3, 511, 2048, 2049, 8193, 1 << 20, (1 << 22) + 5):
        x, y = rng.integers(-9, 9, n).astype(dt), rng.integers(-9, 9, n).astype(dt)
        a, b = _dev(queue, x, aoff), _dev(queue, y, boff)
        out = ca.DeviceArray(n + 2, dt, queue)
        one = ca.DeviceArray(1, dt, queue)
        code = ca.DTYPE[x.dtype]
        ca.check(ca.lib().bcmi_transform(queue.h, code, ca.MINUS, a.at(aoff), b.at(boff), out.at(1), n))
        assert np.array_equal(out.to_host(queue)[1:n + 1], x - y), n
        init = np.array([3], dt)
        ca.check(ca.lib().bcmi_reduce(queue.h, code, ca.PLUS, a.at(aoff), n, init.ctypes.data, one.ptr, None,
                                      ca.COMPENSATED))
        assert one.to_host(queue)[0] == x.sum(dtype=dt) + init[0], n  # whole numbers: exact in every type
        sa, sb = ca.Seq(a.at(aoff).value, 0), ca.Seq(b.at(boff).value, 0)
        m = ca.mapping(dt, "id", "multiplies")
        ca.check(ca.lib().bcmi_transform_reduce(queue.h, code, ca.C.byref(sa), ca.C.byref(sb), n, ca.C.byref(m),
                                                ca.PLUS, None, one.ptr, None, ca.COMPENSATED))
        assert one.to_host(queue)[0] == (x * y).sum(dtype=dt), n


@pytest.mark.parametrize("key,shapes", [("__bcmi_scan", [(4, 4), (4, 8), (4, 16), (8, 8), (8, 16)]),
                                        ("__bcmi_reduce_by_key", [(4, 2), (4, 4), (4, 8), (8, 8)])])
def test_tuned_shapes_at_small_sizes(queue, key, shapes):
    """fit_size = 0: the tuned shape at sizes that would take a smaller one."""
    L, rng = ca.lib(), np.random.default_rng(1)
    saved = {}
    for p, d in (("q", 8 if "key" in key else 16), ("waves", 4), ("fit_size", 1)):
        v = ca.C.c_uint()
        ca.check(L.bcmi_tune_get(key.encode(), p.encode(), d, ca.C.byref(v)))
        saved[p] = v.value
    try:
        ca.check(L.bcmi_tune_set(key.encode(), b"fit_size", 0))
        for nw, qq in shapes:
            ca.check(L.bcmi_tune_set(key.encode(), b"q", qq))
            ca.check(L.bcmi_tune_set(key.encode(), b"waves", nw))
            for n in (1000, 32768 * 3 + 5, 300007):
                x = rng.integers(-100, 100, n).astype(np.int32)
                d = ca.DeviceArray.from_host(x, queue)
                if key == "__bcmi_scan":
                    o = ca.DeviceArray(n, np.int32, queue)
                    ca.scan(queue, d, o, True, init=1)
                    assert np.array_equal(o.to_host(queue), O.scan(x, True, 1)), (nw, qq, n)
                else:
                    k = np.cumsum(rng.integers(0, 9, n) == 0).astype(np.int32)
                    heads = np.flatnonzero(np.concatenate([[True], k[1:] != k[:-1]]))
                    ko, vo = ca.DeviceArray(n, np.int32, queue), ca.DeviceArray(n, np.int32, queue)
                    assert ca.reduce_by_key(queue, ca.DeviceArray.from_host(k, queue), d, ko, vo) == heads.size
                    assert np.array_equal(vo.to_host(queue)[:heads.size], np.add.reduceat(x, heads)), (nw, qq, n)
    finally:
        for p, v in saved.items():
            ca.check(L.bcmi_tune_set(key.encode(), p.encode(), v))


@pytest.mark.parametrize("dt", ["int8", "uint8", "int16", "uint16"])
def test_narrow_reduce_off_the_grid(queue, dt):
    """Every offset to a 16-byte boundary, ranges that end before it included."""
    rng = np.random.default_rng(2)
    x = rng.integers(np.iinfo(dt).min, np.iinfo(dt).max, 70000, dtype=dt, endpoint=True)
    d = ca.DeviceArray.from_host(x, queue)
    out = ca.DeviceArray(2, dt, queue)
    code = ca.DTYPE[x.dtype]
    for off in range(17):
        for n in (1, 2, 7, 14, 15, 16, 17, 31, 33, 8191, 65537):
            s = x[off:off + n]
            ca.check(ca.lib().bcmi_reduce(queue.h, code, ca.PLUS, d.at(off), n, None, out.ptr, None, ca.COMPENSATED))
            ca.check(ca.lib().bcmi_reduce(queue.h, code, ca.MIN, d.at(off), n, None, out.at(1), None, ca.COMPENSATED))
            got = out.to_host(queue)
            assert got[0] == s.sum(dtype=dt) and got[1] == s.min(), (off, n)
