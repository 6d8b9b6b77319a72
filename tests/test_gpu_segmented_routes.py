"""Segmented plans large enough that the all-digits passes take a side stream:
both routes of large segments beside each other and small segments beside
both, eager and captured, and plans that share a queue's side streams, against
the oracle's sort of every segment."""
import os
import re

import numpy as np
import pytest

import compute_amd as ca
import oracle as O

pytestmark = pytest.mark.gpu

CSRC = os.path.join(os.path.dirname(ca.LIB_PATH), "csrc")


def _fork_tiles():
    with open(os.path.join(CSRC, "segmented.hpp")) as f:
        return int(re.search(r"kForkLsdTiles = (\d+)", f.read()).group(1))


def _keys(dt, off, crowded, rng):
    """Spread keys, which take the top-digit route; in segments of `crowded`
    the top digit is one value, which sends them through all digits."""
    n, t = int(off[-1]), np.dtype(dt)
    if t.kind == "f":
        k = rng.uniform(1.0, 2.0, n).astype(t)  # one octave: the top byte never changes
        spread = (10.0 ** rng.uniform(-30, 30, n) * rng.choice([-1.0, 1.0], n)).astype(t)
    else:
        k = rng.integers(0, 1 << 20, n).astype(t)
        spread = rng.integers(0, 256, n * t.itemsize, dtype=np.uint8).view(t)
    keep = np.repeat(crowded, np.diff(off).astype(np.int64))
    return np.where(keep, k, spread)


@pytest.mark.parametrize("dt,vdt,small", [("uint64", "uint32", 1500), ("float32", None, 1500), ("int32", "uint64", 0)])
def test_both_routes_beside_each_other(queue, dt, vdt, small):
    rng = np.random.default_rng(len(dt))
    # a segment of 4100 to 6000 elements makes at least one tile of any tile size
    large = rng.integers(4100, 6000, _fork_tiles() + 50)
    lens = np.concatenate([large, rng.integers(0, 2000, small)])
    lens = lens[rng.permutation(lens.size)]
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    n = int(off[-1])
    plan = ca.SegmentedPlan(queue, np.dtype(dt), np.dtype(vdt) if vdt else None, off)
    dk = ca.DeviceArray(n, dt, queue)
    dv = ca.DeviceArray(n, vdt, queue) if vdt else None
    v = np.arange(n, dtype=vdt) if vdt else None
    graph = ca.Graph(queue)
    with graph:
        plan.run(queue, dk, dv)

    def put(d, a):
        ca.check(ca.lib().bcmi_memcpy(queue.h, d.ptr, a.ctypes.data_as(ca.C.c_void_p), a.nbytes, ca.H2D, 1))

    # all segments on one route, half on each, the halves exchanged, all on the other
    half = np.arange(lens.size) % 2 == 0
    for crowded in (np.zeros(lens.size, bool), half, ~half, np.ones(lens.size, bool)):
        k = _keys(dt, off, crowded, rng)
        e = O.segmented_sort(k, v, off)
        ek, ev = e if vdt else (e, None)
        bits = "u%d" % k.dtype.itemsize
        for run in (lambda: plan.run(queue, dk, dv), graph.launch, graph.launch):
            put(dk, k)
            if vdt:
                put(dv, v)
            run()
            queue.finish()
            assert np.array_equal(dk.to_host(queue).view(bits), ek.view(bits))
            if vdt:
                assert np.array_equal(dv.to_host(queue), ev)


def test_plans_share_a_queues_side_streams():
    """Two plans of one queue in turn, and a plan run on a queue it was not
    built on: eagerly, and captured before that queue has side streams."""
    rng = np.random.default_rng(3)
    built, other = ca.Queue(0), ca.Queue(0)
    plans = []
    for _ in range(2):
        lens = np.concatenate([rng.integers(4100, 30000, 20), rng.integers(0, 2000, 300)])
        off = np.concatenate([[0], np.cumsum(lens[rng.permutation(lens.size)])]).astype(np.uint64)
        plans.append((off, ca.SegmentedPlan(built, np.uint32, None, off)))
    captured = ca.DeviceArray(int(plans[0][0][-1]), np.uint32, other)
    other.reserve(1 << 21, 8)  # no call below grows its scratch: that would retire the graph
    graph = ca.Graph(other)
    with graph:
        plans[0][1].run(other, captured)
    for rep in range(3):
        done = []
        for q in (built, other):
            for off, plan in plans:
                k = rng.integers(0, 1 << 32, int(off[-1]), dtype=np.uint64).astype(np.uint32)
                k[: k.size // 3] &= 0xFFFF
                d = ca.DeviceArray.from_host(k, q)
                plan.run(q, d)
                # a plan's temporaries serve one run at a time
                q.finish()
                done.append((d, q, O.segmented_sort(k, None, off)))
        k = rng.integers(0, 1 << 20, captured.size, dtype=np.uint64).astype(np.uint32)
        ca.check(ca.lib().bcmi_memcpy(other.h, captured.ptr, k.ctypes.data_as(ca.C.c_void_p), k.nbytes, ca.H2D, 1))
        graph.launch()
        done.append((captured, other, O.segmented_sort(k, None, plans[0][0])))
        for d, q, e in done:
            q.finish()
            assert np.array_equal(d.to_host(q), e), rep
    for q in (built, other):
        q.close()


@pytest.mark.parametrize("dt", ["uint8", "int16", "uint32", "int32", "uint64", "int64"])
def test_crowded_bins(queue, dt):
    """Small integer segments on both sides of what the bins hold (32 keys
    each): as many values as the segment just needs, one more and one fewer,
    away from zero and at the type's ends; one bin of 31 to 34 keys among
    spread ones; keys spread over octaves; equal keys in input order."""
    rng = np.random.default_rng(np.dtype(dt).itemsize)
    info, parts = np.iinfo(dt), []
    for n in (33, 63, 64, 65, 96, 97, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047, 2048):
        for values in sorted({max(1, -(-n // 32) + d) for d in (-1, 0, 1)} | {2}):
            lo = (info.min, 7, info.max - values + 1)[rng.integers(3)]
            k = (np.arange(n) % values).astype(dt) + np.array(lo, dt)  # as even as it gets
            parts += [k, rng.permutation(k)]
        for crowd in (31, 32, 33, 34):
            k = rng.integers(info.min, info.max, n, dtype=dt, endpoint=True)
            k[rng.permutation(n)[:crowd]] = 3
            parts.append(k)
        parts.append(np.exp2(rng.uniform(0, np.log2(float(info.max)) - 0.01, n)).astype(dt))
    off = np.concatenate([[0], np.cumsum([p.size for p in parts])]).astype(np.uint64)
    k = np.concatenate(parts)
    v = np.arange(k.size, dtype=np.uint32)
    for desc in (False, True):
        dk, dv = ca.DeviceArray.from_host(k, queue), ca.DeviceArray.from_host(v, queue)
        ca.segmented_sort(queue, dk, dv, off, descending=desc)
        ek, ev = O.segmented_sort(k, v, off, descending=desc)
        assert np.array_equal(dk.to_host(queue), ek), desc
        assert np.array_equal(dv.to_host(queue), ev), desc
