"""Performance cases of the data-parallel primitives.

Each case is one algorithm call (preceded, for the in-place sorts, by the
device copy that gives it an unsorted range again) on device-resident data,
through the C-ABI of include/bcmi.h -- the entry points that the
boost::compute templates call -- on one queue kept for the whole program, as
system::default_queue() is.

Families:
  sort      bcmi_sort without values (sort, stable_sort)
  sort_kv   bcmi_sort with values (sort_by_key)
  scan      bcmi_scan: exclusive_scan, inclusive_scan
  fold      bcmi_reduce (reduce, accumulate), bcmi_transform_reduce
            (inner_product), bcmi_count_if
  bykey     bcmi_reduce_by_key, bcmi_segmented_scan
  select    bcmi_copy_if, bcmi_unique, bcmi_partition (partition_copy)
  map       bcmi_saxpy (transform with a*_1+_2)
  segsort   bcmi_segmented_sort_plan over a plan built once

A case's "offset" is the position of the range's first element inside its
allocation (a buffer_iterator that does not start at element 0), so offset 1
or 3 gives a range off the 16-byte grid.
"""
import ctypes as C
import math

import numpy as np
import torch

import compute_amd as ca

# torch element types and dtype codes by name.  torch's unsigned types lack
# most operations, so unsigned elements live in signed tensors of their size
# (the bits are what the library sees and what is compared).
TORCH = {"i32": torch.int32, "u32": torch.int32, "i64": torch.int64, "u64": torch.int64, "f32": torch.float32,
         "f64": torch.float64}
CODE = {"i32": ca.I32, "u32": ca.U32, "i64": ca.I64, "u64": ca.U64, "f32": ca.F32, "f64": ca.F64}
SIZE = {"i32": 4, "u32": 4, "i64": 8, "u64": 8, "f32": 4, "f64": 8}

_queue = None


def _q():
    global _queue
    if _queue is None:
        _queue = ca.Queue(0)
    return _queue


def listed():
    return [
        # a list of a few thousand items put in order: latency of one call
        {"name": "sort_i32_3k", "family": "sort", "dtype": "i32", "keys": "full", "descending": False, "n": 3001,
         "offset": 0},
        # the plain sort of the configurations: 2^20 random uint32 keys
        {"name": "sort_u32_1m", "family": "sort", "dtype": "u32", "keys": "full", "descending": False, "n": 1 << 20,
         "offset": 0},
        # the headline: 2^27 random uint32 keys
        {"name": "sort_u32_128m", "family": "sort", "dtype": "u32", "keys": "full", "descending": False,
         "n": 1 << 27, "offset": 0},
        # float keys with duplicates and signed zeros carrying the element's
        # index, a sort by score whose order is then applied to other columns
        {"name": "sort_kv_f32_u32_33m", "family": "sort_kv", "dtype": "f32", "keys": "full", "value_bytes": 4,
         "descending": False, "n": 33554393, "offset": 0},
        # 64-bit keys (hashes, packed coordinates) with 32-bit payload at an
        # ordinary ragged size
        {"name": "sort_kv_u64_u32_1m5", "family": "sort_kv", "dtype": "u64", "keys": "full", "value_bytes": 4,
         "descending": False, "n": 1500007, "offset": 0},
        # offsets from counts (exclusive scan of int) at an ordinary size
        {"name": "scan_excl_i32_1m", "family": "scan", "dtype": "i32", "exclusive": True, "n": 1000003, "offset": 0},
        # compensated inclusive scan of 2^28 floats with heavy cancellation
        {"name": "scan_incl_f32_268m", "family": "scan", "dtype": "f32", "exclusive": False, "n": 1 << 28,
         "offset": 0},
        # accumulate of a small float range: latency of one call
        {"name": "reduce_f32_65k", "family": "fold", "op": "reduce", "dtype": "f32", "n": 65537, "offset": 0},
        # group-by sums over sorted int keys (runs of mean length 32)
        {"name": "rbk_i32_f32_50m", "family": "bykey", "op": "reduce", "dtype": "f32", "n": 50000017, "offset": 0},
        # filter of a mid-sized column: about half of the elements kept
        {"name": "copy_if_i32_4m", "family": "select", "op": "copy_if", "dtype": "i32", "n": 4194301, "offset": 0},
        # saxpy over ten million elements
        {"name": "saxpy_f32_10m", "family": "map", "dtype": "f32", "n": 10000019, "offset": 0},
        # the batched workload: 65,536 uneven segments of uint64 keys with
        # uint32 payload, about 2^26 pairs
        {"name": "segsort_u64_u32_65k", "family": "segsort", "dtype": "u64", "value_bytes": 4, "segments": 65536,
         "median": 256, "longest": 1 << 20},
    ]


def _log(rng, lo, hi):
    """A size between lo and hi, even over the logarithm, mostly odd."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(hi, n | 1) if rng.random() < 0.8 else n


def draw(rng):
    family = rng.choice(["sort", "sort", "sort_kv", "sort_kv", "scan", "scan", "fold", "bykey", "select", "map",
                         "segsort"])
    offset = rng.choice([0, 0, 0, 1, 3])
    if family == "sort":
        dtype = rng.choice(["u32", "i32", "f32", "u64", "i64", "f64"])
        top = 1 << 27 if SIZE[dtype] == 4 else 1 << 24
        return {"family": family, "dtype": dtype, "keys": rng.choice(["full", "full", "narrow"]),
                "descending": rng.random() < 0.25, "n": _log(rng, 1000, top), "offset": offset}
    if family == "sort_kv":
        dtype = rng.choice(["f32", "u32", "i32", "u64", "i64", "f64"])
        top = 1 << 25 if SIZE[dtype] == 4 else 1 << 23
        return {"family": family, "dtype": dtype, "keys": rng.choice(["full", "full", "narrow"]),
                "value_bytes": rng.choice([4, 4, 8]), "descending": rng.random() < 0.25, "n": _log(rng, 1000, top),
                "offset": offset}
    if family == "scan":
        dtype = rng.choice(["i32", "u32", "f32", "i64", "f64"])
        top = (1 << 30) // SIZE[dtype]
        return {"family": family, "dtype": dtype, "exclusive": rng.random() < 0.5, "n": _log(rng, 1000, top),
                "offset": offset}
    if family == "fold":
        op = rng.choice(["reduce", "inner_product", "count_if"])
        dtype = rng.choice(["f32", "f32", "i32", "f64"])
        return {"family": family, "op": op, "dtype": dtype, "n": _log(rng, 1000, (1 << 30) // SIZE[dtype]),
                "offset": offset}
    if family == "bykey":
        return {"family": family, "op": rng.choice(["reduce", "scan"]), "dtype": rng.choice(["f32", "f32", "i32", "f64"]),
                "n": _log(rng, 1000, 1 << 26), "offset": offset}
    if family == "select":
        return {"family": family, "op": rng.choice(["copy_if", "unique", "partition"]),
                "dtype": rng.choice(["i32", "f32", "i64"]), "n": _log(rng, 1000, 1 << 27), "offset": offset}
    if family == "map":
        return {"family": family, "dtype": "f32", "n": _log(rng, 1000, 1 << 27), "offset": offset}
    return {"family": family, "dtype": rng.choice(["u64", "u64", "u32", "f32"]), "value_bytes": rng.choice([0, 4]),
            "segments": _log(rng, 64, 40000), "median": rng.choice([64, 256]), "longest": 1 << 20}


# ------------------------------------------------------------------ inputs
def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 2654435761 % (1 << 62) + 12345)


def _range(n, dtype, offset):
    """n elements `offset` elements into their allocation."""
    return torch.empty(n + offset, dtype=TORCH[dtype], device="cuda")[offset:]


def _uniform(n, dtype, g, lo, hi):
    return torch.empty(n, dtype=TORCH[dtype], device="cuda").uniform_(lo, hi, generator=g)


def _keys(n, dtype, kind, g):
    """Sort keys.  full: integers over the type's whole range; floats uniform
    in [-1e6, 1e6], 1 % of them replaced by +-0 and every 16th a duplicate of
    the key before it.  narrow: identifiers below 50,000."""
    if kind == "narrow":
        return torch.randint(0, 50000, (n,), device="cuda", generator=g).to(TORCH[dtype])
    if dtype in ("f32", "f64"):
        k = _uniform(n, dtype, g, -1e6, 1e6)
        zero = torch.randint(0, 200, (n,), device="cuda", generator=g)
        k[zero == 0] = 0.0
        k[zero == 1] = -0.0
        sixteens = k[:n - n % 16].view(-1, 16)
        sixteens[:, 1] = sixteens[:, 0]
        return k
    if SIZE[dtype] == 4:
        return torch.randint(-(1 << 31), 1 << 31, (n,), device="cuda", generator=g).to(torch.int32)
    lo = torch.randint(0, 1 << 32, (n,), device="cuda", generator=g)
    hi = torch.randint(-(1 << 31), 1 << 31, (n,), device="cuda", generator=g)
    return (hi << 32) | lo


def _numbers(n, dtype, g):
    """Values to add up.  Floats: lognormal(0, 3) with random signs (heavy
    cancellation, the precision workload); integers: uniform in [-100, 100],
    unsigned in [0, 100]."""
    if dtype in ("f32", "f64"):
        x = torch.empty(n, dtype=TORCH[dtype], device="cuda").log_normal_(0.0, 3.0, generator=g)
        x[torch.randint(0, 2, (n,), device="cuda", generator=g) == 0] *= -1.0
        return x
    return torch.randint(0 if dtype == "u32" else -100, 101, (n,), device="cuda", generator=g).to(TORCH[dtype])


def _runs(n, g):
    """Sorted int32 keys in runs of geometric length, mean 32."""
    heads = torch.randint(0, 32, (n,), device="cuda", generator=g) == 0
    return heads.to(torch.int32).cumsum(0, dtype=torch.int32)


def _placed(x, offset):
    """x copied to a range `offset` elements into its allocation."""
    y = torch.empty(x.numel() + offset, dtype=x.dtype, device="cuda")[offset:]
    y.copy_(x)
    return y


def _inputs(case, seed):
    g, f = _rng(seed), case["family"]
    if f == "segsort":
        # the same lengths for every seed, in another order
        r = np.random.RandomState(case["segments"])
        sigma = math.sqrt(2.0 * math.log(4.0))  # mean = 4 medians
        lens = np.clip(np.rint(r.lognormal(math.log(case["median"]), sigma, case["segments"])), 1, case["longest"])
        lens = np.random.RandomState(int(seed) % (1 << 31)).permutation(lens)
        off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
        n = int(off[-1])
        return {"offsets": off, "keys": _keys(n, case["dtype"], "full", g),
                "values": torch.arange(n, dtype=torch.int32, device="cuda") if case["value_bytes"] else None}
    n, dtype, at = case["n"], case["dtype"], case["offset"]
    if f in ("sort", "sort_kv"):
        v = None
        if f == "sort_kv":
            v = _placed(torch.arange(n, dtype=torch.int32 if case["value_bytes"] == 4 else torch.int64,
                                     device="cuda"), at)
        return {"keys": _placed(_keys(n, dtype, case["keys"], g), at), "values": v}
    if f == "bykey":
        if dtype == "i32":
            v = _numbers(n, dtype, g)
        else:  # N(0, 1) * 10^U(-3, 3)
            v = torch.empty(n, dtype=TORCH[dtype], device="cuda").normal_(generator=g)
            v *= 10.0 ** _uniform(n, dtype, g, -3.0, 3.0)
        return {"keys": _placed(_runs(n, g), at), "values": _placed(v, at)}
    if f == "select":
        if case["op"] == "unique":
            return {"x": _placed(_runs(n, g).to(TORCH[dtype]), at)}
        return {"x": _placed(_keys(n, dtype, "full", g), at)}
    if f == "map" or case.get("op") == "inner_product":
        if dtype == "i32":
            a, b = _numbers(n, dtype, g), _numbers(n, dtype, g)
        else:
            a = torch.empty(n, dtype=TORCH[dtype], device="cuda").normal_(generator=g)
            b = torch.empty(n, dtype=TORCH[dtype], device="cuda").normal_(generator=g)
        return {"x": _placed(a, at), "y": _placed(b, at)}
    return {"x": _placed(_numbers(n, dtype, g), at)}


SAXPY_A = 2.5


# ------------------------------------------------------------ one pass each
def _ptr(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def prepare(case, seed):
    q, f = _q(), case["family"]
    s = {"family": f, "op": case.get("op"), "code": CODE[case["dtype"]], "n": case.get("n", 0)}
    s.update(_inputs(case, seed))
    n, dtype, at = s["n"], case["dtype"], case.get("offset", 0)
    dev = {"device": "cuda"}
    if f in ("sort", "sort_kv", "segsort"):
        n = s["n"] = s["keys"].numel()
        s["vb"] = case.get("value_bytes", 0)
        s["descending"] = int(case.get("descending", False))
        s["out"] = [_range(n, dtype, at)]
        if s["values"] is not None:
            s["out"].append(torch.empty(n + at, dtype=s["values"].dtype, **dev)[at:])
        if f == "segsort":
            s["plan"] = ca.SegmentedPlan(q, np.dtype({"u64": np.uint64, "u32": np.uint32, "f32": np.float32}[dtype]),
                                         np.uint32 if s["vb"] else None, s["offsets"])
    elif f in ("scan", "map"):
        s["exclusive"] = int(case.get("exclusive", False))
        s["out"] = [_range(n, dtype, at)]
        # exclusive_scan's init, as the host value the call takes
        s["init"] = np.zeros(1, {"i32": np.int32, "u32": np.uint32, "i64": np.int64, "f32": np.float32,
                                 "f64": np.float64}[dtype])
    elif f == "fold":
        if s["op"] == "count_if":
            np_t = {"i32": np.int32, "f32": np.float32, "f64": np.float64}[dtype]
            s["pred"] = ca.predicate(np_t, ">", 0)
            s["out"] = [torch.zeros(1, dtype=torch.int64, **dev)]
        else:
            s["out"] = [torch.zeros(1, dtype=TORCH[dtype], **dev)]
            s["f64"] = torch.zeros(1, dtype=torch.float64, **dev)
            if dtype != "i32":
                s["out"].append(s["f64"])
            s["map"] = ca.Map(ca.MULTIPLIES, ca.MAP_ID, 0)
            if "y" in s:
                s["a"], s["b"] = ca.Seq(s["x"].data_ptr(), 0), ca.Seq(s["y"].data_ptr(), 0)
    elif f == "bykey":
        if s["op"] == "reduce":
            s["out"] = [torch.zeros(n, dtype=torch.int32, **dev), torch.zeros(n, dtype=TORCH[dtype], **dev),
                        torch.zeros(1, dtype=torch.int64, **dev)]
        else:
            s["out"] = [_range(n, dtype, at)]
            s["init"] = np.zeros(1, {"i32": np.int32, "f32": np.float32, "f64": np.float64}[dtype])
    else:  # select
        np_t = {"i32": np.int32, "i64": np.int64, "f32": np.float32}[dtype]
        s["pred"] = ca.predicate(np_t, ">=", 0)
        # zeroed once: positions past the count stay as they are
        s["out"] = [torch.zeros(n, dtype=TORCH[dtype], **dev), torch.zeros(1, dtype=torch.int64, **dev)]
        if s["op"] == "partition":
            s["out"].insert(1, torch.zeros(n, dtype=TORCH[dtype], **dev))
    torch.cuda.synchronize()  # the queue's stream does not wait for torch's
    return s


def _copy(q, dst, src):
    ca.check(ca.lib().bcmi_memcpy(q, _ptr(dst), _ptr(src), src.numel() * src.element_size(), ca.D2D, 0))


def run(s):
    q, L, f, out, n = _q().h, ca.lib(), s["family"], s["out"], s["n"]
    if f in ("sort", "sort_kv", "segsort"):
        _copy(q, out[0], s["keys"])
        vals = None
        if s["values"] is not None:
            _copy(q, out[1], s["values"])
            vals = _ptr(out[1])
        if f == "segsort":
            ca.check(L.bcmi_segmented_sort_plan(q, s["plan"].h, _ptr(out[0]), vals))
        else:
            ca.check(L.bcmi_sort(q, ca.SORT_BY_KEY if vals else ca.SORT, s["code"], _ptr(out[0]), vals, s["vb"], n,
                                 s["descending"]))
    elif f == "scan":
        ca.check(L.bcmi_scan(q, s["code"], ca.PLUS, _ptr(s["x"]), _ptr(out[0]), n, s["init"].ctypes.data,
                             s["exclusive"], ca.COMPENSATED))
    elif f == "map":
        ca.check(L.bcmi_saxpy(q, SAXPY_A, _ptr(s["x"]), _ptr(s["y"]), _ptr(out[0]), n))
    elif f == "fold":
        if s["op"] == "count_if":
            ca.check(L.bcmi_count_if(q, s["code"], _ptr(s["x"]), n, C.byref(s["pred"]), _ptr(out[0])))
        elif s["op"] == "reduce":
            ca.check(L.bcmi_reduce(q, s["code"], ca.PLUS, _ptr(s["x"]), n, None, _ptr(out[0]),
                                   C.cast(_ptr(s["f64"]), C.POINTER(C.c_double)), ca.COMPENSATED))
        else:
            ca.check(L.bcmi_transform_reduce(q, s["code"], C.byref(s["a"]), C.byref(s["b"]), n, C.byref(s["map"]),
                                             ca.PLUS, None, _ptr(out[0]),
                                             C.cast(_ptr(s["f64"]), C.POINTER(C.c_double)), ca.COMPENSATED))
    elif f == "bykey":
        if s["op"] == "reduce":
            ca.check(L.bcmi_reduce_by_key(q, ca.I32, s["code"], ca.PLUS, _ptr(s["keys"]), _ptr(s["values"]), n,
                                          _ptr(out[0]), _ptr(out[1]), _ptr(out[2]), ca.COMPENSATED))
        else:
            ca.check(L.bcmi_segmented_scan(q, ca.I32, s["code"], _ptr(s["keys"]), _ptr(s["values"]), _ptr(out[0]), n,
                                           s["init"].ctypes.data, 1, ca.COMPENSATED))
    elif s["op"] == "copy_if":
        ca.check(L.bcmi_copy_if(q, s["code"], _ptr(s["x"]), _ptr(out[0]), n, C.byref(s["pred"]), ca.SELECT_VALUES,
                                _ptr(out[1])))
    elif s["op"] == "unique":
        ca.check(L.bcmi_unique(q, s["code"], _ptr(s["x"]), _ptr(out[0]), n, _ptr(out[1])))
    else:
        ca.check(L.bcmi_partition(q, s["code"], _ptr(s["x"]), _ptr(out[0]), _ptr(out[1]), n, C.byref(s["pred"]),
                                  _ptr(out[2])))
    return out


# ------------------------------------------------------------ work, results
def work(case):
    f, b = case["family"], SIZE[case["dtype"]]
    if f == "segsort":
        # expected total: mean length 4 medians (the clip at `longest` cuts
        # a fraction of a percent)
        return {"bytes": 2.0 * case["segments"] * 4 * case["median"] * (b + case["value_bytes"]), "flops": 0}
    n = case["n"]
    if f == "sort":
        return {"bytes": 2 * n * b, "flops": 0}
    if f == "sort_kv":
        return {"bytes": 2 * n * (b + case["value_bytes"]), "flops": 0}
    if f == "scan":
        return {"bytes": 2 * n * b, "flops": n}
    if f == "map":
        return {"bytes": 3 * n * b, "flops": 2 * n}
    if f == "fold":
        return {"bytes": n * b * (2 if case["op"] == "inner_product" else 1), "flops": n}
    if f == "bykey":
        # one run per 32 elements
        return {"bytes": n * (4 + b) + (n // 32) * (4 + b) if case["op"] == "reduce" else n * (4 + 2 * b), "flops": n}
    kept = {"copy_if": 0.5, "unique": 1 / 32, "partition": 1.0}[case["op"]]
    return {"bytes": n * b * (1 + kept), "flops": 0}


def tolerance(case):
    """Moved and counted values and integer sums are exact.  Float sums are
    compensated and rounded once to float, so two correct orders differ by
    at most one rounding of the result: 2.7e-8 (2-norm) and 6e-8 (largest)
    measured against 64 bits.  FP64 sums in two orders differ by 2.4e-15 and
    1.8e-14 over 2^26 terms."""
    f, dtype = case["family"], case["dtype"]
    if dtype not in ("f32", "f64") or f in ("sort", "sort_kv", "select", "segsort") or case.get("op") == "count_if":
        return "exact"
    if f == "map":
        return "exact"  # one fused multiply-add per element
    if dtype == "f64":
        return {"rel": 2e-14, "max": 1e-13}
    if f == "fold":
        return {"rel": 2.5e-7, "max": 2.5e-7}
    return {"rel": 1.5e-7, "max": 2.5e-7}


def exact(case, seed):
    """The float results in 64 bits.  Integer results, and results that only
    move input values, have no rounding to measure."""
    f, dtype = case["family"], case["dtype"]
    if dtype not in ("f32", "f64") or f in ("sort", "sort_kv", "select", "segsort") or case.get("op") == "count_if":
        return None
    s = _inputs(case, seed)
    if f == "map":
        return [SAXPY_A * s["x"].double() + s["y"].double()]
    if f == "scan":
        c = s["x"].double().cumsum(0)
        if not case["exclusive"]:
            return [c]
        return [torch.cat([torch.zeros(1, dtype=torch.float64, device="cuda"), c[:-1]])]
    if f == "fold":
        t = s["x"].double()
        if case["op"] == "inner_product":
            t = t * s["y"].double()
        # math.fsum of partial sums: the cancellation leaves little of the sum
        t = math.fsum(t.cpu().numpy().tolist()) if t.numel() <= 1 << 22 else float(t.sum())
        return [torch.tensor([t], dtype=torch.float64)] * 2
    # bykey: each run summed by itself
    k, v = s["keys"], s["values"].double()
    group = (k - k[0]).long()
    if case["op"] == "reduce":
        n, runs = case["n"], int(group[-1]) + 1
        sums = torch.zeros(n, dtype=torch.float64, device="cuda")
        sums.index_add_(0, group, v)
        keys = torch.zeros(n, dtype=torch.int32, device="cuda")
        keys[:runs] = torch.arange(runs, dtype=torch.int32, device="cuda") + k[0]
        return [keys, sums, torch.tensor([runs])]
    # exclusive within each run: running sum minus the running sum at the
    # run's head loses digits, so long inputs have no such value
    if case["n"] > 1 << 20:
        return None
    v, group = v.cpu().numpy(), group.cpu().numpy()
    out = np.zeros(case["n"])
    total, last = 0.0, -1
    for i in range(case["n"]):
        if group[i] != last:
            total, last = 0.0, group[i]
        out[i] = total
        total += v[i]
    return [out]
