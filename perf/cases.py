"""The work that a program gives this library, as cases to time and compare.

A case is one call of the public host layer (`rccl_amd.cub`, the asynchronous
calls with caller-owned workspaces, or `rccl_amd.thrust` /
`rccl_amd.record_sort`, which allocate and wait as Thrust does) on inputs with
the benchmark's and the tests' distributions:

  radix       DeviceRadixSort of a copy of a column, keys or stable pairs. The
              sort works in place, so a program that keeps its column copies
              it first; that copy is part of the pass.
  merge_sort  DeviceMergeSort, copy form, keys or pairs, either order
  merge       DeviceMerge of two sorted ranges, keys or pairs
  set         the four set operations, written out (keys or pairs) or counted
  record      record_sort: lexicographic rows of u32 columns with a payload
  reduce      reduce_by_key over runs of equal adjacent keys

Every result is whole numbers, bit patterns or (reduce) a wrapping u64 sum, so
outputs compare exactly. Buffers and workspaces belong to the state: programs
keep them from call to call.
"""
import math

import numpy as np
import torch

from rccl_amd import cub, record_sort, thrust
from rccl_amd.device import DeviceBuffer

DEV = "cuda:0"
SIZE = {"u32": 4, "i32": 4, "f32": 4, "u64": 8, "i64": 8, "f64": 8, "u16": 2}
NP = {"u32": np.uint32, "i32": np.int32, "f32": np.float32, "u64": np.uint64, "i64": np.int64,
      "f64": np.float64, "u16": np.uint16}
TORCH = {2: torch.int16, 4: torch.int32, 8: torch.int64}
VALUE = {0: None, 4: np.uint32, 8: np.uint64}

_program = None


def _launch():
    global _program
    if _program is None:
        _program = cub.Program.load(0)
    return _program.on(torch.cuda.current_stream(0))


def listed():
    return [
        # The smallest sorts: a few thousand index pairs, one launch on one CU.
        {"name": "radix_pairs_2000", "op": "radix", "kind": "u32", "value": 4, "order": "asc",
         "dist": "uniform", "n": 2000},
        # An ordinary latency-bound sort: 2^20 keys, the benchmark's smallest configuration.
        {"name": "radix_u32_2e20", "op": "radix", "kind": "u32", "value": 0, "order": "asc",
         "dist": "uniform", "n": 1 << 20},
        # Floats, descending, with signed zeros, infinities, denormals and NaNs; an odd length.
        {"name": "radix_f32_desc_20m", "op": "radix", "kind": "f32", "value": 0, "order": "desc",
         "dist": "special", "n": 20_000_003},
        # A dictionary-coded column: 64-bit codes, 256 of them, Zipf frequencies; row numbers move.
        {"name": "radix_u64_u32_zipf_2e26", "op": "radix", "kind": "u64", "value": 4,
         "order": "asc", "dist": "zipf", "n": 1 << 26},
        # The headline sort: 2^28 uniform 32-bit keys.
        {"name": "radix_u32_2e28", "op": "radix", "kind": "u32", "value": 0, "order": "asc",
         "dist": "uniform", "n": 1 << 28},
        # A stable comparator sort of a mid-sized odd number of pairs, descending.
        {"name": "merge_sort_u64_u32_50001", "op": "merge_sort", "kind": "u64", "value": 4,
         "order": "desc", "dist": "uniform", "n": 50_001},
        # The large comparator sort: 2^26 keys below 2^24.
        {"name": "merge_sort_u32_2e26", "op": "merge_sort", "kind": "u32", "value": 0,
         "order": "asc", "dist": "low24", "n": 1 << 26},
        # Merging two sorted runs of 2^27 pairs with heavy duplicates.
        {"name": "merge_u32_u32_2e27", "op": "merge", "kind": "u32", "value": 4, "order": "asc",
         "na": 1 << 27, "nb": 1 << 27},
        # Set union of two large sorted multisets of 64-bit keys.
        {"name": "union_u64_2e26", "op": "set", "set": "union", "kind": "u64", "value": 0,
         "write": True, "na": 1 << 26, "nb": 1 << 26},
        # A mid-sized join-like intersection that carries values, ragged and unequal.
        {"name": "intersect_u32_u32_3m", "op": "set", "set": "intersection", "kind": "u32",
         "value": 4, "write": True, "na": 3_000_017, "nb": 1_234_567},
        # A relation's rows in lexicographic order with provenance payloads (record_sort).
        {"name": "record4_u64_2e20", "op": "record", "arity": 4, "value": 8, "n": (1 << 20) + 13},
        # Aggregation after such a sort: sums over runs of equal keys.
        {"name": "reduce_u32_u64_2e20", "op": "reduce", "kind": "u32", "value": 8,
         "n": (1 << 20) + 13},
    ]


def _size(rng, lo, hi):
    """Log-uniform in [lo, hi]; hardly ever a round number."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["radix", "radix", "radix", "merge_sort", "merge_sort", "merge", "set", "set",
                     "record", "reduce"])
    if op in ("radix", "merge_sort"):
        kind = rng.choice(["u32", "u32", "i32", "f32", "u64", "i64", "f64"])
        value = rng.choice([0, 4, 8])
        dist = rng.choice(["uniform", "uniform", "low24", "zipf", "special"])
        if dist == "special" and kind not in ("f32", "f64") or op == "merge_sort" and dist == "special":
            dist = "uniform"
        # At most the bytes of the 2^26-pair case (12 bytes each).
        top = min(1 << 28, (3 << 28) // (SIZE[kind] + value))
        return {"op": op, "kind": kind, "value": value, "order": rng.choice(["asc", "desc"]),
                "dist": dist, "n": _size(rng, 1000, top)}
    if op == "merge":
        kind, value = rng.choice(["u32", "i32", "u64", "f32"]), rng.choice([0, 4, 8])
        top = (1 << 30) // (SIZE[kind] + value)
        return {"op": op, "kind": kind, "value": value, "order": rng.choice(["asc", "desc"]),
                "na": _size(rng, 1000, top), "nb": _size(rng, 1000, top)}
    if op == "set":
        kind, value = rng.choice(["u32", "u64"]), rng.choice([0, 0, 4])
        na = _size(rng, 1000, (1 << 29) // (SIZE[kind] + value))
        nb = max(500, int(na * math.exp(rng.uniform(-2.0, 0.0))))
        if rng.random() < 0.5:
            na, nb = nb, na
        return {"op": op, "kind": kind, "value": value, "write": value > 0 or rng.random() < 0.75,
                "set": rng.choice(["union", "intersection", "difference", "symmetric_difference"]),
                "na": na, "nb": nb}
    if op == "record":
        return {"op": op, "arity": rng.randint(2, 6), "value": rng.choice([0, 8]),
                "n": _size(rng, 2000, 1 << 24)}
    return {"op": op, "kind": rng.choice(["u32", "u64"]), "value": 8, "n": _size(rng, 2000, 1 << 26)}


# ---------------------------------------------------------------------------
# Inputs, made on the GPU.
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1_000_003 + 17)
    return g


def _bits(n, size, g):
    """n uniform bit patterns of `size` bytes, as a signed torch integer type."""
    info = torch.iinfo(TORCH[size])
    t = torch.empty(n, dtype=TORCH[size], device=DEV)
    if size == 8:
        lo = torch.randint(0, 1 << 32, (n,), generator=g, device=DEV, dtype=torch.int64)
        hi = torch.randint(-(1 << 31), 1 << 31, (n,), generator=g, device=DEV, dtype=torch.int64)
        return torch.bitwise_or(hi << 32, lo)
    return t.random_(info.min, info.max + 1, generator=g)


def _column(kind, dist, n, g):
    """A key column: bit patterns in the signed integer type of the key's width."""
    size = SIZE[kind]
    if dist == "zipf":
        weights = torch.arange(1, 257, dtype=torch.float64, device=DEV).pow_(-1.1)
        cdf = torch.cumsum(weights / weights.sum(), 0)
        u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
        at = torch.searchsorted(cdf, u, right=True).clamp_(max=255)
        if kind[0] == "f":
            book = torch.randn(256, generator=g, device=DEV, dtype=torch.float64)
            return book.to(_float(size))[at].view(TORCH[size])
        return _bits(256, size, g)[at]
    if kind[0] == "f":
        x = torch.randn(n, generator=g, device=DEV, dtype=_float(size)).mul_(1000.0)
        if dist == "low24":
            x.round_()
        x = x.view(TORCH[size])
        if dist == "special":
            _specials(x, size, g)
        return x
    if dist == "low24":
        return torch.randint(0, 1 << 24, (n,), generator=g, device=DEV, dtype=TORCH[size])
    return _bits(n, size, g)


def _float(size):
    return torch.float32 if size == 4 else torch.float64


def _specials(bits, size, g):
    """1% of each zero, 0.1% infinities of each sign and denormals, 0.01% NaNs."""
    n = bits.numel()
    sign = -(1 << (8 * size - 1))
    one = torch.tensor([math.inf], dtype=_float(size)).view(TORCH[size]).item()
    quiet = one | (1 << (22 if size == 4 else 51))
    for share, pattern in ((0.01, 0), (0.01, sign), (0.001, one), (0.001, one + sign),
                           (0.001, 12345), (0.0001, quiet)):
        at = torch.randint(0, n, (max(1, int(n * share)),), generator=g, device=DEV)
        bits[at] = pattern


def _sorted(kind, n, order, g):
    """A sorted run: u32 / i32 below 2^24 with heavy duplicates, 64-bit below 2^28, floats normal."""
    if kind[0] == "f":
        x = torch.randn(n, generator=g, device=DEV, dtype=_float(SIZE[kind])).mul_(1000.0)
    else:
        x = torch.randint(0, 1 << (24 if SIZE[kind] == 4 else 28), (n,), generator=g, device=DEV,
                          dtype=TORCH[SIZE[kind]])
    x = torch.sort(x, descending=order == "desc").values
    return x.view(TORCH[SIZE[kind]])


def _multiset(kind, n, pool, g):
    """A sorted multiset: half its keys from a shared pool, a tenth of them repeated 2-4 times."""
    half = n // 2
    side = torch.cat([pool[torch.randint(0, pool.numel(), (half,), generator=g, device=DEV)],
                      _keys31(kind, n - half, g)])
    side = torch.sort(side).values
    src = torch.randint(0, max(1, n - 4), (n // 10,), generator=g, device=DEV)
    for k in (1, 2, 3):
        s = src[: src.numel() // k]
        side[s + k] = side[s]
    return torch.sort(side).values


def _keys31(kind, n, g):
    bits = 31 if SIZE[kind] == 4 else 62
    return torch.randint(0, 1 << bits, (n,), generator=g, device=DEV, dtype=torch.int64).to(
        TORCH[SIZE[kind]])


def _buffer(tensor, dtype):
    return DeviceBuffer(tensor, dtype, tensor.numel())


def _values(value, n, start=0):
    if not value:
        return None
    t = torch.arange(start, start + n, dtype=torch.int64, device=DEV).to(TORCH[value])
    return _buffer(t, VALUE[value])


def prepare(case, seed):
    g = _gen(seed)
    return {"radix": _prepare_radix, "merge_sort": _prepare_merge_sort, "merge": _prepare_merge,
            "set": _prepare_set, "record": _prepare_record, "reduce": _prepare_reduce}[
                case["op"]](case, g, _launch())


def run(state):
    return state["call"](state)


def _prepare_radix(c, g, launch):
    n, dt = c["n"], NP[c["kind"]]
    s = {"launch": launch, "column": _column(c["kind"], c["dist"], n, g),
         "keys": DeviceBuffer.empty(dt, n)}
    desc = c["order"] == "desc"
    if c["value"]:
        s["rows"] = _values(c["value"], n)
        s["values"] = DeviceBuffer.empty(VALUE[c["value"]], n)
        s["ws"] = cub.device_radix_sort_pairs_workspace(launch, dt, VALUE[c["value"]], n)
        s["sort"] = cub.device_radix_sort_pairs_descending if desc else cub.device_radix_sort_pairs
        s["call"] = _radix_pairs
    else:
        s["ws"] = cub.device_radix_sort_workspace(launch, dt, n)
        s["sort"] = cub.device_radix_sort_keys_descending if desc else cub.device_radix_sort_keys
        s["call"] = _radix_keys
    return s


def _radix_keys(s):
    s["keys"].tensor.copy_(s["column"])
    s["sort"](s["launch"], s["keys"], s["ws"])
    return s["keys"].tensor


def _radix_pairs(s):
    s["keys"].tensor.copy_(s["column"])
    s["values"].copy_from(s["rows"])
    s["sort"](s["launch"], s["keys"], s["values"], s["ws"])
    return [s["keys"].tensor, s["values"].tensor]


def _prepare_merge_sort(c, g, launch):
    n, dt = c["n"], NP[c["kind"]]
    s = {"launch": launch, "keys": _buffer(_column(c["kind"], c["dist"], n, g), dt),
         "out": DeviceBuffer.empty(dt, n),
         "order": cub.descending if c["order"] == "desc" else cub.ascending}
    if c["value"]:
        s["values"] = _values(c["value"], n)
        s["out_values"] = DeviceBuffer.empty(VALUE[c["value"]], n)
        s["ws"] = cub.device_merge_sort_pairs_workspace(launch, dt, VALUE[c["value"]], n)
        s["call"] = _merge_sort_pairs
    else:
        s["ws"] = cub.device_merge_sort_workspace(launch, dt, n)
        s["call"] = _merge_sort_keys
    return s


def _merge_sort_keys(s):
    cub.device_merge_sort_keys_copy(s["launch"], s["keys"], s["ws"], s["out"], s["order"])
    return s["out"].tensor


def _merge_sort_pairs(s):
    cub.device_merge_sort_pairs_copy(s["launch"], s["keys"], s["values"], s["ws"], s["out"],
                                     s["out_values"], s["order"])
    return [s["out"].tensor, s["out_values"].tensor]


def _prepare_merge(c, g, launch):
    na, nb, dt = c["na"], c["nb"], NP[c["kind"]]
    s = {"launch": launch, "a": _buffer(_sorted(c["kind"], na, c["order"], g), dt),
         "b": _buffer(_sorted(c["kind"], nb, c["order"], g), dt),
         "out": DeviceBuffer.empty(dt, na + nb),
         "order": cub.descending if c["order"] == "desc" else cub.ascending}
    if c["value"]:
        vt = VALUE[c["value"]]
        s["av"], s["bv"] = _values(c["value"], na), _values(c["value"], nb, na)
        s["out_values"] = DeviceBuffer.empty(vt, na + nb)
        s["ws"] = cub.device_merge_pairs_workspace(launch, dt, vt, na, nb)
        s["call"] = _merge_pairs
    else:
        s["ws"] = cub.device_merge_workspace(launch, dt, na, nb)
        s["call"] = _merge_keys
    return s


def _merge_keys(s):
    cub.device_merge_keys(s["launch"], s["a"], s["b"], s["ws"], s["out"], s["order"])
    return s["out"].tensor


def _merge_pairs(s):
    cub.device_merge_pairs(s["launch"], s["a"], s["av"], s["b"], s["bv"], s["ws"], s["out"],
                           s["out_values"], s["order"])
    return [s["out"].tensor, s["out_values"].tensor]


def _prepare_set(c, g, launch):
    na, nb, dt = c["na"], c["nb"], NP[c["kind"]]
    pool = _keys31(c["kind"], max(na, nb), g)
    s = {"launch": launch, "op": c["set"], "a": _buffer(_multiset(c["kind"], na, pool, g), dt),
         "b": _buffer(_multiset(c["kind"], nb, pool, g), dt)}
    cap = cub.set_output_capacity(c["set"], na, nb)
    # Zeroed: the places past the result's length are never written.
    s["out"] = DeviceBuffer.zeroed(dt, cap) if c["write"] else None
    if c["value"]:
        vt = VALUE[c["value"]]
        s["av"], s["bv"] = _values(c["value"], na), _values(c["value"], nb, na)
        s["out_values"] = DeviceBuffer.zeroed(vt, cap)
        s["ws"] = cub.device_set_pairs_workspace(launch, c["set"], dt, vt, na, nb)
        s["call"] = _set_pairs
    else:
        s["ws"] = cub.device_set_workspace(launch, c["set"], dt, na, nb)
        s["call"] = _set_keys
    return s


def _set_keys(s):
    cub.device_set_keys(s["launch"], s["op"], s["a"], s["b"], s["ws"], s["out"])
    count = s["ws"].output_count.tensor
    return [count] if s["out"] is None else [count, s["out"].tensor]


def _set_pairs(s):
    cub.device_set_pairs(s["launch"], s["op"], s["a"], s["av"], s["b"], s["bv"], s["ws"],
                         s["out"], s["out_values"])
    return [s["ws"].output_count.tensor, s["out"].tensor, s["out_values"].tensor]


def _prepare_record(c, g, launch):
    n, arity = c["n"], c["arity"]
    # Interned ids: every column holds small numbers, later columns more of them.
    cols = [torch.randint(0, 1 << min(20, 4 + 4 * k), (n,), generator=g, device=DEV,
                          dtype=torch.int32) for k in range(arity)]
    rows = torch.stack(cols, 1).reshape(-1).contiguous()
    s = {"execution": thrust.Program.load(0).par(torch.cuda.current_stream(0)),
         "rows": record_sort.RowBuffer(_buffer(rows, np.uint32), arity, n),
         "out": record_sort.RowBuffer(DeviceBuffer.empty(np.uint32, arity * n), arity, n),
         "call": _record}
    if c["value"]:
        s["payload"] = _values(8, n)
        s["out_payload"] = DeviceBuffer.empty(np.uint64, n)
        s["call"] = _record_payload
    return s


def _record(s):
    record_sort.sort_rows_lexicographic_into(s["execution"], s["rows"], s["out"])
    return s["out"].words.tensor


def _record_payload(s):
    record_sort.sort_rows_with_payload_lexicographic_into(
        s["execution"], s["rows"], s["payload"], s["out"], s["out_payload"])
    return [s["out"].words.tensor, s["out_payload"].tensor]


def _prepare_reduce(c, g, launch):
    n, dt = c["n"], NP[c["kind"]]
    # Runs of one to five equal keys, three on average.
    run = torch.randint(1, 6, (n // 2 + 16,), generator=g, device=DEV)
    first = torch.cumsum(run, 0)
    keys = torch.searchsorted(first, torch.arange(n, device=DEV), right=True).to(
        TORCH[SIZE[c["kind"]]])
    return {"execution": thrust.Program.load(0).par(torch.cuda.current_stream(0)),
            "keys": _buffer(keys, dt), "values": _buffer(_bits(n, 8, g), np.uint64),
            "out": DeviceBuffer.zeroed(dt, n), "sums": DeviceBuffer.zeroed(np.uint64, n),
            "count": DeviceBuffer.zeroed(np.uint64, 1), "call": _reduce}


def _reduce(s):
    thrust.reduce_by_key(s["execution"], s["keys"], s["values"], s["out"], s["sums"], s["count"])
    return [s["count"].tensor, s["out"].tensor, s["sums"].tensor]


def work(case):
    """Every input item read once and every output item written once. Set operations: about
    half of either side is shared."""
    op = case["op"]
    if op in ("radix", "merge_sort"):
        return {"bytes": 2 * case["n"] * (SIZE[case["kind"]] + case["value"]), "flops": 0}
    if op == "merge":
        return {"bytes": 2 * (case["na"] + case["nb"]) * (SIZE[case["kind"]] + case["value"]),
                "flops": 0}
    if op == "set":
        na, nb = case["na"], case["nb"]
        both = min(na, nb) // 4
        out = {"union": na + nb - both, "intersection": both, "difference": na - both,
               "symmetric_difference": na + nb - 2 * both}[case["set"]]
        item = SIZE[case["kind"]]
        # Only the values of kept items are read; a count reads keys alone.
        return {"bytes": (na + nb) * item +
                (out * (item + 2 * case["value"]) if case["write"] else 0), "flops": 0}
    if op == "record":
        return {"bytes": 2 * case["n"] * (4 * case["arity"] + case["value"]), "flops": 0}
    n = case["n"]
    return {"bytes": n * (SIZE[case["kind"]] + 8) + n // 3 * (SIZE[case["kind"]] + 8), "flops": 0}


def tolerance(case):
    return "exact"


# ---------------------------------------------------------------------------
# The same results from plain torch.
# ---------------------------------------------------------------------------
def exact(case, seed):
    g = _gen(seed)
    op = case["op"]
    if op in ("radix", "merge_sort"):
        if case["n"] * SIZE[case["kind"]] > 1 << 28:
            return None
        x = _column(case["kind"], case["dist"], case["n"], g)
        at = torch.sort(_rank(x, case["kind"], case["order"] == "desc"), stable=True).indices
        if not case["value"]:
            return x[at]
        return [x[at], _values(case["value"], case["n"]).tensor[at]]
    if op == "merge":
        if case["na"] + case["nb"] > 1 << 26:
            return None
        a = _sorted(case["kind"], case["na"], case["order"], g)
        b = _sorted(case["kind"], case["nb"], case["order"], g)
        x = torch.cat([a, b])
        at = torch.sort(_rank(x, case["kind"], case["order"] == "desc"), stable=True).indices
        if not case["value"]:
            return x[at]
        v = _values(case["value"], case["na"] + case["nb"]).tensor
        return [x[at], v[at]]
    if op == "set":
        return _exact_set(case, g)
    if op == "record":
        return None if case["n"] > 1 << 22 else _exact_record(case, g)
    return _exact_reduce(case, g)


def _rank(bits, kind, desc):
    """int64 numbers in the order of the keys: unsigned and float orders (both zeros alike)."""
    x = bits.to(torch.int64)
    if kind == "u32":
        x = x & 0xFFFFFFFF
    elif kind == "u64":
        x = x ^ -(1 << 63)
    elif kind[0] == "f":
        low = (1 << (8 * SIZE[kind] - 1)) - 1
        x = torch.where(x < 0, -1 - (x & low), x)
        x = torch.where(x == -1, torch.zeros_like(x), x)
    return ~x if desc else x


def _exact_set(case, g):
    na, nb = case["na"], case["nb"]
    if na + nb > 1 << 25:
        return None
    pool = _keys31(case["kind"], max(na, nb), g)
    a, b = _multiset(case["kind"], na, pool, g), _multiset(case["kind"], nb, pool, g)

    def nth(x):
        """Which of its run of equal keys an item is."""
        return torch.arange(x.numel(), device=DEV) - torch.searchsorted(x, x)

    def times(x, y):
        """How often x's keys are in y."""
        return torch.searchsorted(y, x, right=True) - torch.searchsorted(y, x)

    op = case["set"]
    a_in_b, b_in_a = nth(a) < times(a, b), nth(b) < times(b, a)
    keep_a = {"union": torch.ones_like(a_in_b), "intersection": a_in_b,
              "difference": ~a_in_b, "symmetric_difference": ~a_in_b}[op]
    keep_b = ~b_in_a if op in ("union", "symmetric_difference") else torch.zeros_like(b_in_a)
    if op in ("difference", "symmetric_difference"):
        # A key's surplus is the end of its run in A.
        left = torch.searchsorted(a, a, right=True) - torch.arange(na, device=DEV)
        keep_a = left <= times(a, a) - times(a, b)
    if op in ("union", "symmetric_difference"):
        left = torch.searchsorted(b, b, right=True) - torch.arange(nb, device=DEV)
        keep_b = left <= times(b, b) - times(b, a)
    keys = torch.cat([a[keep_a], b[keep_b]])
    at = torch.sort(keys, stable=True).indices
    count = torch.tensor([keys.numel()], dtype=torch.int64, device=DEV)
    if not case["write"]:
        return [count]
    cap = cub.set_output_capacity(op, na, nb)
    out = torch.zeros(max(cap, 1), dtype=a.dtype, device=DEV)
    out[: keys.numel()] = keys[at]
    if not case["value"]:
        return [count, out]
    vals = torch.cat([_values(case["value"], na).tensor[keep_a],
                      _values(case["value"], nb, na).tensor[keep_b]])
    outv = torch.zeros(max(cap, 1), dtype=vals.dtype, device=DEV)
    outv[: keys.numel()] = vals[at]
    return [count, out, outv]


def _exact_record(case, g):
    s = _prepare_record(case, g, None)
    rows = s["rows"].words.tensor.view(case["n"], case["arity"])
    at = torch.arange(case["n"], device=DEV)
    for k in range(case["arity"] - 1, -1, -1):
        at = at[torch.sort(rows[at, k], stable=True).indices]
    out = rows[at].reshape(-1)
    return [out, at.to(torch.int64)] if case["value"] else out


def _exact_reduce(case, g):
    s = _prepare_reduce(case, g, None)
    keys, vals = s["keys"].tensor, s["values"].tensor
    uniq, inverse = torch.unique_consecutive(keys, return_inverse=True)
    out, sums = torch.zeros_like(keys), torch.zeros_like(vals)
    out[: uniq.numel()] = uniq
    sums.scatter_add_(0, inverse, vals)
    return [torch.tensor([uniq.numel()], dtype=torch.int64, device=DEV), out, sums]
