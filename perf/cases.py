"""Performance cases of the relational operators.

Each case is one call sequence a program makes through the public entry points
(the C ABI over ctypes, device pointers in and out) on tables that already lie
in HBM.  Seven kinds of work:

  agg     fused filter + COUNT / SUM of two int32 columns      qo_filter_agg
  select  range selection of Records with compaction           qo_filter_records
  group   hash group-by (COUNT, SUM, MIN, MAX), optionally
          with the filter fused                                qo_groupby_agg(_filtered)
  sort    the sort-based group-by chain over Records: copy,
          sort, group start positions, per-group SUM           qo_sort_records,
                                                               qo_group_startpos,
                                                               qo_aggregate_groups
  join    filter + hash join + sort of the joined rows         qo_hj_filter_sort
  star    build a dimension table, probe it with filtered
          facts, aggregate the matches per dimension
          attribute                                            qo_hash_build, qo_hash_probe,
                                                               qo_groupby_agg
  batch   many filtered joins planned once and launched as
          one graph                                            JoinBatch (qo_batch_*)

``listed`` holds the named cases, ``draw`` more of the same ranges: rows from
2^12 to 2^28, groups from 16 to 2^20, uniform to Zipf(1) groups, dense keys and
keys spread over 31 or 32 bits, uniform and skewed foreign keys, 5 to 100 % of
the rows selected.  Inputs come from torch generators seeded with the case's
seed alone.
"""
from __future__ import annotations

import ctypes as C
import math

import torch

from query_on_opencl_fpga_amd import _lib, operators
from query_on_opencl_fpga_amd.device import DeviceBuffer

INT_MIN = -(1 << 31)


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # A full-table scan with a predicate: the filter + aggregation of the benchmark at its size.
        {"name": "agg_2e28", "kind": "agg", "n": 1 << 28, "sel": 0.5},
        # A selection that materialises half of a large table, ragged size.
        {"name": "select_50m", "kind": "select", "n": 50_000_003, "sel": 0.5},
        # A dashboard query: a small table, a few hundred groups, a date-range filter.  Latency counts.
        {"name": "group_small", "kind": "group", "n": 100_003, "groups": 500, "z": 0.5, "sel": 0.3},
        # Group-by of the benchmark at its two group counts: few groups of skewed sizes ...
        {"name": "group_2e10_skewed", "kind": "group", "n": 1 << 28, "groups": 1 << 10, "z": 1.0, "sel": 1.0},
        # ... and many groups (per customer).
        {"name": "group_2e20", "kind": "group", "n": 1 << 28, "groups": 1 << 20, "z": 0.5, "sel": 1.0},
        # The reference's group-by pipeline (sort, start positions, aggregate) at the benchmark's size.
        {"name": "sort_group_2e26", "kind": "sort", "n": 1 << 26, "groups": 1 << 20, "keys": "dense"},
        # A lookup-sized join: the smallest query of the benchmark's batch, alone.  Latency counts.
        {"name": "join_small", "kind": "join", "nr": 4096, "ratio": 4, "sel": 0.5, "keys": "sparse", "fk": "uniform"},
        # An ordinary join on scattered 31-bit keys, ragged sizes.
        {"name": "join_sparse", "kind": "join", "nr": 1_500_001, "ratio": 8, "sel": 0.5, "keys": "sparse",
         "fk": "uniform"},
        # Popular products: some build keys are referenced thousands of times.
        {"name": "join_skewed", "kind": "join", "nr": 200_003, "ratio": 15, "sel": 0.6, "keys": "dense",
         "fk": "skewed"},
        # Filter + hash join of the benchmark at its size, rows sorted.
        {"name": "join_2e28", "kind": "join", "nr": 1 << 24, "ratio": 16, "sel": 0.5, "keys": "dense",
         "fk": "uniform"},
        # The same tables in a star query: build, probe, aggregate per attribute of the dimension.
        {"name": "star_2e28", "kind": "star", "nr": 1 << 24, "ratio": 16, "sel": 0.5, "keys": "dense",
         "groups": 1000},
        # A dashboard's worth of small joins in one launch: the benchmark's batch of small queries.
        {"name": "batch_512", "kind": "batch", "queries": 512, "nr_lo": 1 << 12, "nr_hi": 1 << 16},
    ]


def _log_int(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["agg", "select", "group", "group", "sort", "join", "join", "star", "batch"])
    sel = round(rng.uniform(0.05, 1.0), 2)
    if kind in ("agg", "select"):
        return {"kind": kind, "n": _log_int(rng, 1 << 12, 1 << 27), "sel": sel}
    if kind == "group":
        n = _log_int(rng, 1 << 12, 1 << 27)
        return {"kind": kind, "n": n, "groups": _log_int(rng, 16, min(1 << 20, n)),
                "z": round(rng.uniform(0.0, 1.0), 2), "sel": rng.choice([1.0, sel])}
    if kind == "sort":
        n = _log_int(rng, 1 << 12, 1 << 26)
        return {"kind": kind, "n": n, "groups": _log_int(rng, 16, min(1 << 20, n)),
                "keys": rng.choice(["dense", "wide"])}
    if kind == "join":
        return {"kind": kind, "nr": _log_int(rng, 1 << 12, 1 << 22), "ratio": rng.randint(4, 16), "sel": sel,
                "keys": rng.choice(["dense", "sparse"]), "fk": rng.choice(["uniform", "skewed"])}
    if kind == "star":
        return {"kind": kind, "nr": _log_int(rng, 1 << 12, 1 << 23), "ratio": rng.randint(4, 16), "sel": sel,
                "keys": rng.choice(["dense", "sparse"]), "groups": _log_int(rng, 16, 1 << 12)}
    return {"kind": kind, "queries": rng.randint(8, 400), "nr_lo": 1 << 12, "nr_hi": _log_int(rng, 1 << 13, 1 << 16)}


# ---------------------------------------------------------------------------
# Inputs (torch only; the device and a seeded generator)
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _uniform(n, lo, hi, g):
    return torch.randint(lo, hi, (n,), generator=g, device="cuda", dtype=torch.int32)


def _payload(n, g):
    return _uniform(n, INT_MIN, (1 << 31) - 1, g)


def _zipf(n, groups, z, g):
    """Group ids in [0, groups): Zipf(z) ranks mapped through a permutation."""
    if z == 0.0:
        return _uniform(n, 0, groups, g)
    w = torch.arange(1, groups + 1, device="cuda", dtype=torch.float64).pow(-z)
    cdf = w.cumsum(0)
    cdf = cdf / cdf[-1]
    perm = torch.randperm(groups, generator=g, device="cuda").to(torch.int32)
    out = torch.empty(n, dtype=torch.int32, device="cuda")
    step = 1 << 26
    for i in range(0, n, step):
        u = torch.rand(min(step, n - i), generator=g, device="cuda", dtype=torch.float64)
        out[i:i + step] = perm[torch.searchsorted(cdf, u).clamp_(max=groups - 1)]
    return out


def _filter_column(n, sel, g):
    """(filter column uniform in [0, 1000), upper bound that selects the fraction sel)."""
    return _uniform(n, 0, 1000, g), int(round(1000 * sel)) - 1


def _build_keys(nr, keys, seed, g):
    """nr distinct keys: a permutation of [0, nr), or spread over 31 bits (an odd multiple modulo 2^31)."""
    k = torch.randperm(nr, generator=g, device="cuda")
    if keys == "sparse":
        k = (k * 1_640_531_527 + (int(seed) * 104_729 + 5)) & 0x7FFFFFFF
    return k.to(torch.int32)


def _foreign_keys(rkey, ns, fk, g):
    """ns references to rows of R: uniform, or skewed (density falls as 1 / sqrt(rank))."""
    nr = rkey.numel()
    out = torch.empty(ns, dtype=torch.int32, device="cuda")
    step = 1 << 26
    for i in range(0, ns, step):
        m = min(step, ns - i)
        if fk == "skewed":
            u = torch.rand(m, generator=g, device="cuda", dtype=torch.float64)
            at = (u * u * nr).long().clamp_(max=nr - 1)
        else:
            at = torch.randint(0, nr, (m,), generator=g, device="cuda")
        out[i:i + step] = rkey[at]
    return out


def _batch_sizes(case):
    """|R| of every query, log-uniform over [nr_lo, nr_hi], and |S| = 4..16 |R|."""
    q = int(case["queries"])
    lo, hi = math.log(case["nr_lo"]), math.log(case["nr_hi"])
    nr = [int(round(math.exp(lo + (hi - lo) * ((i * 0.6180339887) % 1.0)))) for i in range(q)]
    return nr, [n * (4, 8, 16)[i % 3] for i, n in enumerate(nr)]


def _zeros(n, dtype=torch.int32):
    return torch.zeros(max(int(n), 1), dtype=dtype, device="cuda")


def _group_outputs(groups):
    return {"key": _zeros(groups), "count": _zeros(groups, torch.int64), "sum": _zeros(groups, torch.int64),
            "min": _zeros(groups), "max": _zeros(groups), "groups": _zeros(1, torch.int64)}


def _ptrs(out):
    return [out[c].data_ptr() for c in ("key", "count", "sum", "min", "max", "groups")]


class _Column:
    """A column as JoinBatch takes it: an object with the device pointer `ptr`."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()


class _Batch:
    """A planned batch and the tensors it reads and writes; gives the plan back with itself."""

    def __init__(self, case, g, seed):
        nrs, nss = _batch_sizes(case)
        at = lambda sizes: [sum((s + 63) // 64 * 64 for s in sizes[:i]) for i in range(len(sizes) + 1)]
        ro, so = at(nrs), at(nss)
        self.rkey, self.skey = _zeros(ro[-1]), _zeros(so[-1])
        self.rpay, self.spay = _payload(ro[-1], g), _payload(so[-1], g)
        self.sfilt = _uniform(so[-1], 0, 1000, g)
        self.out = {c: _zeros(so[-1]) for c in ("key", "rpay", "spay")}
        self.queries = []
        for i, (nr, ns) in enumerate(zip(nrs, nss)):
            rk = _build_keys(nr, "sparse", int(seed) + i, g)
            self.rkey[ro[i]:ro[i] + nr] = rk
            self.skey[so[i]:so[i] + ns] = _foreign_keys(rk, ns, "uniform", g)
            r, s = slice(ro[i], ro[i] + nr), slice(so[i], so[i] + ns)
            self.queries.append({
                "rkey": _Column(self.rkey[r]), "rpay": _Column(self.rpay[r]), "skey": _Column(self.skey[s]),
                "spay": _Column(self.spay[s]), "sfilt": _Column(self.sfilt[s]), "nr": nr, "ns": ns, "flo": INT_MIN,
                "fhi": (49, 199, 499)[i % 3], "okey": _Column(self.out["key"][s]),
                "orpay": _Column(self.out["rpay"][s]), "ospay": _Column(self.out["spay"][s]), "cap": ns})
        torch.cuda.synchronize()
        self.plan = operators.JoinBatch(self.queries)

    def __del__(self):
        if getattr(self, "plan", None) is not None:
            self.plan.destroy()


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    s = {"kind": kind}
    if kind == "agg":
        n = case["n"]
        s.update(n=n, key=_uniform(n, 0, (1 << 31) - 1, g), val=_uniform(n, 0, 1000, g),
                 hi=int(case["sel"] * ((1 << 31) - 1)), out=_zeros(3, torch.int64))
    elif kind == "select":
        n = case["n"]
        rows = torch.stack([torch.arange(n, device="cuda", dtype=torch.int32),
                            _uniform(n, 0, 1000, g)], dim=1).contiguous()
        s.update(n=n, rows=rows, hi=int(round(1000 * case["sel"])) - 1, out=_zeros(2 * n).view(n, 2),
                 count=_zeros(1, torch.int64))
    elif kind == "group":
        n, groups = case["n"], case["groups"]
        s.update(n=n, cap=groups, key=_zipf(n, groups, case["z"], g), val=_uniform(n, 0, 1 << 16, g),
                 out=_group_outputs(groups))
        if case["sel"] < 1.0:
            s["filt"], s["hi"] = _filter_column(n, case["sel"], g)
    elif kind == "sort":
        n, groups = case["n"], case["groups"]
        y = _uniform(n, 0, groups, g).long()
        if case["keys"] == "wide":
            y = (y * 2_654_435_761) & 0xFFFFFFFF
            y = torch.where(y >= 1 << 31, y - (1 << 32), y)
        rows = torch.stack([_uniform(n, 0, 1 << 16, g), y.to(torch.int32)], dim=1).contiguous()
        s.update(n=n, rows=rows, sorted=_zeros(2 * n).view(n, 2), start=_zeros(n), sums=_zeros(groups),
                 num=DeviceBuffer(8), h_num=C.c_uint64())
    elif kind in ("join", "star"):
        nr, ns = case["nr"], case["nr"] * case["ratio"]
        rkey = _build_keys(nr, case["keys"], seed, g)
        rpay = _payload(nr, g) if kind == "join" else _uniform(nr, 0, case["groups"], g)
        spay = _payload(ns, g) if kind == "join" else _uniform(ns, 0, 1 << 16, g)
        filt, hi = _filter_column(ns, case["sel"], g)
        bytes_ = _lib.load().qo_join_table_bytes(nr)
        s.update(nr=nr, ns=ns, rkey=rkey, rpay=rpay, skey=_foreign_keys(rkey, ns, case.get("fk", "uniform"), g),
                 spay=spay, filt=filt, hi=hi, table=_zeros(bytes_ // 4 + 1), table_bytes=bytes_,
                 okey=_zeros(ns), orpay=_zeros(ns), ospay=_zeros(ns), h_count=C.c_uint64())
        if kind == "star":
            s.update(count=DeviceBuffer(8), cap=case["groups"], out=_group_outputs(case["groups"]))
    elif kind == "batch":
        s["batch"] = _Batch(case, g, seed)
    torch.cuda.synchronize()
    return s


def _read_u64(buf, host):
    """A device counter the program needs on the host."""
    _lib.call("qo_memcpy_d2h", C.addressof(host), buf.ptr, 8)
    return host.value


def run(s):
    kind = s["kind"]
    if kind == "agg":
        _lib.call("qo_filter_agg", s["key"].data_ptr(), s["val"].data_ptr(), s["n"], 0, s["hi"],
                  s["out"].data_ptr(), None)
        return s["out"]
    if kind == "select":
        _lib.call("qo_filter_records", s["rows"].data_ptr(), s["n"], 0, s["hi"], s["out"].data_ptr(),
                  s["count"].data_ptr(), None)
        return s["out"], s["count"]
    if kind == "group":
        if "filt" in s:
            _lib.call("qo_groupby_agg_filtered", s["key"].data_ptr(), s["val"].data_ptr(), s["filt"].data_ptr(),
                      s["n"], 0, s["hi"], s["cap"], *_ptrs(s["out"]), None)
        else:
            _lib.call("qo_groupby_agg", s["key"].data_ptr(), s["val"].data_ptr(), s["n"], s["cap"],
                      *_ptrs(s["out"]), None)
        return s["out"]
    if kind == "sort":
        rows, n = s["sorted"].data_ptr(), s["n"]
        _lib.call("qo_memcpy_d2d", rows, s["rows"].data_ptr(), 8 * n, None)
        _lib.call("qo_sort_records", rows, n, None)
        _lib.call("qo_group_startpos", rows, n, s["start"].data_ptr(), s["num"].ptr, None)
        groups = _read_u64(s["num"], s["h_num"])
        _lib.call("qo_aggregate_groups", rows, n, s["start"].data_ptr(), groups, operators.REDUCE_SUM,
                  s["sums"].data_ptr(), None)
        return s["sorted"], s["start"], s["sums"], groups
    if kind == "join":
        _lib.call("qo_hj_filter_sort", s["table"].data_ptr(), s["table_bytes"], s["rkey"].data_ptr(),
                  s["rpay"].data_ptr(), s["nr"], s["skey"].data_ptr(), s["spay"].data_ptr(), s["filt"].data_ptr(),
                  s["ns"], 0, s["hi"], s["okey"].data_ptr(), s["orpay"].data_ptr(), s["ospay"].data_ptr(), s["ns"],
                  C.byref(s["h_count"]), None)
        return s["okey"], s["orpay"], s["ospay"], s["h_count"].value
    if kind == "star":
        _lib.call("qo_hash_build", s["table"].data_ptr(), s["table_bytes"], s["rkey"].data_ptr(),
                  s["rpay"].data_ptr(), s["nr"], None)
        _lib.call("qo_hash_probe", s["table"].data_ptr(), s["table_bytes"], s["skey"].data_ptr(),
                  s["spay"].data_ptr(), s["filt"].data_ptr(), s["ns"], 0, s["hi"], s["okey"].data_ptr(),
                  s["orpay"].data_ptr(), s["ospay"].data_ptr(), s["ns"], s["count"].ptr, None)
        m = _read_u64(s["count"], s["h_count"])
        _lib.call("qo_groupby_agg", s["orpay"].data_ptr(), s["ospay"].data_ptr(), m, s["cap"], *_ptrs(s["out"]),
                  None)
        return s["out"], m
    s["batch"].plan.launch()
    return s["batch"].out


# ---------------------------------------------------------------------------
# work / exact
# ---------------------------------------------------------------------------
def work(case):
    """Bytes each entry point's contract moves: every input once, every output row once."""
    kind = case["kind"]
    if kind == "agg":
        b = 8 * case["n"]
    elif kind == "select":
        b = 8 * case["n"] * (1 + case["sel"])
    elif kind == "group":
        b = case["n"] * (8 if case["sel"] >= 1.0 else 12) + 28 * case["groups"]
    elif kind == "sort":
        b = 16 * case["n"] + 8 * case["groups"]  # records in and out, start positions and sums
    elif kind == "join":
        ns = case["nr"] * case["ratio"]
        b = 8 * case["nr"] + 12 * ns + 12 * ns * case["sel"]
    elif kind == "star":
        ns = case["nr"] * case["ratio"]
        b = 8 * case["nr"] + 12 * ns + (12 + 8) * ns * case["sel"] + 28 * case["groups"]
    else:
        nr, ns = _batch_sizes(case)
        b = sum(8 * r + 12 * s + 12 * s * (0.05, 0.2, 0.5)[i % 3] for i, (r, s) in enumerate(zip(nr, ns)))
    return {"bytes": b, "flops": 0}


def _aggregate(key, val, groups):
    """Per present key ascending: (key, COUNT, SUM, MIN, MAX), padded with zeros to `groups` rows."""
    k = key.long()
    count = torch.bincount(k, minlength=groups)
    total = torch.zeros(groups, dtype=torch.int64, device=k.device).index_add_(0, k, val.long())
    low = torch.full((groups,), (1 << 31) - 1, dtype=torch.int32, device=k.device)
    high = torch.full((groups,), INT_MIN, dtype=torch.int32, device=k.device)
    low.scatter_reduce_(0, k, val, "amin")
    high.scatter_reduce_(0, k, val, "amax")
    present = count.nonzero().flatten()
    out = _group_outputs(groups)
    m = present.numel()
    out["key"][:m] = present.to(torch.int32)
    for name, col in (("count", count), ("sum", total), ("min", low), ("max", high)):
        out[name][:m] = col[present]
    out["groups"][0] = m
    return out


def exact(case, seed):
    """The outputs of `run` from plain torch on the same inputs (whole numbers throughout)."""
    kind = case["kind"]
    if kind not in ("agg", "select", "group") or case["n"] > 1 << 24:
        return None
    s = prepare(case, seed)
    if kind == "agg":
        v = s["val"][s["key"] <= s["hi"]].long()
        total = v.sum()
        low = total & 0xFFFFFFFF
        return torch.stack([torch.tensor(v.numel(), device="cuda"), total,
                            torch.where(low >= 1 << 31, low - (1 << 32), low)])
    if kind == "select":
        sel = s["rows"][s["rows"][:, 1] <= s["hi"]]
        out = torch.zeros_like(s["rows"])
        out[:sel.shape[0]] = sel
        return out, torch.tensor([sel.shape[0]], device="cuda")
    keep = s["filt"] <= s["hi"] if "filt" in s else slice(None)
    return _aggregate(s["key"][keep], s["val"][keep], case["groups"])
