"""Performance cases: the passes a program runs with this library, over the
sizes, key widths and options it is used with.

A case is a dict of plain values; its "kind" names the pass:
  probe    build a table, probe raw keys against it, matched keys written
  join     build two tables, join them, matched keys written
  rowid    build two index-carrying tables, join them to pairs of positions
  rle      one GPU's share of a partitioned table: split points, partitioned
           builds of both sides, run-length join of every partition
  learned  as probe, under a learned hash trained beforehand
  batch    one replay of a captured plan: build every table, count its matches
  staged   tables in pinned host memory: two builds and the join

All outputs are whole numbers, so exact() has nothing to add: they are equal
or wrong.  The order of the keys inside a bin, and of a match list, is left
open by the library (the entries of a bin are a multiset), so run() hands
these outputs back as they were written, in a Bags, and reading one from there
gives its entries in ascending order.
"""
import math

import torch

import hashgraph_amd as hg
from hashgraph_amd import workloads as wl


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a lookup table of a few hundred rows, rebuilt for each request: launches and latency only
        {"name": "probe_u32_1k", "kind": "probe", "key_bytes": 4, "offset_bytes": 4, "n_a": 1000, "n_b": 1500,
         "n_bins": 1000, "hit": 0.5, "kept": False},
        # the smallest benchmark configuration (2^20 keys a side, half of B drawn from A)
        {"name": "probe_u32_1m", "kind": "probe", "key_bytes": 4, "offset_bytes": 4, "n_a": 1 << 20, "n_b": 1 << 20,
         "n_bins": 1 << 20, "hit": 0.5, "kept": False},
        # a mid-sized table of 64-bit ids, ragged sizes, a prime number of bins, 64-bit offsets, fewer probes than rows
        {"name": "probe_u64_5m", "kind": "probe", "key_bytes": 8, "offset_bytes": 8, "n_a": 5000011, "n_b": 3000017,
         "n_bins": 4194301, "hit": 0.25, "kept": False},
        # the headline configuration: 2^28 32-bit keys a side, 25% overlap, buffers kept by the program
        {"name": "probe_u32_268m", "kind": "probe", "key_bytes": 4, "offset_bytes": 4, "n_a": 1 << 28,
         "n_b": 1 << 28, "n_bins": 1 << 28, "hit": 0.25, "kept": True},
        # its 64-bit form: 2^27 keys a side
        {"name": "probe_u64_134m", "kind": "probe", "key_bytes": 8, "offset_bytes": 4, "n_a": 1 << 27,
         "n_b": 1 << 27, "n_bins": 1 << 27, "hit": 0.25, "kept": True},
        # the driver program's input (sequential keys, both tables the same range), joined table against table
        {"name": "join_u32_100m", "kind": "join", "key_bytes": 4, "offset_bytes": 4, "n_a": 100000000,
         "n_b": 100000000, "n_bins": 100000000},
        # a join whose consumer needs row numbers
        {"name": "rowid_u32_50m", "kind": "rowid", "key_bytes": 4, "offset_bytes": 4, "n_a": 50000000,
         "n_b": 50000000, "n_bins": 1 << 26, "hit": 0.25},
        # heavy duplicates: Zipf(1.1) values over 2^32, 16 partitions, records instead of pairs
        {"name": "rle_zipf_u64_33m", "kind": "rle", "key_bytes": 8, "offset_bytes": 4, "n_a": 1 << 25,
         "n_b": 1 << 24, "n_bins": 1 << 25, "parts": 16},
        # skewed 64-bit keys under the learned hash
        {"name": "learned_u64_33m", "kind": "learned", "key_bytes": 8, "offset_bytes": 4, "n_a": 1 << 25,
         "n_b": 1 << 25, "n_bins": 1 << 25, "hit": 0.5},
        # many uneven small tables at once, every other one Zipf(1.2)
        {"name": "batch_u32_1024", "kind": "batch", "key_bytes": 4, "tables": 1024, "lo_bits": 8.0, "hi_bits": 20.0,
         "hit": 0.3},
        # tables in host memory through a device budget of about an eighth of one of them
        {"name": "staged_u32_16m", "kind": "staged", "key_bytes": 4, "offset_bytes": 4, "n_a": 1 << 24,
         "n_b": 1 << 24, "n_bins": 1 << 24, "hit": 0.25, "budget_mib": 24},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["probe", "probe", "probe", "probe", "join", "rowid", "rle", "learned", "batch", "staged"])
    kb = rng.choice([4, 4, 8])
    if kind == "batch":
        lo = rng.uniform(6.0, 10.0)
        return {"kind": kind, "key_bytes": 4, "tables": _log_int(rng, 16, 1024), "lo_bits": lo,
                "hi_bits": rng.uniform(lo + 4.0, 20.0), "hit": rng.uniform(0.1, 0.9)}
    top = {"probe": 1 << 28, "join": 100000000, "rowid": 50000000, "rle": 1 << 25, "learned": 1 << 25,
           "staged": 1 << 24}[kind]
    low = {"probe": 300, "join": 300, "rowid": 300, "rle": 1 << 18, "learned": 1 << 16, "staged": 1 << 20}[kind]
    if kind in ("rle", "learned"):
        kb = 8
    elif kind == "staged":
        kb = 4
    elif kb == 8:
        top //= 2
    n_a = _log_int(rng, low, top)
    n_b = max(1, min(top, int(n_a * math.exp(rng.uniform(-1.0, 0.3)))))
    n_bins = max(1, min(top, int(n_a * math.exp(rng.uniform(-0.7, 0.7)))))
    case = {"kind": kind, "key_bytes": kb, "offset_bytes": rng.choice([4, 4, 8]) if kind == "probe" else 4,
            "n_a": n_a, "n_b": n_b, "n_bins": n_bins}
    if kind in ("probe", "rowid", "learned", "staged"):
        case["hit"] = rng.uniform(0.05, 0.95)
    if kind == "probe":
        case["kept"] = rng.random() < 0.5
    if kind == "rle":
        case["parts"] = rng.choice([2, 4, 8, 16])
    if kind == "staged":
        case["budget_mib"] = rng.choice([8, 16, 32])
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _uniform_pair(case, seed):
    dev = _device()
    A = wl.uniform_keys(4 * seed + 1, case["n_a"], case["key_bytes"], device=dev)
    return A, wl.probe_keys(A, 4 * seed + 2, case["n_b"], case["hit"], case["key_bytes"], device=dev)


def _prepare_probe(case, seed):
    A, B = _uniform_pair(case, seed)
    s = {"A": A, "B": B, "table": None, "matches": None}
    if case["kept"]:  # the program's own table and result buffers
        ot = torch.int32 if case["offset_bytes"] == 4 else torch.int64
        s["table"] = (torch.empty(case["n_bins"] + 1, dtype=ot, device=A.device), torch.empty_like(A))
        s["matches"] = torch.empty(2 * case["n_b"], dtype=A.dtype, device=A.device)
    return s


def _prepare_join(case, seed):
    # a range of row numbers that starts anywhere, the same for both tables
    dev, kb = _device(), case["key_bytes"]
    first = wl.mix64_int(seed) % (1 << 30)
    dt = torch.int32 if kb == 4 else torch.int64
    return {"A": torch.arange(first, first + case["n_a"], dtype=torch.int64, device=dev).to(dt),
            "B": torch.arange(first, first + case["n_b"], dtype=torch.int64, device=dev).to(dt)}


def _prepare_rle(case, seed):
    dev = _device()
    return {"A": wl.zipf_keys(4 * seed + 1, case["n_a"], 1.1, device=dev),
            "B": wl.zipf_keys(4 * seed + 2, case["n_b"], 1.1, device=dev)}


def _prepare_learned(case, seed):
    dev = _device()
    A = wl.lognormal_keys(4 * seed + 1, case["n_a"], device=dev)
    B = wl.mixed_probe(A, wl.lognormal_keys(4 * seed + 2, case["n_b"], device=dev), 4 * seed + 3, case["hit"])
    # the sampled check is close to even on these keys: the model is used whatever it says, so that the case is what
    # its name says for every seed
    model, _ = hg.rmi_train(A, case["n_bins"], n_sample=max(1, case["n_a"] // 100), seed=24)
    return {"A": A, "B": B, "hash": {"hash_kind": hg.HG_HASH_RMI, "rmi_model": model}}


def _batch_sizes(case):
    return wl.batch_sizes(5, case["tables"], case["lo_bits"], case["hi_bits"])


def _prepare_batch(case, seed):
    # even tables uniform, odd ones Zipf(1.2); both from one stream cut into tables
    dev = _device()
    sizes = _batch_sizes(case).tolist()
    off = [0]
    for n in sizes:
        off.append(off[-1] + n)
    uni = wl.uniform_keys(4 * seed + 1, off[-1], 4, device=dev)
    z = wl.zipf_keys(4 * seed + 2, off[-1], 1.2, device=dev)
    odd = torch.repeat_interleave((torch.arange(len(sizes), device=dev) & 1).bool(),
                                  torch.tensor(sizes, device=dev))
    A = torch.where(odd, (z - ((z >> 31) << 32)).to(torch.int32), uni)
    B = torch.cat([wl.probe_keys(A[off[t]:off[t + 1]], 8 * seed + 8 * t + 3, n, case["hit"], 4, device=dev)
                   for t, n in enumerate(sizes)])
    return {"plan": hg.BatchPlan(A, off, sizes, B, off)}


def _prepare_staged(case, seed):
    A, B = _uniform_pair(case, seed)

    def pin(n):
        return torch.empty(n, dtype=torch.int32, pin_memory=True)

    def host(x):
        return pin(x.numel()).copy_(x)

    return {"A": host(A), "B": host(B), "ta": (pin(case["n_bins"] + 1), pin(case["n_a"])),
            "tb": (pin(case["n_bins"] + 1), pin(case["n_b"])), "matches": pin(2 * case["n_b"])}


_PREPARE = {"probe": _prepare_probe, "rowid": lambda case, seed: dict(zip("AB", _uniform_pair(case, seed))),
            "join": _prepare_join, "rle": _prepare_rle, "learned": _prepare_learned, "batch": _prepare_batch,
            "staged": _prepare_staged}


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    s["case"] = case
    return s


# ---------------------------------------------------------------------------
# passes
# ---------------------------------------------------------------------------
def _run_probe(s, case):
    kw = s.get("hash", {})
    off, csr = hg.build(s["A"], case["n_bins"], case["offset_bytes"], out=s.get("table"), **kw)
    count, matches = hg.probe(off, csr, case["n_bins"], s["B"], out=s.get("matches"), **kw)
    return Bags(count=count, offsets=off, keys=lambda: _csr(off, csr),
                matches=lambda: _ascending(matches, 2 * case["n_b"]))


def _run_join(s, case):
    ta, tb = (hg.build(s[x], case["n_bins"], case["offset_bytes"]) for x in "AB")
    count, matches = hg.intersect(*ta, *tb, case["n_bins"])
    return Bags(count=count, offsets_a=ta[0], keys_a=lambda: _csr(*ta), offsets_b=tb[0], keys_b=lambda: _csr(*tb),
                matches=lambda: _ascending(matches, 2 * case["n_b"]))


def _run_rowid(s, case):
    ta, tb = (hg.build_indexed(s[x], case["n_bins"], case["offset_bytes"]) for x in "AB")
    count, pa, pb = hg.intersect_indexed(*ta, *tb, case["n_bins"])
    return Bags(count=count, offsets_a=ta[0], entries_a=lambda: _entries(*ta), offsets_b=tb[0],
                entries_b=lambda: _entries(*tb), pairs=lambda: _ascending((pa << 32) | pb, 2 * case["n_b"]))


def _run_rle(s, case):
    M, P = case["n_bins"], case["parts"]
    splits = hg.find_splits(s["A"], M, 16000, P)
    ta, tb = (hg.build_partitioned(s[x], M, splits, case["offset_bytes"]) for x in "AB")
    total, recs = 0, []
    for p in range(P):
        lo, hi = splits[p], splits[p + 1]
        if hi == lo:  # repeated split point: no bins
            continue
        oa, ob = (t[0][lo + p: hi + p + 1] for t in (ta, tb))
        ka, kb = (t[1][t[2][p]: t[2][p + 1]] for t in (ta, tb))
        # a record per value in both: never more than either side's keys
        count, *rec = hg.intersect_rle(oa, ka, ob, kb, hi - lo, capacity=min(ka.numel(), kb.numel()))
        total += count
        recs.append(rec)
    return Bags(count=total, splits=lambda: torch.tensor(splits), offsets_a=ta[0], offsets_b=tb[0],
                keys_a=lambda: _csr_parts(splits, *ta), keys_b=lambda: _csr_parts(splits, *tb),
                records=lambda: _records(recs, min(case["n_a"], case["n_b"])))


def _run_batch(s, case):
    plan = s["plan"]
    plan.run()
    return Bags(offsets=plan.offsets, counts=plan.counts, keys=lambda: _csr_batch(plan, _batch_sizes(case).tolist()))


def _run_staged(s, case):
    kw = {"device_budget": case["budget_mib"] << 20, "device": torch.cuda.current_device()}
    for x, t in (("A", "ta"), ("B", "tb")):
        hg.build_staged(s[x], case["n_bins"], case["offset_bytes"], out=s[t], **kw)
    count, matches = hg.intersect_staged(*s["ta"], *s["tb"], case["n_bins"], out=s["matches"], **kw)
    return Bags(count=count, offsets_a=s["ta"][0], keys_a=lambda: _csr(*s["ta"]), offsets_b=s["tb"][0],
                keys_b=lambda: _csr(*s["tb"]), matches=lambda: _ascending(matches, 2 * case["n_b"]))


_RUN = {"probe": _run_probe, "learned": _run_probe, "join": _run_join, "rowid": _run_rowid, "rle": _run_rle,
        "batch": _run_batch, "staged": _run_staged}


def run(state):
    return _RUN[state["case"]["kind"]](state, state["case"])


# ---------------------------------------------------------------------------
# outputs
# ---------------------------------------------------------------------------
class Bags(dict):
    """A pass's outputs.  One whose order is open is held as a function that
    reads it in ascending order; the reader's cost is not the pass's.  A list
    whose length depends on the keys is read with zeros behind it, up to a
    length that depends on the sizes alone."""

    def __getitem__(self, k):
        v = super().__getitem__(k)
        return v() if callable(v) else v

    def values(self):
        return [self[k] for k in self]

    def items(self):
        return [(k, self[k]) for k in self]


def _ascending(x, length):
    return _padded(torch.sort(x.to(_device())).values, length)


def _padded(x, length):
    return torch.cat([x, x.new_zeros(max(0, length - x.numel()))])


def _bins(degrees):
    return torch.repeat_interleave(torch.arange(degrees.numel(), device=degrees.device), degrees)


def _by_bin(degrees, keys):
    """keys (bin after bin, degrees[b] in bin b), ascending inside each bin."""
    order = torch.sort(keys, stable=True).indices
    bins = _bins(degrees)[order]
    return keys[order[torch.sort(bins, stable=True).indices]]


def _degrees(offsets):
    o = offsets.to(_device()).to(torch.int64)
    return o[1:] - o[:-1]


def _csr(offsets, keys):
    return _by_bin(_degrees(offsets), keys.to(_device()))


def _csr_parts(splits, offsets, keys, part_offsets):
    deg = [_degrees(offsets[splits[p] + p: splits[p + 1] + p + 1]) for p in range(len(splits) - 1)]
    return _by_bin(torch.cat(deg), keys[: part_offsets[-1]])


def _csr_batch(plan, sizes):
    deg = [_degrees(plan.offsets[o: o + n + 1]) for o, n in zip(plan.off_off, sizes)]
    return _by_bin(torch.cat(deg), plan.csr)


def _entries(offsets, keys, index):
    """(key, input position) of every entry, by position inside each bin."""
    order = torch.sort((_bins(_degrees(offsets)) << 32) | index).indices
    return [keys[order], index[order]]


def _records(recs, length):
    keys, ca, cb = (torch.cat([r[i] for r in recs]) for i in range(3))
    order = torch.sort(keys).indices
    return [_padded(x[order], length) for x in (keys, ca, cb)]


def exact(case, seed):
    return None


# ---------------------------------------------------------------------------
# work: every input read once, every output written once
# ---------------------------------------------------------------------------
def work(case):
    s, o = case["key_bytes"], case.get("offset_bytes", 4)
    if case["kind"] == "batch":
        n, t = int(_batch_sizes(case).sum()), case["tables"]
        # both key sets; CSR keys, offsets (n + 1 a table), counts
        return {"bytes": 2 * n * s + n * s + (n + t) * 4 + 8 * t, "flops": 0}
    a, b, m = case["n_a"], case["n_b"], case["n_bins"]
    hits = case["hit"] * b if "hit" in case else min(a, b)
    table = o * (m + 1)
    if case["kind"] in ("probe", "learned"):
        return {"bytes": s * (a + b) + table + s * a + s * hits, "flops": 0}
    if case["kind"] == "rowid":
        return {"bytes": s * (a + b) + 2 * table + (s + 8) * (a + b) + 16 * hits, "flops": 0}
    if case["kind"] == "rle":  # about a record per 30 keys of B
        return {"bytes": s * (a + b) + 2 * (table + o * case["parts"]) + s * (a + b) + (s + 16) * (b // 30), "flops": 0}
    return {"bytes": s * (a + b) + 2 * table + s * (a + b) + s * hits, "flops": 0}
