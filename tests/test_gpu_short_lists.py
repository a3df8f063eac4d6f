"""Probes and joins into lists shorter than their matches: the count stays
exact, every place of the list holds a match (none more often than it occurs)
and nothing is written behind it."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

from hashgraph_amd import workloads as wl

GUARD = 4096


def _tables(n, copies, kb, dev):
    """Keys of n // copies values on both sides, half as many in B, and one
    value with a bin beyond the walk limits."""
    A = wl.uniform_keys(3, n, kb, device=dev) % max(1, n // copies) + 5
    B = wl.uniform_keys(4, max(1, n // 2), kb, device=dev) % max(1, n // copies) + 5
    A[: min(n // 4, 4000)] = 2
    B[: min(n // 8, 2000)] = 2
    return A, B


def _matches(A, B):
    """Matched keys of both sides, ascending."""
    import torch
    ua, ca = torch.unique(A, return_counts=True)
    ub, cb = torch.unique(B, return_counts=True)
    pos = torch.searchsorted(ua, ub).clamp(max=ua.numel() - 1)
    hit = ua[pos] == ub
    return ub[hit], (ca[pos] * cb)[hit]


def _capacities(total):
    return sorted({0, 1, total // 50, total // 2, total - 1, total, total + 3})


def _check_keys(out, cap, total, vals, counts):
    import torch
    assert bool((out[min(cap, total):] == -1).all())  # nothing behind the list or the last match
    u, c = torch.unique(out[: min(cap, total)], return_counts=True)
    pos = torch.searchsorted(vals, u).clamp(max=vals.numel() - 1)
    assert torch.equal(vals[pos], u) and bool((c <= counts[pos]).all())


@pytest.mark.parametrize("switch", [None, "HG_TILE_ROUNDS"])
@pytest.mark.parametrize("kb", [4, 8])
@pytest.mark.parametrize("n,copies", [(3000, 4), (100000, 9), (3000000, 5), (3000000, 40), (20000000, 4)])
def test_short_probe_and_join(n, copies, kb, switch, dev, monkeypatch):
    import torch
    import hashgraph_amd as hg
    if switch:
        monkeypatch.setenv(switch, "1")
    A, B = _tables(n, copies, kb, dev)
    M = n
    vals, counts = _matches(A, B)
    total = int(counts.sum())
    ta, tb = hg.build(A, M), hg.build(B, M)
    c, P = hg.context(), hg._p
    dA, dB = hg._desc(A.numel(), M, kb), hg._desc(B.numel(), M, kb)
    for cap in _capacities(total):
        print(f"short lists n={n} copies={copies} kb={kb} {switch} matches={total} capacity={cap}", flush=True)
        for what in ("probe", "join"):
            out = torch.full((cap + GUARD,), -1, dtype=A.dtype, device=dev)
            cnt = ctypes.c_uint64(0)
            if what == "probe":
                st = c.lib.hg_probe(c.bind_stream(), ctypes.byref(dA), P(ta[0]), P(ta[1]), P(B), B.numel(), P(out), cap,
                                    ctypes.byref(cnt))
            else:
                st = c.lib.hg_intersect(c.bind_stream(), ctypes.byref(dA), P(ta[0]), P(ta[1]), ctypes.byref(dB),
                                        P(tb[0]), P(tb[1]), P(out), cap, ctypes.byref(cnt))
            assert cnt.value == total, what
            assert st == (0 if cap >= total else 4), what
            _check_keys(out, cap, total, vals, counts)


@pytest.mark.parametrize("kb", [4, 8])
@pytest.mark.parametrize("n,copies", [(3000, 4), (100000, 9), (1000000, 3)])
def test_short_rowid_join(n, copies, kb, dev):
    import torch
    import hashgraph_amd as hg
    A, B = _tables(n, copies, kb, dev)
    M = n
    vals, counts = _matches(A, B)
    total = int(counts.sum())
    ta, tb = hg.build_indexed(A, M), hg.build_indexed(B, M)
    c, P = hg.context(), hg._p
    dA, dB = hg._desc(A.numel(), M, kb), hg._desc(B.numel(), M, kb)
    for cap in _capacities(total):
        print(f"short row-id list n={n} copies={copies} kb={kb} matches={total} capacity={cap}", flush=True)
        pa, pb = (torch.full((cap + GUARD,), -1, dtype=torch.int64, device=dev) for _ in range(2))
        cnt = ctypes.c_uint64(0)
        st = c.lib.hg_intersect_indexed(c.bind_stream(), ctypes.byref(dA), P(ta[0]), P(ta[1]), P(ta[2]),
                                        ctypes.byref(dB), P(tb[0]), P(tb[1]), P(tb[2]), P(pa), P(pb), cap,
                                        ctypes.byref(cnt))
        assert cnt.value == total
        assert st == (0 if cap >= total else 4)
        w = int((pa != -1).sum())  # a call that knows beforehand that the list is short may leave places out
        assert w == total if cap >= total else w <= cap
        assert bool((pa[cap:] == -1).all()) and bool((pb[cap:] == -1).all())
        pa, pb = pa[pa != -1], pb[pb != -1]
        assert torch.equal(A[pa], B[pb])
        assert torch.unique((pa << 32) | pb).numel() == w  # no pair twice
