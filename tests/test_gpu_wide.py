"""The wide partition pass, one level and two, at sizes that otherwise take a
shorter way (the tuning switches send every build and probe through it):
builds, index-carrying builds and probes against the CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from hashgraph_amd import workloads as wl
from oracle import oracle as o

ONE, TWO, BIG = {"HG_TILE_ROUNDS": "1"}, {"HG_L1_FANOUT": "4"}, {"HG_BUILD_FILL": "2"}
SIZES = [(1, 1), (1000, 97), (100003, 65536), (300000, 299993), (1 << 20, 1 << 20), (200000, 3000000)]


def _to_dev(a, dev):
    import torch
    return torch.from_numpy(a.view(np.int32 if a.dtype == np.uint32 else np.int64).copy()).to(dev)


def _keys(n, kb, hot):
    k = wl.uniform_keys(n, n, kb)
    if hot:
        k[::3] = k[0]
    return k


class Wide:
    """Profiles the calls inside; they must have taken the wide pass `levels`
    times (its column scan runs once a level)."""

    def __init__(self, levels):
        import hashgraph_amd as hg
        self.c, self.levels = hg.context(), levels

    def __enter__(self):
        self.c.profile(True)
        self.c.profile_read()

    def __exit__(self, kind, *rest):
        seen = self.c.profile_read()
        self.c.profile(False)
        if kind is None:
            assert seen.get("col_scan", (0,))[0] == self.levels, seen


def _levels(switch, n, M):
    """Two levels from twice as many buckets as the fan-out on; a bucket has at
    most 65535 bins, and 28672 keys or fewer."""
    return 2 if switch is TWO and max(M / 65535, n / 28672) > 8 else 1


@pytest.mark.parametrize("hot", [False, True])
@pytest.mark.parametrize("kb,ob", [(4, 4), (8, 8)])
@pytest.mark.parametrize("n,M", SIZES)
@pytest.mark.parametrize("switch", [ONE, TWO, BIG], ids=["one level", "two levels", "oversized"])
def test_wide_build(switch, n, M, kb, ob, hot, dev, monkeypatch):
    import hashgraph_amd as hg
    for k, v in switch.items():
        monkeypatch.setenv(k, v)
    print(f"wide build {switch} n={n} M={M} kb={kb} hot={hot}", flush=True)
    keys = _keys(n, kb, hot)
    with Wide(_levels(switch, n, M)):
        off, csr = hg.build(_to_dev(keys, dev), M, offset_bytes=ob)
    goff = off.cpu().numpy().view(np.uint32 if ob == 4 else np.uint64).astype(np.uint64)
    gcsr = csr.cpu().numpy().view(keys.dtype).copy()
    eoff, ecsr = o.build_csr(keys, M)
    assert np.array_equal(goff, eoff)
    o.canon(goff, gcsr)
    o.canon(eoff, ecsr)
    assert np.array_equal(gcsr, ecsr)


@pytest.mark.parametrize("kb", [4, 8])
@pytest.mark.parametrize("n,M", SIZES)
@pytest.mark.parametrize("switch", [ONE, TWO], ids=["one level", "two levels"])
def test_wide_indexed_build(switch, n, M, kb, dev, monkeypatch):
    import hashgraph_amd as hg
    keys = _keys(n, kb, True)
    want = hg.build(_to_dev(keys, dev), M)[0].cpu().numpy()
    for k, v in switch.items():
        monkeypatch.setenv(k, v)
    print(f"wide indexed build {switch} n={n} M={M} kb={kb}", flush=True)
    with Wide(_levels(switch, n, M)):
        off, csr, ind = hg.build_indexed(_to_dev(keys, dev), M)
    assert np.array_equal(off.cpu().numpy(), want)
    ind = ind.cpu().numpy()
    assert np.array_equal(np.sort(ind), np.arange(n))
    assert np.array_equal(csr.cpu().numpy().view(keys.dtype), keys[ind])
    assert np.array_equal(hg.hash_bins(csr, M).cpu().numpy(), np.repeat(np.arange(M, dtype=np.int32), np.diff(want)))


@pytest.mark.parametrize("ob", [4, 8])
@pytest.mark.parametrize("kb", [4, 8])
@pytest.mark.parametrize("n,M", SIZES)
@pytest.mark.parametrize("switch", [ONE, TWO], ids=["one level", "two levels"])
def test_wide_probe(switch, n, M, kb, ob, dev, monkeypatch):
    import hashgraph_amd as hg
    A = _keys(n, kb, False)
    B = wl.probe_keys(A, n + 1, n, 0.4, kb)
    B[: n // 50] = A[0]
    off, csr = hg.build(_to_dev(A, dev), M, offset_bytes=ob)
    dB = _to_dev(B, dev)
    for k, v in switch.items():
        monkeypatch.setenv(k, v)
    print(f"wide probe {switch} n={n} M={M} kb={kb} ob={ob}", flush=True)
    with Wide(2 * _levels(switch, n, M)):
        only = hg.probe(off, csr, M, dB, emit=False)[0]
        cnt, out = hg.probe(off, csr, M, dB)
    assert only == cnt == o.bag_intersect_count(A, B)
    ua, ca = np.unique(A, return_counts=True)
    pos = np.minimum(np.searchsorted(ua, B), len(ua) - 1)
    want = np.repeat(B, np.where(ua[pos] == B, ca[pos], 0))
    assert np.array_equal(np.sort(out.cpu().numpy().view(A.dtype)), np.sort(want))
