"""Two-step partitions of keys with hot values, whose buckets skip the second
step: one hot bucket, many, several of them in one group of buckets, at the
edges of the bins.  Results against the keys' bins computed apart."""
import pytest

pytestmark = pytest.mark.gpu

from hashgraph_amd import workloads as wl

N = 16000001  # beyond the narrow pass


def _values_in(lo, hi, M, count, dev):
    """Keys whose bins lie in [lo, hi) (murmur3 over M bins), in bin order."""
    import torch
    import hashgraph_amd as hg
    v = torch.arange(1, 8000001, dtype=torch.int32, device=dev)
    b = hg.hash_bins(v, M).to(torch.int64) & 0xFFFFFFFF
    at = torch.nonzero((b >= lo) & (b < hi)).flatten()
    at = at[torch.argsort(b[at])]
    assert at.numel() >= count
    return v[at[torch.linspace(0, at.numel() - 1, count, device=dev).long()]]


def _hot_values(kind, M, dev):
    import torch
    if kind == "one":
        return _values_in(0, M, M, 1, dev)
    if kind == "many":
        return _values_in(0, M, M, 60, dev)
    if kind == "neighbours":  # a group of the 2^24-bin table has about 49 buckets of 7168 bins
        return _values_in(M // 3, M // 3 + 7168 * 12, M, 6, dev)
    return torch.cat([_values_in(0, 3000, M, 1, dev), _values_in(M - 3000, M, M, 1, dev)])  # first and last bucket


def _keys(kind, share, kb, n, M, dev):
    """n uniform keys, `share` of them replaced by the hot values in turn."""
    import torch
    k = wl.uniform_keys(17, n, kb, device=dev)
    hot = _hot_values(kind, M, dev).to(k.dtype)
    at = torch.nonzero(torch.rand(n, generator=torch.Generator(dev).manual_seed(5), device=dev) < share).flatten()
    k[at] = hot[at % hot.numel()]
    return k


def _check_table(off, csr, keys, bins, M):
    import torch
    deg = torch.bincount(bins, minlength=M)
    assert int(off[0]) == 0 and torch.equal(off[1:].to(torch.int64), torch.cumsum(deg, 0))
    assert torch.equal(torch.sort(csr).values, torch.sort(keys).values)


def _bins(keys, M):
    import torch
    import hashgraph_amd as hg
    return hg.hash_bins(keys, M).to(torch.int64) & 0xFFFFFFFF


@pytest.mark.parametrize("kb,ob", [(4, 4), (8, 8)])
@pytest.mark.parametrize("kind,share", [("one", 0.05), ("one", 1.0), ("many", 0.6), ("neighbours", 0.9), ("ends", 0.3)])
def test_hot_builds(kind, share, kb, ob, dev):
    import torch
    import hashgraph_amd as hg
    M = 1 << 24
    print(f"hot build {kind} share={share} kb={kb} ob={ob}", flush=True)
    keys = _keys(kind, share, kb, N, M, dev)
    bins = _bins(keys, M)
    off, csr = hg.build(keys, M, offset_bytes=ob)
    _check_table(off, csr, keys, bins, M)
    order = torch.repeat_interleave(torch.arange(M, device=dev), off.diff().to(torch.int64))
    assert torch.equal(_bins(csr, M), order)
    off2, ck, ind = hg.build_indexed(keys, M, offset_bytes=ob)
    assert torch.equal(off2, off)
    assert torch.equal(torch.sort(ind).values, torch.arange(N, device=dev)) and torch.equal(ck, keys[ind])
    assert torch.equal(bins[ind], order)
    own = keys.clone()
    hg.build(own, M, out=(off2, own), offset_bytes=ob)  # in place
    assert torch.equal(off2, off) and torch.equal(_bins(own, M), order)
    assert torch.equal(torch.sort(own).values, torch.sort(keys).values)


@pytest.mark.parametrize("kb", [4, 8])
@pytest.mark.parametrize("kind,share", [("one", 1.0), ("many", 0.6), ("neighbours", 0.5)])
def test_hot_probes(kind, share, kb, dev):
    import torch
    import hashgraph_amd as hg
    M = 1 << 24
    print(f"hot probe {kind} share={share} kb={kb}", flush=True)
    B = _keys(kind, share, kb, N, M, dev)
    picked = torch.unique(B[:: N // 500])  # a copy each: as many matches as keys that have one
    A = torch.cat([wl.uniform_keys(23, N - picked.numel(), kb, device=dev), picked])
    off, csr = hg.build(A, M)
    ua, ca = torch.unique(A, return_counts=True)
    pos = torch.searchsorted(ua, B).clamp(max=ua.numel() - 1)
    want = torch.repeat_interleave(B, torch.where(ua[pos] == B, ca[pos], 0))
    cnt, out = hg.probe(off, csr, M, B)
    assert cnt == want.numel() == hg.probe(off, csr, M, B, emit=False)[0]
    assert torch.equal(torch.sort(out).values, torch.sort(want).values)


def test_hot_learned_build(dev):
    import torch
    import hashgraph_amd as hg
    M = 1 << 24
    keys = wl.lognormal_keys(3, N, device=dev)
    model, _ = hg.rmi_train(keys, M, n_sample=200000, seed=1, n_leaves=4096)
    keys[::3] = keys[7]
    keys[1::5] = keys[11]
    kw = {"hash_kind": hg.HG_HASH_RMI, "rmi_model": model}
    bins = hg.table_bins(keys, M, **kw).to(torch.int64)
    off, csr = hg.build(keys, M, **kw)
    _check_table(off, csr, keys, bins, M)
    order = torch.repeat_interleave(torch.arange(M, device=dev), off.diff().to(torch.int64))
    assert torch.equal(hg.table_bins(csr, M, **kw).to(torch.int64), order)


def test_hot_slabs_of_a_staged_build(dev):
    """Slabs of more keys than the narrow pass takes, the later ones beginning
    at a bin other than 0."""
    import torch
    import hashgraph_amd as hg
    n, M = 1 << 25, 1 << 25
    keys = _keys("many", 0.2, 4, n, M, dev)
    host = torch.empty(n, dtype=torch.int32, pin_memory=True).copy_(keys)
    out = (torch.empty(M + 1, dtype=torch.int32, pin_memory=True), torch.empty(n, dtype=torch.int32, pin_memory=True))
    off, csr = hg.build_staged(host, M, out=out, device_budget=720 << 20, device=0)
    off, csr = off.to(dev), csr.to(dev)
    _check_table(off, csr, keys, _bins(keys, M), M)
    assert torch.equal(_bins(csr, M), torch.repeat_interleave(torch.arange(M, device=dev), off.diff().to(torch.int64)))


@pytest.mark.parametrize("kb,ob", [(4, 4), (8, 8)])
@pytest.mark.parametrize("copies", [1, 64, 300])
@pytest.mark.parametrize("n,M", [(40000, 40000), (1 << 18, 1 << 18), (3 << 20, 3 << 20), (4194305, 1 << 22),
                                 (14600000, 14600000), (1 << 20, 1 << 25), (1 << 21, 1 << 13)])
def test_narrow_builds_of_copies(n, M, copies, kb, ob, dev):
    """The narrow pass's widths, from the fewest buckets of a class to all of
    its columns; copies of the keys fill the buckets unevenly."""
    import torch
    import hashgraph_amd as hg
    print(f"narrow n={n} M={M} copies={copies} kb={kb} ob={ob}", flush=True)
    keys = wl.uniform_keys(29, n, kb, device=dev)
    if copies > 1:
        keys = keys % (n // copies)
    bins = _bins(keys, M)
    off, csr = hg.build(keys, M, offset_bytes=ob)
    _check_table(off, csr, keys, bins, M)
    order = torch.repeat_interleave(torch.arange(M, device=dev), off.diff().to(torch.int64))
    assert torch.equal(_bins(csr, M), order)
    off2, ck, ind = hg.build_indexed(keys, M, offset_bytes=ob)
    assert torch.equal(off2, off) and torch.equal(torch.sort(ind).values, torch.arange(n, device=dev))
    assert torch.equal(ck, keys[ind]) and torch.equal(bins[ind], order)


@pytest.mark.parametrize("kb", [4, 8])
@pytest.mark.parametrize("per", [0.1, 1, 4, 16, 17.5, 18, 24.9, 25, 40, 300])
@pytest.mark.parametrize("n", [2500000, 12582912, 20000003])
def test_dense_probes(n, per, kb, dev):
    """Keys of A a bin on both sides of the lines between the probe's ways."""
    import torch
    import hashgraph_amd as hg
    M = int(n / per)
    print(f"dense probe n={n} M={M} kb={kb}", flush=True)
    A = wl.uniform_keys(31, n, kb, device=dev)
    B = wl.probe_keys(A, 32, n // 2, 0.4, kb, device=dev)
    off, csr = hg.build(A, M)
    ua, ca = torch.unique(A, return_counts=True)
    pos = torch.searchsorted(ua, B).clamp(max=ua.numel() - 1)
    want = torch.repeat_interleave(B, torch.where(ua[pos] == B, ca[pos], 0))
    cnt, out = hg.probe(off, csr, M, B)
    assert cnt == want.numel() and torch.equal(torch.sort(out).values, torch.sort(want).values)
