"""Small and mid-sized tables, which take shorter kernel sequences than large
ones: edges of every size class against the CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from hashgraph_amd import workloads as wl
from oracle import oracle as o


def _to_dev(a, dev):
    import torch
    return torch.from_numpy(a.view(np.int32 if a.dtype == np.uint32 else np.int64).copy()).to(dev)


def _same(off, csr, keys, M, ob):
    goff = off.cpu().numpy().view(np.uint32 if ob == 4 else np.uint64).astype(np.uint64)
    gcsr = csr.cpu().numpy().view(keys.dtype).copy()
    eoff, ecsr = o.build_csr(keys, M)
    assert np.array_equal(goff, eoff), "offsets differ"
    o.canon(goff, gcsr)
    o.canon(eoff, ecsr)
    assert np.array_equal(gcsr, ecsr), "bin contents differ"


@pytest.mark.parametrize("kb,ob", [(4, 4), (8, 8)])
@pytest.mark.parametrize("n,M", [(1, 1), (1, 65535), (1024, 4096), (1024, 4097), (1025, 1000), (4096, 65535),
                                 (4097, 3), (16384, 16384), (16384, 65536), (16385, 16385)])
def test_one_workgroup_build(n, M, kb, ob, dev):
    import hashgraph_amd as hg
    print(f"one-workgroup build n={n} M={M} kb={kb} ob={ob}", flush=True)
    keys = wl.uniform_keys(n + M, n, kb)
    off, csr = hg.build(_to_dev(keys, dev), M, offset_bytes=ob)
    _same(off, csr, keys, M, ob)


@pytest.mark.parametrize("kb", [4, 8])
def test_one_workgroup_build_in_place_and_hot_key(kb, dev):
    """The CSR written over the input keys; a table of one repeated key."""
    import torch
    import hashgraph_amd as hg
    n, M = 16384, 5000
    for keys in (wl.uniform_keys(9, n, kb), np.full(n, 12345, dtype=np.uint32 if kb == 4 else np.uint64)):
        dk = _to_dev(keys, dev)
        off = torch.empty(M + 1, dtype=torch.int32, device=dev)
        hg.build(dk, M, out=(off, dk))
        _same(off, dk, keys, M, 4)


def test_one_workgroup_build_learned(dev):
    """A learned table of one workgroup: every key in the bin its hash gives."""
    import torch
    import hashgraph_amd as hg
    keys = wl.lognormal_keys(3, 16000)
    dk = _to_dev(keys, dev)
    M = 12000
    model, _ = hg.rmi_train(dk, M, n_sample=4000, seed=1, n_leaves=1024)
    off, csr = hg.build(dk, M, hash_kind=hg.HG_HASH_RMI, rmi_model=model)
    bins = hg.table_bins(dk, M, hash_kind=hg.HG_HASH_RMI, rmi_model=model).to(torch.int64)
    deg = torch.bincount(bins, minlength=M)
    assert torch.equal(off[1:].to(torch.int64), torch.cumsum(deg, 0)) and int(off[0]) == 0
    cb = hg.table_bins(csr, M, hash_kind=hg.HG_HASH_RMI, rmi_model=model).to(torch.int64)
    assert torch.equal(cb, torch.repeat_interleave(torch.arange(M, device=dev), deg))
    assert torch.equal(torch.sort(csr).values, torch.sort(dk).values)


def _probe_equal(hg, off, csr, M, A, B, dev, ob=4):
    dB = _to_dev(B, dev)
    eo, ek = o.build_csr(A, M)
    bo, bk = o.build_csr(B, M)
    ecnt, elst = o.intersect(eo, ek, bo, bk)
    assert hg.probe(off, csr, M, dB, emit=False)[0] == ecnt
    cnt, out = hg.probe(off, csr, M, dB)
    assert cnt == ecnt
    assert np.array_equal(np.sort(out.cpu().numpy().view(A.dtype)), np.sort(elst))
    return ecnt


@pytest.mark.parametrize("kb,ob", [(4, 4), (8, 8)])
@pytest.mark.parametrize("nB", [1, 255, 257, 65536, 65537, (1 << 18) + 1, (1 << 21) - 1])
def test_direct_probe_sizes(nB, kb, ob, dev):
    """Every workgroup size of the direct probe, with a remainder."""
    import hashgraph_amd as hg
    print(f"direct probe nB={nB} kb={kb} ob={ob}", flush=True)
    A = wl.uniform_keys(5, 100003, kb)
    M = 65537
    off, csr = hg.build(_to_dev(A, dev), M, offset_bytes=ob)
    _probe_equal(hg, off, csr, M, A, wl.probe_keys(A, 6, nB, 0.5, kb), dev, ob)


@pytest.mark.parametrize("kb", [4, 8])
def test_direct_probe_long_bins_short_output_and_overlap(kb, dev):
    """Keys of long bins (answered by the partitioned probe) beside keys of
    short ones; a buffer one match short; matches written over the probe keys."""
    import torch
    import hashgraph_amd as hg
    A = wl.uniform_keys(11, 50000, kb)
    A[:700] = A[0]
    A[1000:1033] = A[1000]
    M = 50000
    B = wl.probe_keys(A, 12, 20000, 0.6, kb)
    B[:40] = A[0]
    B[50:60] = A[1000]
    off, csr = hg.build(_to_dev(A, dev), M)
    n = _probe_equal(hg, off, csr, M, A, B, dev)
    dB = _to_dev(B, dev)
    short = torch.zeros(n - 1, dtype=dB.dtype, device=dev)
    with pytest.raises(hg.HGError):
        hg.probe(off, csr, M, dB, out=short)
    full = hg.probe(off, csr, M, dB)[1]
    both = torch.zeros(n + len(B), dtype=dB.dtype, device=dev)
    both[100:100 + len(B)] = dB
    cnt, _ = hg.probe(off, csr, M, both[100:100 + len(B)], out=both)
    assert cnt == n and torch.equal(torch.sort(both[:n]).values, torch.sort(full).values)


@pytest.mark.parametrize("kb", [4, 8])
def test_matches_beyond_the_first_buffers(kb, dev):
    """Calls that name no capacity and match more often than either side has
    keys: short bins, then one value in thousands of copies on both sides."""
    import torch
    import hashgraph_amd as hg
    for reps, one in ((3, 0), (1, 3000)):
        base = wl.uniform_keys(21, 4000, kb)
        A = np.concatenate([np.repeat(base, reps), np.full(one, base[0], dtype=base.dtype)])
        B = A[::-1].copy()
        M = 5000
        ta, tb = hg.build_indexed(_to_dev(A, dev), M), hg.build_indexed(_to_dev(B, dev), M)
        eo, ek = o.build_csr(A, M)
        bo, bk = o.build_csr(B, M)
        ecnt, elst = o.intersect(eo, ek, bo, bk)
        assert ecnt > len(A)
        _probe_equal(hg, ta[0], ta[1], M, A, B, dev)
        cnt, out = hg.intersect(ta[0], ta[1], tb[0], tb[1], M)
        assert cnt == ecnt and np.array_equal(np.sort(out.cpu().numpy().view(A.dtype)), np.sort(elst))
        cnt, pa, pb = hg.intersect_indexed(*ta, *tb, M)
        assert cnt == ecnt == pa.numel() == pb.numel()
        assert np.array_equal(A[pa.cpu().numpy()], B[pb.cpu().numpy()])
        assert torch.unique((pa << 32) | pb).numel() == cnt


# keys at the edges of the final stage's size classes (0.875 of the class times
# the 512 buckets of a narrow pass), ragged ranges, sparse and dense tables
@pytest.mark.parametrize("kb,ob", [(4, 4), (8, 8)])
@pytest.mark.parametrize("n,M", [(16385, 65537), (20011, 3000017), (70001, 70001), (300007, 40009), (1835007, 1835009),
                                 (1835009, 1835007), (3670021, 3670013), (7340041, 7340033)])
def test_narrow_build(n, M, kb, ob, dev):
    import hashgraph_amd as hg
    print(f"narrow build n={n} M={M} kb={kb} ob={ob}", flush=True)
    keys = wl.uniform_keys(n + M, n, kb)
    off, csr = hg.build(_to_dev(keys, dev), M, offset_bytes=ob)
    _same(off, csr, keys, M, ob)


@pytest.mark.parametrize("kb", [4, 8])
def test_narrow_build_oversized_buckets(kb, dev):
    """Hot keys: buckets beyond every size class, beside ordinary ones."""
    import hashgraph_amd as hg
    dt = np.uint32 if kb == 4 else np.uint64
    keys = wl.uniform_keys(31, 900000, kb)
    keys[100:300000] = keys[0]
    keys[400000:420000] = keys[1]
    for M in (900000, 65537):
        off, csr = hg.build(_to_dev(keys.astype(dt), dev), M)
        _same(off, csr, keys, M, 4)


@pytest.mark.parametrize("kb", [4, 8])
@pytest.mark.parametrize("n", [20011, 1835009])
def test_narrow_indexed_build(n, kb, dev):
    import torch
    import hashgraph_amd as hg
    keys = wl.uniform_keys(n, n, kb)
    keys[5:4000] = keys[5]
    dk = _to_dev(keys, dev)
    off, csr, ind = hg.build_indexed(dk, n)
    _same(off, csr, keys, n, 4)
    assert torch.equal(dk[ind], csr) and torch.equal(torch.sort(ind).values, torch.arange(n, device=dev))


def test_narrow_learned_build(dev):
    import torch
    import hashgraph_amd as hg
    n, M = 1000003, 900001
    dk = wl.lognormal_keys(8, n, device=dev)
    model, _ = hg.rmi_train(dk, M, seed=2)
    kw = {"hash_kind": hg.HG_HASH_RMI, "rmi_model": model}
    off, csr = hg.build(dk, M, **kw)
    deg = torch.bincount(hg.table_bins(dk, M, **kw).to(torch.int64), minlength=M)
    assert torch.equal(off[1:].to(torch.int64), torch.cumsum(deg, 0)) and int(off[0]) == 0
    assert torch.equal(hg.table_bins(csr, M, **kw).to(torch.int64),
                       torch.repeat_interleave(torch.arange(M, device=dev), deg))
    assert torch.equal(torch.sort(csr).values, torch.sort(dk).values)


@pytest.mark.parametrize("kb,ob", [(4, 4), (8, 8)])
@pytest.mark.parametrize("nA,nB,M", [(1310723, 1310721, 1310719), (100003, 3000017, 65537), (3000017, 1400003, 1000003),
                                     (200003, 1500007, 5000011), (6000011, 6000007, 6000013)])
def test_narrow_probe(nA, nB, M, kb, ob, dev):
    """Every bucket class of the narrow probe: balanced, many more probe keys
    than table keys, long and sparse bins."""
    import hashgraph_amd as hg
    print(f"narrow probe nA={nA} nB={nB} M={M} kb={kb} ob={ob}", flush=True)
    A = wl.uniform_keys(41, nA, kb)
    off, csr = hg.build(_to_dev(A, dev), M, offset_bytes=ob)
    _probe_equal(hg, off, csr, M, A, wl.probe_keys(A, 42, nB, 0.4, kb), dev, ob)


@pytest.mark.parametrize("kb", [4, 8])
def test_narrow_probe_skewed(kb, dev):
    """Buckets of B beyond every class, of A beyond the LDS, and long bins."""
    import hashgraph_amd as hg
    n = 1400003
    A = wl.uniform_keys(43, n, kb)
    A[10:40000] = A[10]
    B = wl.probe_keys(A, 44, n, 0.4, kb)
    B[1000:200000] = A[50000]   # a hot key with a short bin
    B[300000:300040] = A[10]    # a few of the long bin
    off, csr = hg.build(_to_dev(A, dev), n)
    _probe_equal(hg, off, csr, n, A, B, dev)


def test_narrow_probe_learned(dev):
    import torch
    import hashgraph_amd as hg
    n, M = 1500007, 1400003
    A = wl.lognormal_keys(51, n, device=dev)
    B = wl.mixed_probe(A, wl.lognormal_keys(52, n, device=dev), 53, 0.5)
    model, _ = hg.rmi_train(A, M, seed=2)
    kw = {"hash_kind": hg.HG_HASH_RMI, "rmi_model": model}
    cnt, out = hg.probe(*hg.build(A, M, **kw), M, B, **kw)
    ecnt, eout = hg.probe(*hg.build(A, M), M, B)
    assert cnt == ecnt and torch.equal(torch.sort(out).values, torch.sort(eout).values)


@pytest.mark.parametrize("kb", [4, 8])
def test_batch_of_many_tables_skewed(kb, dev):
    """A batch of more than 256 tables whose buckets fall into every size tier:
    ordinary, between the small and the largest class, beyond both; long bins."""
    import hashgraph_amd as hg
    T = 260
    sizes = [100 + 37 * t for t in range(T)]
    sizes[7], sizes[100], sizes[200] = 60000, 90000, 45000
    tabs, probes = [], []
    for t, n in enumerate(sizes):
        a = wl.uniform_keys(900 + t, n, kb)
        if t == 7:
            a[:12000] = a[0]          # one bucket between the classes
        elif t == 100:
            a[:50000] = a[0]          # one bucket beyond both
        elif t == 200:
            a[:300], a[300:700] = a[0], a[300]
        tabs.append(a)
        probes.append(wl.probe_keys(a, 5000 + 2 * t, n // 2 + 1, 0.4, kb))
        if t in (7, 100):
            probes[-1][:40] = a[0]
    ko = np.concatenate([[0], np.cumsum(sizes)])
    po = np.concatenate([[0], np.cumsum([len(b) for b in probes])])
    off, csr, oo = hg.batch_build(_to_dev(np.concatenate(tabs), dev), ko, sizes)
    total, counts = hg.batch_probe(off, csr, ko, sizes, oo, _to_dev(np.concatenate(probes), dev), po)
    goff, gcsr = off.cpu().numpy().view(np.uint32), csr.cpu().numpy().view(tabs[0].dtype)
    exp = []
    for t, n in enumerate(sizes):
        eo, ek = o.build_csr(tabs[t], n)
        assert np.array_equal(goff[oo[t]:oo[t] + n + 1].astype(np.uint64), eo), f"table {t}: offsets differ"
        g = gcsr[ko[t]:ko[t + 1]].copy()
        o.canon(eo, g)
        o.canon(eo, ek)
        assert np.array_equal(g, ek), f"table {t}: bins differ"
        bo, bk = o.build_csr(probes[t], n)
        exp.append(o.intersect(eo, ek, bo, bk)[0])
    assert counts.cpu().numpy().tolist() == exp and total == sum(exp)


def _csr_matches(hg, dk, off, csr, M, **kw):
    """Table of dk on the device: degrees, bins in order, the same keys."""
    import torch
    deg = torch.bincount(hg.table_bins(dk, M, **kw).to(torch.int64) & 0xFFFFFFFF, minlength=M)
    assert int(off[0]) == 0 and torch.equal(off[1:].to(torch.int64) & 0xFFFFFFFF, torch.cumsum(deg, 0))
    assert torch.equal(hg.table_bins(csr, M, **kw).to(torch.int64) & 0xFFFFFFFF,
                       torch.repeat_interleave(torch.arange(M, device=dk.device), deg))
    assert torch.equal(torch.sort(csr).values, torch.sort(dk).values)


# two-step partitions: as many keys as bins, long bins, a table of few keys a
# bin (every bucket at its widest), sizes that leave short rows and tiles
@pytest.mark.parametrize("kb,ob", [(4, 4), (8, 8)])
@pytest.mark.parametrize("n,M", [(15000011, 15000017), (20000003, 1000003), (16777217, 900000011), (40000003, 39999983)])
def test_two_step_build_and_probe(n, M, kb, ob, dev):
    import torch
    import hashgraph_amd as hg
    print(f"two-step n={n} M={M} kb={kb} ob={ob}", flush=True)
    dk = wl.uniform_keys(n, n, kb, device=dev)
    dk[5:3000] = dk[5]                 # a long bin
    dk[1000000:1009000] = dk[1000000]  # a bucket beyond the small class
    off, csr = hg.build(dk, M, offset_bytes=ob)
    _csr_matches(hg, dk, off, csr, M)
    q = wl.probe_keys(dk, n + 1, n // 2 + 1, 0.3, kb, device=dev)
    q[100:50000] = dk[77]              # a bucket of B beyond every class
    cnt, out = hg.probe(off, csr, M, q)
    vals, num = torch.unique(csr, return_counts=True)
    at = torch.searchsorted(vals, q).clamp_(max=vals.numel() - 1)
    m = torch.where(vals[at] == q, num[at], 0)
    assert cnt == int(m.sum())
    assert torch.equal(torch.sort(out).values, torch.sort(torch.repeat_interleave(q, m)).values)


@pytest.mark.parametrize("kb", [4, 8])
def test_two_step_build_in_place_and_indexed(kb, dev):
    """The CSR written over the input keys; the index-carrying form; one value
    in more copies than a bucket, a group's share of them, half the table."""
    import torch
    import hashgraph_amd as hg
    n, M = 16000001, 15000013
    dk = wl.uniform_keys(3, n, kb, device=dev)
    off, csr, ind = hg.build_indexed(dk, M)
    _csr_matches(hg, dk, off, csr, M)
    assert torch.equal(dk[ind], csr) and torch.equal(torch.sort(ind).values, torch.arange(n, device=dev))
    dk[::2] = dk[1]
    keep = dk.clone()
    off = torch.empty(M + 1, dtype=torch.int32, device=dev)
    hg.build(dk, M, out=(off, dk))
    _csr_matches(hg, keep, off, dk, M)


def test_two_step_learned(dev):
    """Skewed keys under a learned hash: the same matches as under murmur3."""
    import torch
    import hashgraph_amd as hg
    n, M = 15000013, 15000001
    A = wl.lognormal_keys(61, n, device=dev)
    B = wl.mixed_probe(A, wl.lognormal_keys(62, n, device=dev), 63, 0.5)
    model, _ = hg.rmi_train(A, M, seed=2)
    kw = {"hash_kind": hg.HG_HASH_RMI, "rmi_model": model}
    off, csr = hg.build(A, M, **kw)
    _csr_matches(hg, A, off, csr, M, **kw)
    cnt, out = hg.probe(off, csr, M, B, **kw)
    ecnt, eout = hg.probe(*hg.build(A, M), M, B)
    assert cnt == ecnt and torch.equal(torch.sort(out).values, torch.sort(eout).values)


@pytest.mark.parametrize("kb,n", [(4, 28000001), (4, 30500003), (8, 28000001)])
def test_partitions_around_the_few_column_scatter(kb, n, dev):
    """Second partition levels just below and above its 512 columns."""
    import torch
    import hashgraph_amd as hg
    M = n
    dk = wl.uniform_keys(71, n, kb, device=dev)
    off, csr, po = hg.build_partitioned(dk, M, [0, M // 2, M])
    whole = hg.build(dk, M)[0].to(torch.int64)
    for p, (lo, hi) in enumerate(((0, M // 2), (M // 2, M))):
        assert torch.equal(off[lo + p:hi + p + 1].to(torch.int64), whole[lo:hi + 1] - whole[lo])
    deg = whole[1:] - whole[:-1]
    assert torch.equal(hg.table_bins(csr[:po[2]], M).to(torch.int64) & 0xFFFFFFFF,
                       torch.repeat_interleave(torch.arange(M, device=dev), deg))
    assert torch.equal(torch.sort(csr[:po[2]]).values, torch.sort(dk).values)


# keys a bin around what the join stages: a bin number per key of B fits behind
# the keys, then only the keys do, then not even they
@pytest.mark.parametrize("kb,ob", [(4, 4), (8, 8)])
@pytest.mark.parametrize("per", [0.3, 1.0, 1.4, 2.2, 2.6, 3.3, 5.0])
def test_join_keys_per_bin(per, kb, ob, dev):
    import hashgraph_amd as hg
    M = 6145
    n = int(per * M)
    A = wl.uniform_keys(81, n, kb)
    A[: n // 3] = A[n // 3: 2 * (n // 3)]   # every second match twice
    A[5:140] = A[5]                         # a bin beyond the pair limit
    B = wl.probe_keys(A, 82, n + 77, 0.9, kb)
    B[300:400] = A[5]
    ta, tb = (hg.build_indexed(_to_dev(x, dev), M, offset_bytes=ob) for x in (A, B))
    eo, ek = o.build_csr(A, M)
    bo, bk = o.build_csr(B, M)
    ecnt, elst = o.intersect(eo, ek, bo, bk)
    assert hg.intersect(ta[0], ta[1], tb[0], tb[1], M, emit=False)[0] == ecnt
    cnt, out = hg.intersect(ta[0], ta[1], tb[0], tb[1], M)
    assert cnt == ecnt and np.array_equal(np.sort(out.cpu().numpy().view(A.dtype)), np.sort(elst))
    cnt, pa, pb = hg.intersect_indexed(*ta, *tb, M)
    pa, pb = pa.cpu().numpy(), pb.cpu().numpy()
    assert cnt == ecnt and np.array_equal(A[pa], B[pb]) and len(np.unique((pa << 32) | pb)) == cnt


def test_two_step_larger_buckets(dev):
    """More keys than 8 K-key buckets can be counted for: the next class."""
    import torch
    import hashgraph_amd as hg
    n = M = 302000011
    dk = wl.uniform_keys(91, n, 4, device=dev)
    off, csr = hg.build(dk, M)
    deg = torch.bincount(hg.table_bins(dk, M), minlength=M)
    assert int(off[0]) == 0 and torch.equal(off[1:].to(torch.int64), torch.cumsum(deg, 0))
    assert torch.equal(hg.table_bins(csr, M).to(torch.int64), torch.repeat_interleave(torch.arange(M, device=dev), deg))
    assert torch.equal(torch.sort(csr).values, torch.sort(dk).values)
    q = wl.probe_keys(dk, 92, n // 2, 0.3, 4, device=dev)
    cnt, out = hg.probe(off, csr, M, q)
    tq = hg.build(q, M)
    assert (cnt, int(out.to(torch.int64).sum())) == (lambda c, o: (c, int(o.to(torch.int64).sum())))(
        *hg.intersect(off, csr, *tq, M))
