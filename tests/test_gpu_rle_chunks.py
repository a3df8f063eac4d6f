"""Run-length join at the edges of its chunks: chunk remainders, chunks whose
light keys need several rounds, light and heavy bins side by side."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from hashgraph_amd import workloads as wl
from oracle import oracle as o


def _to_dev(a, dev):
    import torch
    return torch.from_numpy(a.view(np.int32 if a.dtype == np.uint32 else np.int64).copy()).to(dev)


@pytest.mark.parametrize("kb,ob", [(4, 4), (8, 8)])
@pytest.mark.parametrize("n,M,values", [(600, 511, 300), (20000, 512, 9000), (40000, 513, 15000), (40000, 1025, 2000),
                                        (30000, 1, 50), (65536, 1024, 1 << 30)])
def test_rle_rounds(n, M, values, kb, ob, dev):
    """values: distinct values the keys are drawn from (copies on both sides)."""
    import hashgraph_amd as hg
    print(f"rle rounds n={n} M={M} values={values} kb={kb} ob={ob}", flush=True)
    pool = wl.uniform_keys(71, min(values, 1 << 16), kb)
    A = pool[(wl.stream_np(72, n) % np.uint64(len(pool))).astype(np.int64)]
    B = pool[(wl.stream_np(73, n) % np.uint64(len(pool))).astype(np.int64)]
    A[:64], A[64:129] = pool[0], pool[1]   # 64 or more and 65 or more copies of two values
    ta, tb = hg.build(_to_dev(A, dev), M, offset_bytes=ob), hg.build(_to_dev(B, dev), M, offset_bytes=ob)
    oa, ka = o.build_csr(A, M)
    ob_, kb_ = o.build_csr(B, M)
    o.canon(oa, ka)  # the oracle counts runs of canonical bins
    o.canon(ob_, kb_)
    expected = o.intersect_rle(oa, ka, ob_, kb_)
    ecnt, ek, eca, ecb = expected
    for cap in (None, len(ek)):
        cnt, rk, ca, cb = hg.intersect_rle(*ta, *tb, M, capacity=cap)
        assert cnt == ecnt and rk.numel() == len(ek)
        g = np.argsort(rk.cpu().numpy().view(A.dtype))
        e = np.argsort(ek)
        assert np.array_equal(rk.cpu().numpy().view(A.dtype)[g].astype(np.uint64), ek[e])
        assert np.array_equal(ca.cpu().numpy()[g].astype(np.uint64), np.asarray(eca)[e].astype(np.uint64))
        assert np.array_equal(cb.cpu().numpy()[g].astype(np.uint64), np.asarray(ecb)[e].astype(np.uint64))


def _check_rle(A, B, M, dev):
    import torch
    import hashgraph_amd as hg
    ua, ca = torch.unique(A, return_counts=True)
    ub, cb = torch.unique(B, return_counts=True)
    pos = torch.searchsorted(ua, ub).clamp(max=ua.numel() - 1)
    hit = ua[pos] == ub
    want = (ub[hit], ca[pos[hit]], cb[hit])
    ta, tb = hg.build(A, M), hg.build(B, M)
    for cap in (None, want[0].numel(), want[0].numel() + 7):
        cnt, rk, ra, rb = hg.intersect_rle(*ta, *tb, M, capacity=cap)
        assert cnt == int((want[1] * want[2]).sum())
        o = torch.argsort(rk)
        for x, y in zip((rk, ra, rb), want):
            assert torch.equal(x[o], y.to(x.dtype))


@pytest.mark.parametrize("kb", [4, 8])
@pytest.mark.parametrize("M", [(1 << 25) + 1, (1 << 25) + 8192 * 512 + 1])
def test_rle_more_chunks_than_one_scan(M, kb, dev):
    """Tables of more than 2^16 chunks of 512 bins, most of them empty."""
    print(f"rle many chunks M={M} kb={kb}", flush=True)
    pool = wl.uniform_keys(81, 300000, kb, device=dev)
    A = pool.repeat(3)
    B = pool[100000:].repeat(2)
    A[:100000] = pool[200001]
    _check_rle(A, B, M, dev)


@pytest.mark.parametrize("values,copies", [(63, 40000), (64, 40000), (65, 40000), (140, 40000), (400, 270000)])
def test_rle_many_giant_bins(values, copies, dev):
    """Bins of more than 2^15 keys, more of them than a wave has lanes and than
    their share of the places; bins of more than 2^18, more than there are places."""
    import torch
    print(f"rle giant bins values={values} copies={copies}", flush=True)
    pool = wl.uniform_keys(91, values, 4, device=dev)
    A = torch.cat([pool.repeat(copies), wl.uniform_keys(92, 100000, 4, device=dev)])
    B = torch.cat([pool.repeat(70), A[-50000:]])
    _check_rle(A, B, 1 << 20, dev)
