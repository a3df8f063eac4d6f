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
