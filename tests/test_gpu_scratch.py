"""Scratch memory of builds and probes: what hg_scratch_bytes states, what
hg_ctx_reserve covers, and what happens when there is no more."""
import ctypes

import pytest
import torch

import hashgraph_amd as hg
from hashgraph_amd import _lib
from hashgraph_amd import workloads as wl

P = hg._p


def _scratch(n, M, kb, ob=4):
    b = ctypes.c_size_t(0)
    assert _lib.load().hg_scratch_bytes(ctypes.byref(hg._desc(n, M, kb, ob)), 0, ctypes.byref(b)) == 0
    return b.value


@pytest.mark.parametrize("kb", [4, 8])
@pytest.mark.parametrize("n,M", [(1000, 1000), (1 << 16, 1 << 16), (1 << 20, 1 << 20), (1 << 20, 1 << 25)])
def test_stated_scratch_holds_a_direct_probe(kb, n, M):
    """Half of it (hg_ctx_reserve's share of each arena) holds the listed keys
    and their partitioned copy, and a build's per-bin counters."""
    assert _scratch(n, M, kb) // 2 >= 2 * n * kb
    if n > 16384:
        assert _scratch(n, M, kb) // 2 >= 4 * M


def _keys(kind, n, kb):
    if kind == "uniform":
        return wl.uniform_keys(1, n, kb, device="cuda")
    k = wl.zipf_keys(1, n, 1.1, device="cuda")
    return k if kb == 8 else k.to(torch.int32)


def _build_probe(c, A, B, M, off, csr):
    d = hg._desc(A.numel(), M, A.element_size(), 4)
    cnt = ctypes.c_uint64(0)
    hg.check(c.lib.hg_build(c.bind_stream(), ctypes.byref(d), P(A), P(off), P(csr)), "hg_build")
    hg.check(c.lib.hg_probe(c.bind_stream(), ctypes.byref(d), P(off), P(csr), P(B), B.numel(), None, 0,
                            ctypes.byref(cnt)), "hg_probe")
    return cnt.value


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["uniform", "zipf"])
@pytest.mark.parametrize("kb", [4, 8])
@pytest.mark.parametrize("n,M", [(1 << 20, 1 << 20), (1 << 22, 1 << 22), (3000001, 1 << 20), (1 << 25, 1 << 25),
                                 (1 << 22, 1 << 17)])
def test_reserved_context_allocates_nothing(kind, kb, n, M):
    A, B = _keys(kind, n, kb), _keys(kind, n, kb).flip(0).contiguous()
    fewer = B[: n // 3].clone()
    off = torch.empty(M + 1, dtype=torch.int32, device="cuda")
    csr = torch.empty_like(A)
    want = _build_probe(hg.context(), A, B, M, off, csr)  # the kernels are loaded
    c = hg.Context(0)
    try:
        c.reserve(_scratch(n, M, kb))
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        assert _build_probe(c, A, B, M, off, csr) == want
        assert _build_probe(c, A, fewer, M, off, csr) <= want
        torch.cuda.synchronize()
        assert torch.cuda.mem_get_info()[0] == free
    finally:
        c.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kb", [4, 8])
def test_keys_listed_by_a_direct_probe_survive_a_growing_arena(kb):
    """Every probe key is listed (long bins only), so the partitioned probe
    that follows needs more of the arena than the list did."""
    n, M = 1 << 19, 1 << 17
    A = _keys("uniform", n, kb)[: n // 64].repeat(64)
    B = A.flip(0).contiguous()
    off = torch.empty(M + 1, dtype=torch.int32, device="cuda")
    csr = torch.empty_like(A)
    c = hg.Context(0)
    try:
        d = hg._desc(n, M, kb, 4)
        hg.check(hg.context().lib.hg_build(hg.context().bind_stream(), ctypes.byref(d), P(A), P(off), P(csr)), "hg_build")
        torch.cuda.synchronize()
        cnt = ctypes.c_uint64(0)
        out = torch.empty(n * 64, dtype=A.dtype, device="cuda")
        hg.check(c.lib.hg_probe(c.bind_stream(), ctypes.byref(d), P(off), P(csr), P(B), n, P(out), n * 64,
                                ctypes.byref(cnt)), "hg_probe")
        assert cnt.value == n * 64
        assert torch.equal(out.sort().values, B.repeat_interleave(64).sort().values)
    finally:
        c.close()


class Room:
    """While entered, holds the device's memory but for `nbytes`."""

    def __init__(self, nbytes):
        self.nbytes = nbytes

    def __enter__(self):
        torch.cuda.empty_cache()
        torch.cuda.synchronize()
        block = 64 << 20
        self.held = [torch.empty(torch.cuda.mem_get_info()[0] - self.nbytes, dtype=torch.uint8, device="cuda")]
        spare = []
        try:  # what is free beyond the stated bytes, and inside cached segments (the first blocks), too
            while len(spare) < 1024:
                spare.append(torch.empty(block, dtype=torch.uint8, device="cuda"))
        except torch.OutOfMemoryError:
            pass
        self.held += spare[: -(self.nbytes // block)]
        del spare
        torch.cuda.empty_cache()

    def __exit__(self, *exc):
        self.held.clear()
        torch.cuda.empty_cache()


@pytest.mark.gpu
def test_build_in_place_without_memory_takes_one_copy():
    """2^26 uint32 keys: 256 MiB a copy, as much again for the bins' counters.
    The two-step partition needs two copies in place, the wide pass one."""
    n = 1 << 26
    keys = wl.uniform_keys(1, n, 4, device="cuda")
    off, csr = hg.build(keys, n, 4)
    off2 = torch.empty_like(off)
    c = hg.Context(0)
    try:
        with Room(640 << 20):
            hg.check(c.lib.hg_build(c.bind_stream(), ctypes.byref(hg._desc(n, n, 4, 4)), P(keys), P(off2), P(keys)),
                     "hg_build")
            torch.cuda.synchronize()
    finally:
        c.close()
    assert torch.equal(off, off2)
    bins = torch.repeat_interleave(torch.arange(n, dtype=torch.int32, device="cuda"), off.diff())
    assert torch.equal(hg.hash_bins(keys, n), bins)
    assert torch.equal(keys.sort().values, csr.sort().values)


@pytest.mark.gpu
def test_probe_without_memory_takes_one_copy():
    """2^26 uint64 keys, 512 MiB a copy."""
    n = 1 << 26
    A = wl.uniform_keys(1, n, 8, device="cuda")
    off, csr = hg.build(A, n, 4)
    cnt = ctypes.c_uint64(0)
    c = hg.Context(0)
    try:
        with Room(900 << 20):
            hg.check(c.lib.hg_probe(c.bind_stream(), ctypes.byref(hg._desc(n, n, 8, 4)), P(off), P(csr), P(A), n, None,
                                    0, ctypes.byref(cnt)), "hg_probe")
    finally:
        c.close()
    assert cnt.value == hg.probe(off, csr, n, A, emit=False)[0] >= n


@pytest.mark.gpu
@pytest.mark.parametrize("kb", [4, 8])
def test_run_length_join_keeps_to_its_bounds(kb):
    """Tables of 2^24 keys without a common bin: no record, so no room for one
    per key (335 MiB for uint32 keys, 403 for uint64)."""
    n = M = 1 << 24
    keys = wl.uniform_keys(1, 3 * n, kb, device="cuda")
    low = hg.hash_bins(keys, M) < M // 2
    ta, tb = (hg.build(k[:n].clone(), M, 4) for k in (keys[low], keys[~low]))
    rk, ca, cb = (torch.empty(n, dtype=d, device="cuda") for d in (keys.dtype, torch.int64, torch.int64))
    cnt, nrec = ctypes.c_uint64(1), ctypes.c_uint64(1)

    def join(c):
        d = hg._desc(n, M, kb, 4)
        hg.check(c.lib.hg_intersect_rle(c.bind_stream(), ctypes.byref(d), P(ta[0]), P(ta[1]), ctypes.byref(d), P(tb[0]),
                                        P(tb[1]), P(rk), P(ca), P(cb), n, ctypes.byref(nrec), ctypes.byref(cnt)), "rle")
        assert (cnt.value, nrec.value) == (0, 0)
        torch.cuda.synchronize()

    join(hg.context())  # the kernels are loaded
    c = hg.Context(0)
    try:
        free = torch.cuda.mem_get_info()[0]
        join(c)
        assert free - torch.cuda.mem_get_info()[0] < 200 << 20
    finally:
        c.close()


@pytest.mark.gpu
def test_context_created_while_a_stream_captures():
    """A context made by one thread neither waits for another thread's capture
    nor spoils it."""
    import threading
    x = torch.zeros(1000, device="cuda")
    made, g = [], torch.cuda.CUDAGraph()

    def make():
        try:
            made.append(hg.Context(0))
        except hg.HGError as e:
            made.append(e)

    with torch.cuda.graph(g, stream=torch.cuda.Stream(), capture_error_mode="thread_local"):
        x += 1
        t = threading.Thread(target=make)
        t.start()
        t.join()
        x += 1
    assert isinstance(made[0], hg.Context), made[0]
    for i in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert bool((x == 2 * (i + 1)).all())
    keys = torch.arange(1000, dtype=torch.int32, device="cuda")
    off, csr = hg.build(keys, 1000)
    cnt = ctypes.c_uint64(0)
    c = made[0]
    for _ in range(3):
        hg.check(c.lib.hg_probe(c.bind_stream(), ctypes.byref(hg._desc(1000, 1000, 4)), P(off), P(csr), P(keys), 1000,
                                None, 0, ctypes.byref(cnt)), "hg_probe")
        assert cnt.value == 1000
    c.close()
