"""The buffers of a join or probe whose caller names no capacity, when memory
is short: the library and the allocator are stood in for, so that each of them
can refuse."""
import ctypes

import pytest
import torch

import hashgraph_amd as hg
from hashgraph_amd import _lib


class Library:
    """Writes min(matches, capacity) numbers; refuses with HG_ERR_OOM while
    more than `room` matches of buffers are held."""

    def __init__(self, matches, room):
        self.matches, self.room, self.cnt, self.calls = matches, room, ctypes.c_uint64(0), []

    def call(self, bufs, capacity):
        self.calls.append(capacity)
        if capacity > self.room:
            return _lib.HG_ERR_OOM
        self.cnt.value = self.matches
        for b in bufs or []:
            b[: min(self.matches, capacity)] = torch.arange(min(self.matches, capacity), dtype=b.dtype)
        return _lib.HG_OK if not bufs or self.matches <= capacity else _lib.HG_ERR_CAPACITY


class NoClone(torch.Tensor):
    """A buffer that nothing can be copied out of (no memory for the copy)."""

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        if func is torch.Tensor.clone:
            raise torch.OutOfMemoryError("no memory for a copy")
        return super().__torch_function__(func, types, args, kwargs or {})


def _alloc(n):
    return [torch.full((n,), -1, dtype=torch.int64) for _ in range(2)]


def _check(out, matches):
    assert len(out) == 2
    for b in out:
        assert torch.equal(torch.as_tensor(b).as_subclass(torch.Tensor), torch.arange(matches))


@pytest.mark.parametrize("matches", [0, 3, 100])
def test_library_out_of_memory_beside_the_guess(matches):
    """The guess took the room that the library's scratch needs: it is given
    back, and the counting pass and the exact buffers follow."""
    lib = Library(matches, room=max(matches, 1))
    _check(hg._emit(lib.call, 1000, _alloc, lib.cnt, "x"), matches)
    assert lib.calls == [1000, 0, matches]


def test_no_memory_for_the_copy():
    """The result is whole before the copy that gives the spare room back."""
    lib = Library(7, room=1000)
    _check(hg._emit(lib.call, 1000, lambda n: [b.as_subclass(NoClone) for b in _alloc(n)], lib.cnt, "x"), 7)
    assert lib.calls == [1000]


def test_no_memory_for_the_guess():
    def alloc(n):
        if n > 50:
            raise torch.OutOfMemoryError("no memory")
        return _alloc(n)

    lib = Library(7, room=1000)
    _check(hg._emit(lib.call, 1000, alloc, lib.cnt, "x"), 7)
    assert lib.calls == [0, 7]


@pytest.mark.parametrize("matches,calls", [(7, [10]), (10, [10]), (25, [10, 25])])
def test_enough_memory(matches, calls):
    lib = Library(matches, room=1000)
    _check(hg._emit(lib.call, 10, _alloc, lib.cnt, "x"), matches)
    assert lib.calls == calls


def test_other_errors_are_raised():
    cnt = ctypes.c_uint64(0)
    for guess in (10, 0):
        with pytest.raises(hg.HGError):
            hg._emit(lambda bufs, cap: 3, guess, _alloc, cnt, "x")
    with pytest.raises(hg.HGError):  # no scratch even without the guess
        hg._emit(lambda bufs, cap: _lib.HG_ERR_OOM, 10, _alloc, cnt, "x")
