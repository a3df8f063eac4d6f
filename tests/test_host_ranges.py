"""A staged build's kernels write host memory only where one pinned range
covers all of it (hg_common.hpp: covers), also with other memory between two
pinned ends, which they must not touch."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hashgraph_amd", "csrc")
CASES = """
  // start, size, p, bytes, covered
  CHECK(4096, 8192, 4096, 8192, true)
  CHECK(4096, 8192, 4100, 8188, true)
  CHECK(4096, 8192, 12284, 4, true)
  CHECK(4096, 8192, 4096, 0, true)
  CHECK(4096, 8192, 4095, 8, false)          // begins before it
  CHECK(4096, 8192, 4100, 8192, false)       // ends behind it
  CHECK(4096, 8192, 12288, 4, false)         // begins behind it
  CHECK(4096, 8192, 4096, 24576, false)      // its end is in another range (20480 ..)
  CHECK(~0ull - 4095, 4096, ~0ull - 7, 8, true)   // at the end of the addresses
  CHECK(~0ull - 4095, 4096, ~0ull - 7, 16, false)
  CHECK(4096, 8192, 8192, ~0ull - 8191, false)    // a length that wraps around
  CHECK(4096, 0, 4096, 1, false)
"""


def test_covers(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text('#include "hg_common.hpp"\n#define CHECK(s, n, p, b, want) '
                   'static_assert(hg::covers(s, n, p, b) == want, "covers");\n' + CASES + "int main() { return 0; }\n")
    r = subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-fsyntax-only", str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr


@pytest.mark.gpu
def test_pinned_slices_take_the_kernels(dev):
    """Slices of pinned tensors are written by kernels (one column scan a chunk,
    of the counting pass), pageable memory by copies (two)."""
    import torch
    import hashgraph_amd as hg
    n, M = 1 << 20, 1 << 20
    keys = torch.randint(-2**31, 2**31 - 1, (n,), dtype=torch.int32)
    want = hg.build(keys.to(dev), M)
    c, scans = hg.context(), []
    for pinned in (True, False):
        def host(k):
            return torch.empty(k + 100, dtype=torch.int32, pin_memory=pinned)[60:60 + k]

        off, csr = host(M + 1), host(n)
        c.profile(True)
        c.profile_read()
        hg.build_staged(host(n).copy_(keys), M, out=(off, csr), device_budget=4 << 20, device=0)
        scans.append(c.profile_read()["col_scan"][0])
        c.profile(False)
        assert torch.equal(off, want[0].cpu())
        assert torch.equal(csr.sort().values, keys.sort().values)
    assert scans[1] == 2 * scans[0] > 2
