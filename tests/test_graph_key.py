"""Keys of the captured PCG graphs: two MAS hierarchies that launch differently
have different keys.  The key is host code of the library's own header; a small
program here compiles it (host side only) and prints keys of made-up tables."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "context.hpp"
#include <cstdio>
using namespace sgipc;
static void tables(MasState& m, std::vector<int> ls) {
    m.n = 500; m.M = 512; m.bank = 16; m.L = (int)ls.size() / 2 - 1; m.level_size_h = ls;
    m.total = ls[2 * m.L + 1]; m.nbanks = m.total / m.bank; m.nb1 = (ls[2] + 15) / 16;
    std::printf("%d %d %d ", m.nbanks, m.nb1, mas_top_bank0(m));
}
static void put(const MasState& m) {
    GraphKey k;
    k.mix(m);
    std::printf("%zu\n", k.h);
}
int main() {
    { MasState m; tables(m, {0, 0, 64, 512, 40, 576, 16, 624, 1, 640}); put(m); }   // 48 + 16 nodes on levels 2, 3
    { MasState m; tables(m, {0, 0, 64, 512, 20, 576, 20, 608, 1, 640}); put(m); }   // 32 + 32 nodes
    { MasState m; tables(m, {0, 0, 64, 512, 40, 576, 16, 624, 1, 640}); put(m); }   // the first again
    // pointers that one of the two engines' launches take
    { MasState m; tables(m, {0, 0, 64, 512, 40, 576, 16, 624, 1, 640}); m.comp_mask.p = (unsigned*)8; put(m);
      m.comp_mask.p = nullptr; }
    { MasState m; tables(m, {0, 0, 64, 512, 40, 576, 16, 624, 1, 640}); m.l1hi.p = (int*)8; put(m);
      m.l1hi.p = nullptr; }
}
"""


def test_graph_keys_tell_hierarchies_apart(tmp_path):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not (os.path.exists(hipcc) or shutil.which(hipcc)):
        pytest.skip("no hipcc")
    src = tmp_path / "key.hip"
    src.write_text(SRC)
    exe = tmp_path / "key"
    p = subprocess.run([hipcc, "-std=c++17", "-O1", "--offload-arch=gfx950", "--offload-host-only", "-x", "hip",
                        "-I", os.path.join(ROOT, "stiff-gipc_amd", "csrc"), str(src), "-o", str(exe)],
                       capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stderr[-2000:]
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stderr
    rows = [list(map(int, ln.split())) for ln in out.stdout.split("\n") if ln]
    a, b, again, mask, hi = rows
    assert a[:2] == b[:2] == [40, 4] and a[2] != b[2]       # the same totals, another boundary
    assert a[3] != b[3]
    assert again == a
    assert len({a[3], mask[3], hi[3]}) == 3
