"""Buffers that are only of use together (lumen_amd/csrc/alloc_set.h) are
allocated all or none, whichever allocation fails, and a retry after a failure
completes the set; compiled for the host with an allocator that fails at a
given call."""
import shutil
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "alloc_set.h"
int main() {
    for (int fail = 0; fail <= 4; fail++) {  // the call that fails; 4: none
        void *a = nullptr, *b = nullptr, *c = nullptr, *d = nullptr;
        int call = 0, live = 0;
        const BufferReq set[] = {{&a, 8}, {&b, 16}, {&c, 24}, {&d, 32}};
        auto alloc = [&](void** p, size_t n) {
            if (call++ == fail) {
                *p = (void*)1;  // a failing allocator may leave anything there
                return 2;
            }
            *p = malloc(n);
            live++;
            return 0;
        };
        auto release = [&](void* p) {
            free(p);
            live--;
        };
        const int first = alloc_set(set, alloc, release);
        if (fail < 4) {
            if (first != 2 || live != 0 || a || b || c || d) return 1 + fail;
            if (alloc_set(set, alloc, release) != 0) return 11 + fail;
        } else if (first != 0) {
            return 20;
        }
        if (live != 4 || !a || !b || !c || !d) return 21 + fail;
        for (const BufferReq& r : set) release(*r.ptr);
    }
    return 0;
}
"""


def test_all_or_none(tmp_path):
    (tmp_path / "a.cpp").write_text(SRC)
    subprocess.run([shutil.which("g++") or "g++", "-O1", "-std=c++17", f"-I{ROOT / 'lumen_amd' / 'csrc'}",
                    str(tmp_path / "a.cpp"), "-o", str(tmp_path / "a")], check=True)
    assert subprocess.run([str(tmp_path / "a")]).returncode == 0


def test_the_merge_buffers_are_one_set():
    """The buffers that k_vcm_merge and the eye pass use without a check of their own."""
    src = (ROOT / "lumen_amd" / "csrc" / "vcm.hip").read_text()
    body = src[src.index("if (merge_pass && !b.queries)"):]
    body = body[:body.index("const uint32_t merge_blocks")]
    assert "alloc_set(" in body
    for name in ("fcol", "queries", "tasks", "qctr"):
        assert f"&b.{name}," in body, name
    assert "LT_HIP(ctx, hipMalloc" not in body
