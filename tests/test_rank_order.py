"""Rows of the resident solve's ranks by recursive bisection (csrc/order.cpp,
host code): a permutation whose parts lie on the two sides of each cut, the
same when no memory is left for its threads."""
import os
import shutil
import subprocess

import pytest

from tests.conftest import ROOT

SRC = r"""
#include <cstdio>
#include <cstdlib>
#include <new>
static thread_local bool main_thread = false;
static int left = -1;   // allocations the main thread may still make (-1: any number)
void *operator new(std::size_t n)
{
    if (main_thread && left >= 0 && left-- == 0) throw std::bad_alloc();
    if (void *p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }
#include "order.cpp"
int main()
{
    const int n = 40000, dim = 3;
    std::vector<double> x(n * dim);
    unsigned s = 1;
    for (double &v : x) { s = s * 1664525u + 1013904223u; v = s / 4294967296.0; }
    std::vector<int> node(n), ref, row(n);
    std::iota(node.begin(), node.end(), 0);
    main_thread = true;
    for (int fail = -1; fail < 4; fail++) {
        std::iota(row.begin(), row.end(), 0);
        left = fail;
        tmi::split_ranks(dim, n, 256, 0, 256, x.data(), node, row);
        left = -1;
        if (fail < 0) ref = row;
        else if (row != ref) return 1;
    }
    std::vector<int> c(ref);
    std::sort(c.begin(), c.end());
    if (c != node) return 2;
    // the first cut: one coordinate separates the halves
    bool cut = false;
    for (int d = 0; d < dim; d++) {
        double hi = 0.0, lo = 1.0;
        for (int i = 0; i < n / 2; i++) hi = std::max(hi, x[ref[i] * dim + d]);
        for (int i = n / 2; i < n; i++) lo = std::min(lo, x[ref[i] * dim + d]);
        cut |= hi <= lo;
    }
    if (!cut) return 3;
    printf("ok\n");
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("hipcc", path="/opt/rocm/bin") is None, reason="no hipcc")
def test_rank_order_without_memory_for_threads(tmp_path):
    src, exe = tmp_path / "ranks.cpp", tmp_path / "ranks"
    src.write_text(SRC)
    lib = os.path.join(ROOT, "toastpp_amd")
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-std=c++17", "-O1",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(lib, "csrc"), str(src), "-o", str(exe),
                    "-L" + lib, "-l:libtoastpp_amd.so", "-Wl,-rpath," + lib], check=True, capture_output=True, text=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
