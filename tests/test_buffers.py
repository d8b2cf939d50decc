"""Owning device buffers (csrc/common.hpp) where an allocation fails, with or
without a GPU: the buffer is empty afterwards, so that a later size check
allocates again instead of handing out a null pointer."""
import os
import shutil
import subprocess

import pytest

from tests.conftest import ROOT

SRC = r"""
#include <cstdio>
#include "common.hpp"
int main()
{
    tmi::DBuf<double> b;
    for (int way = 0; way < 2; way++) {
        // more than any device holds; then the limit of the tests
        const size_t count = way ? 1000 : (size_t)1 << 56;
        if (way) tmi::g_alloc_limit = 4096;
        try {
            b.alloc(count);
            return 1;
        } catch (const tmi::Error &) {
        }
        if (b.p || b.n || b.bytes()) return 2 + way;
    }
    printf("empty\n");
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("hipcc", path="/opt/rocm/bin") is None, reason="no hipcc")
def test_failed_allocation_leaves_buffer_empty(tmp_path):
    src, exe = tmp_path / "buffers.cpp", tmp_path / "buffers"
    src.write_text(SRC)
    lib = os.path.join(ROOT, "toastpp_amd")
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-std=c++17", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(lib, "csrc"), str(src), "-o", str(exe), "-L" + lib, "-l:libtoastpp_amd.so",
                    "-Wl,-rpath," + lib], check=True, capture_output=True, text=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "empty\n", (r.returncode, r.stdout, r.stderr)
