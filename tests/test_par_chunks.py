"""The host's threaded loop (csrc/hip/par.hpp): every index once, and an
exception of a worker (an allocation that fails while a context is created)
reaches the caller, which turns it into a status, instead of ending the
process."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "par.hpp"
#include <cstdio>
#include <new>
int main() {
    for (int64_t n : {0, 1, 63, 64, 65, 1000, 4097})
        for (int64_t chunk : {1, 64, 5000}) {
            std::vector<int> hit(n, 0);
            tfd::par_chunks(n, chunk, [&](int64_t lo, int64_t hi) { for (int64_t i = lo; i < hi; ++i) ++hit[i]; });
            for (int h : hit) if (h != 1) return 1;
        }
    for (int64_t bad : {0, 500, 999}) {
        bool got = false;
        try {
            tfd::par_chunks(1000, 10, [&](int64_t lo, int64_t hi) { if (lo <= bad && bad < hi) throw std::bad_alloc(); });
        } catch (const std::bad_alloc&) { got = true; }
        if (!got) return 2;
    }
    std::puts("ok");
}
"""


def test_par_chunks(tmp_path):
    src, exe = tmp_path / "p.cpp", tmp_path / "p"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "tetfit_amd/csrc/hip"), str(src),
                    "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout == "ok\n"
