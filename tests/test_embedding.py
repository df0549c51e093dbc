"""Wrap-around embedding of the free-space kernel table, on the CPU: the index
rule both row kernels read the table by (csrc/embed.hpp) over every grid side
the spectral backend takes and the torus side the library embeds it in. A host
program includes the header and calls the library for the torus side."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "embed.hpp"
#include "spectral.hpp"
#include <cstdio>
using namespace aspher;

static int check(int Ns, int n) {
    if (n < 2 * Ns - 1 || n % 2) { printf("Ns %d: side %d\n", Ns, n); return 1; }
    for (int i = 0; i < n; ++i) {
        const int d = embed_offset(i, Ns, n);
        // inside the table (or a zero), even, and the offset itself up to Ns
        const bool held = i < Ns || n - i < Ns;
        const int want = !held ? -1 : i < Ns ? i : n - i;
        if (d < -1 || d >= Ns || d != want || d != embed_offset((n - i) % n, Ns, n)) {
            printf("Ns %d side %d index %d: offset %d, expected %d\n", Ns, n, i, d, want);
            return 1;
        }
    }
    return 0;
}

int main() {
    int bad = 0, wider = 0;
    for (int Ns = 1; Ns <= 2559; ++Ns) {
        const int n = free_space_side(Ns);
        bad += check(Ns, n);
        wider += is_pow2(n) && n != 2 * Ns;
    }
    for (int Ns = 4; Ns <= 4096; Ns *= 2) bad += check(Ns, 2 * Ns);
    printf("sides on a wider power of two: %d\n", wider);
    return bad || !wider;
}
"""


def _hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    pytest.skip("no hipcc")


def run_host(program, tmp_path):
    """Builds a host program against the library and its headers and runs it."""
    from aspher_amd import _capi, build
    _capi.lib()
    src, exe = tmp_path / "host.hip", tmp_path / "host"
    src.write_text(program)
    subprocess.run([_hipcc(), "--offload-host-only", "-std=c++17", "-O1", "-w", "-I" + build.CSRC,
                    "-x", "hip", str(src), "-x", "none", build.LIB, "-Wl,-rpath," + build.HERE,
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_embedding_stays_inside_the_table(tmp_path):
    run_host(PROGRAM, tmp_path)
