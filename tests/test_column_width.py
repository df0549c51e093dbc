"""Columns per workgroup of the register-blocked column pass, on the CPU. Its
wave-local exchanges hold only where a group of neighbouring threads of a
transform lies in one wave, and columns are interleaved over the lanes: thread
th of column c is lane th W + c. Every width the plan may take is checked for
every group of 64 / Wmax threads (csrc/fft_rb.hpp, wave_local)."""
from test_embedding import run_host

PROGRAM = r"""
#include "spectral.hpp"
#include <algorithm>
#include <cstdio>
using namespace aspher;

int main() {
    int bad = 0;
    for (int logn = 5; logn <= 13; ++logn)
        for (int le : {2, 4})
            for (std::size_t elt : {8, 16})
                for (int want = 1; want <= 64; ++want) {
                    const int n = 1 << logn, T = n >> le;
                    const std::size_t lds = elt * (n + n / 16 + 1);
                    if (T > 512) continue;
                    const int W = column_width(want, T, lds);
                    bool ok = W >= 1 && W <= want && W * T <= 512 && (W == 1 || W * lds <= 98304);
                    const int lanes = 64 / std::max(1, 512 / T);
                    for (int g = 0; T >= 64 && g < T; g += lanes)
                        ok = ok && g * W / 64 == ((g + lanes - 1) * W + W - 1) / 64;
                    if (!ok) {
                        printf("n %d le %d elt %d want %d: width %d\n", n, le, (int)elt, want, W);
                        ++bad;
                    }
                }
    return bad != 0;
}
"""


def test_column_groups_stay_in_a_wave(tmp_path):
    run_host(PROGRAM, tmp_path)
