"""Row index of the streaming kernels (phx_row_wrap.h) against the remainder, on the host: the header is plain C++.

One row (the quotient's factor does not fit 32 bits rounded up) and more than 2^32 / Nr rows past 37837 (where a
rounded-up factor is no longer exact) included; every tile row from the halo above the grid to 128 rows below it."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include "phx_row_wrap.h"
int main() {
    const int sizes[] = {1, 2, 3, 4, 5, 6, 7, 8, 9, 16, 31, 150, 1000, 1024, 4096, 37837, 37839, 46341, 46349, 60000, 65535, 65536,
                         65537, 100003, 1000003, 16777259, 268435399};
    for (int Nr : sizes)
        for (int halo : {4, 6, 7, 8}) {
            const phx::RowWrap w = phx::make_row_wrap(Nr, halo);
            auto check = [&](int g) {
                bool in = false;
                const unsigned row = phx::tile_row(g, w, 1, in);
                const int want = (int)((((long)g % Nr) + Nr) % Nr);
                if (!in || row != (unsigned)want) {
                    std::printf("Nr %d halo %d: row %d -> %u, not %d\n", Nr, halo, g, row, want);
                    return false;
                }
                bool zin = true;
                (void)phx::tile_row(g, w, 0, zin);
                return zin == (g >= 0 && g < Nr);
            };
            for (int g = -halo; g < 128; g++)
                if (!check(g)) return 1;
            for (int g = Nr > 128 ? Nr - 128 : 0; g < Nr + 128; g++)
                if (!check(g)) return 1;
        }
    return 0;
}
"""


def test_rows_wrap_exactly(tmp_path):
    src = tmp_path / "wrap.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "wrap"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "phoenix_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
