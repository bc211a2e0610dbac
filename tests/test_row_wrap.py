"""Grid rows of a tile's rows in the streaming kernels (phx_row_wrap.h) against the remainder, on the host: the header is
plain C++.

One row and more than 37837 rows (where a 32-bit reciprocal rounded up, as it once was, gives no row of the grid) included;
tiles in both directions, from the halo above the grid to past its end."""
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
        for (int halo : {4, 6, 7, 8})
            for (int dir : {1, -1}) {
                /* a tile of up to 120 rows and its halos, anywhere in the grid */
                auto tile = [&](int low) {
                    const int count = 136, first = dir > 0 ? low : low + count - 1;
                    phx::RowWalk p = phx::make_row_walk(first, dir, Nr, halo, true), z = phx::make_row_walk(first, dir, Nr, halo, false);
                    for (int k = 0, g = first; k < count; k++, g += dir) {
                        const unsigned want = (unsigned)((((long)g % Nr) + Nr) % Nr);
                        if (!phx::next_row(p) || p.row != want) {
                            std::printf("Nr %d halo %d: row %d -> %u, not %u\n", Nr, halo, g, p.row, want);
                            return false;
                        }
                        const bool in = g >= 0 && g < Nr;
                        if (phx::next_row(z) != in || (in && z.row != (unsigned)g)) {
                            std::printf("Nr %d halo %d, zero boundary: row %d\n", Nr, halo, g);
                            return false;
                        }
                    }
                    return true;
                };
                for (int low = -halo; low < 130 && low < Nr; low++)
                    if (!tile(low)) return 1;
                for (int low = Nr > 300 ? Nr - 150 : 0; low < Nr; low++)
                    if (!tile(low)) return 1;
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
