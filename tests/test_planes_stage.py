"""The bit-plane kernel's staging arithmetic (csrc/tdd_planes_stage.h), the
header the kernel itself uses, enumerated on the host: a GPU is not needed."""
import subprocess
from pathlib import Path

REPO = Path(__file__).resolve().parents[1]

SRC = r'''
#include "tdd_planes_stage.h"
#include <cstdio>
#include <vector>
// Every lane of a window of P positions from sample a on: each position is
// written once, from the row words and by the shift that hold it, inside its
// slot, and the third row word only where it was loaded.
static int window(uint32_t a, uint32_t P, uint32_t nbits, uint32_t slots, uint32_t stride)
{
    const uint32_t T = DD_TDD_PLANES_T;
    const bool third = planes_needs_third(a, P);
    for (uint32_t slot = 0; slot < slots; slot += slots - 1) {
        std::vector<int> seen(P, 0);
        int bad = 0;
        for (uint32_t p = 0; p < T; ++p)
            planes_stage(a, P, p, [&](int k, uint32_t shift, uint32_t u, bool in) {
                const uint32_t pos = planes_window_pos(a, p, u);
                if (!in) { bad |= pos < P; return; }
                if (pos >= P) { bad |= 2; return; }
                ++seen[pos];
                const uint32_t run = (a + pos) / T - 32 * (a / T / 32);  // from the start tile's first run on
                if ((a + pos) % T != p || 32 * k + shift % 32 != run) bad |= 4;
                if (k == 1 && shift % 32 && !third) bad |= 8;
                const uint32_t word = planes_lds_word(planes_lds_first(slot, stride, a, p, nbits), u, nbits);
                if (word != (slot * stride + pos) * nbits) bad |= 64;
                if (word < slot * stride * nbits || word + nbits > (slot + 1) * stride * nbits) bad |= 16;
            });
        for (uint32_t i = 0; i < P; ++i) bad |= (seen[i] != 1) * 32;
        if (bad) { std::printf("a %u P %u slot %u: %d\n", a, P, slot, bad); return 1; }
    }
    return 0;
}
int main()
{
    const uint32_t shape[4][2] = {{1, 16}, {2, 8}, {4, 4}, {8, 4}};  // width, slots
    int bad = 0;
    for (auto& s : shape)
        // the longest window: that of one workgroup per CU, two for 8-bit
        for (uint32_t P = 128; P <= (s[0] == 8 ? 640u : 2496u); P += (P < 512 ? 64 : 320))
            for (uint32_t a = 0; a < 2 * 4096 + 256; a += (a % 128 < 3 || a % 128 > 124) ? 1 : 13)
                bad += window(a, P, s[0], s[1], P + 64);
    // a start far into a long series
    for (uint32_t a : {2147483000u, 2146435072u}) bad += window(a, 448, 4, 4, 448);
    return bad != 0;
}
'''


def test_planes_staging_stays_inside_the_windows(tmp_path):
    src = tmp_path / "stage.cpp"
    src.write_text(SRC)
    exe = tmp_path / "stage"
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include", f"-I{REPO / 'dedisp_tests_amd' / 'csrc'}", str(src), "-o", str(exe)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.stdout, r.stderr)

