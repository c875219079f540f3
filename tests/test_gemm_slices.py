"""The prompt GEMM's cut of its tile grid into one slice per XCD
(libcmol_amd/csrc/hip/gemm_slices.h), compiled for the host: every tile once,
and no XCD far above its share at prompt lengths whose vector tiles do not
divide by eight."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "gemm_slices.h"
#include <cstdio>
#include <vector>
int main()
{
    for (int mt = 1; mt <= 70; mt++)
        for (int nt : {1, 2, 5, 8, 16, 24, 33, 172, 345, 1002})
            for (int ks : {1, 2, 8}) {
                const GemmSlices s = gemm_slices(mt, nt, ks, 16 / ks, 32);
                std::vector<int> seen(mt * nt);
                long fullest = 0;
                for (int xcd = 0; xcd < 8; xcd++) {
                    long mine = 0;
                    for (int i = 0; i < s.mts * s.nts; i++) {   // as the kernel walks its slice
                        const int m = (xcd % s.ga) * s.mts + i % s.mts, n = (xcd / s.ga) * s.nts + i / s.mts;
                        if (m >= mt || n >= nt) continue;
                        seen[m * nt + n]++;
                        mine++;
                    }
                    if (mine > fullest) fullest = mine;
                }
                for (int x : seen)
                    if (x != 1) { std::printf("mt %d nt %d: a tile %d times\n", mt, nt, x); return 1; }
                std::printf("%d %d %d %ld\n", mt, nt, ks, fullest);
            }
    return 0;
}
"""


def test_every_tile_once_and_no_xcd_far_above_its_share(tmp_path):
    src, exe = tmp_path / "t.cc", tmp_path / "t"
    src.write_text(SOURCE)
    inc = os.path.join(ROOT, "libcmol_amd", "csrc", "hip")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", inc, "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-300:]
    for line in r.stdout.split("\n")[:-1]:
        mt, nt, ks, fullest = map(int, line.split())
        # 22016 rows (172 row tiles) up to 512 vectors: what the cuts of ceil(mt
        # / 8) or ceil(mt / 4) tiles took was up to 1.6 of the even share
        if nt >= 172 and 2 <= mt <= 16:
            assert fullest * 8 <= 1.15 * mt * nt, line
