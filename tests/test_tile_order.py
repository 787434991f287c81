"""The order of a prefill GEMM's tiles (xcd_tile, compiled for the host from the kernels' source): every tile once, whatever the
grid, and no XCD with more tiles than its share."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <vector>
#define __device__
#define __host__
#define __forceinline__ inline
static long round_up(long v, long m) { return (v + m - 1) / m * m; }
%s
int main() {
    for (int RT = 1; RT <= 70; ++RT)
        for (int CT = 1; CT <= 45; CT += (RT > 20 ? 11 : 1))
            for (int band : {1, 2, 4, 8})
                for (int spare : {0, 16}) {       // (a grid made for more tiles than there are)
                    std::vector<int> seen(RT * CT, 0); int per[8] = {};
                    const long blocks = xcd_tile_blocks((long)RT * CT + spare);
                    for (long b = 0; b < blocks; ++b) {
                        int r = -1, c = -1;
                        if (!xcd_tile((unsigned)b, RT, CT, band, r, c)) continue;
                        if (r < 0 || r >= RT || c < 0 || c >= CT) { printf("outside %%d %%d %%d\n", RT, CT, band); return 1; }
                        ++seen[r * CT + c]; ++per[b & 7];
                    }
                    for (int n : seen) if (n != 1) { printf("times %%d: %%d %%d %%d\n", n, RT, CT, band); return 1; }
                    for (int n : per) if (n > (RT * CT + 7) / 8) { printf("share %%d: %%d %%d %%d\n", n, RT, CT, band); return 1; }
                }
    return 0;
}
"""


def test_every_tile_once_and_equal_shares(tmp_path):
    text = open(os.path.join(ROOT, "seq2seqsharp_amd", "csrc", "tship_gpt_kernels.h")).read()
    fn = re.search(r"__host__ __device__ inline long xcd_tile_blocks.*?\n}\n", text, re.S).group(0)
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM % fn)
    subprocess.run(["g++", "-O2", "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout


def test_kernels_hand_over_the_block_id_itself():
    """xcd_tile covers every tile for block ids 0 ... xcd_tile_blocks - 1 only: shifted ids leave tiles out."""
    text = open(os.path.join(ROOT, "seq2seqsharp_amd", "csrc", "tship_gpt_kernels.h")).read()
    first = re.findall(r"!xcd_tile\(([^,]*),", text)
    assert len(first) >= 3 and set(first) == {"blockIdx.x"}
