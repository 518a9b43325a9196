"""The static scratch of clk_lloyd_step_noalloc holds as many partial rows of
8k(d+1) bytes as 8 MiB held of k(8d+4) (masses of 4 bytes), so that no size
runs on fewer work-groups; and at least one of every size that the LDS tiles
admit."""
import os
import re

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "clkmeans.h")


def test_rows():
    text = open(HEADER).read()
    mib = int(re.search(r"#define CLK_NOALLOC_SCRATCH_BYTES \((\d+)u << 20\)", text).group(1))
    for d in range(1, 65):
        head = ((d + 1) * 4 + 255) // 256 * 256  # the call's sum grid
        for k in (1, 2, 3, 7, 10, 33, 100, 129, 256, 300, 1000, 2500, 8000):
            if d * k * 12 > 160 * 1024:  # beyond the LDS
                continue
            now = ((mib << 20) - head) // (8 * k * (d + 1))
            assert now >= ((8 << 20) - head) // (k * (8 * d + 4)) and now >= 1, (d, k)
