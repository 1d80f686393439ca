"""The rule that splits the scatter of the tile-segment binning into bands of
tile rows (splat.js_amd/csrc/gs_bands.h) against measurements on an MI355X: the
whole binning of scenes of 100k to 10M Gaussians at three view sizes, in one
band and in as many as the open lines ask for. The rule may not take bands
where they cost more than 5% (it may pass over a gain: short runs of keys)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROBE = r"""
#include <stdio.h>
#include <stdlib.h>
#include "gs_bands.h"
int main(int argc, char** argv) {
  for (int i = 1; i + 4 < argc; i += 5)
    printf("%d ", gs_band_rows(strtoull(argv[i], 0, 10), atoll(argv[i + 1]), atoi(argv[i + 2]), atoi(argv[i + 3]),
                             atoi(argv[i + 3]) * atoi(argv[i + 4])));
  return 0;
}
"""

# width, height, Gaussians, keys, us in one band, us in bands
MEASURED = [
    (1920, 1080, 100000, 67299498, 1864.3, 1521.4), (1920, 1080, 100000, 183586093, 5167.5, 4214.5),
    (1920, 1080, 300000, 32475622, 919.4, 725.9), (1920, 1080, 300000, 201362254, 5594.5, 4532.7),
    (1920, 1080, 1000000, 26158232, 751.9, 696.9), (1920, 1080, 1000000, 52449934, 1448.4, 1244.6),
    (1920, 1080, 1000000, 108343145, 2911.4, 2412.8), (1920, 1080, 3000000, 30102569, 891.8, 1276.4),
    (1920, 1080, 3000000, 56245401, 1550.9, 1888.3), (1920, 1080, 3000000, 92994370, 2481.4, 2594.0),
    (1920, 1080, 3000000, 157296368, 4234.0, 3970.6), (1920, 1080, 10000000, 35360085, 1252.3, 2803.1),
    (1920, 1080, 10000000, 65483368, 1979.0, 3449.7), (1920, 1080, 10000000, 116733329, 3267.8, 4624.3),
    (1920, 1080, 10000000, 187549205, 5186.5, 6340.5), (1280, 720, 100000, 30567984, 868.8, 740.9),
    (1280, 720, 300000, 37740208, 1078.9, 932.8), (1280, 720, 1000000, 13439904, 394.8, 372.7),
    (1280, 720, 1000000, 51516320, 1526.2, 1295.9), (1280, 720, 3000000, 16985212, 532.8, 658.9),
    (1280, 720, 3000000, 29710467, 878.6, 1041.0), (1280, 720, 3000000, 47195732, 1388.1, 1364.8),
    (1280, 720, 3000000, 77282153, 2317.8, 2199.0), (1280, 720, 10000000, 23608803, 936.7, 1511.0),
    (1280, 720, 10000000, 64691157, 2107.5, 2584.5), (1280, 720, 10000000, 99049828, 3157.1, 3515.4),
    (2048, 2048, 100000, 248173712, 7177.3, 5392.0), (2048, 2048, 300000, 99889440, 2842.3, 2115.0),
    (2048, 2048, 1000000, 62059683, 1811.3, 1530.0), (2048, 2048, 3000000, 65559474, 1972.6, 2242.8),
    (2048, 2048, 3000000, 109242876, 3146.2, 3454.8), (2048, 2048, 3000000, 186094791, 5394.4, 4690.6),
    (2048, 2048, 10000000, 74453067, 2555.5, 5186.9), (2048, 2048, 10000000, 218656762, 6597.2, 8215.2),
]


def _rows(tmp_path, cases):
    """gs_band_rows of (keys, n, nb, tilesX, tilesY) tuples (0: one band)."""
    src = tmp_path / "bands.c"
    src.write_text(PROBE)
    exe = tmp_path / "bands"
    subprocess.check_call(["gcc", "-O2", "-I", os.path.join(ROOT, "splat.js_amd", "csrc"), "-o", str(exe), str(src), "-lm"])
    args = [str(int(v)) for c in cases for v in c]
    return [int(v) for v in subprocess.check_output([str(exe), *args], text=True).split()]


def test_bands_where_they_were_measured_to_pay(tmp_path):
    cases = []
    for W, H, n, keys, one, banded in MEASURED:
        cases.append((keys, n, min(256, -(-n // 256)), -(-W // 16), -(-H // 16)))
    for m, c, rows in zip(MEASURED, cases, _rows(tmp_path, cases)):
        assert 0 <= rows < c[4]
        if m[5] < 0.97 * m[4]:      # paid in these: all hold full runs of keys
            assert rows > 0, m
        if m[5] > 1.05 * m[4]:
            assert rows == 0, m


def test_band_sizes_at_the_ends_of_their_range(tmp_path):
    big = 1 << 40
    cases = [(0, 1, 1, 1, 1), (big, 1, 1, 1, 1),                       # one tile
             (big, 1 << 19, 256, 120, 68),                             # 24576 lines / 32 / 120 = 6 rows
             (big, 1 << 19, 256, 16384, 1), (big, 1 << 19, 256, 800, 20),   # a row is past the lines: one row
             (big, 3000, 12, 40, 30),                                  # 24576 / 2 / 40: every row
             (12 * 256 * 8160 - 1, 1000, 256, 120, 68), (12 * 256 * 8160, 1000, 256, 120, 68),
             (3 * 12 * 10000000 - 1, (1 << 19) + 10000000, 256, 120, 68), (3 * 12 * 10000000, (1 << 19) + 10000000, 256, 120, 68)]
    assert _rows(tmp_path, cases) == [0, 0, 6, 0, 1, 0, 0, 6, 0, 6]
