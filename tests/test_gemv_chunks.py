"""Tiles of a chunk of the one-token GEMV (blok_amd/csrc/kx_gemv_chunks.h), on the host.  The reference has no such choice (src/kimi_exec.cu:272-323: a
workgroup per row)."""
import random
import subprocess

import pytest

import tile_share as T

# rows, columns, rows of a tile, workgroups that run at once; us with chunks of one to eight tiles
MEASURED = [
    (131073, 512, 32, 512, (26.99, 24.01, 24.37, 24.95, 25.11, 24.61, 27.33, 28.40)), (66000, 1024, 16, 512, (28.34, 24.48, 24.60, 26.72, 25.34, 24.84, 27.49, 30.21)),
    (66000, 1536, 16, 256, (48.52, 39.84, 37.66, 38.96, 38.34, 34.47, 37.97, 42.13)), (151316, 1536, 16, 256, (101.39, 81.27, 78.46, 78.34, 76.64, 77.80, 76.68, 75.57)),
    (36864, 2048, 8, 512, (30.78, 25.83, 26.01, 27.56, 26.26, 25.68, 27.91, 31.00)), (66000, 2048, 8, 512, (52.53, 43.50, 43.59, 45.55, 45.06, 43.70, 45.17, 48.81)),
    (33824, 2560, 8, 256, (46.08, 36.86, 33.69, 34.73, 34.13, 30.77, 34.08, 37.07)), (50000, 2560, 8, 256, (65.80, 51.66, 48.58, 47.70, 43.61, 48.20, 45.72, 49.58)),
    (87515, 2560, 8, 256, (110.16, 85.62, 79.67, 75.05, 75.50, 77.64, 78.72, 76.28)), (160633, 2560, 8, 256, (200.16, 152.78, 140.62, 133.68, 132.56, 134.32, 134.56, 129.38)),
    (37190, 3072, 8, 256, (54.73, 44.41, 43.38, 40.19, 39.43, 43.63, 38.99, 43.26)), (119347, 3072, 8, 256, (160.52, 126.55, 120.15, 117.79, 116.33, 112.21, 116.15, 119.09)),
    (20000, 3584, 4, 512, (31.44, 25.37, 26.31, 24.99, 24.91, 25.53, 26.09, 28.33)), (33000, 3584, 4, 512, (49.02, 39.08, 39.53, 40.62, 40.74, 38.74, 41.06, 44.17)),
    (18432, 4096, 4, 512, (31.15, 25.54, 26.21, 26.85, 26.25, 25.68, 27.96, 31.72)), (25411, 4096, 4, 512, (40.96, 34.05, 35.31, 35.68, 34.08, 37.87, 34.84, 37.24)),
    (32768, 4096, 4, 512, (51.81, 42.76, 42.82, 41.74, 44.68, 42.98, 44.74, 43.53)), (37447, 5120, 8, 256, (82.84, 71.02, 69.88, 66.05, 64.98, 73.38, 66.20, 72.10)),
    (24843, 6144, 8, 256, (62.93, 56.69, 57.21, 59.35, 54.89, 62.90, 50.59, 56.83)), (45667, 6144, 8, 256, (110.77, 97.71, 95.67, 94.15, 96.01, 93.45, 101.17, 94.75)),
    (18432, 7168, 4, 512, (46.79, 43.01, 42.10, 45.87, 43.27, 43.29, 48.33, 53.09)), (32768, 7168, 4, 512, (79.87, 72.26, 73.96, 72.08, 77.84, 74.24, 78.04, 73.16)),
    (59039, 7168, 4, 512, (140.54, 127.17, 130.02, 130.77, 129.21, 129.74, 136.06, 131.90)), (16887, 9216, 8, 256, (61.63, 57.95, 51.59, 62.31, 52.70, 58.29, 66.50, 73.03)),
]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return T.build(tmp_path_factory.mktemp("chunks"), "gemv_chunks")


def _tiles(exe, cases):
    text = "".join(" ".join(map(str, c)) + "\n" for c in cases)
    return list(map(int, subprocess.run([exe], input=text, capture_output=True, text=True, timeout=60, check=True).stdout.split()))


def test_chunks_are_those_that_take_least(exe):
    """Every number of tiles was timed.  A rule that only evens out the rows takes one tile for fourteen of these, up to 55 % longer than eight."""
    for (rows, cols, _, _, us), n in zip(MEASURED, _tiles(exe, [(r, t, 8, s) for r, _, t, s, _ in MEASURED]), strict=True):
        assert us[n - 1] <= min(1.05 * min(us), us[7] + 0.3), (rows, cols, n)


def test_chunks_are_one_to_as_many_tiles_as_are_given(exe):
    rng = random.Random(1)
    cases = [(rng.randint(1, 300000), rng.choice((1, 2, 4, 8, 16, 32)), rng.randint(1, 8), rng.choice((1, 256, 512, 2048))) for _ in range(20000)]
    assert all(1 <= n <= c[2] for c, n in zip(cases, _tiles(exe, cases), strict=True))
