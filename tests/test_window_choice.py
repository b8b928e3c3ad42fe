"""Whether 32-bit attention of several positions goes over the keys on the matrix cores or in parts (blok_amd/csrc/kx_window_choice.h), on the host.  The
reference has no such choice (src/kimi_exec.cu:692-716: one kernel for every length)."""
import subprocess

import pytest

import tile_share as T

# heads, key heads, columns of a key and a value, sequences, positions, keys of the last position and on average, keys of a part, parts, tokens whose parts
# the scratch holds; us in parts and on the matrix cores
MEASURED = [
    ((32, 8, 256, 1, 20, 520, 510.5, 256, 3, 20), 32, 56), ((8, 2, 256, 32, 4, 204, 202.5, 256, 1, 128), 26, 37), ((32, 8, 384, 1, 20, 520, 510.5, 256, 3, 20), 42, 87),
    ((16, 4, 256, 2, 21, 482, 472.0, 256, 2, 42), 27, 45), ((64, 64, 256, 1, 4, 34, 32.5, 256, 1, 4), 39, 50), ((16, 4, 256, 1, 3, 3, 2.0, 64, 1, 3), 16, 25),
    ((2, 1, 256, 1, 24, 24, 12.5, 64, 1, 16), 25, 25), ((16, 16, 256, 1, 53, 53, 27.0, 256, 1, 16), 47, 29), ((40, 5, 256, 14, 6, 6, 3.5, 256, 1, 16), 94, 60),
    ((8, 2, 256, 1, 100, 100, 50.5, 64, 2, 16), 93, 33), ((2, 1, 384, 1, 258, 64, 64.0, 256, 1, 16), 194, 31), ((8, 2, 256, 16, 50, 50, 25.5, 256, 1, 16), 558, 35),
]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return T.build(tmp_path_factory.mktemp("choice"), "window_choice")


def test_the_sooner_way_is_taken(exe):
    """Both ways were timed; an estimate by tokens and heads alone took the slower one for the first five, which was up to 2.1 times as long."""
    text = "".join(" ".join(map(str, m[0])) + f" {T.CUS}\n" for m in MEASURED)
    got = list(map(int, subprocess.run([exe], input=text, capture_output=True, text=True, timeout=60, check=True).stdout.split()))
    for (step, parts, cores), c in zip(MEASURED, got, strict=True):
        assert (cores if c else parts) <= 1.1 * min(parts, cores), (step, parts, cores, c)
