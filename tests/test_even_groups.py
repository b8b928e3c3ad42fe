"""Equal shares of the rows for products of 5 to 64 tokens (kxtile::even_groups of blok_amd/csrc/kx_tile_share.h), on the host.  The reference has no such
choice (src/kimi_exec.cu:272-323: a workgroup per row)."""
import random
import subprocess

import pytest

import tile_share as T

# rows, columns, tokens; us by workgroups, groups of 64 rows first
MEASURED = [
    (9344, 2048, 64, {146: 16.11, 256: 15.05, 512: 24.44}), (11584, 2048, 32, {181: 14.34, 256: 14.24, 512: 16.98}), (17472, 2048, 5, {273: 22.23, 512: 18.67, 1024: 27.83}),
    (17472, 2048, 64, {273: 30.88, 512: 28.09, 1024: 46.35}), (24576, 2048, 33, {384: 30.24, 512: 29.22, 1024: 43.79}), (33000, 2048, 32, {516: 38.42, 768: 34.17, 1024: 36.41}),
    (33000, 2048, 64, {516: 48.94, 768: 46.16, 1024: 52.63}), (40000, 1024, 5, {625: 20.25, 768: 19.00, 1024: 20.68}), (40000, 1024, 32, {625: 21.27, 768: 20.93, 1024: 23.33}),
    (40000, 1024, 64, {625: 30.28, 768: 30.17, 1024: 35.86}), (40000, 2048, 33, {625: 46.07, 768: 44.88, 1024: 49.99}), (40000, 4096, 64, {625: 88.33, 768: 84.82, 1024: 93.05}),
    (50000, 2048, 64, {782: 66.66, 1024: 65.09, 1536: 78.09}), (66000, 2048, 33, {1032: 78.43, 1280: 74.70, 1536: 79.98}),
]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return T.build(tmp_path_factory.mktemp("groups"), "even_groups")


def _groups(exe, cases):
    text = "".join(" ".join(map(str, c)) + f" {T.CUS}\n" for c in cases)
    return list(map(int, subprocess.run([exe], input=text, capture_output=True, text=True, timeout=60, check=True).stdout.split()))


def test_shares_are_those_that_take_least(exe):
    """Whole rounds of two workgroups per CU, which is what a CU holds with up to 32 tokens, take up to 18 % longer than groups of 64 rows for seven of these."""
    got = _groups(exe, [(r, c, -(-r // 64), 1, 1 << 40, r) for r, c, _, _ in MEASURED])
    for (r, c, t, us), n in zip(MEASURED, got, strict=True):
        assert us[n] == min(us.values()), (r, c, t, n)


def test_shares_have_at_most_64_rows_and_fit_the_scratch(exe):
    rng = random.Random(3)
    cases = []
    for _ in range(20000):
        rows, parts = rng.randint(1, 70000), rng.choice((1, 1, 2, 3, 5, 16))
        cases.append((rows, 64 * rng.randint(1, 300), -(-rows // 64), parts, rng.choice((1 << 40, 512, 300, 0)), rng.choice((512, 100, 70000))))
    changed = 0
    for (rows, cols, groups, parts, room, arrivals), n in zip(cases, _groups(exe, cases), strict=True):
        assert n >= groups
        if n > groups:
            changed += 1
            assert rows // n + (rows % n > 0) <= 64 and rows // n >= 1 and n <= arrivals and n * parts <= room and cols >= 1024 * parts, (rows, cols, parts)
    assert changed > 1000
