"""What is copied nontemporally (blok_amd/csrc/kx_read_once.h), on the host.  The reference has no such choice (src/kimi_exec.cu:272-323 loads into registers)."""
import subprocess

import pytest

import tile_share as T

# latent decode attention of 64 heads: sequences, positions; us with plain and nontemporal copies, the same cache again and again and then over 1.4 GB of caches
LATENT = [
    (8, 128, (17.10, 17.09), None), (8, 512, (20.78, 20.77), None), (32, 300, (24.11, 25.47), (24.61, 25.39)), (16, 1024, (23.90, 25.24), (24.40, 25.20)),
    (32, 1024, (29.69, 30.80), (30.17, 30.57)), (1, 4096, (22.72, 22.71), None), (4, 4096, (26.20, 28.05), (26.78, 28.19)), (16, 2048, (29.21, 30.26), (29.77, 30.18)),
    (8, 4096, (29.42, 32.27), (29.96, 32.23)), (1, 32768, (35.41, 38.74), (36.60, 38.98)), (32, 2048, (37.90, 37.79), (38.32, 37.87)),
    (16, 4096, (37.12, 37.60), (37.01, 36.83)),
    (1, 131072, (63.70, 66.22), (65.00, 66.44)), (2, 65536, (54.37, 56.56), (55.79, 56.64)), (4, 32768, (50.82, 51.36), (52.05, 52.13)),
    (16, 8192, (47.84, 48.73), (49.52, 49.00)), (32, 4096, (50.27, 50.09), (51.10, 49.82)), (4, 46000, (65.02, 66.71), (65.46, 67.30)),
    (1, 200000, (77.02, 79.89), (78.08, 79.56)), (24, 8192, (65.41, 64.71), (65.13, 64.46)),
    (32, 6000, (64.41, 64.16), (66.09, 63.90)), (2, 114000, (75.92, 76.43), (75.87, 75.91)), (8, 28000, (71.98, 68.35), (71.26, 68.67)),
    (16, 14000, (69.72, 67.91), (72.09, 68.50)), (32, 7000, (70.58, 68.98), (71.71, 70.88)), (1, 262144, (89.42, 88.54), (89.31, 89.28)),
    (4, 65536, (79.75, 78.09), (78.71, 77.48)), (16, 16384, (77.96, 76.04), (78.11, 75.50)), (8, 32768, (79.47, 76.59), (77.59, 76.63)),
    (4, 100000, (120.60, 115.40), (116.26, 111.50)), (16, 32768, (135.91, 129.35), (135.23, 128.23)),
]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return T.build(tmp_path_factory.mktemp("once"), "read_once")


def _nontemporal(exe, what, sizes):
    text = "".join(f"{what} {n}\n" for n in sizes)
    return list(map(int, subprocess.run([exe], input=text, capture_output=True, text=True, timeout=60, check=True).stdout.split()))


def test_latent_caches_are_copied_as_takes_less(exe):
    """Nontemporal copies of every cache take up to 10 % longer, more than 4 % for six of these.  What is chosen is never slower by more than that."""
    for (seqs, n, *times), once in zip(LATENT, _nontemporal(exe, "latent", [s * n * 576 * 2 for s, n, *_ in LATENT]), strict=True):
        for us in filter(None, times):
            assert us[once] <= 1.04 * us[1 - once], (seqs, n, once, us)


def test_no_launch_of_a_few_sequences_of_ordinary_length_is_nontemporal(exe):
    assert not any(_nontemporal(exe, "latent", [s * n * 576 * 2 for s in (1, 2, 8, 16, 32) for n in (100, 1500, 4096)]))
