"""The choice of tiles and parts for a product, on the host.  The reference has no such choice (src/kimi_exec.cu:272-323: a matrix-vector
product per token)."""
import random

import pytest

import tile_share as T


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return T.build(tmp_path_factory.mktemp("share"))


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def test_32_bit_products_of_few_tiles_fill_two_workgroups_per_cu(exe):
    """As many parts as fill them, of at least 8 blocks, as the scratch allows: 32-bit sums are as short as they can be."""
    rng = random.Random(5)
    products = [(64, 1024, 8192), (64, 1024, 16384), (5, 512, 11008), (16, 1024, 8192)]
    products += [(_log(rng, 5, 2048), _log(rng, 64, 20000), 64 * _log(rng, 1, 512)) for _ in range(20000)]
    for (t, r, c), got in zip(products, T.choices(exe, True, products, T.F32)):
        fill = min(2 * T.CUS // got.tiles, c // 32 // 8, T.F32[0] // (64 * 128) // got.tiles)
        if got.tiles <= T.F32[1] and fill > 1:
            assert got.whole == 0 and got.parts >= fill, (t, r, c, got)
        if got.whole < got.tiles:                                                     # the scratch holds the parts
            assert got.tiles - got.whole <= T.F32[1] and (got.tiles - got.whole) * got.parts * 64 * 128 <= T.F32[0], (t, r, c, got)
            assert got.parts <= max(1, c // 32 // 8), (t, r, c, got)


def test_32_bit_parts_beside_one_round_of_whole_tiles_are_one_round(exe):
    rng = random.Random(6)
    products = [(464, 6396, 1024), (488, 6250, 2816), (777, 2560, 1024)] + [(_log(rng, 64, 2048), _log(rng, 128, 20000), 64 * _log(rng, 4, 256)) for _ in range(20000)]
    got = T.choices(exe, True, products, T.F32)
    assert got[0].parts == got[1].parts == 1 and got[2].whole == T.CUS and got[2].parts == 4
    for p, c in zip(products, got):
        if c.whole == T.CUS and c.parts > 1:
            assert (c.tiles - c.whole) * c.parts <= T.CUS, (p, c)
