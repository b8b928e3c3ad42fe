"""Products whose last round of tiles is shared by several workgroups each (kx_tile_share.h): more tiles than one round holds, a few
left over, columns enough for parts.  With the bars of the whole-model tests, twice or with both libraries for the same bits; each test
asks the rule whether its products are shared."""
import os

import numpy as np
import pytest

import kagalorn_case as KC
import kagalorn_oracle as K
import blok_amd.lib as kxl
import oracle as O
import tile_share as TS
from blok_amd.lib import check
from kxt import say
from test_gpu_kagalorn import BF16_LOGITS, F32_LOGITS
from test_gpu_kimi_prompt import _config
from test_gpu_model import KxModel

pytestmark = pytest.mark.gpu


# tokens, width, ff: f32 4 x 66 tiles of 64 x 128 and 5 x 67 with their edges inside; bf16 5 x 130 tiles of 128 x 128, whole, and few-tile
# products in parts
@pytest.mark.parametrize("dtype, tokens, width, ff, bar", [("float32", 256, 512, 4200, F32_LOGITS), ("float32", 261, 544, 4260, F32_LOGITS),
                                                           ("bfloat16", 577, 2048, 8290, BF16_LOGITS)])
def test_last_round_in_parts(kxlib, tmp_path, dtype, tokens, width, ff, bar):
    cfg = KC.config([KC.delta(heads=4, kv_heads=2, dim=32, vdim=64, ff=ff)], width=width, vocab=300)
    w = KC.weights(cfg, ff)
    if dtype == "float32":
        (c,) = TS.choices(TS.build(tmp_path), True, [(tokens, 2 * ((ff + 31) // 32 * 32), (width + 63) // 64 * 64)], TS.F32)
        assert c.whole == TS.CUS and c.parts > 1
    ids = KC.tokens(cfg, tokens, 7)[None]
    want = K.forward(cfg, w, ids[0])[:, None]
    with KC.Model(KC.write(tmp_path, cfg, w), dtype, batch=1, context=tokens) as m:
        first = m.run(ids, [tokens], 1)
        assert KC.logit_error(first, want).max() < bar
        assert (m.run(ids, [tokens], 1) == first).all()


def test_more_than_16_parts_in_32_bits(kxlib, tmp_path):
    """The down product of a decode step: 16 x 512 x 8200, 4 tiles in 32 parts."""
    cfg = KC.config([KC.delta(heads=4, kv_heads=2, dim=32, vdim=64, ff=8200)], width=512, vocab=300)
    w = KC.weights(cfg, 8)
    ids = np.stack([KC.tokens(cfg, 3, 40 + b) for b in range(16)])
    want = np.stack([K.forward(cfg, w, s) for s in ids], 1)
    assert TS.choices(TS.build(tmp_path), True, [(16, 512, 8256)], TS.F32) == [(0, 0, 32, 4)]
    with KC.Model(KC.write(tmp_path, cfg, w), "float32", batch=16, context=3) as m:
        first = m.run(ids, [1], 16)
        assert KC.logit_error(first, want).max() < F32_LOGITS
        assert (m.run(ids, [1], 16) == first).all()


@pytest.fixture(scope="module")
def strict():
    """The library with the hand-over between workgroups in its memory-model form (kx_arrive.h)."""
    return kxl.load_library(os.path.join(os.path.dirname(kxl.lib_path()), "libkx_strict.so"))


# gate and up: 528 medium tiles, the last 16 shared, 352 large ones, the last 96, and 280 twin ones, the last 24; down: all of 72 large tiles shared
@pytest.mark.parametrize("hidden, inter, tokens, product, tile, choice",
                         [(2048, 16896, 187, "gate and up", "medium", (0, 512, 2, 528)), (4096, 11264, 900, "gate and up", "large", (1, 256, 2, 352)),
                          (3072, 8192, 1300, "down", "large", (1, 0, 3, 72)), (7168, 3584, 515, "gate and up", "twin", (0, 256, 5, 280))])
def test_kimi_shares_large_and_medium_tiles(kxlib, strict, ox, tmp_path, hidden, inter, tokens, product, tile, choice):
    """A prompt in one step against itself in steps whose products are whole or few-tile ones."""
    shape = (tokens, 2 * inter, hidden) if product == "gate and up" else (tokens, hidden, inter)
    exe = TS.build(tmp_path)
    assert TS.choices(exe, False, [shape], TS.KIMI) == [choice] and TS.tiles(exe, [shape], TS.KIMI) == [tile]
    cfg = _config(16, 1, tokens + 1)
    cfg.hidden, cfg.dense_inter = hidden, inter
    ids = O.tokens_u32(tokens, cfg.seed, 4, cfg.vocab).reshape(1, tokens)
    got = []
    for lib, chunk in ((kxlib, tokens), (strict, tokens), (kxlib, 100)):
        km = KxModel(lib, cfg)
        check(lib.kx_model_set_prefill_chunk(km.h, chunk))
        rc, _, _ = km.generate(ids, 1)
        assert rc == 0, lib.kx_last_error()
        got.append((O.bf16_to_f32(km.latent(1, 0, tokens)).astype(np.float64), km.logits(1)))
        km.close()
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1].view(np.uint32), got[1][1].view(np.uint32)), "both forms of the hand-over"
    row_err, log_err = np.abs(got[0][0] - got[2][0]).max() / np.abs(got[2][0]).max(), O.max_rel(got[0][1][0], got[2][1][0])
    say(f"kimi {shape}: cache rows {row_err:.1e}, logits {log_err:.1e}")
    assert row_err < 2e-2 and log_err < 3e-2


@pytest.mark.parametrize("width, ff, tokens, tile, choice", [(2048, 16450, 187, "medium", (0, 512, 2, 516)), (4096, 11264, 900, "large", (1, 256, 2, 352)),
                                                             (6144, 3290, 515, "twin", (0, 256, 5, 260))])
def test_hybrid_decoder_shares_large_and_medium_tiles(kxlib, strict, tmp_path, monkeypatch, width, ff, tokens, tile, choice):
    exe, shape = TS.build(tmp_path), (tokens, 2 * ((ff + 31) // 32 * 32), width)
    assert TS.choices(exe, False, [shape], TS.HYBRID) == [choice] and TS.tiles(exe, [shape], TS.HYBRID) == [tile]
    cfg = KC.config([KC.delta(heads=4, kv_heads=2, dim=32, vdim=64, ff=ff)], width=width, vocab=300)
    path, ids, got = KC.write(tmp_path / "m", cfg, {}), KC.tokens(cfg, tokens, 5)[None], []
    for lib, cuts in ((kxlib, [tokens]), (strict, [tokens]), (kxlib, [100])):
        monkeypatch.setattr(KC, "kx", lambda lib=lib: lib)
        with KC.Model(path, "bfloat16", batch=1, context=tokens, random_init=1, seed=9) as m:
            got.append(m.run(ids, cuts, 1))
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32)), "both forms of the hand-over"
    assert KC.logit_error(got[0], got[2]).max() < BF16_LOGITS
