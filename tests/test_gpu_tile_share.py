"""Products whose last round of tiles is shared by several workgroups each (kxtile::share): more tiles than one round holds, a few
left over, columns enough for parts.  Against the plain forward pass, with the bars of the whole-model tests, twice for the same bits."""
import numpy as np
import pytest

import kagalorn_case as KC
import kagalorn_oracle as K
import tile_share as TS
from test_gpu_kagalorn import BF16_LOGITS, F32_LOGITS

pytestmark = pytest.mark.gpu


# tokens, width, ff: f32 4 x 66 tiles of 64 x 128 and 5 x 67 with their edges inside; bf16 5 x 130 tiles of 128 x 128
@pytest.mark.parametrize("dtype, tokens, width, ff, bar", [("float32", 256, 512, 4200, F32_LOGITS), ("float32", 261, 544, 4260, F32_LOGITS),
                                                           ("bfloat16", 577, 2048, 8290, BF16_LOGITS)])
def test_last_round_in_parts(kxlib, tmp_path, dtype, tokens, width, ff, bar):
    cfg = KC.config([KC.delta(heads=4, kv_heads=2, dim=32, vdim=64, ff=ff)], width=width, vocab=300)
    w = KC.weights(cfg, ff)
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
