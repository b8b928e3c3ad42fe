"""Products whose last round of tiles is shared by several workgroups each (kxtile::share): more tiles than one round holds, a few
left over, columns enough for parts.  Against the plain forward pass, with the bars of the whole-model tests, twice for the same bits."""
import numpy as np
import pytest

import kagalorn_case as KC
import kagalorn_oracle as K
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
