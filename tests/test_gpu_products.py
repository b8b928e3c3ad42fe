"""Products of the hybrid decoder where their kernels change: few tokens with the columns split over workgroups, experts with
few slots.  Against the plain forward passes, with the bars of the whole-model tests."""
import numpy as np
import pytest

import kagalorn_case as KC
import kagalorn_oracle as K
from test_gpu_kagalorn import BF16_LOGITS, rel
from test_gpu_rapitar import Experts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ff", [4200, 4130], ids=["whole blocks", "half a block left"])
def test_few_tokens_against_wide_matrices(kxlib, tmp_path, ff):
    """5 to 64 tokens a step: up to eight parts of 66 and 65 pieces of 64 columns, and the last part shorter than the others."""
    cfg = KC.config([KC.delta(heads=4, kv_heads=2, dim=32, vdim=640, ff=ff), KC.attention(ff=ff)], width=192, vocab=300)
    w = KC.weights(cfg, ff)
    ids = np.stack([KC.tokens(cfg, 6, 100 + b) for b in range(64)])
    want = np.stack([K.forward(cfg, w, s) for s in ids], 1)
    with KC.Model(KC.write(tmp_path, cfg, w), "bfloat16", batch=64, context=6) as m:
        for batch, cuts in ((5, [1]), (8, [4, 1]), (31, [2, 1]), (33, [1]), (63, [1]), (64, [1]), (5, [1])):
            first = m.run(ids[:batch], cuts, batch)
            assert KC.logit_error(first, want[:, :batch]).max() < BF16_LOGITS, (batch, cuts)
            assert (m.run(ids[:batch], cuts, batch) == first).all(), "the parts' order does not depend on who comes last"


@pytest.mark.parametrize("tokens", [31, 32, 33, 200])
def test_experts_of_more_slots_than_a_small_tile(kxlib, tokens):
    """All tokens on three of 100 experts: one to seven tiles of 32 slots each, the last one short."""
    a = Experts(kxlib, 192, 72, 100, 3, 64, 0, 200)
    a.router[:], a.bias[:] = 0.0, 0.0
    a.bias[[99, 5, 40]] = 3.0
    a.push()
    r = np.random.default_rng(tokens)
    x, rows = r.standard_normal((tokens, 192)).astype(np.float32), KC.bf16(r.standard_normal((tokens, 64)))
    got, ids = a.run(x, rows)
    assert (np.sort(ids, 1) == [5, 40, 99]).all()
    assert rel(got, a.oracle(x, rows, ids)) < 2e-2
    a.close()
