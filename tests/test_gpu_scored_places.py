"""Logits that kx_extend hands back for the last place and for others: the last one's are those of the position that is sampled from
(kx_model_logits, kx_greedy_sample), whatever else is asked for, at any number of sequences up to the model's."""
import numpy as np
import pytest

import kagalorn_case as KC
import kagalorn_oracle as K
import oracle as O
from blok_amd.lib import check
from test_gpu_kagalorn import BF16_LOGITS, F32_LOGITS
from test_gpu_kimi_prompt import _config
from test_gpu_model import KxModel

pytestmark = pytest.mark.gpu


def _sampled(lib, h, batch, vocab):
    logits, ids = np.empty((batch, vocab), np.float32), np.empty(batch, np.uint32)
    check(lib.kx_model_logits(h, logits.ctypes.data))
    check(lib.kx_greedy_sample(h, ids.ctypes.data))
    return logits, ids


@pytest.mark.parametrize("batch, n, chunk", [(1, 40, 40), (1, 90, 33), (3, 20, 20), (5, 4, 1)])
def test_kimi_with_as_many_sequences_as_it_holds(kxlib, ox, batch, n, chunk):
    cfg = _config(16, batch, n)
    ids = O.tokens_u32(batch * n, 21, 4, cfg.vocab).reshape(batch, n).astype(np.uint32)
    km = KxModel(kxlib, cfg)
    check(kxlib.kx_model_set_prefill_chunk(km.h, chunk))
    got = []
    for want in ([n - 1], [0, n - 1], [n - 1, n // 2, n - 2, n - 1]):
        w, out = np.array(want, np.int32), np.empty((len(want), batch, cfg.vocab), np.float32)
        check(kxlib.kx_restart(km.h, batch))
        check(kxlib.kx_extend(km.h, ids.ctypes.data, n, w.ctypes.data, len(w), out.ctypes.data))
        logits, sampled = _sampled(kxlib, km.h, batch, cfg.vocab)
        for at, row in zip(want, out):
            if at == n - 1:
                assert np.array_equal(row.view(np.uint32), logits.view(np.uint32)) and (sampled == logits.argmax(1)).all(), want
        got.append(logits)
    km.close()
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])


@pytest.mark.parametrize("dtype, bar", [("bfloat16", BF16_LOGITS), ("float32", F32_LOGITS)])
def test_places_of_many_sequences(kxlib, tmp_path, dtype, bar):
    """48, 63 and 64 sequences in one step: 64 rows are made at a time."""
    cfg = KC.config([KC.delta(heads=4, kv_heads=2, dim=32, vdim=64, ff=200)], width=192, vocab=301)
    w = KC.weights(cfg, 4)
    ids = np.stack([KC.tokens(cfg, 5, 70 + b) for b in range(64)])
    full = np.stack([K.forward(cfg, w, s) for s in ids], 1)
    path = KC.write(tmp_path, cfg, w)
    for batch in (48, 63, 64):
        with KC.Model(path, dtype, batch=batch, context=5) as m:
            for want in ([4], [0, 4], [3, 4, 1, 3, 2, 0], [2]):
                m.restart(batch)
                got = m.extend(ids[:batch], want)
                assert KC.logit_error(got, full[want][:, :batch]).max() < bar, (batch, want)
                logits, sampled = _sampled(m.lib, m.h, batch, cfg["vocab"])
                assert (sampled == logits.argmax(1)).all()
                if 4 in want:
                    assert np.array_equal(got[want.index(4)].view(np.uint32), logits.view(np.uint32)), (batch, want)
