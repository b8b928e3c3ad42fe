"""What is not finite at a position of a prompt step stays with the positions that see it: those before it, and those whose window
has left it, come out to the bit as without it."""
import numpy as np
import pytest

import ckpt
import kagalorn_case as KC
import oracle as O
from blok_amd import model_index as MI
from blok_amd.lib import check
from kxt import say
from test_gpu_kagalorn import Window
from test_gpu_load import KxLoaded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("dim, vdim", [(32, 32), (40, 70), (190, 120), (256, 200)])
def test_value_in_the_window_attention(kxlib, dim, vdim, bad):
    heads, kv, size, n = 4, 2, 100, 300
    for pool in (0, 8):
        w = Window(kxlib, heads, kv, dim, vdim, size, pool, 0)
        clean = np.random.default_rng(dim).standard_normal((1, n, w.cols[-1])).astype(np.float32)
        for at, cuts in ((170, [n]), (191, [n]), (192, [130, n]), (0, [n]), (255, [200, n])):
            say(f"window {dim} {vdim} pool={pool} {bad} at {at} in steps of {cuts}")
            want = w.run(clean, cuts)[0].reshape(n, heads, vdim)
            proj = clean.copy()
            proj[0, at, w.cols[2] + 5] = bad                                     # column 5 of key head 0
            got = w.run(proj, cuts)[0].reshape(n, heads, vdim)
            hit = np.zeros(got.shape, bool)
            hit[at:n if pool else at + size, :2, 5] = True                      # a pooled block is seen from then on
            assert np.isfinite(want).all() and np.array_equal(got[~hit], want[~hit])
            assert not np.isfinite(got[at:at + size, :2, 5]).any()
        w.close()


def test_token_in_a_long_step_of_kimi(kxlib, ox, tmp_path, monkeypatch):
    """A token whose embedding is not finite, in steps that attend to expanded keys and values."""
    cfg = O.small_config(n_layers=2, first_dense=2, context=400)
    tensors = ckpt.model_tensors

    def spoiled(c, seed):
        out = tensors(c, seed)
        assert out[0][0].endswith("embed_tokens.weight")
        out[0][3].reshape(c.vocab, c.hidden)[77, 3] = 0x7fc0                     # a NaN
        return out

    monkeypatch.setattr(ckpt, "model_tensors", spoiled)
    ckpt.write_checkpoint(tmp_path / "hf", cfg, seed=9)
    km = KxLoaded(kxlib, cfg, MI.materialize(tmp_path / "hf", tmp_path / "meta")["index"])
    n, at = 300, 170
    clean = O.tokens_u32(n, 9, 4, cfg.vocab).astype(np.uint32)
    clean[clean == 77] = 78
    dirty = clean.copy()
    dirty[at] = 77
    for chunk in (256, 100, 1):
        check(kxlib.kx_model_set_prefill_chunk(km.h, chunk))
        got = []
        for ids in (clean, dirty):
            places, logits = np.arange(at, dtype=np.int32), np.empty((at, 1, cfg.vocab), np.float32)
            check(kxlib.kx_restart(km.h, 1))
            check(kxlib.kx_extend(km.h, ids.ctypes.data, n, places.ctypes.data, at, logits.ctypes.data))
            rows = np.stack([km.latent(l, 0, n) for l in range(2)])
            check(kxlib.kx_model_rewind(km.h, n - at))                         # and on without it
            check(kxlib.kx_extend(km.h, clean[at:].ctypes.data, n - at, None, 0, None))
            got.append((logits, rows, km.logits(1), np.stack([km.latent(l, 0, n) for l in range(2)])))
        (logits, rows, last, after), (logits1, rows1, last1, after1) = got
        assert np.isfinite(logits).all() and np.isfinite(last).all()
        assert not np.isfinite(O.bf16_to_f32(rows1[:, at])).all()
        assert np.array_equal(rows1[:, :at], rows[:, :at]) and np.array_equal(logits1, logits), chunk
        assert np.array_equal(after1, after) and np.array_equal(last1, last), chunk
    km.close()


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_token_in_a_long_step_of_kagalorn(kxlib, tmp_path, dtype):
    cfg = KC.config([KC.attention(), KC.delta(), KC.attention(), KC.delta()], vocab=200)
    w = KC.weights(cfg, 5)
    w["embed"][77, 3] = np.nan
    n, at = 200, 139
    clean = np.asarray(KC.tokens(cfg, n, 8), np.uint32)
    clean[clean == 77] = 78
    dirty = clean.copy()
    dirty[at] = 77
    with KC.Model(KC.write(tmp_path, cfg, w), dtype, context=n) as m:
        for cuts in ([n], [130, n]):
            want, got = m.run(clean, cuts), m.run(dirty, cuts)
            assert np.isfinite(want).all() and not np.isfinite(got[at]).all()
            assert np.array_equal(got[:at], want[:at]), cuts
