"""Products of the hybrid decoder where their kernels change: few tokens with the columns split over workgroups, experts with
few slots, large tiles.  Against the plain forward passes, with the bars of the whole-model tests."""
import ctypes as C
import os

import numpy as np
import pytest

import blok_amd.lib as kxl
import kagalorn_case as KC
import kagalorn_oracle as K
import oracle as O
import tile_share as TS
from blok_amd.lib import DevBuf, KxLinearArgs, check
from kxt import dev, say
from test_gpu_kagalorn import BF16_LOGITS, F32_LOGITS, _matrix, rel
from test_gpu_kimi_prompt import _config
from test_gpu_model import KxModel
from test_gpu_rapitar import Experts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype, bar", [("bfloat16", BF16_LOGITS), ("float32", F32_LOGITS)])
@pytest.mark.parametrize("ff", [4200, 4130], ids=["whole blocks", "half a block left"])
def test_few_tokens_against_wide_matrices(kxlib, tmp_path, ff, dtype, bar):
    """5 to 64 tokens a step: up to eight parts of 66 and 65 pieces of 64 columns, and the last part shorter than the others;
    66 to 192 tokens: tiles in up to four parts.  In 32 bits tiles in up to 16 parts throughout."""
    cfg = KC.config([KC.delta(heads=4, kv_heads=2, dim=32, vdim=640, ff=ff), KC.attention(ff=ff)], width=192, vocab=300)
    w = KC.weights(cfg, ff)
    ids = np.stack([KC.tokens(cfg, 6, 100 + b) for b in range(64)])
    want = np.stack([K.forward(cfg, w, s) for s in ids], 1)
    with KC.Model(KC.write(tmp_path, cfg, w), dtype, batch=64, context=6) as m:
        for batch, cuts in ((5, [1]), (8, [4, 1]), (31, [2, 1]), (33, [1]), (63, [1]), (64, [1]), (5, [1]), (33, [2]), (64, [2]), (43, [3]), (64, [3])):
            first = m.run(ids[:batch], cuts, batch)
            assert KC.logit_error(first, want[:, :batch]).max() < bar, (batch, cuts)
            assert (m.run(ids[:batch], cuts, batch) == first).all(), "the parts' order does not depend on who comes last"


@pytest.fixture(scope="module")
def strict():
    """The library with the hand-over between workgroups in its memory-model form (kx_arrive.h)."""
    return kxl.load_library(os.path.join(os.path.dirname(kxl.lib_path()), "libkx_strict.so"))


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_parts_of_the_hybrid_decoder_in_both_forms_of_the_hand_over(kxlib, strict, tmp_path, monkeypatch, dtype):
    """All tokens against 64 rows in parts of the columns, and tiles in parts, bf16 and f32."""
    cfg = KC.config([KC.delta(heads=4, kv_heads=2, dim=32, vdim=640, ff=4200), KC.attention(ff=4130)], width=192, vocab=300)
    path, ids = KC.write(tmp_path, cfg, KC.weights(cfg, 3)), np.stack([KC.tokens(cfg, 6, 50 + b) for b in range(64)])
    got = []
    for lib in (kxlib, strict):
        monkeypatch.setattr(KC, "kx", lambda lib=lib: lib)
        with KC.Model(path, dtype, batch=64, context=6) as m:
            got.append([m.run(ids[:b], cuts, b) for b, cuts in ((5, [1]), (8, [4, 1]), (33, [2]), (64, [1]), (64, [3]))])
    for a, b in zip(*got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_parts_of_kimi_in_both_forms_of_the_hand_over(kxlib, strict, ox):
    """Steps of 40 to 300 tokens: short and medium tiles in parts."""
    cfg = _config(16, 1, 310)
    ids = O.tokens_u32(300, 9, 4, cfg.vocab).reshape(1, 300)
    for chunk in (300, 129, 40):
        got = []
        for lib in (kxlib, strict):
            km = KxModel(lib, cfg)
            check(lib.kx_model_set_prefill_chunk(km.h, chunk))
            rc, _, _ = km.generate(ids, 1)
            assert rc == 0, lib.kx_last_error()
            got.append((km.logits(1), km.latent(1, 0, 300)))
            km.close()
        say(f"kimi, steps of {chunk}")
        assert np.array_equal(got[0][0].view(np.uint32), got[1][0].view(np.uint32)) and np.array_equal(got[0][1], got[1][1]), chunk


@pytest.mark.parametrize("tokens", [31, 32, 33, 96, 97, 200])
def test_experts_of_more_slots_than_a_small_tile(kxlib, tokens):
    """All tokens on three of 100 experts: one to three tiles of 32 slots each, and from 97 tokens on of 64, the last one short."""
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


def _put(x):
    """bf16 values in memory as the rows of a product"""
    return dev((np.ascontiguousarray(x, np.float32).view(np.uint32) >> 16).astype(np.uint16))


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    return TS.build(tmp_path_factory.mktemp("share"))


@pytest.mark.parametrize("tokens, rows, cols, tile", [(1985, 8000, 64, "medium"), (2048, 8192, 128, "medium"), (1793, 7937, 192, "medium"), (2048, 8192, 384, "large"),
                                                      (1985, 8000, 448, "large"), (1793, 7937, 576, "large")], ids=lambda v: str(v))
def test_large_tiles(kxlib, rule, tokens, rows, cols, tile):
    """Tiles of few blocks, 128 x 128 and, from six on, 256 x 256, whole and with remainders of tokens and rows, through every epilogue that a prompt meets."""
    assert TS.tiles(rule, [(tokens, rows, (cols + 63) // 64 * 64)]) == [tile]
    r = np.random.default_rng(rows)
    w, x = KC.bf16(r.standard_normal((rows, cols)) * cols ** -0.5), KC.bf16(r.standard_normal((tokens, cols)))
    dw, ld = _matrix(w, 0)
    dx, y = _put(x), (x @ w.T).astype(np.float64)
    scratch = DevBuf(64)

    def run(out, m=dw, n=rows, **kw):
        a = KxLinearArgs(f32=0, tokens=tokens, rows=n, cols=cols, ld=ld, row_kind=0, streams=1, groups=1, d_w=m.ptr, d_x=dx.ptr, x_ld=ld)
        for k, v in kw.items():
            setattr(a, k, v)
        a.d_out = out.ptr
        check(kxlib.kx_linear_run(C.byref(a), scratch.ptr, None))
        check(kxlib.kx_sync(None))

    # stored; the last rows through gelu
    acts = 70
    out, mid = dev(np.full((tokens, rows), 7.0, np.float32)), dev(np.zeros((tokens, 96), np.uint16))
    run(out, epilogue=0, out_ld=rows, act_rows=acts, d_mid=mid.ptr, mid_ld=96)
    got, act = out.to_numpy(np.float32, (tokens, rows)), mid.to_numpy(np.uint16, (tokens, 96))
    assert rel(got[:, :rows - acts], y[:, :rows - acts]) < 1e-5 and (got[:, rows - acts:] == 7.0).all()
    z = y[:, rows - acts:]
    gelu = 0.5 * z * (1 + np.tanh(np.sqrt(2 / np.pi) * (z + 0.044715 * z ** 3)))
    assert rel((act[:, :acts].astype(np.uint32) << 16).view(np.float32), gelu) < 1e-2 and not act[:, acts:].any()
    # two streams, and one
    for streams in (2, 1):
        s0 = r.standard_normal((tokens, streams, rows)).astype(np.float32)
        mix, ow = r.standard_normal((streams, streams)).astype(np.float32), r.standard_normal(streams).astype(np.float32)
        ds, dm, do = dev(s0), dev(mix), dev(ow)
        run(ds, epilogue=2, streams=streams, d_mix=dm.ptr, d_outw=do.ptr)
        want = K.hyper_write(s0.transpose(1, 0, 2).astype(np.float64), mix, ow, y).transpose(1, 0, 2)
        assert rel(ds.to_numpy(np.float32, s0.shape), want) < 1e-5
    # gate and up
    ff = rows // 64 * 32
    g, u = w[:ff], w[ff:2 * ff]
    packed = np.stack([g.reshape(-1, 32, cols), u.reshape(-1, 32, cols)], 1).reshape(2 * ff, cols)
    out = dev(np.zeros((tokens, ff), np.uint16))
    run(out, m=_matrix(packed, 0)[0], n=2 * ff, epilogue=1, out_ld=ff, limit=1.5, alpha=1.702, bias=1.0)
    gv, uv = np.minimum(y[:, :ff], 1.5), np.clip(y[:, ff:2 * ff], -1.5, 1.5)
    want = gv * K.sigmoid(1.702 * gv) * (uv + 1.0)
    assert rel((out.to_numpy(np.uint16, (tokens, ff)).astype(np.uint32) << 16).view(np.float32), want) < 1e-2


@pytest.mark.parametrize("tokens, rows, cols, tile", [(300, 1000, 640, "twin"), (129, 4100, 704, "twin"), (66, 129, 1280, "twin"), (2047, 2048, 832, "twin"), (1793, 8191, 1024, "large"),
                                                      (2048, 7424, 1088, "large")], ids=["twin, 10 blocks", "twin, 11", "twin, a few", "twin, 13", "large, 16", "large, 17"])
def test_tiles_whose_groups_take_turns(kxlib, rule, tokens, rows, cols, tile):
    """Even and odd numbers of blocks, tiles with remainders of tokens and rows, every epilogue: the bars of the large tiles, 32-bit sums of up to
    1088 products (about 1e-6)."""
    test_large_tiles(kxlib, rule, tokens, rows, cols, tile)


@pytest.mark.parametrize("f32", [0, 1], ids=["bf16", "f32"])
@pytest.mark.parametrize("tokens", [2, 3, 4])
@pytest.mark.parametrize("cols, streams, groups, heads", [(96, 1, 1, 3), (1000, 2, 4, 8), (2048, 2, 2, 16), (4097, 3, 1, 17)])
def test_rows_in_a_launch_of_their_own(kxlib, tokens, cols, streams, groups, heads, f32):
    """Two to four tokens: with room for them the rows are built in front of the product, without in it, and the results are the same to the bit."""
    r = np.random.default_rng(cols + tokens)
    rows = 70
    w, ld = _matrix(KC.bf16(r.standard_normal((rows, cols)) * cols ** -0.5), f32)
    vdim = cols // heads
    x, win = dev(r.standard_normal((tokens, streams, cols)).astype(np.float32)), dev(r.standard_normal(streams).astype(np.float32))
    norm = dev((1 + 0.3 * r.standard_normal(cols)).astype(np.float32))
    o, gate = dev(r.standard_normal((tokens, cols)).astype(np.float32)), dev(r.standard_normal((tokens, cols + 5)).astype(np.float32))
    scratch = DevBuf(tokens * ld * 4)
    forms = [dict(row_kind=1, streams=streams, groups=groups, d_streams_in=x.ptr, d_in=win.ptr)]
    if vdim * heads == cols:
        forms += [dict(row_kind=2, streams=1, groups=1, heads=heads, vdim=vdim, d_o=o.ptr, d_gate=gate.ptr, gate_ld=cols + 5, gate_first=first) for first in (0, 1)]
    for form in forms:
        got = []
        for room in (None, scratch.ptr):
            out = dev(np.full((tokens, rows), 7.0, np.float32))
            a = KxLinearArgs(f32=f32, tokens=tokens, rows=rows, cols=cols, ld=ld, eps=1e-5, d_w=w.ptr, d_norm=norm.ptr, epilogue=0, out_ld=rows)
            for k, v in form.items():
                setattr(a, k, v)
            a.d_out = out.ptr
            check(kxlib.kx_linear_run(C.byref(a), room, None))
            check(kxlib.kx_sync(None))
            got.append(out.to_numpy(np.float32, (tokens, rows)))
        assert np.isfinite(got[0]).all() and (got[0] != 7.0).any() and np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32)), form


@pytest.mark.parametrize("tokens", [5, 33, 64])
@pytest.mark.parametrize("rows, cols", [(8192, 1024), (8193, 1024), (8256, 1088), (16387, 1600), (16448, 2100), (33001, 1024), (40000, 1030)])
def test_few_tokens_on_workgroups_with_equal_shares(kxlib, rows, cols, tokens):
    """Rows for half of the CUs and more, one column part: one workgroup per CU, rounds of two per CU, shares of 32 to 64 rows that do not come out even, stored and
    through two streams.  32-bit sums of bf16 products."""
    r = np.random.default_rng(rows)
    w, x = KC.bf16(r.standard_normal((rows, cols)) * cols ** -0.5), KC.bf16(r.standard_normal((tokens, cols)))
    y = x @ w.T
    dw, ld = _matrix(w, 0)
    dx, scratch = _matrix(x, 0)[0], DevBuf(64)
    base = dict(f32=0, tokens=tokens, rows=rows, cols=cols, ld=ld, row_kind=0, groups=1, d_w=dw.ptr, d_x=dx.ptr, x_ld=ld)
    out = dev(np.full((tokens, rows + 1), 7.0, np.float32))
    a = KxLinearArgs(**base, streams=1, epilogue=0, out_ld=rows + 1)
    a.d_out = out.ptr
    check(kxlib.kx_linear_run(C.byref(a), scratch.ptr, None))
    check(kxlib.kx_sync(None))
    got = out.to_numpy(np.float32, (tokens, rows + 1))
    assert rel(got[:, :rows], y) < 1e-5 and (got[:, rows:] == 7.0).all()
    s0 = r.standard_normal((tokens, 2, rows)).astype(np.float32)
    mix, ow = r.standard_normal((2, 2)).astype(np.float32), r.standard_normal(2).astype(np.float32)
    ds, dm, do = dev(s0), dev(mix), dev(ow)
    a = KxLinearArgs(**base, streams=2, epilogue=2, d_mix=dm.ptr, d_outw=do.ptr)
    a.d_out = ds.ptr
    check(kxlib.kx_linear_run(C.byref(a), scratch.ptr, None))
    check(kxlib.kx_sync(None))
    assert rel(ds.to_numpy(np.float32, s0.shape), K.hyper_write(s0.transpose(1, 0, 2).astype(np.float64), mix, ow, y.astype(np.float64)).transpose(1, 0, 2)) < 1e-5


@pytest.mark.parametrize("vocab, width", [(11003, 2048), (15003, 2048), (7003, 4096), (4003, 8192)], ids=["two parts of 256 shares", "nearly whole groups", "four of 128", "eight of 64"])
def test_equal_shares_with_parts_of_the_columns(kxlib, strict, tmp_path, monkeypatch, vocab, width):
    """A head whose rows come out uneven on the shares, with its columns in parts as well: partial sums and counters of arrivals are numbered by shares.  The layer
    adds nothing, so the head's rows are the normed embeddings and every logit is compared with its 64-bit sum: a rounding of a row's element to the other bf16
    value moves a logit by about 1e-4 of their root mean square, sums of 32 bits by less.  The same bits whoever comes last, and in both forms of the hand-over."""
    cfg = KC.config([KC.delta(heads=1, kv_heads=1, dim=8, vdim=8, ff=None)], width=width, vocab=vocab, streams=1, groups=1)
    w = KC.weights(cfg, vocab)
    w["l0.mix.o"][:] = 0.0
    for k in ("in", "out", "mix"):
        w["l0.hc1." + k][:] = 1.0
    path, batches = KC.write(tmp_path, cfg, w), (5, 32, 33, 64)
    ids = KC.tokens(cfg, 64, 7)
    x = w["embed"][ids]
    x = KC.bf16(x / np.sqrt((x * x).mean(-1, keepdims=True) + 1e-5) * w["final.norm"]).astype(np.float64)
    want = x @ w["head"].T
    got = []
    for lib in (kxlib, strict):
        monkeypatch.setattr(KC, "kx", lambda lib=lib: lib)
        with KC.Model(path, "bfloat16", batch=64, context=4) as m:
            for b in batches + batches:
                m.restart(b)
                got.append(m.extend(ids[:b, None])[0])
    for i, y in enumerate(got):
        b = batches[i % 4]
        assert np.abs(y - want[:b]).max() < 2e-3 * np.sqrt((want * want).mean()), (b, i)
        assert np.array_equal(y.view(np.uint32), got[i % 4].view(np.uint32)), (b, i)
