"""Prompts of the Kimi-K2 design in long steps on dense layers, against the token-by-token prefill of the same model: the
tiles of the dense products (short, medium and large ones, columns in parts) and the attention of a step."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from blok_amd.lib import DevBuf, check, default_config
from kxt import say
from test_gpu_model import KxModel

pytestmark = pytest.mark.gpu


def _config(heads, batch, context):
    cfg = default_config()
    cfg.n_layers = cfg.first_dense = 2
    cfg.hidden, cfg.heads, cfg.dense_inter, cfg.vocab = 1024, heads, 8192, 3000
    cfg.max_batch, cfg.max_context, cfg.seed = batch, context, 11
    return cfg


@pytest.mark.parametrize("heads, batch, prompt, chunks", [
    (16, 1, 1801, (1801, 1000, 129, 40)),   # large tiles for gate and up, medium ones in parts, short ones; a step that ends with one position
    (64, 1, 700, (700, 333, 64)),
    (20, 3, 301, (301, 100, 17)),           # several sequences, a number of heads that is no multiple of 16
    (4, 33, 40, (40, 7, 1)),                # a batch that takes the step kernels of long prompts
], ids=lambda v: str(v))
def test_long_steps_against_token_by_token(kxlib, ox, heads, batch, prompt, chunks):
    cfg = _config(heads, batch, prompt + 4)
    ids = O.tokens_u32(batch * prompt, cfg.seed, 4, cfg.vocab).reshape(batch, prompt)
    km = KxModel(kxlib, cfg)
    check(kxlib.kx_model_set_exact(km.h, 15))
    got = {}
    for c in (0,) + chunks:
        if c:
            check(kxlib.kx_model_set_exact(km.h, 0))
            check(kxlib.kx_model_set_prefill_chunk(km.h, c))
        rc, out, _ = km.generate(ids, 1)
        assert rc == 0, kxlib.kx_last_error()
        got[c] = O.bf16_to_f32(np.stack([km.latent(1, b, prompt) for b in range(batch)])).astype(np.float64), km.logits(batch)
    km.close()
    rows, logits = got[0]
    for c in chunks:
        row_err = np.abs(got[c][0] - rows).max() / np.abs(rows).max()
        log_err = max(O.max_rel(got[c][1][b], logits[b]) for b in range(batch))
        say(f"heads={heads} batch={batch} prompt={prompt} chunk={c}: cache rows {row_err:.1e}, logits {log_err:.1e}")
        assert row_err < 2e-2 and log_err < 3e-2, c


@pytest.mark.parametrize("heads, batch, prompt, kernel", [(64, 1, 27000, 2), (60, 40, 750, 1), (64, 1, 62000, 2)],
                         ids=["all at once", "sequences in groups", "heads in groups"])
def test_expanded_keys_that_do_not_fit_at_once(kxlib, ox, heads, batch, prompt, kernel):
    """A context whose expanded keys and values take more than their room: fewer heads, or fewer sequences, at a time.
    Against the decode form of the attention in the same steps."""
    cfg = _config(heads, batch, prompt + 1)
    ids = O.tokens_u32(batch * prompt, cfg.seed, 4, cfg.vocab).reshape(batch, prompt)
    assert batch * heads * ((prompt + 63) // 64 * 64) * 640 > 1 << 30
    km = KxModel(kxlib, cfg)
    check(kxlib.kx_model_set_prefill_chunk(km.h, 2048))
    got = []
    for k in (kernel, 0):
        check(kxlib.kx_model_set_attention_kernel(km.h, k))
        rc, _, _ = km.generate(ids, 1)
        assert rc == 0, kxlib.kx_last_error()
        got.append((O.bf16_to_f32(np.stack([km.latent(1, b, prompt) for b in range(batch)])).astype(np.float64), km.logits(batch)))
    km.close()
    assert (got[0][0] != got[1][0]).any(), "the same bits: both runs took the decode form"
    row_err = np.abs(got[1][0] - got[0][0]).max() / np.abs(got[0][0]).max()
    log_err = max(O.max_rel(got[1][1][b], got[0][1][b]) for b in range(batch))
    say(f"heads={heads} batch={batch} prompt={prompt}: cache rows {row_err:.1e}, logits {log_err:.1e}")
    assert row_err < 2e-2 and log_err < 3e-2


@pytest.mark.parametrize("heads, kernel, short, long", [(64, 2, 100, 600), (8, 1, 40, 300)], ids=lambda v: str(v))
def test_short_steps_behind_a_long_context_take_the_decode_form(kxlib, heads, kernel, short, long):
    """Which of the two forms a step took shows in its bits: those of the decode form where that is the shorter one, others where not."""
    behind = 16000
    cfg = _config(heads, 1, behind + long)
    ids = O.tokens_u32(behind + long, cfg.seed, 4, cfg.vocab).astype(np.uint32)
    km = KxModel(kxlib, cfg)
    check(kxlib.kx_model_set_prefill_chunk(km.h, 2048))
    check(kxlib.kx_restart(km.h, 1))
    check(kxlib.kx_extend(km.h, ids.ctypes.data, behind, None, 0, None))
    for n, decode in ((short, True), (long, False)):
        got = []
        for k in (kernel, 0):
            check(kxlib.kx_model_set_attention_kernel(km.h, k))
            check(kxlib.kx_extend(km.h, ids[behind:].ctypes.data, n, None, 0, None))
            got.append(km.latent(1, 0, behind + n)[behind:])
            check(kxlib.kx_model_rewind(km.h, n))
        assert np.array_equal(got[0], got[1]) == decode, (n, decode)
    km.close()


def _free(lib):
    free, total = C.c_size_t(), C.c_size_t()
    assert lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_a_model_takes_the_memory_that_its_size_is_given_as(kxlib):
    """Also where a prompt's expanded keys and values would take a gigabyte."""
    cfg = _config(64, 33, 1000)
    parts = [C.c_uint64() for _ in range(3)]
    check(kxlib.kx_model_bytes(C.byref(cfg), *map(C.byref, parts)))
    KxModel(kxlib, _config(16, 1, 64)).close()                    # what the first model of a process loads
    before = _free(kxlib)
    km = KxModel(kxlib, cfg)
    check(kxlib.kx_model_set_prefill_chunk(km.h, 2048))
    rc, _, _ = km.generate(O.tokens_u32(33 * 130, 3, 4, cfg.vocab).reshape(33, 130), 1)
    assert rc == 0, kxlib.kx_last_error()
    taken = before - _free(kxlib)
    km.close()
    assert taken < sum(p.value for p in parts) + (64 << 20)


@pytest.mark.parametrize("batch", [5, 16, 17, 32])
@pytest.mark.parametrize("ff, vocab", [(8704, 9001), (2048, 4097), (4608, 33000)], ids=["two and three tiles a workgroup", "a tile or a few rows each", "five tiles"])
def test_products_of_a_batch_on_as_many_workgroups_as_run_at_once(kxlib, ox, batch, ff, vocab):
    """One position of 5 to 32 sequences a step, 16 and 17 on either side of the kernel's two forms: rows that do not come out even on 256 workgroups, against the
    same model's GEMVs.  The bars are those of long steps."""
    prompt = 6
    cfg = _config(16, batch, prompt + 4)
    cfg.dense_inter, cfg.vocab = ff, vocab
    ids = O.tokens_u32(batch * prompt, cfg.seed, 4, cfg.vocab).reshape(batch, prompt)
    km = KxModel(kxlib, cfg)
    got = []
    for exact in (15, 0):
        check(kxlib.kx_model_set_exact(km.h, exact))
        check(kxlib.kx_model_set_prefill_chunk(km.h, 1))
        rc, out, _ = km.generate(ids, 1)
        assert rc == 0, kxlib.kx_last_error()
        got.append((O.bf16_to_f32(np.stack([km.latent(1, b, prompt) for b in range(batch)])).astype(np.float64), km.logits(batch)))
    km.close()
    (rows, logits), (rows1, logits1) = got
    assert np.abs(rows1 - rows).max() / np.abs(rows).max() < 2e-2
    assert max(O.max_rel(logits1[b], logits[b]) for b in range(batch)) < 3e-2


@pytest.mark.parametrize("batch", [5, 16, 17, 32])
@pytest.mark.parametrize("vocab", [8449, 4097, 33000], ids=["shares of 33 and 34", "of 16 and 17", "of 128 and 129"])
def test_head_and_residual_of_a_batch_element_by_element(kxlib, vocab, batch):
    """A last tile of one row, and rows that do not come out even.  Every logit against its 64-bit sum over the device's own normed row: sums of 32 bits and a rounding to bf16, which
    may fall to the other side.  The residual rows, which every projection adds to, against those of the GEMVs: 2^-8 at each of four sums, and what the layers before differ by."""
    cfg = _config(16, batch, 8)
    cfg.dense_inter, cfg.vocab = 8704, vocab
    ids = O.tokens_u32(batch * 3, cfg.seed, 4, vocab).reshape(batch, 3)
    km = KxModel(kxlib, cfg)
    check(kxlib.kx_model_set_prefill_chunk(km.h, 1))
    hidden = []
    for exact in (15, 0):
        check(kxlib.kx_model_set_exact(km.h, exact))
        check(kxlib.kx_prefill(km.h, ids.ctypes.data, batch, 3))
        hidden.append(km.hidden(batch))
    logits = km.logits(batch)
    km.close()
    H = cfg.hidden
    norm, head, dn = DevBuf(2 * H), DevBuf(2 * H * vocab), DevBuf(2 * H * batch)
    check(kxlib.kx_fill_affine_bf16(norm.ptr, H, cfg.seed, 2, 1.0, 0.02, None))
    check(kxlib.kx_fill_normal_bf16(head.ptr, H * vocab, cfg.seed, 3, cfg.init_sigma, 0, None))
    dx = DevBuf.from_numpy(hidden[1])
    check(kxlib.kx_rmsnorm(dx.ptr, norm.ptr, dn.ptr, batch, H, cfg.rms_eps, None))
    check(kxlib.kx_sync(None))
    f64 = lambda b, shape: O.bf16_to_f32(b.to_numpy(np.uint16, shape)).astype(np.float64)
    want = f64(dn, (batch, H)) @ f64(head, (vocab, H)).T
    assert O.elem_err(logits, want) < 5e-3
    assert O.elem_err(*map(O.bf16_to_f32, hidden[::-1])) < 2e-2
