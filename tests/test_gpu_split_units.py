"""Up to four tokens against matrices of few rows: two or four waves share a unit of two rows (gemv_split in kx_linear.hip).  The
activations are given, so a product of n columns differs from 64 bits by its 32-bit sums alone; the bars are those of the other
operator tests."""
import ctypes as C

import numpy as np
import pytest

import kagalorn_case as KC
import kagalorn_oracle as K
from blok_amd.lib import DevBuf, KxLinearArgs, check
from kxt import dev
from test_gpu_kagalorn import _matrix, rel
from test_gpu_rapitar import Experts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("rows, cols", [(2, 5000), (67, 1025), (1024, 1024), (1030, 4097), (1536, 2048), (2047, 3100), (4097, 1088)])
def test_streams_of_few_rows(kxlib, rows, cols, f32):
    r = np.random.default_rng(rows)
    w = KC.bf16(r.standard_normal((rows, cols)) * cols ** -0.5)
    dw, ld = _matrix(w, f32)
    for tokens, streams in ((1, 1), (1, 2), (2, 2), (3, 1), (4, 2)):
        x = KC.bf16(r.standard_normal((tokens, cols)))
        s0 = r.standard_normal((tokens, streams, rows)).astype(np.float32)
        mix, ow = r.standard_normal((streams, streams)).astype(np.float32), r.standard_normal(streams).astype(np.float32)
        dx, ds, dm, do, scratch = _matrix(x, f32)[0], dev(s0), dev(mix), dev(ow), DevBuf(64)
        a = KxLinearArgs(f32=f32, tokens=tokens, rows=rows, cols=cols, ld=ld, row_kind=0, streams=streams, groups=1, d_w=dw.ptr, d_x=dx.ptr, x_ld=ld,
                         epilogue=2, d_mix=dm.ptr, d_outw=do.ptr)
        a.d_out = ds.ptr
        check(kxlib.kx_linear_run(C.byref(a), scratch.ptr, None))
        check(kxlib.kx_sync(None))
        want = K.hyper_write(s0.transpose(1, 0, 2).astype(np.float64), mix, ow, x.astype(np.float64) @ w.T).transpose(1, 0, 2)
        assert rel(ds.to_numpy(np.float32, s0.shape), want) < 1e-5, (tokens, streams)


@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("width, cols", [(192, 2500), (1056, 4100)])
def test_experts_behind_a_wide_product(kxlib, width, cols, f32):
    """The residual update's own columns and the chosen experts' as one sum, shared by two and four waves."""
    a = Experts(kxlib, width, 72, 16, 3, cols, f32, 4)
    r = np.random.default_rng(cols)
    for tokens in (1, 2, 4):
        x, rows = r.standard_normal((tokens, width)).astype(np.float32), KC.bf16(r.standard_normal((tokens, cols)))
        got, ids = a.run(x, rows)
        assert rel(got, a.oracle(x, rows, ids)) < (1e-5 if f32 else 2e-2), tokens
    a.close()
