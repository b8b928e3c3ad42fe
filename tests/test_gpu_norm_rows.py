"""RMSNorm at the row lengths where its kernel changes, and beside them: bit-exact with the oracle (src/kimi_exec.cu:258-270)."""
import numpy as np
import pytest

import oracle as O
from blok_amd.lib import check
from kxt import dev, say
from test_gpu_dense import ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 2040, 2048, 2056, 4096, 4104, 6136, 8192, 8200, 12304])
@pytest.mark.parametrize("tokens", [1, 37])
def test_rows_of_every_form(kxlib, ox, n, tokens):
    say(f"rmsnorm n={n} tokens={tokens}")
    x, w = O.normal_bf16(tokens * n, 3, 1, 1.0), O.normal_bf16(n, 3, 2, 1.0)
    guard = 0x1234
    dx, dw, dy = dev(x), dev(w), dev(np.full(tokens * n + 64, guard, np.uint16))
    check(kxlib.kx_rmsnorm(dx.ptr, dw.ptr, dy.ptr, tokens, n, 1e-5, None))
    check(kxlib.kx_sync(None))
    want = np.empty(tokens * n, np.uint16)
    ox.ox_rmsnorm(ptr(x), ptr(w), ptr(want), tokens, n, 1e-5, 1)
    got = dy.to_numpy(np.uint16, (tokens * n + 64,))
    assert np.array_equal(got[:-64], want) and (got[-64:] == guard).all()
