"""The delta rule where its blocks of 16 tokens, its rows of 64 and its slices of 16 columns end."""
import numpy as np
import pytest

from kxt import say
from test_gpu_kagalorn import Delta, rel

pytestmark = pytest.mark.gpu
# keys have unit length, so a sum of 256 products is off by at most 256 * 2^-24 of its terms, in what a token takes
# out of the state and again in what it reads
TOLERANCE = 2 * 256 * 2.0 ** -24


@pytest.mark.parametrize("shape", [(2, 1, 16, 15), (3, 1, 64, 16), (2, 2, 65, 17), (4, 2, 128, 33), (1, 1, 192, 1), (2, 1, 256, 16), (32, 2, 70, 80)], ids=lambda c: "-".join(map(str, c)))
def test_delta_blocks(kxlib, shape):
    d = Delta(kxlib, *shape, 3, batch=2)
    for n in (2, 15, 16, 17, 32, 33, 49):
        say(f"delta blocks {shape} {n}")
        proj = np.random.default_rng(n).standard_normal((2, n + 5, d.cols[-1])).astype(np.float32)
        got = d.run(proj, [n, 5], 2)
        for b in range(2):
            assert rel(got[b], d.oracle(proj[b])) < TOLERANCE, (n, b)
    d.close()


@pytest.mark.parametrize("shape", [(1, 1, 3, 1, 2), (3, 1, 5, 7, 4)], ids=lambda c: "-".join(map(str, c)))
def test_delta_state_that_is_no_multiple_of_16_bytes(kxlib, shape):
    """The scratch, which is accessed in pieces of 16 bytes, does not begin where the state and the inputs end."""
    d = Delta(kxlib, *shape)
    proj = np.random.default_rng(5).standard_normal((1, 40, d.cols[-1])).astype(np.float32)
    for cuts in ([40], [2, 17, 1, 20]):
        assert rel(d.run(proj, cuts)[0], d.oracle(proj[0])) < TOLERANCE
    d.close()


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_delta_value_that_is_not_finite_reaches_no_token_before_it(kxlib, bad):
    heads, kv, dim, vdim = 2, 1, 40, 20
    d = Delta(kxlib, heads, kv, dim, vdim, 1)
    proj = np.random.default_rng(1).standard_normal((1, 45, d.cols[-1])).astype(np.float32)
    d.conv[:] = np.abs(d.conv)
    d.d[0].upload(d.conv)
    clean = d.run(proj, [45])[0].reshape(45, heads, vdim)
    proj[0, 21, d.cols[2] + vdim + 3] = bad                       # head 1, column 3
    got = d.run(proj, [45])[0].reshape(45, heads, vdim)
    hit = np.zeros(got.shape, bool)
    hit[21:, 1, 3] = True
    assert np.array_equal(got[~hit], clean[~hit]) and not np.isfinite(got[hit]).any()
    d.close()


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("at", [0, 16, 21, 31, 44])
def test_delta_token_that_is_not_finite_reaches_no_token_before_it(kxlib, at, bad):
    """The query, the key, a value, the step size, the decay or the whole row of a token at the first, a middle or the last place
    of a block or of the step; with more heads than key heads, so that a key head's neighbour has to stay as it is too."""
    heads, kv, dim, vdim = 4, 2, 40, 20
    d = Delta(kxlib, heads, kv, dim, vdim, 1)
    clean = np.random.default_rng(2).standard_normal((1, 45, d.cols[-1])).astype(np.float32)
    want = d.run(clean, [45])[0].reshape(45, heads, vdim)
    assert np.isfinite(want).all()
    c = [int(x) for x in d.cols]
    # columns of a token, and the heads that read them
    cases = {"query": (c[0] + 3, [0, 1]), "key": (c[1] + dim + 5, [2, 3]), "value": (c[2] + vdim + 3, [1]), "step size": (c[3] + 2, [2]), "decay": (c[4] + 3, [3]),
             "row": (slice(None), [0, 1, 2, 3])}
    for name, (col, hit) in cases.items():
        say(f"delta {name} {bad} at {at}")
        proj = clean.copy()
        proj[0, at, col] = bad
        got = d.run(proj, [45])[0].reshape(45, heads, vdim)
        others = [h for h in range(heads) if h not in hit]
        assert np.array_equal(got[:at], want[:at]) and np.array_equal(got[:, others], want[:, others]), name
        if name in ("query", "key", "value", "row"):  # the sigmoid and the decay are finite for every number and for none
            assert not np.isfinite(got[at, hit]).all(), name
        if name == "query":  # is read by its own token alone
            assert np.array_equal(got[at + 1:], want[at + 1:]), name
    d.close()
