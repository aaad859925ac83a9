"""The forms that fast FP32 streaming evaluates expressions in (paraiso_amd/schemes/rewrites.py)
on every pair of zeros, infinities, NaN, subnormal, tiny, ordinary and large values.

The limiter is compared with its definition on the exact product: in FP32 a product of two tiny
values underflows to 0, where the general form gives 0 and the median the smaller value.  The
quotients and the maximum are the bits of the tile form of the same build."""
import numpy as np
import pytest

from paraiso_amd import variants
from paraiso_amd.schemes.rewrites import OUT

pytestmark = pytest.mark.gpu
SPECIAL = [0.0, -0.0, 1.0, -1.0, 0.5, 2.5, -3.25, np.inf, -np.inf, np.nan, 1e-45, -1e-45, 3e-39,
           -7e-39, 1.2e-38, 1e-30, -2e-30, 1e-23, -1e-22, 1e19, -2e20, 3e38, -3.4e38, 1e-7]


def limited(x, y):
    with np.errstate(all="ignore"):
        p = x.astype(np.float64) * y.astype(np.float64)      # exact: 48 bits, no underflow
        return np.where(p <= 0, np.float32(0), np.where(np.abs(x) < np.abs(y), x, y))


def fields():
    s = np.array(SPECIAL, dtype=np.float32)
    n = len(s)
    rng = np.random.default_rng(7)
    a = np.tile(s[:, None], (4, 3 * n))
    b = np.tile(s[None, :], (4 * n, 3))
    c = rng.permutation(np.resize(s, a.size)).reshape(a.shape)
    d = rng.permutation(np.resize(s, a.size)).reshape(a.shape)
    rest = rng.standard_normal((4, 3 * n, a.shape[1])).astype(np.float32)
    return [np.concatenate([x, y]) for x, y in zip((a, b, c, d), rest)]


def test_special_values(require_gpu):
    print("fast FP32 rewrites", flush=True)
    ins = fields()
    shape = ins[0].shape
    got = {}
    for v in ("rewrites_f32", "rewrites_f32_tiles"):
        m = variants.machine(v, shape[::-1])
        for name, x in zip("abcd", ins):
            m.set(name, x)
        m.run("apply")
        got[v] = {o: m.get(o) for o in OUT}
    a, b = ins[:2]
    fast, tiles = got["rewrites_f32"], got["rewrites_f32_tiles"]
    assert np.array_equal(fast["limited"], limited(a, b), equal_nan=True)
    assert np.array_equal(fast["shifted"], limited(a, np.roll(b, -1, 1)), equal_nan=True)
    for o in OUT[2:]:
        assert np.array_equal(fast[o], tiles[o], equal_nan=True), o
