"""The library's own sine, cosine and logarithm of fp32 values against the host's Float64 functions, rounded: every exponent,
both sides of the switch of reductions at 2^20 (also in one wavefront), the neighbours of multiples of pi / 2 and of 1, the
argument closest to a tie, subnormals, infinities and NaN."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def device(mrl, x, want):
    ctx = mrl.DeviceContext("cuda:0")
    d = torch.from_numpy(x).cuda()
    out = [torch.full_like(d, 7.0) if w else None for w in want]
    mrl._lib.call("mrl_math32", ctx.handle, d.data_ptr(), d.numel(), *[None if o is None else o.data_ptr() for o in out])
    ctx.synchronize()
    return [None if o is None else o.cpu().numpy() for o in out]


def rounded(f, x):
    return np.array([f(v) for v in x.astype(np.float64).tolist()]).astype(np.float32)


def every_exponent(rng, per):
    m = rng.integers(0, 1 << 23, (255, per), dtype=np.uint32) | (np.arange(255, dtype=np.uint32)[:, None] << 23)
    m[:, 0] &= 0xFF800000
    m[:, 1] |= 0x007FFFFF
    return m.reshape(-1).view(np.float32)


def neighbours(x, k=3):
    b = x.astype(np.float32).view(np.int32)
    return np.concatenate([(b + i).view(np.float32) for i in range(-k, k + 1)])


def angles():
    rng = np.random.default_rng(1)
    q = np.concatenate([np.arange(1, 2000), rng.integers(1, 1 << 53, 3000)]) * (math.pi / 2)
    x = np.concatenate([every_exponent(rng, 1500), neighbours(q), neighbours(np.array([2.0 ** 20, 2.0 ** 23, 2.0 ** 24]), 200),
                        np.array([0x5922AA80], np.uint32).view(np.float32)])
    return np.where(rng.random(x.size) < 0.5, x, -x).astype(np.float32)


@pytest.mark.parametrize("order", ["mixed", "sorted"])   # near and far angles in one wavefront, and wavefronts of one kind
def test_sine_and_cosine(mrl, order):
    print("math32 angles", order, flush=True)
    x = angles()
    x = np.sort(x) if order == "sorted" else np.random.default_rng(2).permutation(x)
    s, c, _ = device(mrl, x, (1, 1, 0))
    np.testing.assert_array_equal(s, rounded(math.sin, x))
    np.testing.assert_array_equal(c, rounded(math.cos, x))


def test_angles_without_a_sine(mrl):
    x = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1.0, 1e30, -1e-45] * 9, np.float32)
    s, c, _ = device(mrl, x, (1, 1, 0))
    ok = np.isfinite(x)
    assert np.isnan(s[~ok]).all() and np.isnan(c[~ok]).all()
    np.testing.assert_array_equal(s[ok].view(np.uint32), rounded(math.sin, x[ok]).view(np.uint32))   # (the sign of zero too)
    np.testing.assert_array_equal(c[ok], rounded(math.cos, x[ok]))


def test_logarithm(mrl):
    print("math32 log", flush=True)
    rng = np.random.default_rng(3)
    x = np.concatenate([every_exponent(rng, 3000), neighbours(np.array([1.0, 0.5, 2.0, math.sqrt(0.5), math.sqrt(2.0)]), 500)])
    x = x[x > 0]
    _, _, l = device(mrl, np.concatenate([x, np.array([0.0, -0.0, -1.0, -1e-45, np.inf, -np.inf, np.nan], np.float32)]), (0, 0, 1))
    np.testing.assert_array_equal(l[:x.size], rounded(math.log, x))
    np.testing.assert_array_equal(l[x.size:], np.array([-np.inf, -np.inf, np.nan, np.nan, np.inf, np.nan, np.nan], np.float32))
