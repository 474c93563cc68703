"""normalize_advantages on buffers on and off 16 bytes, sizes around a 16-byte piece, a block and the grid, values far from
zero, a first value far from the others, all values alike, and values that are not finite."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("off", [0, 1, 3])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 1023, 1025, 131072 * 4 - 1, 131072 * 4 + 1, 4 * 131072 * 4 + 5])
@pytest.mark.parametrize("mean, first", [(1.5, None), (3000.0, None), (0.0, 1e4)])
def test_against_float64(mrl, n, off, mean, first):
    ctx = mrl.DeviceContext("cuda:0")
    a = np.random.default_rng(n + off).normal(mean, 2.5, n).astype(np.float32)
    if first is not None:
        a[0] = first
    buf = torch.full((n + off + 4,), 7.0, device="cuda")
    buf[off:off + n] = torch.from_numpy(a).cuda()
    mrl.ppo.normalize_advantages(ctx, buf[off:off + n])
    ctx.synchronize()
    a64 = a.astype(np.float64)
    den = np.sqrt(a64.var() + 1e-8) + 1e-8
    want = (a64 - a64.mean()) / den
    # the fp32 mean is off by 2^-25 |mean| (a little where the Float64 sums round), x - mean by 2^-24 |x - mean|, the square
    # root, its two sums and the quotient by 2^-24 each of the result
    got = buf[off:off + n].cpu().numpy()
    bound = 2.0 ** -24 * abs(a64.mean()) / den + 8 * 2.0 ** -24 * np.abs(want) + 1e-12
    assert (np.abs(got - want) <= bound).all()
    assert (buf[:off] == 7.0).all() and (buf[off + n:] == 7.0).all()


@pytest.mark.parametrize("n", [1, 6, 70000])
def test_equal_values_give_zero(mrl, n):
    ctx = mrl.DeviceContext("cuda:0")
    x = torch.full((n,), 0.1, device="cuda")
    mrl.ppo.normalize_advantages(ctx, x)
    ctx.synchronize()
    assert (x == 0).all()


@pytest.mark.parametrize("at", [0, 5])
def test_an_infinity_makes_all_nan(mrl, at):
    ctx = mrl.DeviceContext("cuda:0")
    x = torch.arange(40, device="cuda", dtype=torch.float32)
    x[at] = float("inf")
    mrl.ppo.normalize_advantages(ctx, x)
    ctx.synchronize()
    assert torch.isnan(x).all()
