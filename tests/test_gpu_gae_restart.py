"""compute_gae where an episode's end meets values that are not finite, and zeros: the sum restarts there as if nothing had
come after, whatever had."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# (the last two pairs: a decay of zero, which keeps an infinity of a later step as NaN, and an infinite one; N = 16385: the
# plain scan, one lane per env)
@pytest.mark.parametrize("gamma,lam", [(0.99, 0.95), (0.99, 0.0), (0.0, 0.95), (1e20, 1e20)])
@pytest.mark.parametrize("T,N", [(16, 16), (65, 33), (130, 100), (64, 4097), (70, 9000), (40, 16385)])
def test_gae_restarts_at_episode_ends(mrl, orc, T, N, gamma, lam):
    print("gae restarts", T, N, gamma, lam, flush=True)
    ctx = mrl.DeviceContext("cuda:0")
    rng = np.random.default_rng(T + N)
    r, v = rng.normal(size=(T, N)).astype(np.float32), rng.normal(size=(T, N)).astype(np.float32)
    odd = np.array([np.inf, -np.inf, np.nan, 0.0, -0.0, 3.0e38], np.float32)
    hit = rng.random((T, N)) < 0.1
    r[hit] = rng.choice(odd, hit.sum())
    d = np.where(rng.random((T, N)) < 0.3, 1.0, rng.choice(np.array([0.0, 0.5, 0.25], np.float32), (T, N))).astype(np.float32)
    boot = rng.choice(odd, N).astype(np.float32)
    r, v, d = r.reshape(-1), v.reshape(-1), d.reshape(-1)
    adv_h, ret_h = np.zeros(T * N, np.float32), np.zeros(T * N, np.float32)
    orc.orc_gae(T, N, r, v, d, boot, gamma, lam, adv_h, ret_h)
    dev = lambda a: torch.from_numpy(a).cuda()
    adv, ret = torch.zeros(T * N, device="cuda"), torch.zeros(T * N, device="cuda")
    mrl.ppo.compute_gae(ctx, dev(r), dev(v), dev(d), dev(boot), gamma, lam, adv, ret)
    ctx.synchronize()
    np.testing.assert_array_equal(adv.cpu().numpy(), adv_h)      # same fp32 operations in the same order; NaN equals NaN
    np.testing.assert_array_equal(ret.cpu().numpy(), ret_h)
    assert np.isnan(adv_h).any() and (gamma > 1 or np.isfinite(adv_h).any())   # (an infinite decay: NaN from the first step on)


@pytest.mark.parametrize("N", [33, 4097, 16385])
def test_gae_of_subnormal_values(mrl, orc, N):
    """Values and products below the smallest normal float are kept."""
    print("gae subnormal", N, flush=True)
    ctx, T = mrl.DeviceContext("cuda:0"), 70
    rng = np.random.default_rng(N)
    r, v = ((rng.normal(size=T * N) * 1e-39).astype(np.float32) for _ in range(2))
    d, boot = (rng.random(T * N) < 0.1).astype(np.float32), (rng.normal(size=N) * 1e-39).astype(np.float32)
    adv_h, ret_h = np.zeros(T * N, np.float32), np.zeros(T * N, np.float32)
    orc.orc_gae(T, N, r, v, d, boot, 0.99, 0.95, adv_h, ret_h)
    dev = lambda a: torch.from_numpy(a).cuda()
    adv, ret = torch.zeros(T * N, device="cuda"), torch.zeros(T * N, device="cuda")
    mrl.ppo.compute_gae(ctx, dev(r), dev(v), dev(d), dev(boot), 0.99, 0.95, adv, ret)
    ctx.synchronize()
    np.testing.assert_array_equal(adv.cpu().numpy(), adv_h)
    np.testing.assert_array_equal(ret.cpu().numpy(), ret_h)
    assert (np.abs(adv_h) < 1e-37).all() and (adv_h != 0).mean() > 0.99
