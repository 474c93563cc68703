"""compute_gae where an episode's end meets values that are not finite, and zeros: the sum restarts there as if nothing had
come after, whatever had."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,N", [(16, 16), (65, 33), (130, 100), (64, 4097), (70, 9000)])
def test_gae_restarts_at_episode_ends(mrl, orc, T, N):
    print("gae restarts", T, N, flush=True)
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
    orc.orc_gae(T, N, r, v, d, boot, 0.99, 0.95, adv_h, ret_h)
    dev = lambda a: torch.from_numpy(a).cuda()
    adv, ret = torch.zeros(T * N, device="cuda"), torch.zeros(T * N, device="cuda")
    mrl.ppo.compute_gae(ctx, dev(r), dev(v), dev(d), dev(boot), 0.99, 0.95, adv, ret)
    ctx.synchronize()
    np.testing.assert_array_equal(adv.cpu().numpy(), adv_h)      # same fp32 operations in the same order; NaN equals NaN
    np.testing.assert_array_equal(ret.cpu().numpy(), ret_h)
    assert np.isfinite(adv_h).any() and np.isnan(adv_h).any()
