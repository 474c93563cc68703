"""compute_gae at the edges of its groups of envs and chunks of steps; normalize_advantages at sizes of a
hundred thousand values and more."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(mrl):
    return mrl.DeviceContext("cuda:0")


def d(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# groups of 16, 32 and 64 envs (chunks of 64, 64 and 32 steps), the plain scan: one below, at and above a chunk, ragged last groups,
# the last N of a group width and the first of the next on 256 CUs (plain from 16385)
@pytest.mark.parametrize("T,N", [(63, 15), (64, 16), (65, 17), (513, 33), (3, 4096), (127, 4097), (64, 5000),
                                 (129, 8192), (31, 8193), (32, 9000), (33, 8256), (65, 16384), (17, 16385), (65, 20001)])
@pytest.mark.parametrize("in_place", [False, True])
def test_gae_chunks(mrl, orc, ctx, T, N, in_place):
    print("gae chunks", T, N, in_place, flush=True)
    rng = np.random.default_rng(T * 7 + N)
    r, v = rng.normal(size=T * N).astype(np.float32), rng.normal(size=T * N).astype(np.float32)
    dn, boot = (rng.random(T * N) < 0.02).astype(np.float32), rng.normal(size=N).astype(np.float32)
    adv_h, ret_h = np.zeros(T * N, np.float32), np.zeros(T * N, np.float32)
    orc.orc_gae(T, N, r, v, dn, boot, 0.99, 0.95, adv_h, ret_h)
    rd, vd = d(r), d(v)
    adv, ret = (rd, vd) if in_place else (torch.zeros_like(rd), torch.zeros_like(vd))
    mrl.ppo.compute_gae(ctx, rd, vd, d(dn), d(boot), 0.99, 0.95, adv, ret)
    ctx.synchronize()
    np.testing.assert_array_equal(adv.cpu().numpy(), adv_h)      # same fp32 operations in the same order
    np.testing.assert_array_equal(ret.cpu().numpy(), ret_h)


@pytest.mark.parametrize("n", [255, 257, 262144, 4 * 262144 - 1, 4 * 262144 + 3, 5 * 262144])
def test_normalize_blocks(mrl, ctx, n):
    a = np.random.default_rng(n).normal(1.5, 2.5, n).astype(np.float32)
    a64 = a.astype(np.float64)
    want = (a64 - a64.mean()) / (np.sqrt(a64.var() + 1e-8) + 1e-8)
    x = d(a)
    mrl.ppo.normalize_advantages(ctx, x)
    ctx.synchronize()
    # sums in Float64; the fp32 mean is off by 2^-25 |mean|, and x - mean, the variance's root, its two sums and the quotient
    # by 2^-24 each of the result (test_gpu_normalize.py takes the pieces, blocks and grid apart)
    den = np.sqrt(a64.var() + 1e-8) + 1e-8
    bound = 2.0 ** -24 * abs(a64.mean()) / den + 8 * 2.0 ** -24 * np.abs(want) + 1e-12
    assert (np.abs(x.cpu().numpy() - want) <= bound).all()
