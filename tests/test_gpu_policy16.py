"""GPU: the policy step gives a row the same action, log-probability, value and stored observation, bit for bit, whether its
batch goes through the 16-row tiles (few rows) or the 32-row tiles (many)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

BIG = 9001      # beyond what the 16-row tiles take at any hidden width


@pytest.mark.parametrize("H, n", [(H, n) for H in (64, 128, 256) for n in (1, 15, 16, 17, 33, 1000)] +
                         [(64, 8192), (64, 8193), (128, 4096), (128, 4097), (256, 2048), (256, 2049)])
@pytest.mark.parametrize("env", ["CartPoleEnv", "LunarLanderV2", "PendulumV2", "BipedalWalkerV2", "HalfCheetahPlanarV2"])
def test_small_batch_equals_rows_of_a_large_one(mrl, env, H, n):
    E = getattr(mrl, env)
    ctx = mrl.DeviceContext("cuda:0")
    lay = mrl.LinearReLU if E.NUM_ACTIONS else mrl.LinearTanh
    head = mrl.Linear(H, E.NUM_ACTIONS) if E.NUM_ACTIONS else mrl.StochasticActor(H, E.ACTION_DIM)
    actor = mrl.seq(lay(E.OBS_DIM, H), lay(H, H), head)
    critic = mrl.seq(lay(E.OBS_DIM, H), lay(H, H), mrl.Linear(H, 1))
    g = torch.Generator(device="cuda").manual_seed(n + H)
    rnd = lambda k, s: (torch.rand(k, device="cuda", generator=g) - 0.5) * 2 * s
    pa, pc, obs = rnd(actor.PARAM_SIZE, 0.2), rnd(critic.PARAM_SIZE, 0.2), rnd(BIG * E.OBS_DIM, 2.0)
    out = []
    for rows in (n, BIG):
        rb = mrl.ppo.RolloutBuffers(ctx, E, actor, critic, rows, 1)
        rb.actor_params, rb.critic_params = pa, pc
        rb.obs.copy_(obs[:rows * E.OBS_DIM])
        actions = torch.full((rows * rb.act_width,), 9.0, device="cuda")
        mrl.ppo.policy_step(ctx, rb, 0, 77, actions)
        out.append([t.view(rows, -1)[:n].clone() for t in (actions, rb.r_obs, rb.r_actions, rb.r_log_probs, rb.r_values)])
    ctx.synchronize()
    for a, b in zip(*out):
        assert torch.equal(a, b)
