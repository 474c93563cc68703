"""The fused CartPole and Pendulum kernels over launches long enough that a workgroup hands over its finished episodes several
times, and with a list too short for them."""
import pytest
import torch

import test_gpu_collect
from test_gpu_collect import ctx, mrl  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("env,N,T,hidden,kind", [
    ("cartpole", 33, 300, 64, "relu"), ("cartpole", 16, 201, 64, "tanh"), ("cartpole", 17, 300, 128, "tanh"), ("cartpole", 15, 200, 256, "relu"),
    ("cartpole", 1, 1, 64, "relu"), ("cartpole", 32769, 3, 64, "relu"), ("pendulum", 20, 410, 64, "tanh"), ("pendulum", 1, 1, 64, "relu"),
    ("pendulum", 31, 205, 128, "relu"), ("pendulum", 32769, 3, 64, "tanh"),
])
def test_long_launches_equal_single_steps(mrl, ctx, env, N, T, hidden, kind):  # noqa: F811
    E = {"cartpole": mrl.CartPoleEnv, "pendulum": mrl.PendulumV2}[env]
    lay = mrl.LinearReLU if kind == "relu" else mrl.LinearTanh
    head = mrl.Linear(hidden, 2) if env == "cartpole" else mrl.StochasticActor(hidden, 1)
    actor = mrl.seq(lay(E.OBS_DIM, hidden), lay(hidden, hidden), head)
    critic = mrl.seq(lay(E.OBS_DIM, hidden), lay(hidden, hidden), mrl.Linear(hidden, 1))
    g = torch.Generator().manual_seed(5)
    pa, pc = ((torch.rand(m.PARAM_SIZE, generator=g) - 0.5).mul_(0.3).cuda() for m in (actor, critic))
    cap = max(1, N * T // 64)     # a third of CartPole's episodes, or fewer
    both = []
    for fused in (True, False):
        rb = mrl.ppo.RolloutBuffers(ctx, E, actor, critic, N, T, done_cap=cap if N < 1000 else None)
        rb.actor_params, rb.critic_params = pa, pc
        if env == "cartpole":
            rb.keep = torch.zeros(N, dtype=torch.int32, device="cuda")
            E.bind_step_counters(ctx, rb.states, rb.keep)
        E.reset_kernel_gpu(ctx, rb.states, 3)
        rb.obs.copy_(rb.states.view(N, E.STATE_SIZE)[:, :E.OBS_DIM].reshape(-1))
        d = rb.descriptor()
        if fused:
            assert mrl.ppo.rollout_fused(d) == 1
            mrl.ppo.rollout_steps(ctx, d, 0, T, 11, 7919, 0, 0, 17, 104729)
        else:
            for t in range(T):
                mrl.ppo.rollout_step(ctx, d, t, 11 + 7919 * t, 0, 17 + 104729 * t)
        ctx.synchronize()
        both.append(rb)
    one, many = both
    for name in ("states", "obs", "r_obs", "r_actions", "r_log_probs", "r_values", "r_rewards", "r_dones", "ep_return", "ep_length"):
        assert torch.equal(getattr(one, name), getattr(many, name)), name
    if env == "cartpole":
        assert torch.equal(one.keep, many.keep)
    count = int(many.done_count.item())
    assert int(one.done_count.item()) == count and (T < 200 or count >= N)
    # the list: as many entries as fit, every one an episode of this rollout
    dones, rewards = (x.view(T, N).cpu() for x in (one.r_dones, one.r_rewards))
    ends, total, length = [], torch.zeros(N), torch.zeros(N)
    for t in range(T):
        total, length = total + rewards[t], length + 1
        for e in torch.nonzero(dones[t] > 0.5).flatten().tolist():
            ends.append((total[e].item(), length[e].item()))
            total[e] = length[e] = 0
    assert len(ends) == count
    got = list(zip(one.done_returns[:min(count, one.done_cap)].tolist(), one.done_lengths[:min(count, one.done_cap)].tolist()))
    for entry in got:
        ends.remove(entry)
    if one.done_cap > count:
        assert not ends and not one.done_lengths[count:].any()
