"""GPU: an update of many minibatches whose KL stop fires early leaves launches away once the host has seen the stop.  What it
leaves in the caller's buffers is what the same minibatches leave one call at a time, also where the last minibatch's
advantage statistics are of another launch than the first's, and a stop reported for one call ends no other."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_mb", [40, 2049, 2100])
def test_long_epochs_behind_the_stop(mrl, n_mb):
    print("long epoch", n_mb, flush=True)
    ctx = mrl.DeviceContext("cuda:0")
    E, H, A, MB = mrl.CartPoleEnv, 64, 2, 16
    actor = mrl.seq(mrl.LinearReLU(4, H), mrl.LinearReLU(H, H), mrl.Linear(H, A))
    critic = mrl.seq(mrl.LinearReLU(4, H), mrl.LinearReLU(H, H), mrl.Linear(H, 1))
    total = n_mb * MB
    g = torch.Generator(device="cuda").manual_seed(n_mb)
    rnd = lambda n, s: (torch.rand(n, device="cuda", generator=g) - 0.5) * 2 * s
    params = rnd(actor.PARAM_SIZE, 0.1), rnd(critic.PARAM_SIZE, 0.1)
    data = rnd(total * 4, 1), torch.randint(0, A, (total,), device="cuda", generator=g).float(), rnd(total, 0.02) - 0.7, rnd(total, 1)
    adv, ret = rnd(total, 1), rnd(total, 1)
    perm = torch.randperm(total, device="cuda", generator=g).to(torch.int32)

    def build(target):
        rb = mrl.ppo.RolloutBuffers(ctx, E, actor, critic, MB, n_mb)
        rb.actor_params, rb.critic_params = params[0].clone(), params[1].clone()
        for dst, src in zip((rb.r_obs, rb.r_actions, rb.r_log_probs, rb.r_values), data):
            dst.copy_(src)
        upd = mrl.ppo.DiscreteUpdate(ctx, rb, MB, mrl.Adam(lr=1e-2), mrl.Adam(lr=1e-2), target_kl=target)
        upd.advantages.copy_(adv)
        upd.returns.copy_(ret)
        upd.reset_kl()
        return rb, upd

    def same(one, whole, rb1, rb2):
        ctx.synchronize()
        assert torch.equal(rb1.actor_params, rb2.actor_params) and torch.equal(rb1.critic_params, rb2.critic_params)
        for name in ("kl_flag", "actor_state", "critic_state", "actor_grads", "critic_grads", "kl", "g_actor_out", "g_values",
                     "actor_out", "values"):
            assert torch.equal(getattr(one, name), getattr(whole, name)), name

    (rb1, one), (rb2, whole) = build(1e-4), build(1e-4)
    for k in range(n_mb):
        one.minibatch_step(perm[k * MB:(k + 1) * MB])
    assert whole.run_epoch(perm)[0]
    assert int(one.kl_flag[0]) == 1 and int(one.kl_flag[2]) < n_mb // 2
    same(one, whole, rb1, rb2)
    # the stop still raised: nothing is applied; then cleared and out of reach: every minibatch is
    assert whole.run_epoch(perm)[0]
    for k in range(n_mb):
        one.minibatch_step(perm[k * MB:(k + 1) * MB])
    same(one, whole, rb1, rb2)
    for u in (one, whole):
        u.actor_opt.t = u.critic_opt.t = 0
        u.target_kl = 1e30
        u.reset_kl()
    for k in range(n_mb):
        one.minibatch_step(perm[k * MB:(k + 1) * MB])
    whole.run_epoch(perm)
    assert int(whole.kl_flag[2]) == n_mb
    same(one, whole, rb1, rb2)
