"""GPU: an epoch in which the KL stop fires part of the way through leaves, in every buffer that the caller can see, what the
same minibatches leave one call at a time (where each is computed): parameters, optimiser state, gradients, outputs, loss
gradients, KL estimates and the flag words, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_mb", [1, 2, 7])
@pytest.mark.parametrize("H", [64, 128, 256])
@pytest.mark.parametrize("cont", [False, True], ids=["discrete", "continuous"])
def test_epoch_equals_single_minibatches_across_the_stop(mrl, cont, H, n_mb):
    ctx = mrl.DeviceContext("cuda:0")
    E = mrl.HalfCheetahPlanarV2 if cont else mrl.LunarLanderV2
    A = E.ACTION_DIM if cont else E.NUM_ACTIONS
    lay = mrl.LinearTanh if cont else mrl.LinearReLU
    actor = mrl.seq(lay(E.OBS_DIM, H), lay(H, H), mrl.StochasticActor(H, A) if cont else mrl.Linear(H, A))
    critic = mrl.seq(lay(E.OBS_DIM, H), lay(H, H), mrl.Linear(H, 1))
    N, T, MB = 100, 7, 100
    total = N * T
    g = torch.Generator(device="cuda").manual_seed(5 + H)
    rnd = lambda n, s: (torch.rand(n, device="cuda", generator=g) - 0.5) * 2 * s
    params = rnd(actor.PARAM_SIZE, 0.1), rnd(critic.PARAM_SIZE, 0.1)
    obs, lp, val, adv, ret = rnd(total * E.OBS_DIM, 1), rnd(total, 0.02) - 1.4, rnd(total, 1), rnd(total, 1), rnd(total, 1)
    acts = rnd(total * A, 1) if cont else torch.randint(0, A, (total,), device="cuda", generator=g).float()
    perm = torch.randperm(total, device="cuda", generator=g).to(torch.int32)[:n_mb * MB].contiguous()

    def build(target):
        rb = mrl.ppo.RolloutBuffers(ctx, E, actor, critic, N, T)
        rb.actor_params, rb.critic_params = params[0].clone(), params[1].clone()
        for dst, src in ((rb.r_obs, obs), (rb.r_actions, acts), (rb.r_log_probs, lp), (rb.r_values, val)):
            dst.copy_(src)
        cls = mrl.ppo.ContinuousUpdate if cont else mrl.ppo.DiscreteUpdate
        upd = cls(ctx, rb, MB, mrl.Adam(lr=1e-2), mrl.Adam(lr=1e-2), target_kl=target)
        upd.advantages.copy_(adv)
        upd.returns.copy_(ret)
        upd.reset_kl()
        return rb, upd

    # a target between the mean KLs of the first minibatches, taken from a run that never stops
    _, probe = build(1e30)
    means = []
    for k in range(n_mb):
        probe.minibatch_step(perm[k * MB:(k + 1) * MB])
        means.append(float(probe.kl_flag.cpu()[1:2].view(torch.float32)))
    target = max(1e-6, 0.5 * (max(means[:3]) + min(means[:3])))
    (rb1, one), (rb2, whole) = build(target), build(target)
    for k in range(n_mb):
        one.minibatch_step(perm[k * MB:(k + 1) * MB])
    whole.run_epoch(perm)
    ctx.synchronize()
    if n_mb == 7:
        assert int(one.kl_flag[0]) == 1 and int(one.kl_flag[2]) < n_mb - 1
    assert torch.equal(rb1.actor_params, rb2.actor_params) and torch.equal(rb1.critic_params, rb2.critic_params)
    for name in ("kl_flag", "actor_state", "critic_state", "actor_grads", "critic_grads", "kl", "g_actor_out", "g_values",
                 "actor_out", "values"):
        assert torch.equal(getattr(one, name), getattr(whole, name)), name
