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


@pytest.mark.parametrize("H", [64, 128, 256])
@pytest.mark.parametrize("cont", [False, True], ids=["discrete", "continuous"])
def test_the_stop_of_a_minibatch_holds_for_every_workgroup_of_its_own_update(mrl, cont, H):
    """The launch that would apply a minibatch is the one that raises the flag.  None of its workgroups may take part of the
    update, whichever of them runs late: other work shares the chip, and parameters and moments must not move by a bit."""
    ctx = mrl.DeviceContext("cuda:0")
    E = mrl.HalfCheetahPlanarV2 if cont else mrl.LunarLanderV2
    A = E.ACTION_DIM if cont else E.NUM_ACTIONS
    lay = mrl.LinearTanh if cont else mrl.LinearReLU
    actor = mrl.seq(lay(E.OBS_DIM, H), lay(H, H), mrl.StochasticActor(H, A) if cont else mrl.Linear(H, A))
    critic = mrl.seq(lay(E.OBS_DIM, H), lay(H, H), mrl.Linear(H, 1))
    N, T = 97, 5
    g = torch.Generator(device="cuda").manual_seed(H)
    rb = mrl.ppo.RolloutBuffers(ctx, E, actor, critic, N, T)
    rb.actor_params = (torch.rand(actor.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.2
    rb.critic_params = (torch.rand(critic.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.2
    rb.r_obs.normal_(generator=g)
    if not cont:
        rb.r_actions.copy_(torch.randint(0, A, (N * T,), device="cuda", generator=g).float())
    rb.r_log_probs.fill_(9.0)                                  # a mean KL far above any target
    cls = mrl.ppo.ContinuousUpdate if cont else mrl.ppo.DiscreteUpdate
    upd = cls(ctx, rb, N * T, mrl.Adam(lr=1e-2), mrl.Adam(lr=1e-2), target_kl=0.01)
    upd.advantages.normal_(generator=g)
    upd.returns.normal_(generator=g)
    upd.actor_state.uniform_(generator=g)
    upd.critic_state.uniform_(generator=g)
    kept = [t.clone() for t in (rb.actor_params, rb.critic_params, upd.actor_state, upd.critic_state)]
    perm = torch.randperm(N * T, device="cuda", generator=g).to(torch.int32)
    side, filler = torch.cuda.Stream(), torch.zeros(1 << 24, device="cuda")
    side.wait_stream(torch.cuda.current_stream())
    for k in range(20):
        with torch.cuda.stream(side):
            for _ in range(4):
                filler.add_(1.0)
        upd.reset_kl()
        upd.minibatch_step(perm)
        ctx.synchronize()
        assert upd.kl_flag.tolist()[0] == 1 and upd.kl_flag.tolist()[2] == 0
        for was, now in zip(kept, (rb.actor_params, rb.critic_params, upd.actor_state, upd.critic_state)):
            assert torch.equal(was, now), k
    side.synchronize()
