"""GPU: an update of many minibatches whose KL stop fires early leaves launches away once the host has seen the stop.  What it
leaves in the caller's buffers is what the same minibatches leave one call at a time, also where the last minibatch's
advantage statistics are of another launch than the first's, and a stop reported for one call ends no other.  A captured
update records every minibatch."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


MB = 16


def case(mrl, n_mb, ctx=None):
    """(build, same, perm) of n_mb minibatches over fixed data: build(target_kl) makes buffers and an update, same(...) compares
    what two of them have left."""
    ctx = ctx or mrl.DeviceContext("cuda:0")
    E, H, A = mrl.CartPoleEnv, 64, 2
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

    return build, same, perm


@pytest.mark.parametrize("n_mb", [40, 2049, 2100])
def test_long_epochs_behind_the_stop(mrl, n_mb):
    print("long epoch", n_mb, flush=True)
    ctx = mrl.DeviceContext("cuda:0")
    build, same, perm = case(mrl, n_mb, ctx)
    (rb1, one), (rb2, whole) = build(0.05), build(0.05)   # (reached within the first ten minibatches, but not at once)
    for k in range(n_mb):
        one.minibatch_step(perm[k * MB:(k + 1) * MB])
        assert ctx.update_enqueued() == 1
    assert whole.run_epoch(perm)[0]
    # (enqueueing 2048 minibatches takes the host over ten milliseconds, the device reports within one: the jump goes into
    # the second launch of advantage statistics, minibatches 2048 and on)
    assert ctx.update_enqueued() <= n_mb if n_mb < 1000 else ctx.update_enqueued() <= 2048
    assert int(one.kl_flag[0]) == 1 and 0 < int(one.kl_flag[2]) < n_mb // 2
    same(one, whole, rb1, rb2)
    # the stop still raised: nothing is applied; then cleared and out of reach: every minibatch is
    assert whole.run_epoch(perm)[0]
    assert 1 <= ctx.update_enqueued() <= min(n_mb, 2048)
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
    assert int(whole.kl_flag[2]) == n_mb and ctx.update_enqueued() == n_mb
    same(one, whole, rb1, rb2)


def test_captured_update_records_every_minibatch(mrl):
    print("captured update", flush=True)
    n_mb, side = 60, torch.cuda.Stream()
    ctx, gctx = mrl.DeviceContext("cuda:0"), mrl.DeviceContext("cuda:0", stream=side)
    build, same, perm = case(mrl, n_mb, ctx)
    gbuild, _, _ = case(mrl, n_mb, gctx)
    (rb1, one), (rb2, rec) = build(0.05), gbuild(0.05)
    torch.cuda.synchronize()

    def epoch(u):   # (run_epoch without its look at the flag)
        d = u.descriptor()
        mrl._lib.call("mrl_ppo_update_epoch", u.ctx.handle, ctypes.byref(d), perm.data_ptr(), n_mb, 0, 0)

    names = ("kl_flag", "actor_state", "critic_state")
    first = [rb2.actor_params.clone(), rb2.critic_params.clone()] + [getattr(rec, n).clone() for n in names]
    epoch(rec)          # (the workspaces are there before the capture)
    gctx.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        epoch(rec)
    assert gctx.update_enqueued() == n_mb
    for replay in range(3):
        for rb, u in ((rb1, one), (rb2, rec)):
            for dst, src in zip([rb.actor_params, rb.critic_params] + [getattr(u, n) for n in names], first):
                dst.copy_(src)
        torch.cuda.synchronize()
        epoch(one)      # eager work of another context between the replays, with a stop of its own
        ctx.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert int(one.kl_flag[0]) == 1 and 0 < int(one.kl_flag[2]) < n_mb, replay
        same(one, rec, rb1, rb2)
    del graph
    gctx.close()
    ctx.close()


@pytest.mark.parametrize("busy", [False, True])
def test_the_host_stays_a_few_minibatches_ahead(mrl, busy):
    """What is enqueued behind the stop is a few minibatches; and where the device does not come to the update for longer than
    the host waits, all of them are, with the same results."""
    print("ahead", busy, flush=True)
    n_mb, ctx = 400, mrl.DeviceContext("cuda:0")
    build, same, perm = case(mrl, n_mb, ctx)
    (rb1, one), (rb2, whole) = build(0.05), build(0.05)
    for k in range(n_mb):
        one.minibatch_step(perm[k * MB:(k + 1) * MB])
    ctx.synchronize()
    if busy:
        filler = torch.zeros(1 << 28, device="cuda")
        for _ in range(400):        # 2 GiB of traffic each, a third of a millisecond and more
            filler.add_(1.0)
    assert whole.run_epoch(perm)[0]
    applied = int(whole.kl_flag[2])
    assert 0 < applied < n_mb // 2
    # the minibatch that raised the stop, the six that the host may be ahead, the one that it was about to enqueue, the last
    assert ctx.update_enqueued() <= (n_mb if busy else applied + 9)
    same(one, whole, rb1, rb2)
