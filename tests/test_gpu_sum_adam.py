"""The update whose sums, clip and Adam are one launch against the two launches that a stream with few CUs takes, at sizes where
the workgroups' shares end unevenly; and the one launch's wait, which no other work on the device can keep from ending."""
import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def build(mrl, ctx, E, H, MB, target, max_norm=0.5):
    A = E.ACTION_DIM if E.ACTION_DIM else E.NUM_ACTIONS
    lay = mrl.LinearTanh if E.ACTION_DIM else mrl.LinearReLU
    head = mrl.StochasticActor(H, A) if E.ACTION_DIM else mrl.Linear(H, A)
    actor = mrl.seq(lay(E.OBS_DIM, H), lay(H, H), head)
    critic = mrl.seq(lay(E.OBS_DIM, H), lay(H, H), mrl.Linear(H, 1))
    g = torch.Generator(device="cuda").manual_seed(H + MB)
    n = 3 * MB
    rb = mrl.ppo.RolloutBuffers(ctx, E, actor, critic, MB, 3)
    rb.actor_params = (torch.rand(actor.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.2
    rb.critic_params = (torch.rand(critic.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.2
    rb.r_obs.normal_(generator=g)
    # about what these policies give, so that not every sample is clipped
    rb.r_log_probs.normal_(mean=-1.4 * A if E.ACTION_DIM else -math.log(A), std=0.1, generator=g)
    if E.ACTION_DIM:
        rb.r_actions.normal_(generator=g)
    else:
        rb.r_actions.copy_(torch.randint(0, A, (n,), device="cuda", generator=g).float())
    upd = mrl.ppo.PPOUpdate(ctx, rb, MB, mrl.Adam(lr=1e-3), mrl.Adam(lr=1e-3), target_kl=target, max_grad_norm=max_norm)
    upd.advantages.normal_(generator=g)
    upd.returns.normal_(generator=g)
    perm = torch.randperm(n, device="cuda", generator=g).to(torch.int32)
    torch.cuda.synchronize()
    return rb, upd, perm


def masked_stream(cus):
    hip = ctypes.CDLL("libamdhip64.so")     # the runtime that torch has loaded
    mask = (ctypes.c_uint32 * 8)(*[(1 << min(32, max(0, cus - 32 * k))) - 1 for k in range(8)])
    s = ctypes.c_void_p()
    assert hip.hipExtStreamCreateWithCUMask(ctypes.byref(s), 8, mask) == 0
    return torch.cuda.ExternalStream(s.value)


@pytest.mark.parametrize("env,H,MB", [("CartPoleEnv", 64, 2), ("PendulumV2", 64, 257), ("LunarLanderV2", 128, 1000),
                                      ("Walker2dPlanar", 128, 2100), ("HopperPlanar", 256, 17), ("BipedalWalkerV2", 256, 1050),
                                      ("BipedalWalkerV2", 256, 4100)])
@pytest.mark.parametrize("target,max_norm", [(0.0, 0.5), (1e30, 0.5), (0.0, 0.0), (0.0, 1e9)])
def test_one_launch_equals_two(mrl, env, H, MB, target, max_norm):
    """Same sums, terms and Adam; only the sum of squares is added up in another order: the factor of the clip, and with it
    gradients, moments and steps, move by a few 2^-24."""
    print("one launch", env, H, MB, target, max_norm, flush=True)
    E, got = getattr(mrl, env), []
    few = masked_stream(32)     # (the smallest grid is 36 workgroups: width 64, 3 inputs)
    for launches, stream in ((1, None), (2, few)):
        ctx = mrl.DeviceContext("cuda:0", stream=stream)
        rb, upd, perm = build(mrl, ctx, E, H, MB, target, max_norm)
        upd.run_epoch(perm)
        ctx.synchronize()
        assert ctx.update_end_launches() == launches
        got.append([t.clone() for t in (upd.actor_grads, upd.critic_grads, upd.actor_state, upd.critic_state, rb.actor_params,
                                        rb.critic_params)])
        ctx.close()
    for a, b in zip(*got):
        assert torch.isfinite(a).all() and float(a.abs().max()) > 0
        # (three steps of 1e-3 from weights of 0.1, moments up to 1e-3: differences of 1e-6 of the largest value at most)
        assert float((a - b).abs().max()) <= 2e-6 * float(b.abs().max())


def left(rb, upd):
    return [t.clone() for t in (upd.actor_grads, upd.critic_grads, upd.actor_state, upd.critic_state, rb.actor_params, rb.critic_params,
                                upd.kl_flag)]


@pytest.mark.parametrize("env,H,MB", [("CartPoleEnv", 64, 2), ("PendulumV2", 64, 4200), ("LunarLanderV2", 128, 1000),
                                      ("Walker2dPlanar", 128, 4100), ("HopperPlanar", 256, 17), ("BipedalWalkerV2", 256, 4100)])
@pytest.mark.parametrize("target", [0.0, 1e30, 1e-30])
def test_sums_that_are_not_there_are_worked_out(mrl, env, H, MB, target):
    """A workgroup that does not wait for the others' sums takes them itself: the same bits, and nothing to report, also where the
    limit of polls is one that a wait would not keep."""
    print("no patience", env, H, MB, target, flush=True)
    E, got = getattr(mrl, env), []
    for patience in (0, 1):
        ctx = mrl.DeviceContext("cuda:0")
        rb, upd, perm = build(mrl, ctx, E, H, MB, target)
        ctx.set_update_patience(patience)
        if patience:
            ctx.set_spin_limit(1)
        upd.run_epoch(perm)
        ctx.synchronize()
        got.append(left(rb, upd))
        ctx.close()
    for a, b in zip(*got):
        assert torch.equal(a, b)
    assert torch.isfinite(got[0][4]).all()


def test_places_for_a_part_of_the_grid(mrl):
    """An update captured where every workgroup has a CU, replayed where the stream has eight of them; and six updates on streams of
    their own."""
    print("few places", flush=True)
    E, streams = mrl.HalfCheetahPlanarV2, [torch.cuda.Stream() for _ in range(6)]
    parts = []
    for s in streams:
        ctx = mrl.DeviceContext("cuda:0", stream=s)
        parts.append((ctx,) + build(mrl, ctx, E, 256, 512, 0.0))
    ctx, rb, upd, perm = parts[0]
    first = left(rb, upd)

    def restart(rb, upd):
        for dst, src in zip((upd.actor_grads, upd.critic_grads, upd.actor_state, upd.critic_state, rb.actor_params, rb.critic_params), first):
            dst.copy_(src)
        torch.cuda.synchronize()

    def epoch(upd, perm):   # (run_epoch with the step counts of a first one)
        d = upd.descriptor()
        mrl._lib.call("mrl_ppo_update_epoch", upd.ctx.handle, ctypes.byref(d), perm.data_ptr(), 3, 0, 0)

    epoch(upd, perm)
    ctx.synchronize()
    want = left(rb, upd)
    for c, r, u, p in parts:
        restart(r, u)
    for c, r, u, p in parts:
        epoch(u, p)
    for c, r, u, p in parts:
        c.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(left(r, u), want))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=streams[0]):
        epoch(upd, perm)
    few = masked_stream(8)
    for replay in range(3):
        restart(rb, upd)
        with torch.cuda.stream(few):
            graph.replay()
        torch.cuda.synchronize()
        ctx.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(left(rb, upd), want)), replay
    del graph


def test_a_wait_that_gives_up_is_reported(mrl):
    ctx = mrl.DeviceContext("cuda:0")
    rb, upd, perm = build(mrl, ctx, mrl.HalfCheetahPlanarV2, 256, 512, 0.0)
    ctx.set_spin_limit(1)
    upd.run_epoch(perm)
    with pytest.raises(mrl.MrlError):
        ctx.synchronize()
    ctx.set_spin_limit(0)
    rb, upd, perm = build(mrl, ctx, mrl.HalfCheetahPlanarV2, 256, 512, 0.0)
    before = rb.actor_params.clone()
    upd.run_epoch(perm)
    ctx.synchronize()
    assert torch.isfinite(rb.actor_params).all() and not torch.equal(before, rb.actor_params)
