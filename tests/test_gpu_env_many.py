"""BipedalWalker's and HalfCheetah's step for batches of several wavefronts per SIMD: the same bits as the workgroup form
that smaller batches take (which is held against the oracle), for rows in every state that the new form treats apart."""
import numpy as np
import pytest
import torch

from test_gpu_collect import ctx, mrl  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


def bits(t):
    t = torch.where(torch.isnan(t), torch.full_like(t, float("nan")), t)     # one NaN for all
    return t.view(torch.int32)


def odd_rows(name, s, rng):
    """Every ninth row into one of the states below."""
    n = s.shape[0]
    if name == "HalfCheetahPlanarV2":
        s[0::9, 17 + 91 + 21 + 102] = 5.0                                    # a joint missing: stepped by the second launch
        s[3::9, 17 + 1] -= 0.6                                               # torso deep in the ground
        s[6::9, 17 + 3] = torch.from_numpy(rng.normal(0, 20, len(range(6, n, 9))).astype(np.float32))
        s[1::9, 245] = 999.0                                                 # the step limit, also of rows with a missing
        s[0::18, 245] = 999.0                                                # joint and of the last, started group of eight
        s[-1, 245] = 999.0
        return
    bodies, joints, edges = 24, 104, 173
    ec = edges + 128 * 6
    E = s[:, edges:ec].view(n, 128, 6)
    s[0::9, 172] = 3.0                                                       # a joint missing
    for b in range(5):
        s[1::9, bodies + 13 * b + 1] -= 1.5                                  # sunk: many contacts
        s[2::9, bodies + 13 * b] += 3.0 * b                                  # strewn: many edges near the bodies
    E[3::9, :, [0, 2]] = E[3::9][:, :, [0, 2]] * 0.1 + float(s[0, bodies])   # crowded edges: a vertex over dozens
    E[4::9] = E[4::9][:, :, [2, 3, 0, 1, 4, 5]]                              # edges from right to left
    s[5::9, ec] = 37.0                                                       # few edges
    s[6::9, bodies] = float("nan")                                           # no hull position
    s[7::9, bodies + 13 + 12] = 0.0                                          # an upper leg with the hull's five vertices
    s[8::9, 942] = 1999.0                                                    # the step limit


@pytest.mark.parametrize("name,batch", [("BipedalWalkerV2", 4097), ("BipedalWalkerV2", 9003),
                                        ("HalfCheetahPlanarV2", 8193), ("HalfCheetahPlanarV2", 12005)])
def test_many_equals_workgroup_form(mrl, ctx, name, batch):  # noqa: F811
    E = getattr(mrl, name)
    rng = np.random.default_rng(batch)
    part = 1024
    assert batch > 4096
    states = torch.zeros(batch * E.STATE_SIZE, device="cuda")
    E.reset_kernel_gpu(ctx, states, 5)
    z = lambda w: torch.zeros(batch * w, device="cuda")  # noqa: E731
    for t in range(60):
        if t in (0, 30, 57):
            odd_rows(name, states.view(batch, -1), rng)
        actions = torch.from_numpy(rng.uniform(-1.3, 1.3, batch * E.ACTION_DIM).astype(np.float32)).cuda()
        ref, r0, d0, o0 = states.clone(), z(1), z(1), z(E.OBS_DIM)
        for i in range(0, batch, part):
            m = min(part, batch - i)
            cut = lambda x, w: x[i * w:(i + m) * w]  # noqa: E731, B023
            E.step_kernel_gpu(ctx, cut(ref, E.STATE_SIZE), cut(actions, E.ACTION_DIM), cut(r0, 1), cut(d0, 1), cut(o0, E.OBS_DIM), 0)
        plain, r1, d1, o1 = states.clone(), z(1), z(1), z(E.OBS_DIM)
        E.step_kernel_gpu(ctx, plain, actions, r1, d1, o1, 0)
        r2, d2, o2 = z(1), z(1), z(E.OBS_DIM)
        E.step_autoreset_kernel_gpu(ctx, states, actions, r2, d2, o2, 0, 77 + t)
        for got, want, what in ((plain, ref, "states"), (r1, r0, "rewards"), (d1, d0, "dones"), (o1, o0, "obs"), (r2, r0, "rewards"), (d2, d0, "dones")):
            same = (bits(got) == bits(want)).view(batch, -1).all(1)
            assert bool(same.all()), (what, t, torch.nonzero(~same).flatten()[:8].tolist())
        if t == 57 or (t > 57 and name == "BipedalWalkerV2"):               # (HalfCheetah ends at the step limit only)
            assert float(d0.sum()) > 1
        E.selective_reset_kernel_gpu(ctx, ref, d0, 77 + t)
        assert torch.equal(bits(states), bits(ref))
        assert torch.equal(bits(o2.view(batch, -1)), bits(ref.view(batch, -1)[:, :E.OBS_DIM].contiguous()))


@pytest.mark.parametrize("name,batch", [("BipedalWalkerV2", 4097), ("HalfCheetahPlanarV2", 8193)])
def test_episode_accounting(mrl, ctx, name, batch):  # noqa: F811
    """rollout_step above the switch: rewards, dones and rows as the workgroup form's on the same actions, running returns and
    lengths and the list of finished episodes as those rewards add up to, for rows of either wiring."""
    E = getattr(mrl, name)
    steps, H, part = 6, 64, 1024
    rng = np.random.default_rng(batch)
    actor = mrl.seq(mrl.LinearTanh(E.OBS_DIM, H), mrl.LinearTanh(H, H), mrl.StochasticActor(H, E.ACTION_DIM))
    critic = mrl.seq(mrl.LinearTanh(E.OBS_DIM, H), mrl.LinearTanh(H, H), mrl.Linear(H, 1))
    g = torch.Generator(device="cuda").manual_seed(3)
    rb = mrl.ppo.RolloutBuffers(ctx, E, actor, critic, batch, steps)
    rb.actor_params = (torch.rand(actor.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.2
    rb.critic_params = (torch.rand(critic.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.2
    E.reset_kernel_gpu(ctx, rb.states, 5)
    desc = rb.descriptor()
    ret, length = torch.zeros(batch, device="cuda"), torch.zeros(batch, device="cuda")
    finished = []
    for t in range(steps):
        if t in (1, 4):
            odd_rows(name, rb.states.view(batch, -1), rng)
        rb.obs.copy_(rb.states.view(batch, -1)[:, :E.OBS_DIM].reshape(-1).nan_to_num())
        ref, r, d = rb.states.clone(), torch.zeros(batch, device="cuda"), torch.zeros(batch, device="cuda")
        o = torch.zeros(batch * E.OBS_DIM, device="cuda")
        mrl.ppo.rollout_step(ctx, desc, t, 100 + t, 0, 77 + t)
        rows = slice(t * batch, (t + 1) * batch)
        actions = rb.r_actions[t * batch * E.ACTION_DIM:(t + 1) * batch * E.ACTION_DIM]
        for i in range(0, batch, part):
            m = min(part, batch - i)
            cut = lambda x, w: x[i * w:(i + m) * w]  # noqa: E731, B023
            E.step_kernel_gpu(ctx, cut(ref, E.STATE_SIZE), cut(actions, E.ACTION_DIM), cut(r, 1), cut(d, 1), cut(o, E.OBS_DIM), 0)
        assert torch.equal(bits(rb.r_rewards[rows]), bits(r)) and torch.equal(rb.r_dones[rows], d)
        ret, length, over = ret + r, length + 1, d > 0.5
        finished += list(zip(ret[over].nan_to_num(7.0).tolist(), length[over].tolist()))
        ret[over], length[over] = 0.0, 0.0
        E.selective_reset_kernel_gpu(ctx, ref, d, 77 + t)
        assert torch.equal(bits(rb.states), bits(ref))
        assert torch.equal(bits(rb.ep_return), bits(ret)) and torch.equal(rb.ep_length, length)
    n = int(rb.done_count)
    assert n == len(finished) and batch // 9 < n <= rb.done_cap
    assert sorted(zip(rb.done_returns[:n].nan_to_num(7.0).tolist(), rb.done_lengths[:n].tolist())) == sorted(finished)
