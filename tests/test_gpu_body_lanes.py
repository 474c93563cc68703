"""GPU: the solver with one lane per body against the oracle, where its lanes can disagree: groups at the end of a batch, rows
of other joint terms and limits among the usual ones (stepped by the second instance of the solver), angles beyond 2^20 (whose sines take
another reduction, found out after the fact), many contacts on one body."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# floats of a body and of a joint in a row, a body's inverse inertia, and a joint's fields
BODY, JOINT, INV_INERTIA = 13, 17, 11
KIND, LO, HI, TORQUE, SPEED, STIFF, DAMP, FLAGS = 0, 8, 9, 10, 11, 12, 13, 14


def layout(mrl, name):   # class, row, observation, offset of body 0, bodies, joints, action components
    if name == "lunarlander":
        return mrl.LunarLanderV2, 192, 8, 8, 3, 2, 0
    if name == "bipedal":
        return mrl.BipedalWalkerV2, 950, 24, 24, 5, 4, 4
    return mrl.HalfCheetahPlanarV2, 253, 17, 17, 7, 6, 6


@pytest.mark.parametrize("name", ["lunarlander", "bipedal", "halfcheetah"])
@pytest.mark.parametrize("n", [1, 7, 17, 50])
def test_mixed_rows_match_the_oracle(mrl, orc, name, n):
    print("body lanes", name, n, flush=True)
    E, S, OBS, b0, nb, nj, aw = layout(mrl, name)
    ctx = mrl.DeviceContext("cuda:0")
    rng = np.random.default_rng(n + S)
    s = torch.zeros(n * S, device="cuda")
    E.reset_kernel_gpu(ctx, s, 5)
    ctx.synchronize()
    rows = s.cpu().numpy().reshape(n, S).copy()
    j0 = b0 + nb * BODY + nb * 3
    for e in range(n):
        kind = e % 6
        if kind == 1:      # falling fast onto the ground, turning
            for b in range(nb):
                rows[e, b0 + b * BODY + 3] = rng.normal() * 3
                rows[e, b0 + b * BODY + 4] = -12 + rng.normal()
                rows[e, b0 + b * BODY + 5] = rng.normal() * 4
        if kind == 2:      # another joint's terms: spring, limit and motor together
            rows[e, j0 + FLAGS] = 7.0
        if kind == 3:      # a joint without a limit
            rows[e, j0 + (nj - 1) * JOINT + FLAGS] = float(int(rows[e, j0 + (nj - 1) * JOINT + FLAGS]) & ~1)
        if kind == 4:      # limits the wrong way round
            lo, hi = rows[e, j0 + LO], rows[e, j0 + HI]
            rows[e, j0 + LO], rows[e, j0 + HI] = hi, lo
        if kind == 5:      # a body torn so far off that the joint's correction turns it by millions
            rows[e, b0 + BODY] += 1e8
    s.copy_(torch.from_numpy(rows.reshape(-1)))
    r, d, o = (torch.zeros(k, device="cuda") for k in (n, n, n * OBS))
    r_h, d_h, o_h = np.zeros(n, np.float32), np.zeros(n, np.float32), np.zeros((n, OBS), np.float32)
    for t in range(40):
        act = (rng.integers(0, 4, n).astype(np.float32) if aw == 0 else rng.uniform(-1.2, 1.2, (n, aw)).astype(np.float32))
        E.step_kernel_gpu(ctx, s, torch.from_numpy(act.reshape(-1)).cuda(), r, d, o, t)
        if name == "lunarlander":
            orc.orc_ll_step_batch(rows, act, r_h, d_h, o_h, n, 1)
        elif name == "bipedal":
            orc.orc_bw_step_batch(rows, act, r_h, d_h, o_h, n, 1)
        else:
            orc.orc_hc_step_batch(rows, act, r_h, d_h, o_h, n, 1)
        ctx.synchronize()
        got = s.cpu().numpy().reshape(n, S)
        # the same fp32 operations in the same order; zeros may differ in sign
        np.testing.assert_array_equal(got, rows, err_msg="step %d" % t)
        np.testing.assert_array_equal(r.cpu().numpy(), r_h)
        np.testing.assert_array_equal(d.cpu().numpy(), d_h)


# every row with terms that its reset does not give (16391 rows: LunarLander's one lane per env, the others' single-wavefront
# workgroups); "torque": a motor that pulls backwards, "torn": a joint of another kind, which the one-lane form steps
@pytest.mark.parametrize("n", [11, 16391])
@pytest.mark.parametrize("terms", ["no limit", "no terms", "spring", "all terms", "reversed", "no inertia", "torque", "torn"])
@pytest.mark.parametrize("name", ["lunarlander", "bipedal", "halfcheetah"])
def test_rows_of_other_terms(mrl, orc, name, n, terms):
    print("other terms", name, n, terms, flush=True)
    E, S, OBS, b0, nb, nj, aw = layout(mrl, name)
    ctx = mrl.DeviceContext("cuda:0")
    rng = np.random.default_rng(n + S)
    s = torch.zeros(n * S, device="cuda")
    E.reset_kernel_gpu(ctx, s, 7)
    ctx.synchronize()
    rows = s.cpu().numpy().reshape(n, S).copy()
    j0 = b0 + nb * BODY + nb * 3
    B, J = rows[:, b0:b0 + nb * BODY].reshape(n, nb, BODY), rows[:, j0:j0 + nj * JOINT].reshape(n, nj, JOINT)
    B, J = B.copy(), J.copy()
    B[:, :, 3:6] += rng.normal(size=(n, nb, 3)) * np.array([2, 3, 3])
    if terms == "no limit":
        J[:, -1, FLAGS] = (J[:, -1, FLAGS].astype(int) & ~1).astype(np.float32)
    if terms == "no terms":
        J[:, :, FLAGS] = 0
    if terms in ("spring", "all terms"):
        J[:, :, FLAGS] = 7 if terms == "all terms" else 4
        J[:, :, STIFF], J[:, :, DAMP] = rng.uniform(1, 40, (n, nj)), rng.uniform(0.1, 2, (n, nj))
        J[:, :, TORQUE], J[:, :, SPEED] = rng.uniform(1, 60, (n, nj)), rng.normal(size=(n, nj)) * 5
    if terms == "reversed":
        J[:, :, [LO, HI]] = J[:, :, [HI, LO]] * rng.uniform(0.2, 1, (n, nj, 1)) + rng.normal(size=(n, nj, 1)) * 0.2
    if terms == "no inertia":
        B[:, :2, INV_INERTIA] = 0
    if terms == "torque":
        J[:, 0, FLAGS], J[:, 0, TORQUE], J[:, 0, SPEED] = 7, -30, 4
    if terms == "torn":
        J[:, -1, KIND] = 1
    rows[:, b0:b0 + nb * BODY], rows[:, j0:j0 + nj * JOINT] = B.reshape(n, -1), J.reshape(n, -1)
    s.copy_(torch.from_numpy(rows.reshape(-1)))
    r, d, o = (torch.zeros(k, device="cuda") for k in (n, n, n * OBS))
    r_h, d_h, o_h = np.zeros(n, np.float32), np.zeros(n, np.float32), np.zeros((n, OBS), np.float32)
    step = {"lunarlander": orc.orc_ll_step_batch, "bipedal": orc.orc_bw_step_batch, "halfcheetah": orc.orc_hc_step_batch}[name]
    for t in range(30 if n < 100 else 3):
        act = (rng.integers(0, 4, n).astype(np.float32) if aw == 0 else rng.uniform(-1.2, 1.2, (n, aw)).astype(np.float32))
        E.step_kernel_gpu(ctx, s, torch.from_numpy(act.reshape(-1)).cuda(), r, d, o, t)
        step(rows, act, r_h, d_h, o_h, n, 8)
        ctx.synchronize()
        # the same fp32 operations in the same order; zeros may differ in sign
        np.testing.assert_array_equal(s.cpu().numpy().reshape(n, S), rows, err_msg="step %d" % t)
        np.testing.assert_array_equal(r.cpu().numpy(), r_h)
        np.testing.assert_array_equal(d.cpu().numpy(), d_h)


@pytest.mark.parametrize("name", ["lunarlander", "bipedal", "halfcheetah"])
def test_fused_rollout_of_mixed_terms(mrl, name):
    """A launch of many steps, which looks at a LunarLander row's joints once and again where it is reset, against the same
    steps one by one: usual rows, rows of other terms and rows for the one-lane form side by side, episodes ending inside."""
    print("fused other terms", name, flush=True)
    E, S, OBS, b0, nb, nj, aw = layout(mrl, name)
    ctx, n, T, H = mrl.DeviceContext("cuda:0"), 83, 14, 64
    head = mrl.StochasticActor(H, aw) if aw else mrl.Linear(H, 4)
    actor = mrl.seq(mrl.LinearTanh(OBS, H), mrl.LinearTanh(H, H), head)
    critic = mrl.seq(mrl.LinearTanh(OBS, H), mrl.LinearTanh(H, H), mrl.Linear(H, 1))
    g = torch.Generator(device="cuda").manual_seed(5)
    params = [(torch.rand(m.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.3 for m in (actor, critic)]
    rbs = []
    for _ in range(2):
        rb = mrl.ppo.RolloutBuffers(ctx, E, actor, critic, n, T)
        rb.actor_params, rb.critic_params = params
        E.reset_kernel_gpu(ctx, rb.states, 3)
        rows = rb.states.view(n, S)
        j0 = b0 + nb * BODY + nb * 3
        rows[::5, j0 + FLAGS] = 7.0
        rows[1::5, j0 + (nj - 1) * JOINT + FLAGS] = 0.0
        rows[2::7, j0 + KIND] = 1.0
        rows[::3, {"lunarlander": 188, "bipedal": 942, "halfcheetah": 245}[name]] = {"bipedal": 1994.0}.get(name, 994.0)
        rb.obs.copy_(rows[:, :OBS].reshape(-1))
        rbs.append(rb)
    s0, ss, r0, rs = 1234567, 2654435761 * n + 7919, 99, 0x9E3779B97F4A7C15
    d1, d2 = rbs[0].descriptor(), rbs[1].descriptor()
    for t in range(T):
        mrl.ppo.rollout_step(ctx, d1, t, s0 + t * ss, 0, r0 + t * rs)
    assert mrl.ppo.rollout_fused(d2)
    mrl.ppo.rollout_steps(ctx, d2, 0, T, s0, ss, 0, 0, r0, rs)
    ctx.synchronize()
    for k in ("r_obs", "r_actions", "r_log_probs", "r_values", "r_rewards", "r_dones", "states", "ep_return", "ep_length"):
        assert torch.equal(getattr(rbs[0], k), getattr(rbs[1], k)), k
    assert int(rbs[0].done_count.item()) == int(rbs[1].done_count.item()) > 0


@pytest.mark.parametrize("n", [8193, 16384, 16385])
def test_lunar_step_where_the_forms_change_over(mrl, orc, n):
    """Up to 16384 envs four lanes an env, beyond one lane an env: the oracle's bits on both sides."""
    print("lunar switch", n, flush=True)
    E = mrl.LunarLanderV2
    ctx = mrl.DeviceContext("cuda:0")
    rng = np.random.default_rng(n)
    rows = np.zeros((n, 192), np.float32)
    orc.orc_ll_reset_batch(rows, n, 3)
    rows[:, 8:47].reshape(n, 3, 13)[:, :, 1] -= rng.uniform(7.5, 9.4, n).astype(np.float32)[:, None]
    s = torch.from_numpy(rows.reshape(-1)).cuda()
    r, d, o = (torch.zeros(k, device="cuda") for k in (n, n, n * 8))
    r_h, d_h, o_h = np.zeros(n, np.float32), np.zeros(n, np.float32), np.zeros((n, 8), np.float32)
    for t in range(4):
        act = rng.integers(0, 4, n).astype(np.float32)
        E.step_kernel_gpu(ctx, s, torch.from_numpy(act).cuda(), r, d, o, t)
        orc.orc_ll_step_batch(rows, act, r_h, d_h, o_h, n, 8)
        ctx.synchronize()
        np.testing.assert_array_equal(s.cpu().numpy().view(np.uint32).reshape(n, 192), rows.view(np.uint32))
        np.testing.assert_array_equal(r.cpu().numpy(), r_h)
        np.testing.assert_array_equal(d.cpu().numpy(), d_h)
