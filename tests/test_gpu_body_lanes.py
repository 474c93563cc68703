"""GPU: the solver with one lane per body against the oracle, where its lanes can disagree: groups at the end of a batch, rows
of other joint flags and limits among the usual ones (stepped in the one-lane form), angles beyond 2^20 (whose sines take
another reduction, found out after the fact), many contacts on one body."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# floats of a body and of a joint in a row, and a joint's limit and flag fields
BODY, JOINT, LO, HI, FLAGS = 13, 17, 8, 9, 14


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
