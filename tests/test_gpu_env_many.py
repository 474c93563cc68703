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
        if t >= 57:
            assert float(d0.sum()) > (1 if name == "BipedalWalkerV2" else -1)
        E.selective_reset_kernel_gpu(ctx, ref, d0, 77 + t)
        assert torch.equal(bits(states), bits(ref))
        assert torch.equal(bits(o2.view(batch, -1)), bits(ref.view(batch, -1)[:, :E.OBS_DIM].contiguous()))
