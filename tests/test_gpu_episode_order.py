"""The finished-episode list of the fused collection kernels: in the order in which episodes end, to within the steps that a
workgroup keeps them back."""
import pytest
import torch

import test_gpu_collect
from test_gpu_collect import ctx, mrl  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("env,N,T,hidden", [
    ("cartpole", 1024, 96, 64), ("cartpole", 512, 96, 128), ("lunar", 777, 128, 64), ("lunar", 512, 128, 256), ("lunar", 4112, 128, 64),
    ("hopper", 1024, 128, 64), ("hopper", 1000, 128, 256), ("bipedal", 512, 160, 64)])
def test_episodes_are_listed_as_they_end(mrl, ctx, env, N, T, hidden):  # noqa: F811
    print("episode order", env, N, T, hidden, flush=True)
    rb, _ = test_gpu_collect._pair(mrl, ctx, N, T, hidden, "relu", env)
    E = rb.env
    if env == "cartpole":
        rb.keep = torch.zeros(N, dtype=torch.int32, device="cuda")
        E.bind_step_counters(ctx, rb.states, rb.keep)
    E.reset_kernel_gpu(ctx, rb.states, 3)
    rows = rb.states.view(N, E.STATE_SIZE)
    rb.obs.copy_(rows[:, :E.OBS_DIM].reshape(-1))
    if env == "bipedal":      # (steps of 2000 left: random policies may stay up for long)
        rows[:, 942] = 2000.0 - 8.0 - torch.arange(N, device="cuda") % 120
    # each env's first episode carries its number in the length: 1000 (e + 1) + its steps, exact in fp32
    rb.ep_length.copy_(1000.0 * torch.arange(1, N + 1, device="cuda"))
    rb.done_count.zero_()
    assert mrl.ppo.rollout_fused(rb.descriptor())
    rb.done_returns, rb.done_lengths = torch.zeros(2, N * T, device="cuda")
    rb.done_cap = N * T
    mrl.ppo.rollout_steps(ctx, rb.descriptor(), 0, T, 11, 7919, 0, 0, 17, 104729)
    ctx.synchronize()
    dones = rb.r_dones.view(T, N).cpu() > 0.5
    first = torch.where(dones.any(0), dones.int().argmax(0), torch.full((N,), -1))
    lengths = rb.done_lengths[:int(rb.done_count.item())].cpu()
    tagged = lengths[lengths >= 1000.0]
    steps = [int(first[int(x) // 1000 - 1]) for x in tagged.tolist()]
    assert sorted(steps) == sorted(first[first >= 0].tolist()) and len(steps) > N // 8
    assert all(int(x) % 1000 == s + 1 for x, s in zip(tagged.tolist(), steps))
    late, newest = 0, 0      # steps by which an episode stands behind one that ended after it
    for s in steps:
        newest = max(newest, s)
        late = max(late, newest - s)
    print("  episodes", len(steps), "last step", max(steps), "late by at most", late, flush=True)
    # sixteen steps kept back, and workgroups that are some steps apart (all of them start together)
    assert late <= 40
