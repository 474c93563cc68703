"""The fused collection kernels at hidden widths 64, 128 and 256: the same bits as single steps, at one env, a full and a
started 16-env workgroup, and past the env counts where a second workgroup shares a CU or another kernel takes over."""
import pytest
import torch

import test_gpu_collect
from test_gpu_collect import ctx, mrl  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("env,N,T,hidden,kind", [
    ("cartpole", 1, 30, 64, "relu"), ("cartpole", 17, 40, 128, "tanh"), ("cartpole", 4097, 8, 128, "relu"),
    ("cartpole", 4096, 8, 64, "tanh"), ("cartpole", 4097, 8, 64, "tanh"), ("cartpole", 4111, 6, 256, "relu"),
    ("pendulum", 1, 9, 128, "tanh"), ("pendulum", 33, 9, 256, "relu"), ("pendulum", 4097, 6, 64, "tanh"), ("pendulum", 4100, 6, 128, "tanh"),
    ("cartpole", 6144, 6, 64, "tanh"), ("cartpole", 6145, 6, 64, "relu"), ("pendulum", 12288, 6, 64, "relu"), ("pendulum", 12289, 6, 64, "tanh"),
    ("lunar", 1, 9, 64, "relu"), ("lunar", 33, 9, 128, "tanh"), ("lunar", 8192, 6, 64, "relu"), ("lunar", 8193, 6, 128, "relu"),
    ("lunarc", 17, 9, 128, "tanh"), ("lunarc", 4099, 6, 64, "tanh"),
    ("bipedal", 17, 9, 64, "tanh"), ("bipedal", 333, 40, 128, "relu"), ("bipedal", 8193, 9, 128, "tanh"), ("bipedal", 12288, 9, 256, "relu"),
    ("cheetah", 16, 9, 128, "tanh"), ("cheetah", 77, 12, 64, "relu"), ("cheetah", 4097, 6, 256, "tanh"),
    ("car", 17, 9, 128, "tanh"), ("car", 50, 12, 64, "relu"),
    ("hopper", 1, 9, 64, "tanh"), ("hopper", 333, 40, 128, "relu"), ("walker2d", 17, 9, 128, "tanh"), ("walker2d", 333, 40, 64, "relu"),
    ("walker2d", 4096, 9, 64, "tanh"), ("walker2d", 4097, 9, 64, "relu"),
])
def test_rollout_steps_equals_single_steps(mrl, ctx, env, N, T, hidden, kind):  # noqa: F811
    test_gpu_collect.test_rollout_steps_equals_single_steps(mrl, ctx, env, N, T, hidden, kind)


@pytest.mark.parametrize("env,hidden,per_cu", [("bipedal", 64, 32), ("bipedal", 128, 32), ("bipedal", 256, 48), ("walker2d", 64, 16),
                                               ("walker2d", 128, 32), ("walker2d", 256, 32)])
def test_one_launch_up_to(mrl, ctx, env, hidden, per_cu):  # noqa: F811
    """As many envs per CU as make the launch of all steps the faster way."""
    n = per_cu * torch.cuda.get_device_properties(0).multi_processor_count
    E = {"bipedal": mrl.BipedalWalkerV2, "walker2d": mrl.Walker2dPlanar}[env]
    actor = mrl.seq(mrl.LinearTanh(E.OBS_DIM, hidden), mrl.LinearTanh(hidden, hidden), mrl.StochasticActor(hidden, E.ACTION_DIM))
    critic = mrl.seq(mrl.LinearTanh(E.OBS_DIM, hidden), mrl.LinearTanh(hidden, hidden), mrl.Linear(hidden, 1))
    for envs, fused in ((n, True), (n + 1, False)):
        rb = mrl.ppo.RolloutBuffers(ctx, E, actor, critic, envs, 1)
        rb.actor_params, rb.critic_params = (torch.zeros(m.PARAM_SIZE, device="cuda") for m in (actor, critic))
        assert mrl.ppo.rollout_fused(rb.descriptor()) == fused
