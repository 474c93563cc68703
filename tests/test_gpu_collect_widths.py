"""The fused collection kernels at hidden widths 64, 128 and 256: the same bits as single steps, at one env, a full and a
started 16-env workgroup, and past the env counts where a second workgroup shares a CU or another kernel takes over."""
import pytest

import test_gpu_collect
from test_gpu_collect import ctx, mrl  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("env,N,T,hidden,kind", [
    ("cartpole", 1, 30, 64, "relu"), ("cartpole", 17, 40, 128, "tanh"), ("cartpole", 4097, 8, 128, "relu"),
    ("cartpole", 4096, 8, 64, "tanh"), ("cartpole", 4097, 8, 64, "tanh"), ("cartpole", 4111, 6, 256, "relu"),
    ("pendulum", 1, 9, 128, "tanh"), ("pendulum", 33, 9, 256, "relu"), ("pendulum", 4097, 6, 64, "tanh"), ("pendulum", 4100, 6, 128, "tanh"),
    ("lunar", 1, 9, 64, "relu"), ("lunar", 33, 9, 128, "tanh"), ("lunar", 8192, 6, 64, "relu"), ("lunar", 8193, 6, 128, "relu"),
    ("lunarc", 17, 9, 128, "tanh"), ("lunarc", 4099, 6, 64, "tanh"),
    ("bipedal", 17, 9, 64, "tanh"), ("bipedal", 333, 40, 128, "relu"),
    ("cheetah", 16, 9, 128, "tanh"), ("cheetah", 77, 12, 64, "relu"), ("cheetah", 4097, 6, 256, "tanh"),
    ("car", 17, 9, 128, "tanh"), ("car", 50, 12, 64, "relu"),
    ("hopper", 1, 9, 64, "tanh"), ("hopper", 333, 40, 128, "relu"), ("walker2d", 17, 9, 128, "tanh"), ("walker2d", 333, 40, 64, "relu"),
])
def test_rollout_steps_equals_single_steps(mrl, ctx, env, N, T, hidden, kind):  # noqa: F811
    test_gpu_collect.test_rollout_steps_equals_single_steps(mrl, ctx, env, N, T, hidden, kind)
