"""LunarLander's fused kernel of eight wavefronts: the same bits as single steps at one env, started and full workgroups, the
last size that takes it and the first that does not, and over enough steps that every env starts again."""
import pytest

import test_gpu_collect
from test_gpu_collect import ctx, mrl  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("env,N,T,hidden,kind", [
    ("lunar", 1, 40, 64, "relu"), ("lunar", 16, 200, 64, "tanh"), ("lunar", 40, 200, 128, "relu"), ("lunar", 17, 150, 256, "tanh"),
    ("lunar", 4096, 6, 64, "relu"), ("lunar", 4096, 6, 128, "tanh"), ("lunar", 4096, 6, 256, "relu"), ("lunar", 4097, 6, 256, "relu"),
    ("lunarc", 1, 40, 64, "relu"), ("lunarc", 15, 150, 128, "tanh"), ("lunarc", 33, 150, 256, "relu"), ("lunarc", 4096, 6, 64, "tanh"),
])
def test_rollout_steps_equals_single_steps(mrl, ctx, env, N, T, hidden, kind):  # noqa: F811
    test_gpu_collect.test_rollout_steps_equals_single_steps(mrl, ctx, env, N, T, hidden, kind)
