"""Nets of hidden width 128 in the fused kernels: the policy step gives the bits of the layer-by-layer kernels (one
chain of fused multiply-adds per output in ascending k), and the fused minibatch update its parts."""
import pytest
import torch

import test_gpu_ppo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(mrl):
    return mrl.DeviceContext("cuda:0")


# one row, a full and a started row tile, both launch forms (up to 4096 rows actor and critic in workgroups of their own)
@pytest.mark.parametrize("n,IN,A,kind", [(1, 8, 4, "relu"), (32, 3, 1, "tanh"), (33, 17, 6, "tanh"), (4097, 32, 8, "tanh")])
def test_policy_step_gives_the_layer_by_layer_bits(mrl, ctx, n, IN, A, kind):
    print("case", n, IN, A, kind, flush=True)
    H = 128
    lin = mrl.LinearReLU if kind == "relu" else mrl.LinearTanh
    gauss = kind == "tanh"
    layers = [lin(IN, H), lin(H, H), mrl.StochasticActor(H, A) if gauss else mrl.Linear(H, A)]
    vlayers = [lin(IN, H), lin(H, H), mrl.Linear(H, 1)]
    g = torch.Generator(device="cuda").manual_seed(n)
    actor, critic = mrl.seq(*layers), mrl.seq(*vlayers)
    ap = (torch.rand(actor.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.3
    cp = (torch.rand(critic.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.3
    E = type("E", (), dict(ENV_ID=-1, STATE_SIZE=IN, OBS_DIM=IN, NUM_ACTIONS=0 if gauss else A, ACTION_DIM=A if gauss else 0))
    rb = mrl.ppo.RolloutBuffers(ctx, E, actor, critic, n, 1)
    rb.actor_params, rb.critic_params = ap, cp
    rb.obs.normal_(generator=g)
    acts = torch.zeros(n * rb.act_width, device="cuda")
    mrl.ppo.policy_step(ctx, rb, 0, 99, acts)

    def layerwise(models, params):
        x, off = rb.obs, 0
        for m in models:
            y = torch.zeros(n * m.OUT_DIM, device="cuda")
            m.forward_gpu_no_cache_ws(ctx, y, x, params[off:off + m.PARAM_SIZE].clone())
            x, off = y, off + m.PARAM_SIZE
        return x

    head, values = layerwise(layers, ap), layerwise(vlayers, cp)
    a2, lp2 = torch.zeros_like(acts), torch.zeros(n, device="cuda")
    (mrl.ppo.sample_continuous_actions if gauss else mrl.ppo.sample_actions)(ctx, head, a2, lp2, 99)
    ctx.synchronize()
    assert torch.equal(rb.r_values, values)
    assert torch.equal(acts, a2) and torch.equal(rb.r_log_probs, lp2) and torch.equal(rb.r_actions, a2)


# the weight gradient of the hidden layer in the row tiles (up to 8192 rows) and in a launch of its own
@pytest.mark.parametrize("env_name,kind,MB", [("CartPoleEnv", "relu", 33), ("Walker2dPlanar", "tanh", 1000), ("HopperPlanar", "tanh", 4096)])
def test_fused_update_minibatch_equals_its_parts(mrl, ctx, env_name, kind, MB):
    test_gpu_ppo.test_fused_update_minibatch_equals_its_parts(mrl, ctx, env_name, kind, MB, 128)


def test_fused_update_weight_gradient_in_its_own_launch(mrl, ctx):
    """8224 rows: the batch gradient against float64 autograd of the value loss (first Adam step from zero moments moves
    nothing but gradients into critic_grads; no clipping at this norm bound)."""
    H, IN, MB = 128, 5, 8224
    E = type("E", (), dict(ENV_ID=-1, STATE_SIZE=IN, OBS_DIM=IN, NUM_ACTIONS=2, ACTION_DIM=0))
    lay = mrl.LinearTanh
    actor = mrl.seq(lay(IN, H), lay(H, H), mrl.Linear(H, 2))
    critic = mrl.seq(lay(IN, H), lay(H, H), mrl.Linear(H, 1))
    g = torch.Generator(device="cuda").manual_seed(3)
    rb = mrl.ppo.RolloutBuffers(ctx, E, actor, critic, MB, 1)
    rb.actor_params = (torch.rand(actor.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.3
    rb.critic_params = (torch.rand(critic.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.3
    rb.r_obs.normal_(generator=g)
    rb.r_log_probs.fill_(-0.7)
    p = rb.critic_params.double().clone().requires_grad_(True)
    upd = mrl.ppo.DiscreteUpdate(ctx, rb, MB, mrl.Adam(lr=3e-4), mrl.Adam(lr=3e-4), target_kl=0.0, clip_value=False, max_grad_norm=1e9)
    upd.returns.normal_(generator=g)
    upd.advantages.normal_(generator=g)
    upd.minibatch_step(torch.arange(MB, dtype=torch.int32, device="cuda"))
    ctx.synchronize()
    o1, o2 = (IN + 1) * H, (IN + 1) * H + (H + 1) * H
    x = rb.r_obs.double().view(MB, IN)
    h1 = torch.tanh(x @ p[:IN * H].view(IN, H) + p[IN * H:o1])
    h2 = torch.tanh(h1 @ p[o1:o1 + H * H].view(H, H) + p[o1 + H * H:o2])
    v = (h2 @ p[o2:o2 + H].view(H, 1)).reshape(-1) + p[o2 + H]
    (0.5 * (v - upd.returns.double())**2).mean().backward()
    # fp32 sums of 8224 terms: sqrt(8224) * 2^-24 of the terms' size is 5e-6; the largest gradient bounds the terms' sum
    # from below by 1e-2 of it
    scale = float(p.grad.abs().max())
    torch.testing.assert_close(upd.critic_grads.double(), p.grad, rtol=0.0, atol=1e-4 * scale)
