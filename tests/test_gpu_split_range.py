"""GPU: the split bf16 products (mlp_split.hpp) at the ends of float32's range: infinities, NaN, values that round to bf16's
infinity, and values whose lower pieces bf16 cannot hold.  What fp32 products give is the yardstick, as IEEE arithmetic has
it: torch in Float64, rounded to float32."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BIG = 3.4e38                # above bf16's largest value (3.3895e38) by more than half its spacing, below float32's


@pytest.fixture(scope="module")
def ctx(mrl):
    return mrl.DeviceContext("cuda:0")


def values_of(mrl, ctx, H, MB, x, w0, w1, w2):
    """The fused update's forward of a critic [1, H, H, 1] without biases: x [MB] -> values."""
    E = type("E", (), dict(ENV_ID=-1, STATE_SIZE=1, OBS_DIM=1, NUM_ACTIONS=2, ACTION_DIM=0))
    actor = mrl.seq(mrl.LinearReLU(1, H), mrl.LinearReLU(H, H), mrl.Linear(H, 2))
    critic = mrl.seq(mrl.LinearReLU(1, H), mrl.LinearReLU(H, H), mrl.Linear(H, 1))
    rb = mrl.ppo.RolloutBuffers(ctx, E, actor, critic, MB, 1)
    zero = torch.zeros(H, device="cuda")
    rb.critic_params = torch.cat([w0, zero, w1.reshape(-1), zero, w2, zero[:1]])
    rb.actor_params = torch.zeros(actor.PARAM_SIZE, device="cuda")
    rb.r_obs.copy_(x)
    rb.r_log_probs.fill_(-0.7)
    upd = mrl.ppo.DiscreteUpdate(ctx, rb, MB, mrl.Adam(lr=0.0), mrl.Adam(lr=0.0), target_kl=0.0, max_grad_norm=1e9,
                                 norm_adv_per_minibatch=False)
    upd.minibatch_step(torch.arange(MB, dtype=torch.int32, device="cuda"))
    ctx.synchronize()
    return upd.values.clone()


def same_kind(got, want):
    """Infinities and NaN where the reference has them."""
    want = want.float()
    return bool((torch.isnan(got) == torch.isnan(want)).all() and
                (torch.where(torch.isinf(want), want, torch.zeros_like(want)) ==
                 torch.where(torch.isinf(got), got, torch.zeros_like(got))).all())


@pytest.mark.parametrize("H,MB", [(64, 19), (128, 33), (256, 45), (256, 4096)])
def test_update_forward(mrl, ctx, H, MB):
    print("case", H, MB, flush=True)
    g = torch.Generator(device="cuda").manual_seed(H + MB)
    u = lambda *n: torch.rand(*n, device="cuda", generator=g)                       # noqa: E731
    # rows: ordinary, infinite, the largest finite ones, NaN (which relu = x > 0 ? x : 0 takes to 0)
    x = u(MB) + 0.5
    x[1::5], x[2::5], x[3::7] = float("inf"), BIG, float("nan")
    w0 = torch.ones(H, device="cuda")
    # the head reads column 4, small enough to stay finite for the largest rows; the others are negative, relu takes them
    # to 0 (magnitudes up to 300: lower pieces above 1; one column exact in bf16: lower pieces 0)
    w1 = -(u(H, H) + 1e-3)
    w1[:, 0::8] *= 300.0
    w1[:, 2] = -0.5
    w1[:, 4] = u(H) * 1e-3 / H
    w2 = torch.where(torch.arange(H, device="cuda") == 4, 1.0, 0.0)
    relu = lambda v: torch.where(v > 0, v, torch.zeros_like(v))                     # noqa: E731
    want = relu(relu(x.double()[:, None] * w0.double()) @ w1.double()) @ w2.double()
    got = values_of(mrl, ctx, H, MB, x, w0, w1, w2)
    assert same_kind(got, want), (got[:8], want[:8])
    assert float(got[1]) == float("inf") and 0 < float(got[2]) < float("inf") and float(got[3]) == 0
    fin = torch.isfinite(want) & (want > 0)
    # h1 is x, layer 1 a sum of H positive terms in fp32 accumulators (H / 32 + 8 roundings at most), bias and head exact
    assert float(((got.double() - want)[fin] / want[fin]).abs().max()) < (H / 32 + 16) * 2.0**-24


@pytest.mark.parametrize("e", [-126, -120, -110, -100])
def test_tiny_weights(mrl, ctx, e):
    """bf16 pieces are multiples of 2^-133: a weight of at least 2^-110 is exact, a smaller one off by half of that."""
    H, MB = 256, 16
    g = torch.Generator(device="cuda").manual_seed(-e)
    x = torch.rand(MB, device="cuda", generator=g) + 1.0
    w1 = (torch.rand(H, H, device="cuda", generator=g) + 1.0) * 2.0**e
    one = torch.ones(H, device="cuda")
    got = values_of(mrl, ctx, H, MB, x, one, w1, one)
    want = x.double() * w1.double().sum()
    # beside the pieces: products of bf16 pieces kept to 2^-24 of a term, fp32 sums of H terms, H columns and the head
    lost = 2.0**-134 * H * H * x.double() if e < -110 else 0.0
    assert bool(((got.double() - want).abs() <= lost + 64 * 2.0**-24 * want).all())


@pytest.mark.parametrize("H,batch,dw_launch", [(256, 45, True), (256, 2065, True), (128, 8200, True), (64, 45, False)])
def test_layer_backward(mrl, ctx, H, batch, dw_launch):
    """dW1 = h1^T g1 with infinite and with the largest gradients in single rows."""
    print("case", H, batch, flush=True)
    g = torch.Generator(device="cuda").manual_seed(batch)
    model = mrl.seq(mrl.LinearTanh(1, H), mrl.LinearTanh(H, H), mrl.Linear(H, 1))
    p = torch.zeros(model.PARAM_SIZE, device="cuda")
    o1, o2 = 2 * H, 2 * H + (H + 1) * H
    p[:H] = torch.rand(H, device="cuda", generator=g) + 0.1                         # h1 in (0, 1)
    p[o2:o2 + H] = 1.0                                                              # g1 = grad_out (h2 = 0: act' = 1)
    x = torch.rand(batch, device="cuda", generator=g) * 1e-2 + 1e-3
    out, cache = torch.empty(batch, device="cuda"), torch.empty(batch * model.CACHE_SIZE, device="cuda")
    model.forward_gpu_ws(ctx, out, x, p, cache)
    h1 = torch.tanh(x.double()[:, None] * p[:H].double())
    for big in (BIG, float("inf"), -float("inf"), float("nan")):
        go = torch.rand(batch, device="cuda", generator=g)
        go[batch // 2] = big
        grads = torch.zeros_like(p)
        model.backward_gpu_ws(ctx, None, go, p, cache, grads)
        ctx.synchronize()
        want = (h1.T @ go.double())[:, None].expand(H, H)
        got = grads[o1:o1 + H * H].view(H, H)
        assert same_kind(got, want), big
        if big == BIG:
            # h1 is off by tanh's few roundings; the sum is its largest term
            assert float(((got.double() - want) / want).abs().max()) < 1e-5
