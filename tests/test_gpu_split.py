"""The minibatch update's products on the bf16 matrix cores with split operands (three bf16 pieces per float, the six
largest of the nine products): against Float64 they must not be further off than the fp32 matrix instructions of the
layer-by-layer kernels.  Both are measured in the same test, on inputs and weights of the agents' size, and
at tile edges (one row, a started 16- and 32-row tile, the sizes where the tile height changes)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(mrl):
    return mrl.DeviceContext("cuda:0")


def _ref(p, IN, H, x, target, relu):
    """Values, gradient of mean((v - target)^2) / 2 with respect to the parameters, in Float64."""
    p = p.double().clone().requires_grad_(True)
    f = torch.relu if relu else torch.tanh
    o1, o2 = (IN + 1) * H, (IN + 1) * H + (H + 1) * H
    h1 = f(x.double() @ p[:IN * H].view(IN, H) + p[IN * H:o1])
    h2 = f(h1 @ p[o1:o1 + H * H].view(H, H) + p[o1 + H * H:o2])
    v = (h2 @ p[o2:o2 + H].view(H, 1)).reshape(-1) + p[o2 + H]
    (0.5 * (v - target.double())**2).mean().backward()
    return v.detach(), p.grad


@pytest.mark.parametrize("H,IN,MB,relu", [(64, 4, 1, True), (64, 3, 2049, False), (128, 17, 33, False), (128, 8, 1025, True),
                                          (256, 8, 17, True), (256, 24, 2048, False), (256, 32, 2049, False), (256, 17, 4096, False)])
def test_split_products_are_as_close_to_float64_as_fp32(mrl, ctx, H, IN, MB, relu):
    print("case", H, IN, MB, relu, flush=True)
    E = type("E", (), dict(ENV_ID=-1, STATE_SIZE=IN, OBS_DIM=IN, NUM_ACTIONS=2, ACTION_DIM=0))
    lay = mrl.LinearReLU if relu else mrl.LinearTanh
    actor = mrl.seq(lay(IN, H), lay(H, H), mrl.Linear(H, 2))
    critic = mrl.seq(lay(IN, H), lay(H, H), mrl.Linear(H, 1))
    g = torch.Generator(device="cuda").manual_seed(MB)
    rb = mrl.ppo.RolloutBuffers(ctx, E, actor, critic, MB, 1)
    rb.actor_params = (torch.rand(actor.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.3
    rb.critic_params = (torch.rand(critic.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.3
    rb.r_obs.normal_(generator=g)
    rb.r_log_probs.fill_(-0.7)
    p0, x = rb.critic_params.clone(), rb.r_obs.clone()
    upd = mrl.ppo.DiscreteUpdate(ctx, rb, MB, mrl.Adam(lr=3e-4), mrl.Adam(lr=3e-4), target_kl=0.0, clip_value=False,
                                 max_grad_norm=1e9, norm_adv_per_minibatch=False)
    upd.returns.normal_(generator=g)
    v64, g64 = _ref(p0, IN, H, x.view(MB, IN), upd.returns, relu)
    upd.minibatch_step(torch.arange(MB, dtype=torch.int32, device="cuda"))
    # the same with the fp32 matrix instructions: a layer per model (the three together would take the fused kernels)
    models = [lay(IN, H), lay(H, H), mrl.Linear(H, 1)]
    acts, caches, parts, off = [x], [], [], 0
    for m in models:
        parts.append(p0[off:off + m.PARAM_SIZE].clone())
        off += m.PARAM_SIZE
        y, cache = torch.zeros(MB * m.OUT_DIM, device="cuda"), torch.zeros(MB * m.CACHE_SIZE, device="cuda")
        m.forward_gpu_ws(ctx, y, acts[-1], parts[-1], cache)
        acts.append(y)
        caches.append(cache)
    v32, grad, g32 = acts[-1], (acts[-1] - upd.returns) / MB, []
    for m, p, cache, below in zip(models[::-1], parts[::-1], caches[::-1], acts[-2::-1]):
        gp, gx = torch.zeros(m.PARAM_SIZE, device="cuda"), torch.zeros(below.numel(), device="cuda")
        m.backward_gpu_ws(ctx, gx, grad, p, cache, gp)
        g32.insert(0, gp)
        grad = gx
    g32 = torch.cat(g32)
    ctx.synchronize()
    err = lambda a, b: float((a.double() - b).norm() / b.norm())
    hh = slice((IN + 1) * H, (IN + 1) * H + H * H)                       # dW1, a split product at H = 256
    ev, ev32, eg, eg32 = err(upd.values, v64), err(v32, v64), err(upd.critic_grads, g64), err(g32, g64)
    ew, ew32 = err(upd.critic_grads[hh], g64[hh]), err(g32[hh], g64[hh])
    print("  values %.2e (fp32 %.2e)  gradients %.2e (fp32 %.2e)  dW1 %.2e (fp32 %.2e)" % (ev, ev32, eg, eg32, ew, ew32), flush=True)
    # Over a thousand rows and more the errors average: the split products may not add to what fp32 shows (a quarter for
    # the spread of two independent sets of roundings).  A handful of rows shows single roundings, half an ulp = 6e-8
    # each: the value is the last of the chain h1, h2, head, bias (four).
    floor = 1e-7 if MB > 1000 else 3e-7
    assert ev <= max(1.25 * ev32, floor)
    if H == 256:
        assert ew <= max(1.25 * ew32, floor)
    # the other gradients are sums over the row tiles, n = MB / 32 pieces one after the other: partial sums of k pieces of
    # either sign are sqrt(k / n) of the result, each rounded with a variance of (2^-24 of it)^2 / 3 at most, which is
    # 2^-24 sqrt(n / 6) together (the layer-by-layer kernels have sums of their own in eg32)
    assert eg <= max(1.25 * eg32 + 2.0**-24 * (MB / 32 / 6)**0.5, floor)
