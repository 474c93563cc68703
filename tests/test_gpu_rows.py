"""GPU parity of the row-tile forward and backward behind Network.forward_gpu / backward_gpu (three-layer nets of the
agents' shapes) against Float64, at the edges of their tiles: one row, a row less or more than a tile of 16 or 32, batches
on either side of the switch between 16 and 32 rows, input widths that leave the cache's rows off 16 bytes, heads of one
to eight outputs and the Gaussian head."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (batch, inputs, outputs, Gaussian head)
SHAPES = [(1, 3, 1, False), (15, 17, 6, True), (16, 24, 8, False), (17, 32, 8, True), (33, 5, 3, False), (1001, 11, 4, True),
          (2049, 8, 4, False), (4097, 3, 1, True)]


def _net(mrl, H, tanh, shape):
    b, i, o, gauss = shape
    lay = mrl.LinearTanh if tanh else mrl.LinearReLU
    return mrl.seq(lay(i, H), lay(H, H), (mrl.StochasticActor if gauss else mrl.Linear)(H, o))


def _split(p, i, H, o):
    out, at = [], 0
    for shape in ((i, H), (H,), (H, H), (H,), (H, o), (o,)):
        n = 1
        for d in shape:
            n *= d
        out.append(p[at:at + n].view(shape))
        at += n
    return out


@pytest.mark.parametrize("tanh", [False, True], ids=["relu", "tanh"])
@pytest.mark.parametrize("H", [64, 128, 256])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "b%d_i%d_o%d%s" % (s[0], s[1], s[2], "_gauss" if s[3] else ""))
def test_forward_backward_against_float64(mrl, shape, H, tanh):
    B, i, o, gauss = shape
    model = _net(mrl, H, tanh, shape)
    ctx = mrl.DeviceContext("cuda:0")
    g = torch.Generator(device="cuda").manual_seed(B * 7 + H)
    p = (torch.rand(model.PARAM_SIZE, device="cuda", generator=g) - 0.5) * (2.0 / H ** 0.5)
    x = torch.randn(B * i, device="cuda", generator=g)
    go = torch.randn(B * model.OUT_DIM, device="cuda", generator=g)
    out, cache, grads, grads2, grad_in = (torch.full((n,), 9.0, device="cuda") for n in
                                          (B * model.OUT_DIM, B * model.CACHE_SIZE, model.PARAM_SIZE, model.PARAM_SIZE, B * i))
    model.forward_gpu_ws(ctx, out, x, p, cache)
    model.backward_gpu_ws(ctx, grad_in, go, p, cache, grads)
    model.backward_gpu_ws(ctx, None, go, p, cache, grads2)
    ctx.synchronize()
    W0, b0, W1, b1, W2, b2 = _split(p.double(), i, H, o)
    X, G = x.double().view(B, i), go.double().view(B, model.OUT_DIM)
    act = torch.tanh if tanh else torch.relu
    pre0 = X @ W0 + b0
    h1 = act(pre0)
    pre1 = h1 @ W1 + b1
    h2 = act(pre1)
    want = h2 @ W2 + b2
    if gauss:
        want = torch.cat([want, p[-o:].double().clamp(-5, 2).expand(B, o)], 1)
    want_cache = [torch.cat([X, h1 if tanh else pre0], 1), torch.cat([h1, h2 if tanh else pre1], 1), h2]
    # sums of up to 256 products each rounded to 2^-24, three layers of them: 1e-5 of the tensor's largest value is eight
    # times what the products alone can show
    close = lambda a, w: torch.testing.assert_close(a.double().view_as(w), w, rtol=0, atol=1e-5 * max(1.0, float(w.abs().max())))
    close(out, want)
    close(cache, torch.cat([c.reshape(-1) for c in want_cache]))
    # act' of what the kernels cached: a pre-activation next to zero may fall on either side of the ReLU
    c1 = cache[B * (i + H):B * (i + 3 * H)].view(B, 2 * H)[:, :H].double()
    c2 = cache[B * (i + 3 * H):].view(B, H).double()
    d = (lambda h: 1 - h * h) if tanh else (lambda h: (h > 0).double())
    g1 = G[:, :o] @ W2.T * d(c2)
    g0 = g1 @ W1.T * d(c1)
    ref = [X.T @ g0, g0.sum(0), c1.T @ g1, g1.sum(0), c2.T @ G[:, :o], G[:, :o].sum(0)] + ([G[:, o:].sum(0)] if gauss else [])
    ref = torch.cat([r.reshape(-1) for r in ref])
    close(grads, ref)
    assert torch.equal(grads, grads2)
    close(grad_in, (g0 @ W0.T).reshape(-1))


def test_grad_in_over_grad_out(mrl):
    """A caller may let the input gradient replace the output gradient in one buffer."""
    B, i, H, o = 200, 8, 64, 4
    model = _net(mrl, H, False, (B, i, o, False))
    ctx = mrl.DeviceContext("cuda:0")
    g = torch.Generator(device="cuda").manual_seed(3)
    p = (torch.rand(model.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.25
    x, go = torch.randn(B * i, device="cuda", generator=g), torch.randn(B * o, device="cuda", generator=g)
    out, cache, grads, grads2, grad_in = (torch.zeros(n, device="cuda") for n in
                                          (B * o, B * model.CACHE_SIZE, model.PARAM_SIZE, model.PARAM_SIZE, B * i))
    model.forward_gpu_ws(ctx, out, x, p, cache)
    model.backward_gpu_ws(ctx, grad_in, go, p, cache, grads)
    buf = torch.zeros(B * i, device="cuda")
    buf[:B * o] = go
    model.backward_gpu_ws(ctx, buf, buf[:B * o], p, cache, grads2)
    ctx.synchronize()
    # two kernels for one sum: rounding of 200-term sums in another order
    torch.testing.assert_close(buf, grad_in, rtol=1e-5, atol=1e-6)
    torch.testing.assert_close(grads2, grads, rtol=1e-5, atol=1e-4)
