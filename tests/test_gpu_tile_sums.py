"""GPU check of the sums over row tiles in the fused backward at numbers of tiles around those that are added up in one
go (8, 16, 32, 64), with a remainder and without.  Inputs, weights and output gradients are small integers, so that every
product and sum is exact in fp32 (below 2^24) and the gradients must equal Float64's."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [64, 128, 256])
@pytest.mark.parametrize("tiles", [1, 7, 8, 9, 15, 17, 31, 40, 63, 64, 65, 79, 127])
def test_integer_gradients_are_exact(mrl, tiles, H):
    B, i, o = 16 * tiles - 3, 5, 3
    model = mrl.seq(mrl.LinearReLU(i, H), mrl.LinearReLU(H, H), mrl.Linear(H, o))
    ctx = mrl.DeviceContext("cuda:0")
    g = torch.Generator(device="cuda").manual_seed(tiles * 1000 + H)
    p = torch.randint(-1, 2, (model.PARAM_SIZE,), device="cuda", generator=g).float()
    p *= (torch.rand(model.PARAM_SIZE, device="cuda", generator=g) < 0.2).float()
    x = torch.randint(-1, 2, (B * i,), device="cuda", generator=g).float()
    go = torch.randint(-1, 2, (B * o,), device="cuda", generator=g).float()
    out, cache, grads = (torch.zeros(n, device="cuda") for n in (B * o, B * model.CACHE_SIZE, model.PARAM_SIZE))
    model.forward_gpu_ws(ctx, out, x, p, cache)
    model.backward_gpu_ws(ctx, None, go, p, cache, grads)
    ctx.synchronize()
    q, at = [], 0
    for shape in ((i, H), (H,), (H, H), (H,), (H, o), (o,)):
        n = shape[0] * (shape[1] if len(shape) > 1 else 1)
        q.append(p[at:at + n].double().view(shape))
        at += n
    W0, b0, W1, b1, W2, b2 = q
    X, G = x.double().view(B, i), go.double().view(B, o)
    h1 = torch.relu(X @ W0 + b0)
    h2 = torch.relu(h1 @ W1 + b1)
    g1 = G @ W2.T * (h2 > 0)
    g0 = g1 @ W1.T * (h1 > 0)
    want = torch.cat([t.reshape(-1) for t in (X.T @ g0, g0.sum(0), h1.T @ g1, g1.sum(0), h2.T @ G, G.sum(0))])
    assert float(want.abs().max()) < 2 ** 24
    assert torch.equal(grads.double(), want)


@pytest.mark.parametrize("tiles,rows", [(64, 16), (127, 16), (4096, 32), (16384, 32)])
def test_rounding_of_many_tiles(mrl, tiles, rows):
    """The head's bias gradient is the sum of the output gradients: rows of a tile one after the other, tiles 64 at a time as
    a tree.  With all terms in [1, 2) every partial sum is below the result, and an addition rounds by 2^-24 of it at most."""
    B, H = rows * tiles, 64
    model = mrl.seq(mrl.LinearReLU(3, H), mrl.LinearReLU(H, H), mrl.Linear(H, 1))
    ctx = mrl.DeviceContext("cuda:0")
    g = torch.Generator(device="cuda").manual_seed(tiles)
    p = (torch.rand(model.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.2
    go = torch.rand(B, device="cuda", generator=g) + 1.0
    out, cache, grads = (torch.zeros(n, device="cuda") for n in (B, B * model.CACHE_SIZE, model.PARAM_SIZE))
    model.forward_gpu_ws(ctx, out, torch.randn(B * 3, device="cuda", generator=g), p, cache)
    model.backward_gpu_ws(ctx, None, go, p, cache, grads)
    ctx.synchronize()
    want = float(go.double().sum())
    # In units of 2^-24 of the result: the tiles' own sums, whose roundings are independent of one another, and the last
    # bias below 4 together, the groups of 64 tiles 1 each at worst, of which independent roundings to nearest leave a
    # sixteenth (their mean is a quarter of the worst, half of it on the way up, and they add up like a root: from 64 groups
    # on an eighth of that), and 1 for the result itself.  One tile after the other would be 64 times the groups.
    groups = max(1, tiles // 64)
    bound = (4 + groups / 16 + 1) * 2.0 ** -24
    assert abs(float(grads[-1]) - want) <= bound * want, (float(grads[-1]) / want - 1) * 2 ** 24
