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


def test_rounding_of_16_row_tiles(mrl):
    """The head's bias gradient is the sum of the output gradients: rows of a tile one after the other, 256 tiles of 16 rows
    in four trees of 64.  With all terms in [1, 2), V the result, a rounded sum v is off by at most 2^-24 v, with a variance of
    a third of that square at most: V / 4 .. V along the four trees 1.9 V^2, within the trees 0.5 V^2, within the tiles 0.02 V^2,
    so a root mean square below 0.9 * 2^-24 V; one tile after the other it would be 5.3.  64 sums estimate it to 9 %: 1.2."""
    B, H, o = 4096, 64, 8
    model = mrl.seq(mrl.LinearReLU(3, H), mrl.LinearReLU(H, H), mrl.Linear(H, o))
    ctx = mrl.DeviceContext("cuda:0")
    g = torch.Generator(device="cuda").manual_seed(5)
    p = (torch.rand(model.PARAM_SIZE, device="cuda", generator=g) - 0.5) * 0.2
    out, cache, grads = (torch.zeros(n, device="cuda") for n in (B * o, B * model.CACHE_SIZE, model.PARAM_SIZE))
    model.forward_gpu_ws(ctx, out, torch.randn(B * 3, device="cuda", generator=g), p, cache)
    off = []
    for _ in range(8):
        go = torch.rand(B * o, device="cuda", generator=g) + 1.0
        model.backward_gpu_ws(ctx, None, go, p, cache, grads)
        ctx.synchronize()
        want = go.double().view(B, o).sum(0)
        off.append((grads[-o:].double() - want) / want * 2 ** 24)
    rms = float(torch.cat(off).pow(2).mean().sqrt())
    print("rms", rms)
    assert rms < 1.2
