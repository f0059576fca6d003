"""The fused training pass against the same network in float64 with the bf16
roundings of the kernels' operands, at one tile, a few and many; also that a
training pass leaves the forward pass of another batch size alone."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _reference(flat, x, t, weight):
    import torch

    from optika_amd import surrogate

    class Bf16(torch.autograd.Function):  # value rounded, and the gradient that flows back
        @staticmethod
        def forward(ctx, v):
            return v.to(torch.bfloat16).to(v.dtype)

        @staticmethod
        def backward(ctx, g):
            return g

    class GradBf16(torch.autograd.Function):  # rounds the gradient only
        @staticmethod
        def forward(ctx, v):
            return v

        @staticmethod
        def backward(ctx, g):
            return g.to(torch.bfloat16).to(g.dtype)

    p = flat.double().cpu().requires_grad_(True)
    part = lambda layer, k: p[(o := surrogate.LAYOUT[layer][k])[0]:  # noqa: E731
                              o[0] + int(np.prod(o[1]))].reshape(o[1])
    h = x.double().cpu()
    for layer in range(4):
        w = part(layer, 0)
        pre = h @ (w if layer == 0 else Bf16.apply(w)).T
        if layer:
            pre = GradBf16.apply(pre)
        pre = pre + part(layer, 1)
        h = Bf16.apply(torch.nn.functional.silu(pre))
    y = h @ part(4, 0).T + part(4, 1)
    loss = (weight.double().cpu() * (y - t.double().cpu()) ** 2).sum() / len(y)
    g, = torch.autograd.grad(loss, p)
    return y.detach().numpy(), loss.item(), g.numpy()


@pytest.mark.parametrize("rows", [128, 384, 16512])
def test_fused_training_pass(rows):
    import torch

    from optika_amd import surrogate

    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(rows)
    net = surrogate.MLP(dev, seed=3)
    flat = net.p + 0.02 * torch.randn(net.p.shape, generator=g).to(dev)
    net.set_params(flat)
    x = (2 * torch.rand((rows, 5), generator=g) - 1).to(dev)
    t = torch.randn((rows, 3), generator=g).to(dev)
    w = torch.tensor([1.0, 0.5, 0.25], device=dev)
    other = x[:64].contiguous()
    before = net.forward(other).clone()
    print(f"case: training pass rows={rows}", flush=True)
    loss = net.loss_grad(x, t, w)
    assert torch.equal(net.forward(other), before) and net.y.shape == (64, 3)
    again = net.loss_grad(x, t, w)
    assert torch.equal(loss, again)  # sums in a fixed order
    y, want, grad = _reference(net.p, x, t, w)
    # a sum in float32 may round a bf16 value the other way: 2^-8 of a few
    # terms, within 2^-8 of a whole in norm
    got = net.g.cpu().numpy().astype(np.float64)
    assert np.linalg.norm(net.y.cpu().numpy() - y) <= 2.0 ** -8 * np.linalg.norm(y)
    assert abs(float(loss) - want) <= 2.0 ** -8 * want
    for layer in range(5):
        for off, shape in surrogate.LAYOUT[layer]:
            k = slice(off, off + int(np.prod(shape)))
            err = np.linalg.norm(got[k] - grad[k]) / np.linalg.norm(grad[k])
            assert err <= 2.0 ** -8, (layer, shape, err)
