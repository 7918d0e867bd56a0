"""Products that a kernel takes over from the library still do what only the library can: gradients, functional
transforms, module hooks."""
import pytest
import torch
from torch import nn

F = torch.nn.functional


@pytest.mark.gpu
@pytest.mark.parametrize("n,K,M", [(65, 64, 32), (192, 64, 32), (2048, 4096, 16128)])
def test_gradients_and_transforms_of_portion_products(n, K, M):
    from dejavu_amd import mixer_ops as ops

    g = torch.Generator(device="cuda").manual_seed(n)
    x, W = (torch.randn(s, generator=g, device="cuda").to(torch.bfloat16) for s in ((n, K), (M, K)))
    assert ops._tiles(x, W) or ops._wide(x, W, True)
    x.requires_grad_()
    ops.linear(x, W).sum().backward()
    got, x.grad = x.grad, None
    F.linear(x, W).sum().backward()
    assert torch.equal(got, x.grad)
    x = x.detach()
    bias = torch.zeros(M, dtype=torch.bfloat16, device="cuda", requires_grad=True)
    assert ops.linear(x, W, bias).requires_grad
    with torch.no_grad():
        assert ops._tiles(x, W, bias) or ops._wide(x, W, True, bias)
    tangent = torch.func.jvp(lambda t: ops.linear(t, W), (x,), (x,))[1]
    assert torch.equal(tangent, F.linear(x, W))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [193, 512])
def test_gradients_and_hooks_of_a_long_prompts_linear(rows):
    from dejavu_amd.modules import decode_linear

    layer = nn.Linear(256, 64, device="cuda", dtype=torch.float16)
    x = torch.randn(1, rows, 256, device="cuda").half()
    decode_linear(layer, x).sum().backward()
    assert torch.equal(layer.bias.grad, torch.full((64,), float(rows), device="cuda").half())
    seen = []
    handle = layer.register_forward_hook(lambda m, i, o: seen.append(o.shape))
    with torch.no_grad():
        decode_linear(layer, x)
        assert seen == [(1, rows, 64)]
        handle.remove()
        y = decode_linear(layer, x)
    assert len(seen) == 1
    torch.testing.assert_close(y, layer(x).detach(), rtol=2e-3, atol=2e-3)  # two results in fp16, below 2 in size
