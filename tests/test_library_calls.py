"""Products and attention that a kernel takes over from the library still do what only the library can: gradients,
functional transforms, tracing, module hooks."""
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


def test_modes_that_watch_library_calls():
    """A kernel's launch is invisible to dispatch and function modes, so none may stand in for a library call under one."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    from torch.utils.flop_counter import FlopCounterMode

    from dejavu_amd._binding import results_only

    assert results_only()
    for mode in (FlopCounterMode(display=False), TorchDispatchMode(), TorchFunctionMode()):
        with mode:
            assert not results_only(), mode
    seen = []
    make_fx(lambda t: [seen.append(results_only()), t + 1][1])(torch.ones(2))
    assert seen == [False]
    with torch.device("cpu"):  # a default device changes what makes tensors, and nothing else
        assert results_only()
    assert results_only()


@pytest.mark.gpu
@torch.no_grad()
def test_traces_of_what_kernels_take_over():
    """Graphs recorded by make_fx compute with the inputs that they are given later."""
    from torch.fx.experimental.proxy_tensor import make_fx

    from dejavu_amd import mixer_ops
    from dejavu_amd.modules import HIP_PROMPT_ATTN_MAX_TOKENS, ParallelMHADejavu, decode_linear

    W = torch.randn(32, 64, device="cuda").bfloat16()
    layer = nn.Linear(256, 64, device="cuda", dtype=torch.float16)
    mha = ParallelMHADejavu(128, 2, causal=True, device="cuda", dtype=torch.float16)
    T = HIP_PROMPT_ATTN_MAX_TOKENS + 8
    for f, shape, dtype in ((lambda t: mixer_ops.linear(t, W), (65, 64), torch.bfloat16),
                            (lambda t: decode_linear(layer, t), (1, 200, 256), torch.float16),
                            (lambda t: mha._dense_context(t, None), (1, T, 3, 2, 64), torch.float16)):
        traced = make_fx(f)(torch.randn(shape, device="cuda").to(dtype))
        x = torch.randn(shape, device="cuda").to(dtype)
        torch.testing.assert_close(traced(x), f(x), rtol=2e-2, atol=2e-2)  # one rounding of each side: 2^-8 and less
