"""Products and attention that a kernel takes over from the library still do what only the library can: gradients,
functional transforms, tracing, module hooks."""
import math

import pytest
import torch
from torch import nn

F = torch.nn.functional


@pytest.mark.gpu
@pytest.mark.parametrize("n,K,M", [(65, 64, 32), (192, 64, 32), (2048, 4096, 22016)])
def test_gradients_and_transforms_of_portion_products(n, K, M):
    from dejavu_amd import mixer_ops as ops

    g = torch.Generator(device="cuda").manual_seed(n)
    x, W = (torch.randn(s, generator=g, device="cuda").to(torch.bfloat16) for s in ((n, K), (M, K)))
    assert ops._tiles(x, W) or ops._wide(x, W)
    x.requires_grad_()
    ops.linear(x, W).sum().backward()
    got, x.grad = x.grad, None
    F.linear(x, W).sum().backward()
    assert torch.equal(got, x.grad)
    x = x.detach()
    bias = torch.zeros(M, dtype=torch.bfloat16, device="cuda", requires_grad=True)
    assert ops.linear(x, W, bias).requires_grad
    with torch.no_grad():
        assert ops._tiles(x, W, bias) or ops._wide(x, W, bias)
    tangent = torch.func.jvp(lambda t: ops.linear(t, W), (x,), (x,))[1]
    assert torch.equal(tangent, F.linear(x, W))


def test_which_products_of_a_portion_are_taken_over():
    """Sizes on both sides of the rules' lines; each was measured against the library with its weights out of the caches."""
    from dejavu_amd.mixer_ops import _tile_rule, _wide_rule

    for n, M, K in ((1603, 22016, 4096), (2048, 22016, 4096), (2000, 22016, 5120), (2000, 18560, 4096), (2000, 18944, 5120),
                    (1918, 20480, 4096), (1862, 21760, 4096)):
        assert _wide_rule(n, M, K), (n, M, K)                    # 1.07 to 1.33 times the library's speed
    for n, M, K in ((1512, 22016, 4096), (1624, 21760, 4096), (1435, 24576, 4096), (1939, 19200, 4096), (1365, 28672, 4096),
                    (2191, 17920, 4096), (1999, 16384, 4096), (1700, 22016, 8192), (12288, 4096, 4096), (8192, 4096, 4096),
                    (6000, 22016, 4096)):
        assert not _wide_rule(n, M, K), (n, M, K)                # 0.75 to 1.07 times
    for n, M, K in ((65, 2048, 2048), (192, 4096, 11008), (192, 12288, 4096), (256, 11264, 2048), (256, 2048, 4096), (256, 4096, 8192)):
        assert _tile_rule(n, M, K, True) and _tile_rule(n, M, K, False)
    for n, M, K in ((129, 22016, 4096), (192, 50000, 2048), (193, 4096, 2048), (256, 2048, 2048), (257, 4096, 8192)):
        assert not _tile_rule(n, M, K, True) and not _tile_rule(n, M, K, False)
    assert _tile_rule(128, 22016, 4096, True) and _tile_rule(193, 22016, 4096, True) and not _tile_rule(65, 22016, 4096, False)


@pytest.fixture(scope="module")
def fc2():
    """A weight whose products of 193..512 rows are this package's, and rows."""
    layer = nn.Linear(16384, 4096, device="cuda", dtype=torch.float16).requires_grad_(False)
    return layer, torch.randn(1, 512, 16384, device="cuda").half()


def _is_ours(layer, x):
    """The two results are fp16 values below 4 of the same sums: a unit of rounding at most between them."""
    from dejavu_amd.modules import _long_product, decode_linear

    y = decode_linear(layer, x)
    torch.testing.assert_close(y, F.linear(x, layer.weight, layer.bias), rtol=2e-3, atol=2e-3)
    return _long_product(layer, x)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [193, 512])
def test_gradients_and_hooks_of_a_long_prompts_linear(fc2, rows):
    from dejavu_amd.modules import decode_linear

    layer, x = nn.Linear(16384, 4096, device="cuda", dtype=torch.float16), fc2[1][:, :rows]
    decode_linear(layer, x).sum().backward()
    assert torch.equal(layer.bias.grad, torch.full((4096,), float(rows), device="cuda").half())
    seen = []
    hook = lambda m, i, o: seen.append(o.shape)  # noqa: E731
    with torch.no_grad():
        for register in (layer.register_forward_hook, nn.modules.module.register_module_forward_hook):
            handle = register(hook)
            try:
                decode_linear(layer, x)
            finally:
                handle.remove()
            assert seen.pop() == (1, rows, 4096)
        assert _is_ours(layer, x) and not seen
        layer.forward = lambda t: t[..., :1]  # as wrappers of a module replace it
        assert decode_linear(layer, x).shape == (1, rows, 1)


def test_rule_of_a_long_prompts_linear():
    """Both sides of each line, in rows and in the weight's size and shape."""
    from dejavu_amd.modules import _long_rule

    for rows, M, K, ours in ((193, 4096, 16384, True), (256, 1024, 8192, True), (256, 1024, 8184, False), (256, 4096, 16376, False),
                             (256, 768, 3072, False), (257, 4096, 16384, True), (257, 4088, 16384, False), (384, 12288, 49152, True),
                             (385, 8192, 32768, True), (385, 8200, 32800, False), (512, 4096, 16384, True), (513, 4096, 16384, False)):
        assert _long_rule(rows, M, K) == ours, (rows, M, K)


@pytest.mark.gpu
@torch.no_grad()
def test_operands_of_a_long_prompts_linear_that_only_the_library_takes(fc2):
    """Weights and rows off a 16-byte boundary or with odd strides, and layers that are no nn.Linear."""
    from dejavu_amd.modules import decode_linear

    layer, x = fc2
    x = x[:, :200]
    assert _is_ours(layer, x)
    M, K = layer.weight.shape
    moved = torch.empty(M * K + 1, device="cuda", dtype=torch.float16)[1:].view(M, K).copy_(layer.weight)
    apart = torch.empty(M, K + 4, device="cuda", dtype=torch.float16)[:, :K].copy_(layer.weight)
    for weight in (moved, apart, layer.weight.t().contiguous().t()):
        other = nn.Linear(1, 1, device="cuda", dtype=torch.float16)
        other.weight, other.bias = nn.Parameter(weight, requires_grad=False), layer.bias
        assert not _is_ours(other, x)
    assert not _is_ours(layer, torch.empty(x.numel() + 1, device="cuda", dtype=torch.float16)[1:].view(x.shape).copy_(x))
    assert _is_ours(layer, torch.randn(1, 200, K + 8, device="cuda").half()[:, :, :K])

    class Duck:
        weight, bias = layer.weight, layer.bias

        def __call__(self, t):
            return t[..., :2]

    assert torch.equal(decode_linear(Duck(), x), x[..., :2])


@pytest.mark.gpu
@torch.no_grad()
@pytest.mark.parametrize("rows,M,K,activation", [(200, 4096, 16384, "id"), (400, 8192, 2048, "relu"), (800, 5120, 20480, "id")])
def test_weights_whose_rows_are_one_row(rows, M, K, activation):
    """An expanded weight, whose rows begin at the same place."""
    from dejavu_amd.modules import _long_product, _wide_product, decode_linear

    layer = nn.Linear(K, M, device="cuda", dtype=torch.float16).requires_grad_(False)
    x = torch.randn(1, rows, K, device="cuda").half()
    assert _long_product(layer, x) or _wide_product(layer, x, activation)
    layer.weight = nn.Parameter(layer.weight[:1].expand(M, K), requires_grad=False)
    want = F.linear(x, layer.weight, layer.bias)
    assert torch.equal(decode_linear(layer, x, activation), F.relu(want) if activation == "relu" else want)


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
def test_traces_of_what_kernels_take_over(fc2):
    """Graphs recorded by make_fx compute with the inputs that they are given later."""
    from torch.fx.experimental.proxy_tensor import make_fx

    from dejavu_amd import mixer_ops
    from dejavu_amd.modules import HIP_PROMPT_ATTN_MAX_TOKENS, ParallelMHADejavu, decode_linear

    W = torch.randn(32, 64, device="cuda").bfloat16()
    layer = fc2[0]
    mha = ParallelMHADejavu(128, 2, causal=True, device="cuda", dtype=torch.float16)
    T = HIP_PROMPT_ATTN_MAX_TOKENS + 8
    for f, shape, dtype in ((lambda t: mixer_ops.linear(t, W), (65, 64), torch.bfloat16),
                            (lambda t: decode_linear(layer, t), (1, 200, 16384), torch.float16),
                            (lambda t: mha._dense_context(t, None), (1, T, 3, 2, 64), torch.float16)):
        traced = make_fx(f)(torch.randn(shape, device="cuda").to(dtype))
        x = torch.randn(shape, device="cuda").to(dtype)
        torch.testing.assert_close(traced(x), f(x), rtol=2e-2, atol=2e-2)  # one rounding of each side: 2^-8 and less


@pytest.mark.gpu
@torch.no_grad()
def test_operands_of_a_long_prompts_attention_that_only_the_library_takes():
    """Caches of a caller's own, of another type, stride, place or length, are filled as ever; so are those that the kernel fills."""
    from dejavu_amd import modules, ops
    from dejavu_amd.modules import HIP_PROMPT_ATTN_MAX_TOKENS, InferenceParams, ParallelMHADejavu

    T, S, H, hd = HIP_PROMPT_ATTN_MAX_TOKENS + 8, HIP_PROMPT_ATTN_MAX_TOKENS + 16, 2, 64
    mha = ParallelMHADejavu(H * hd, H, causal=True, layer_idx=0, device="cuda", dtype=torch.float16)
    qkv = torch.randn(1, T, 3, H, hd, device="cuda").half()
    odd = torch.empty(qkv.numel() + 1, device="cuda", dtype=torch.float16)[1:].view(qkv.shape).copy_(qkv)
    want = mha._dense_context(qkv, None)
    shapes = (1, H, hd // 8, S, 8), (1, H, S, hd)

    def plain(shape, dtype=torch.float16):
        return torch.zeros(shape, device="cuda", dtype=dtype)

    made = {"plain": [plain(s) for s in shapes], "fp32": [plain(s, torch.float32) for s in shapes],
            "moved": [plain(math.prod(s) + 1)[1:].view(s) for s in shapes],
            "strided": [plain(s[:-1] + (s[-1] + 8,))[..., :s[-1]] for s in shapes],
            "longer": [plain((1, H, hd // 8, S + 8, 8)), plain(shapes[1])]}
    for name, (k_cache, v_cache) in made.items():
        for x in (qkv, odd):
            k_cache.zero_(), v_cache.zero_()
            ip = InferenceParams(max_sequence_len=S, max_batch_size=1)
            ip.key_value_memory_dict[0] = k_cache, v_cache
            torch.testing.assert_close(mha._dense_context(x, ip), want, rtol=2e-3, atol=2e-3)
            k = k_cache[:, :, :, :T].permute(0, 3, 1, 2, 4).reshape(1, T, H, hd)
            assert torch.equal(k.half(), qkv[:, :, 1]) and torch.equal(v_cache[:, :, :T].transpose(1, 2).half(), qkv[:, :, 2])
            assert not k_cache[:, :, :, T:].any() and not v_cache[:, :, T:].any()
        assert modules._kernel_takes(qkv, k_cache, v_cache) == (name in ("plain", "longer"))
    assert not modules._kernel_takes(odd)
    torch.testing.assert_close(ops.prefill_attention(qkv), want, rtol=2e-3, atol=2e-3)


@pytest.mark.gpu
@torch.no_grad()
@pytest.mark.parametrize("T,H,hd,ours", [(6144, 1, 64, True), (6145, 1, 64, False), (2048, 41, 128, True), (2049, 41, 128, False),
                                         (2049, 40, 128, True)])
def test_longest_prompts_of_the_attention_kernel(T, H, hd, ours, monkeypatch):
    """On both sides of the lines; the last queries against every key in 64 bits, fp16 weights and results (5e-4 below 5)."""
    from dejavu_amd import ops
    from dejavu_amd.modules import ParallelMHADejavu

    called, kernel = [], ops.prefill_attention
    monkeypatch.setattr(ops, "prefill_attention", lambda *a: [called.append(1), kernel(*a)][1])
    mha = ParallelMHADejavu(H * hd, H, causal=True, device="cuda", dtype=torch.float16)
    qkv = torch.randn(1, T, 3, H, hd, device="cuda").half()
    got = mha._dense_context(qkv, None).view(T, H, hd)[-3:].double()
    assert bool(called) == ours
    q, k, v = (t[0].double().transpose(0, 1) for t in qkv.unbind(2))
    s = (q[:, -3:] @ k.transpose(1, 2).contiguous()) * hd ** -0.5
    s[:, 0, -2:], s[:, 1, -1:] = -math.inf, -math.inf
    torch.testing.assert_close(got, (s.softmax(-1) @ v.contiguous()).transpose(0, 1), rtol=1e-3, atol=5e-3)


@pytest.mark.gpu
@torch.no_grad()
def test_new_windows_that_only_the_library_begins(monkeypatch):
    """A traced reset is in the trace, and trackers and places of a caller's own, of another type, device or stride, are written as
    ever; so are those that the kernel writes."""
    from torch.fx.experimental.proxy_tensor import make_fx

    from dejavu_amd import modules

    launches, kernel = [], modules.lib.dv_window_reset
    monkeypatch.setattr(modules.lib, "dv_window_reset", lambda *a: [launches.append(1), kernel(*a)][1])
    H, here = 3, torch.device("cuda", torch.cuda.current_device())
    mha = modules.ParallelMHASparseAttMlp(192, H, None, dict(embed_dim=192, low_rank_dim=8, out_dim=H, K=1), causal=True, layer_idx=0,
                                          device="cuda", dtype=torch.float16)
    plain, fresh = mha.tracker, torch.arange(16).int().repeat(H, 1)
    new = lambda value, **kw: torch.tensor([value], **{"dtype": torch.int32, "device": "cuda", **kw})  # noqa: E731
    other = {"int64 tracker": (plain.long(), new(-1)), "strided tracker": (torch.zeros(16, H, dtype=torch.int32, device="cuda").t(), new(-1)),
             "tracker on the CPU": (plain.cpu(), None), "int64 place": (plain, new(-1, dtype=torch.int64)),
             "place on the CPU": (plain, new(-1, device="cpu")), "two places": (plain, new(-1).repeat(2))}
    for name, (tracker, place) in [("plain", (plain, new(-1))), ("no place yet", (plain, None)), *other.items()]:
        mha.tracker, mha.cache_offset = tracker.fill_(-7), place
        launches.clear()
        mha.reset_window(123, here)
        assert bool(launches) == (name in ("plain", "no place yet")), name
        assert torch.equal(mha.tracker.cpu(), fresh.to(tracker.dtype)) and (mha.cache_offset.cpu() == 123).all(), name
        assert place is mha.cache_offset or (place is None and mha.cache_offset.device == here), name
        mha.tracker.fill_(-7)
        mha.reset_window()
        assert torch.equal(mha.tracker.cpu(), fresh.to(tracker.dtype)) and (mha.cache_offset.cpu() == 123).all(), name

    mha.tracker, mha.cache_offset = plain, new(-1)
    zero = torch.zeros(1, dtype=torch.int32, device="cuda")
    traced = make_fx(lambda t: [mha.reset_window(7, here), mha.tracker + t, mha.cache_offset + t][1:])(zero)
    plain.fill_(-7), mha.cache_offset.fill_(-1)
    tracker, place = traced(zero)
    assert torch.equal(tracker.cpu(), fresh) and torch.equal(plain.cpu(), fresh) and place.item() == mha.cache_offset.item() == 7
    with monkeypatch.context() as m:  # as on another device than the current one
        m.setattr(modules, "results_only", lambda *tensors: False)
        launches.clear(), plain.fill_(-7)
        mha.reset_window(9, here)
        assert not launches and torch.equal(plain.cpu(), fresh) and mha.cache_offset.item() == 9


@pytest.mark.gpu
@torch.no_grad()
@pytest.mark.parametrize("rows,M,K,kind", [(300, 4096, 16384, "linear"), (300, 2560, 10240, "linear"), (300, 16384, 4096, "linear"),
                                           (100, 4096, 4096, "portion"), (300, 4096, 11008, "portion"), (2048, 22016, 4096, "portion")])
def test_products_in_traced_programs(rows, M, K, kind):
    """Whole graphs and symbolic sizes: what a kernel's rule asks for may not get in the way of the library's product."""
    from torch.fx.experimental.proxy_tensor import make_fx

    from dejavu_amd import mixer_ops
    from dejavu_amd.modules import decode_linear

    dtype = torch.float16 if kind == "linear" else torch.bfloat16
    layer = nn.Linear(K, M, bias=False, device="cuda", dtype=dtype).requires_grad_(False)
    x = torch.randn(1, rows, K, device="cuda").to(dtype)
    if kind == "portion":
        x = x[0]
    want = F.linear(x, layer.weight)

    def f(t, W):
        return decode_linear(layer, t) if kind == "linear" else mixer_ops.linear(t, W)

    torch._dynamo.reset()
    whole = torch.compile(f, backend="eager", fullgraph=True)(x, layer.weight)
    torch.testing.assert_close(whole, want, rtol=2e-2, atol=2e-2)  # (one rounding of each side: 2^-8 and less)
    if kind == "portion":  # (a module's own weight is no input of the graph, and symbolic graphs take such ones only)
        traced = make_fx(f, tracing_mode="symbolic")(x, layer.weight)
        torch.testing.assert_close(traced(x, layer.weight), want, rtol=2e-2, atol=2e-2)


@pytest.mark.gpu
@torch.no_grad()
def test_layers_without_results():
    from dejavu_amd import mixer_ops, ops
    from dejavu_amd.modules import decode_linear

    for K in (4096, 16384):
        layer = nn.Linear(K, 0, device="cuda", dtype=torch.float16)
        assert decode_linear(layer, torch.zeros(1, 300, K, device="cuda").half()).shape == (1, 300, 0)
    W = torch.zeros(0, 11008, device="cuda").bfloat16()
    assert mixer_ops.linear(torch.zeros(300, 11008, device="cuda").bfloat16(), W).shape == (300, 0)
    assert ops.wide_parts(150, 4096, 0) == 0
