"""Products of long rows with K in parts (gemm_wide.hpp): every number of parts, tiles and columns that end within one, what follows the sums."""
import ctypes

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from dejavu_amd import _lib_mixers as L
from dejavu_amd import mixer_ops, modules, ops

pytestmark = pytest.mark.gpu

# (rows, weight rows, columns): six, five, four, three and two parts on tiles of every width, which end in the middle; columns behind the last chunk
SIZES = [(257, 1032, 4168), (300, 520, 2600), (383, 520, 2056), (383, 2056, 2504), (500, 2056, 4168), (700, 4104, 2600), (1300, 1032, 2504)]


def _parts(n, M, K):
    return L.lib.dv_mix_linear_wide_workspace_bytes(n, M, K) // (4 * n * M)


def _operands(n, M, K, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x, W = (torch.randn(r, K, device="cuda", generator=g).to(dtype) for r in (n, M))
    return x, (W * K ** -0.5).to(dtype), torch.randn(M, device="cuda", generator=g).to(dtype)


def _near(got, want, dtype, K):
    """A result is within half a step of its type, and the rounding of fp32 sums of K products of values of about one, of the sum in 64 bits."""
    step = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    bound = step * want.abs() + 2.0 ** -24 * K ** 0.5 * 8
    assert got.shape == want.shape and bool(((got.double() - want).abs() <= bound).all())


def test_every_number_of_parts_is_taken():
    assert {_parts(*s) for s in SIZES} == {2, 3, 4, 5, 6}
    assert _parts(2048, 8192, 4096) == 0 and _parts(300, 512, 960) == 0  # whole rounds of tiles; too few columns
    assert ops.wide_parts(777, 16384, 4096) == _parts(777, 4096, 16384)


@pytest.mark.parametrize("n,M,K", SIZES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_sums_of_parts(n, M, K, dtype):
    x, W, b = _operands(n, M, K, dtype)
    nbytes = L.lib.dv_mix_linear_wide_workspace_bytes(n, M, K)
    assert nbytes > 0
    want = x.double() @ W.double().t() + b.double()
    if dtype == torch.float16:
        got = ops.dense_linear_wide_parts(x, W, b)
    else:
        got = torch.full((n, M), float("nan"), device="cuda", dtype=dtype)
        a = mixer_ops._tile_args(x, W)
        a.out, a.ldo, a.bias = got.data_ptr(), M, b.data_ptr()
        mixer_ops._parts_launch(L.OUT_T, a, nbytes, x.device)
    _near(got, want, dtype, K)


class _Norm:
    def __init__(self, M, seed):
        g = torch.Generator(device="cuda").manual_seed(seed)
        self.w, self.b = (torch.randn(M, device="cuda", generator=g) for _ in range(2))

    def struct(self):
        return L.DynTanh(self.w.data_ptr(), self.b.data_ptr(), 0.6)

    def __call__(self, x):
        return torch.tanh(0.6 * x) * self.w.double() + self.b.double()


@pytest.mark.parametrize("n,M,K", SIZES[:5])
@pytest.mark.parametrize("start,pre", [(False, True), (True, True), (True, False)])
def test_residual_behind_the_parts(n, M, K, start, pre):
    x, W, _ = _operands(n, M, K, torch.bfloat16, 1)
    stream = mixer_ops.ResidualStream(torch.randn(n, M, device="cuda"), torch.randn(n, M, device="cuda"), torch.bfloat16)
    post, following = _Norm(M, 2), _Norm(M, 3)
    want = stream.x.double() + post(x.double() @ W.double().t()) + (stream.start.double() if start else 0.0)
    a, h = mixer_ops._tile_args(x, W), stream.new_h()
    a.res = stream.args(post, following if pre else None, start, h if pre else None)
    mixer_ops._parts_launch(L.OUT_RESIDUAL, a, L.lib.dv_mix_linear_wide_workspace_bytes(n, M, K), x.device)
    # fp32 sums of about one, a tanh of 1e-6 and the rounding of three terms
    assert float((stream.x.double() - want).abs().max()) < 4e-5 * float(want.abs().max())
    if pre:
        assert bool(((h.double() - following(want)).abs() <= 2.0 ** -8 * following(want).abs() + 1e-4).all())


@torch.no_grad()
def test_through_the_layers():
    for n, M, K, ours in ((300, 4096, 8192, False), (300, 4096, 11008, True), (2048, 3072, 12288, True), (256, 4096, 16384, False),
                          (2049, 4096, 16384, False), (600, 1024, 16384, False), (400, 2560, 10240, True), (384, 2560, 10240, False)):
        assert bool(mixer_ops._parts_bytes(torch.empty(n, K, device="cuda", dtype=torch.bfloat16),
                                           torch.empty(M, K, device="cuda", dtype=torch.bfloat16))) == ours
    x, W, b = _operands(400, 2560, 10240, torch.bfloat16)
    _near(mixer_ops.linear(x, W, b), x.double() @ W.double().t() + b.double(), torch.bfloat16, 10240)
    layer = nn.Linear(10240, 2560, device="cuda", dtype=torch.float16)
    x = torch.randn(1, 600, 10240, device="cuda").half()
    want = x.double() @ layer.weight.double().t() + layer.bias.double()
    assert modules._parts_product(layer, x) is not None
    _near(modules.decode_linear(layer, x), want, torch.float16, 10240)
    calls = []
    hook = layer.register_forward_hook(lambda *a: calls.append(1))
    modules.decode_linear(layer, x)
    hook.remove()
    assert calls  # a layer that someone watches is called
    far = torch.zeros(600, 20480, device="cuda").half()
    assert modules._parts_product(layer, far[None, :, ::2]) is None


@torch.no_grad()
def test_replayed_from_a_graph():
    layer = nn.Linear(10240, 2560, device="cuda", dtype=torch.float16)
    x = torch.randn(1, 600, 10240, device="cuda").half()
    modules.decode_linear(layer, x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = modules.decode_linear(layer, x)
    for _ in range(3):
        x.normal_()
        graph.replay()
        assert torch.equal(out, modules.decode_linear(layer, x))


def test_arguments_that_are_refused():
    x, W, _ = _operands(300, 520, 2600, torch.bfloat16)
    out, ws = torch.empty(300, 520, device="cuda", dtype=torch.bfloat16), torch.empty(1 << 24, device="cuda", dtype=torch.uint8)
    a = mixer_ops._tile_args(x, W)
    a.out, a.ldo = out.data_ptr(), 520
    call = lambda after, p, n: L.lib.dv_mix_linear_wide_ws(after, ctypes.byref(a), p, n, mixer_ops._stream())  # noqa: E731
    need = L.lib.dv_mix_linear_wide_workspace_bytes(300, 520, 2600)
    assert call(L.OUT_T, None, 0) == -4 and call(L.OUT_T, ws.data_ptr(), need - 1) == -4 and call(L.OUT_GLU, ws.data_ptr(), need) == -2
    a.ldo = 521
    assert call(L.OUT_T, ws.data_ptr(), need) == -3
    a.ldo, a.ldw = 520, 1 << 25
    assert call(L.OUT_T, ws.data_ptr(), need) == -2
    assert F.linear(x, W).shape == (300, 520)  # nothing was left behind
