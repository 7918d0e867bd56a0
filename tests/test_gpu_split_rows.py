"""Products that merge an attention's splits while they stage their row, against fp64."""
import pytest
import torch

from dejavu_amd import mixer_ops as ops
from dejavu_amd import _lib_mixers as L

pytestmark = pytest.mark.gpu


# rows shorter than one pass of the workgroup, one and several passes; splits of less than a packet of loads, all of it and more
@pytest.mark.parametrize("heads,vdim,splits", [(1, 8, 2), (3, 24, 3), (16, 128, 6), (16, 128, 8), (5, 80, 9), (40, 64, 17), (32, 128, 8)])
@pytest.mark.parametrize("sink,gate", [(True, False), (False, True), (True, True), (False, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_merge_in_the_product(heads, vdim, splits, sink, gate, dtype):
    g = torch.Generator(device="cuda").manual_seed(heads * 1000 + splits)

    def rand(*shape, scale=1.0):
        return torch.randn(*shape, device="cuda", generator=g) * scale

    l = rand(heads, splits).abs() + 0.5
    sums, m = rand(heads, splits, vdim) * l[..., None], rand(heads, splits, scale=4.0)
    sums[0, -1], m[0, -1], l[0, -1] = 0.0, -1e30, 0.0  # a split without keys
    part = torch.cat([sums.reshape(-1), torch.stack([m, l], -1).reshape(-1)])
    sinks, gates = (rand(heads) if sink else None), (rand(heads) if gate else None)
    K, M = heads * vdim, 72
    W = rand(M, K, scale=K ** -0.5).to(dtype)
    out = ops.linear(ops.SplitRow(part, splits, heads, vdim, sinks, gates, dtype), W)
    top = m.double().amax(1, keepdim=True)
    if sink:
        top = torch.maximum(top, sinks.double()[:, None])
    w = (m.double() - top).exp()
    den = (w * l.double()).sum(1) + ((sinks.double() - top[:, 0]).exp() if sink else 0)
    o = (w[..., None] * sums.double()).sum(1) / den[:, None]
    if gate:
        o = o * gates.double().sigmoid()[:, None]
    want = o.reshape(1, K) @ W.double().t()
    # the row is rounded to the weights' type (2^-9 a value, as the merging launch does), then the product
    bound = 2 ** -8 if dtype == torch.bfloat16 else 2e-6
    assert (out.double() - want).norm() <= bound * want.norm()


@pytest.mark.parametrize("window,seen", [(512, 1), (512, 65), (512, 511), (512, 700), (321, 321)])
def test_deferred_row_is_the_row(window, seen):
    H, G, dim = 16, 4, 128
    g = torch.Generator(device="cuda").manual_seed(seen)
    kr, vr = (torch.randn(window, G * dim, device="cuda", generator=g).bfloat16() for _ in range(2))
    row = torch.randn(1, (H + 2 * G) * dim, device="cuda", generator=g)
    sink = torch.randn(H, device="cuda", generator=g)
    W = (torch.randn(256, H * dim, device="cuda", generator=g) * 0.02).bfloat16()
    pos = torch.tensor([seen - 1], dtype=torch.int32, device="cuda")
    rings = [(kr.clone(), vr.clone()) for _ in range(2)]
    got = [ops.window_attention_row(row, *rings[i], H, G, dim, 0.09, 1e-5, sink, window, pos, 0, defer=bool(i)) for i in range(2)]
    assert isinstance(got[0], torch.Tensor) and isinstance(got[1], ops.SplitRow)
    assert all(torch.equal(a, b) for a, b in zip(*rings))  # this token's key and value
    a, b = (ops.linear(x, W).float() for x in got)
    assert (a - b).norm() <= 2 ** -8 * a.norm()


def test_refused():
    part, W = torch.zeros(2 * 16 * 10, device="cuda"), torch.zeros(8, 32, device="cuda")
    for splits, stride in ((1, 16), (129, 16), (2, 12), (2, 24), (2, 0)):
        a = L.RowArgs(part.data_ptr(), W.data_ptr(), 32, 8, 32)
        a.out, a.norm_dim, a.head_stride = W.data_ptr(), splits, stride
        assert L.lib.dv_mix_linear_row(L.F32, L.ROW_SPLITS, L.OUT_T, a, None) != 0
