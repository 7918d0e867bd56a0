"""One row times few long rows of a weight, which two waves share: at the ends of its columns and rows, with what comes before and after."""
import pytest
import torch

from dejavu_amd import _lib_mixers as L
from dejavu_amd import mixer_ops as ops

pytestmark = pytest.mark.gpu


def _weight(M, K):
    g = torch.Generator(device="cuda").manual_seed(M + K)
    return (torch.randn(M, K, device="cuda", generator=g) * K ** -0.5).bfloat16(), torch.randn(1, K, device="cuda", generator=g)


@pytest.mark.parametrize("K", [2048, 2056, 3072, 3080, 5632, 6136, 6144, 6152])
@pytest.mark.parametrize("M", [1, 2, 3, 5, 2047, 2048, 2049])
def test_products_of_shared_rows(M, K):
    W, x = _weight(M, K)
    x = x.bfloat16()
    bias = torch.randn(M, device="cuda").bfloat16()
    want = x.double() @ W.double().t()
    # fp32 sums of K products whose squares add up to about one: 2^-24 sqrt(K) a few times over
    assert float((ops.linear(x, W, f32=True).double() - want).abs().max()) < 2e-5
    assert bool(((ops.linear(x, W, bias).double() - want - bias.double()).abs() <= 2.0 ** -8 * (want + bias.double()).abs() + 2e-5).all())


@pytest.mark.parametrize("M,K", [(2048, 5632), (264, 2056), (1032, 6144)])
def test_what_comes_before_and_after(M, K):
    W, x = _weight(M, K)
    u, weight = x * 3.0, torch.rand(K, device="cuda") + 0.5
    normed = (u / (u.double().square().mean() + 1e-5).sqrt() * weight).bfloat16().double()
    row = ops.RmsRow(u, weight, K, 1e-5, torch.bfloat16)
    want = normed @ W.double().t()
    # the row's entries may round the other way where the norm's last bit decides: 2^-8 of one in K
    assert float((ops.linear(row, W, f32=True).double() - want).abs().max()) < 2e-4
    taps, state = torch.randn(M, 4, device="cuda"), torch.randn(M, 3, device="cuda")
    before = state.double().clone()
    got = ops.row_conv(x.bfloat16(), W, taps, state, silu=False)
    y = (x.bfloat16().double() @ W.double().t())[0]
    assert float((got[0].double() - (before * taps[:, :3]).sum(1) - y * taps[:, 3]).abs().max()) < 1e-4
    assert float((state[:, 2].double() - y).abs().max()) < 2e-5 and torch.equal(state[:, :2].double(), before[:, 1:])
    stream = ops.ResidualStream(torch.randn(1, M, device="cuda"), None, torch.bfloat16)

    class Norm:
        w, b = torch.rand(M, device="cuda"), torch.rand(M, device="cuda")

        def struct(self):
            return L.DynTanh(self.w.data_ptr(), self.b.data_ptr(), 0.7)

    norm, start = Norm(), stream.x.double().clone()
    h = ops.linear_residual(x.bfloat16(), W, stream, norm, norm)
    wanted = start + torch.tanh(0.7 * y) * norm.w + norm.b
    assert float((stream.x.double() - wanted).abs().max()) < 1e-4
    assert float((h.double() - torch.tanh(0.7 * wanted) * norm.w - norm.b).abs().max()) < 2.0 ** -7 + 1e-4
