"""fp32 products by parts in fp16 at the edges of their tiles, chunks and splits, and with values that the parts do not hold,
against float64 products."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

# parts: 2^-24 of a value each; sums of up to 2048 products one after the other, half an ulp of a growing sum each
LIMIT = 6e-7


@pytest.fixture()
def ops(monkeypatch):
    from dejavu_amd import mixer_ops

    for name in ("SPLIT_MIN_ROWS", "SPLIT_COLUMNS", "SPLIT_WORK"):
        monkeypatch.setattr(mixer_ops, name, 1)
    return mixer_ops


def operands(n, M, K, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + n + M + K)
    x = torch.randn(n, K, generator=g, device="cuda")
    W, b = torch.randn(M, K, generator=g, device="cuda") * K ** -0.5, torch.randn(M, generator=g, device="cuda")
    return x, W, b


def close(got, want):
    assert (got.double() - want).norm() <= LIMIT * want.norm()


@pytest.mark.parametrize("n,M,K", [
    (1, 4, 4), (5, 132, 36),        # one tile that is nearly empty, a last chunk of one piece
    (128, 128, 512), (129, 128, 512),  # both tiles of x, two splits
    (256, 260, 2048), (257, 124, 1032),  # a second tile of one row, eight splits; four
    (300, 33000, 64), (600, 8192, 260),  # more than a round of tiles, no split
])
def test_products_at_the_edges(ops, n, M, K):
    x, W, b = operands(n, M, K)
    want = x.double() @ W.double().t()
    close(ops._split_product(x, W), want)
    close(ops._split_product(x, W, b), want + b.double())
    wide, out = torch.randn(n, K + 8, device="cuda"), torch.randn(M, K + 4, device="cuda")
    wide[:, 4:K + 4], out[:, :K] = x, W
    assert torch.equal(ops._split_product(wide[:, 4:K + 4], out[:, :K]), ops._split_product(x, W))


@pytest.mark.parametrize("K", [64, 1032])
def test_values_that_parts_do_not_hold(ops, K):
    """Infinities and NaN reach the results that they reach in the library; rows of any size are as exact as others."""
    x, W, _ = operands(140, 260, K)
    for at, value in (((3, 5), float("inf")), ((130, K - 1), float("-inf")), ((7, 0), float("nan"))):
        bad = x.clone()
        bad[at] = value
        assert torch.equal(ops._split_product(bad, W).nan_to_num(7.0, 8.0, 9.0).abs() > 1e30, F.linear(bad, W).nan_to_num(7.0, 8.0, 9.0).abs() > 1e30)
        for a, b in ((bad, W), (W, bad)):
            got, want = ops._split_product(a, b), F.linear(a, b)
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
            finite = want.isfinite()
            close(torch.where(finite, got, 0.0), torch.where(finite, a.double() @ b.double().t(), 0.0))
    for size in (1e-36, 1e-25, 1e20, 3e37):
        scaled = x.clone()
        scaled[2::3] *= size / x.abs().max()
        got, want = ops._split_product(scaled, W), scaled.double() @ W.double().t()
        for rows in (slice(2, None, 3), slice(0, None, 3)):
            assert (got[rows].double() - want[rows]).norm() <= 2 * LIMIT * want[rows].norm(), size
    ranged = x * torch.logspace(-12, 0, K, device="cuda")
    close(ops._split_product(ranged, W), ranged.double() @ W.double().t())
    assert not ops._split_product(torch.zeros_like(x), W).any()


def test_sums_are_no_further_off_than_the_library(ops):
    for n, M, K in ((500, 1024, 2048), (161, 512, 5632), (300, 256, 4096)):
        x, W, _ = operands(n, M, K)
        want = x.double() @ W.double().t()
        assert (ops._split_product(x, W).double() - want).norm() <= 1.05 * (F.linear(x, W).double() - want).norm()
