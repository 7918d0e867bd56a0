"""fp32 products by parts in bf16 at the edges of their tiles, chunks and splits, and with values of any range, infinite ones
and NaN, against float64 products."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

# parts hold all of a value; sums of up to 2048 products one after the other, half an ulp of a growing sum each
LIMIT = 6e-7
# of the sum of a result's magnitudes: 2^-24 of each product for the parts that are left out, sqrt(2048) / 2 roundings of 2^-24 for the sum,
# of which the values of one result reach a few times as many
SUMS = 2.0 ** -19


@pytest.fixture()
def ops(monkeypatch):
    from dejavu_amd import mixer_ops

    for name in ("SPLIT_MIN_ROWS", "SPLIT_COLUMNS", "SPLIT_RATE"):
        monkeypatch.setattr(mixer_ops, name, 1)
    monkeypatch.setattr(mixer_ops, "_split_us", lambda n, M, K: 1)
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
    (256, 260, 2048), (257, 124, 1032),  # a second tile of four rows, eight splits; of one column, four
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


@pytest.mark.parametrize("K", [36, 64, 1032])
def test_values_that_are_not_finite(ops, K):
    """Infinities and NaN reach the results that they reach in the library, and change no others."""
    x, W, _ = operands(140, 260, K)
    clean = ops._split_product(x, W), ops._split_product(W, x)
    # inf, -inf, NaN, and one that only its lower half tells from an infinity
    for at, bits in (((3, 5), 0x7f800000), ((130, K - 1), -0x800000), ((7, 0), 0x7fc00000), ((9, K // 2), 0x7f800001)):
        bad = x.clone()
        bad.view(torch.int32)[at] = bits
        for (a, b), usual, axis in (((bad, W), clean[0], 0), ((W, bad), clean[1], 1)):
            got, want = ops._split_product(a, b), F.linear(a, b)
            for what in (torch.isnan, torch.isposinf, torch.isneginf):
                assert torch.equal(what(got), what(want)), (at, hex(bits))
            assert not got.select(axis, at[0]).isfinite().any()
            others = [i for i in range(140) if i != at[0]]
            assert torch.equal(got.index_select(axis, torch.tensor(others, device="cuda")),
                               usual.index_select(axis, torch.tensor(others, device="cuda"))), (at, hex(bits))
    assert not ops._split_product(torch.zeros_like(x), W).any()


@pytest.mark.parametrize("K", [64, 1032])
def test_rows_of_any_size(ops, K):
    x, W, _ = operands(140, 260, K)
    for size in (1e-37, 1e-36, 1e-25, 1e20, 3e37):
        scaled = x.clone()
        scaled[2::3] *= size / x.abs().max()
        got, want = ops._split_product(scaled, W), scaled.double() @ W.double().t()
        for rows in (slice(2, None, 3), slice(0, None, 3)):
            assert (got[rows].double() - want[rows]).norm() <= 2 * LIMIT * want[rows].norm(), size
    # products near the largest number, of values whose first parts round up
    for a, b in ((1.9999 * 2.0 ** 63, 1.9999 * 2.0 ** 63), (3.4e38, 1.0), (1.0, 3.4e38), (3.4e38, 0.3)):
        A, B = torch.zeros(4, K, device="cuda"), torch.zeros(4, K, device="cuda")
        A[:, 0], B[:, 0] = a, b
        want = A.double() @ B.double().t()
        assert ((ops._split_product(A, B).double() - want).abs() <= 2.0 ** -22 * want).all() and want.max() > 1e38


def ranges(K):
    """Factors of the columns of x, whose inverse the columns of W have: their products are as large as ever."""
    g = torch.Generator(device="cuda").manual_seed(K)
    for decades in (4, 6, 15, 30):
        yield 10.0 ** (decades * (2 * torch.rand(K, generator=g, device="cuda") - 1))
    for power in (15, 20, 24, 30, 40, 100):
        one = torch.ones(K, device="cuda")
        one[5] = 2.0 ** power
        yield one


@pytest.mark.parametrize("K", [64, 1032, 2048])
def test_rows_of_a_wide_range(ops, K):
    """Values far below the largest of their row keep all their bits: each row is as near as with values of one size, and each
    result within what sums of its products' magnitudes allow."""
    x, W, _ = operands(140, 260, K)
    cases = [(x * r, W / r) for r in ranges(K)] + [(x / r, W * r) for r in ranges(K)]
    for huge in (1e8, 1e12, 1e30):  # a column that counts for nothing
        a, b = x.clone(), W.clone()
        a[:, 7], b[:, 7] = huge, 0.0
        cases += [(a, b), (b, a)]
    cases.append((x * torch.logspace(-12, 0, K, device="cuda"), W))
    for i, (a, b) in enumerate(cases):
        got, want = ops._split_product(a, b).double(), a.double() @ b.double().t()
        assert ((got - want).norm(dim=1) <= LIMIT * want.norm(dim=1)).all(), i
        assert ((got - want).abs() <= SUMS * (a.double().abs() @ b.double().abs().t())).all(), i


def test_sums_are_no_further_off_than_the_library(ops):
    for n, M, K in ((500, 1024, 2048), (161, 512, 5632), (300, 256, 4096)):
        x, W, _ = operands(n, M, K)
        want = x.double() @ W.double().t()
        assert (ops._split_product(x, W).double() - want).norm() <= 1.05 * (F.linear(x, W).double() - want).norm()


def test_the_rule_takes_what_the_kernel_takes(ops, monkeypatch):
    """Sizes, strides and places that the kernel would refuse are the library's."""
    x, W, b = operands(8, 16, 64)
    assert ops._split_product(x, W, b) is not None
    wide, odd = torch.randn(8, 66, device="cuda"), torch.randn(16 * 64 + 1, device="cuda")
    for args in ((x[:, :62], W[:, :62]), (x, W[:14]), (wide[:, :64], W), (x, odd[1:].view(16, 64)), (x, W, odd[1:17]), (x.double(), W.double()),
                 (x, W.clone().requires_grad_())):
        assert ops._split_product(*args) is None
    monkeypatch.setattr(ops, "SPLIT_VALUES", x.numel() - 1)
    assert ops._split_product(x, W) is None


@pytest.mark.parametrize("n,M,K,taken", [(500, 11264, 2048, True), (500, 2048, 5632, True), (384, 4368, 2048, True), (400, 4368, 2048, False), (512, 4368, 2048, True),
                                         (160, 22016, 4096, False), (161, 22016, 4096, False), (500, 2048, 2048, False), (500, 0, 2048, False)])
def test_which_products_are_split(n, M, K, taken):
    from dejavu_amd import mixer_ops

    assert mixer_ops._split_rule(n, M, K) == taken


@pytest.mark.parametrize("stride,taken", [(2 ** 25 - 4, True), (2 ** 25, False)])
def test_rows_of_a_weight_that_are_far_apart(ops, stride, taken):
    """32 rows' bytes are counted in 32 bits."""
    x, W, _ = operands(8, 40, 68)
    room = torch.empty(39 * stride + 68, device="cuda")
    far = room.as_strided((40, 68), (stride, 1))
    far.copy_(W)
    got = ops._split_product(x, far)
    assert (got is not None) == taken
    if taken:
        assert torch.equal(got, ops._split_product(x, W))


@pytest.mark.parametrize("n,M,K,stride", [(130, 40, 68, 2 ** 25), (2 ** 24 + 131, 8, 36, 36), (5, 12, 2 ** 25 + 4, 2 ** 25 + 8)])
def test_strides_and_sizes_beyond_32_bits(n, M, K, stride):
    """Through the entry point itself, which takes what counts more bytes than 32 bits do.  Whole numbers: every sum is exact."""
    from dejavu_amd import mixer_ops as o

    g = torch.Generator(device="cuda").manual_seed(n)
    rand = lambda *s: torch.randint(-2, 3, s, generator=g, device="cuda").float()  # noqa: E731
    x, W, bias = rand(n, K), rand(M, K), rand(M)
    far = torch.empty((M - 1) * stride + K, device="cuda").as_strided((M, K), (stride, 1)).copy_(W)
    out = torch.full((n, M), 77.0, device="cuda")
    nbytes = o.lib.dv_mix_linear_split_workspace_bytes(n, M, K)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    o.check(o.lib.dv_mix_linear_split(x.data_ptr(), K, far.data_ptr(), stride, bias.data_ptr(), n, M, K, out.data_ptr(), M, ws.data_ptr(),
                                      nbytes, o._stream()), "dv_mix_linear_split")
    assert torch.equal(out, F.linear(x.double(), W.double(), bias.double()).float())
