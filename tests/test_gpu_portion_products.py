"""Products of a portion's rows at the edges of their tiles, splits and dispatch rules, against float64 products of the
same bf16 operands."""
import numpy as np
import pytest
import torch

from oracle import vimulorn_oracle as V
from tests.mixer_utils import OP_LIMIT, close, host
from tests.test_gpu_vimulorn import _norm

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


# fp32 sums of K products of bf16 values: rounding stays below sqrt(K) 2^-24 of a row's rms (1e-5 up to K = 28000);
# results in bf16: OP_LIMIT
@pytest.mark.parametrize("n,K,M", [
    (2, 8, 4),            # one piece of a chunk, one lane group of rows
    (16, 520, 30),        # a tile of 32 rows that is not full, two splits, a last chunk of one piece
    (15, 2048, 4100),     # 129 tiles, four splits
    (13, 264, 8202),      # tiles enough for one split
    (17, 2056, 66),       # 32 columns; a second tile of two rows; eight splits
    (32, 136, 18440),     # one split
    (33, 1096, 62),       # 64 columns, four splits
    (64, 4104, 132),      # eight splits
    (47, 264, 16388),     # the taller tile, the last one of four rows
    (64, 72, 16384 + 96 * 3),
    (65, 264, 70), (128, 2056, 4100), (96, 4104, 12296),      # 128 columns: 64, 128 and 192 rows of W
    (129, 1032, 4100), (192, 2048, 5122), (140, 4096, 18436),  # 192 columns
    (193, 8, 1 << 20), (256, 2056, 4100), (256, 1544, 5442),   # 256 columns: 64 and 128 rows
    (256, 264, 72), (257, 520, 72),                            # the library (fp32 results: tiles of 64 columns)
])
def test_edges(n, K, M):
    from dejavu_amd import mixer_ops as ops

    g = torch.Generator().manual_seed(n * 11 + M)
    wide = torch.randn(n, K + 16, generator=g).to(BF16).cuda()
    x = wide[:, 8:8 + K]  # rows further apart than they are long
    W = (torch.randn(M, K, generator=g) * K ** -0.5).to(BF16).cuda()
    bias = torch.randn(M, generator=g).to(BF16).cuda()
    prod = host(x) @ host(W).T
    close(ops.linear(x, W, f32=True), prod, 1e-5, f"{n}x{K}x{M}, fp32 result")
    close(ops.linear(x, W, bias), prod + host(bias), OP_LIMIT[BF16], "with a bias")
    gate, up = np.minimum(prod[:, 0::2], 0.75), np.clip(prod[:, 1::2], -0.75, 0.75)
    close(ops.clamped_glu(x, W, 0.75), gate * V.sigmoid(1.702 * gate) * (up + 1), OP_LIMIT[BF16], "gated unit")
    (post, f_post), (pre, f_pre) = _norm(M, 1), _norm(M, 2)
    x0 = torch.randn(n, M, generator=g).cuda()
    stream = ops.ResidualStream(x0.clone(), None, BF16)
    h = ops.linear_residual(x, W, stream, post, pre)
    want = host(x0) + f_post(prod)
    close(stream.x, want, OP_LIMIT[BF16], "residual")
    close(h, f_pre(want), OP_LIMIT[BF16], "next norm")


@pytest.mark.parametrize("n,K,M", [
    (1, 8, 4), (256, 64, 256), (257, 72, 260), (300, 128, 514), (511, 200, 30),  # edges of tiles and chunks
    (700, 1032, 2564),                                                          # 33 tiles: blocks of eight and a last one
])
def test_wide_tiles(n, K, M):
    from dejavu_amd import _lib_mixers as L
    from dejavu_amd import mixer_ops as ops

    g = torch.Generator().manual_seed(n + M)
    x = torch.randn(n, K + 8, generator=g).to(BF16).cuda()[:, :K]
    W = (torch.randn(M, K, generator=g) * K ** -0.5).to(BF16).cuda()
    bias = torch.randn(M, generator=g).to(BF16).cuda()
    prod = host(x) @ host(W).T
    for after, want in ((L.OUT_T, prod + host(bias)), (L.OUT_GLU, np.maximum(prod[:, 0::2], 0) * prod[:, 1::2])):
        out = torch.empty(n, want.shape[1], dtype=BF16, device="cuda")
        a = ops._tile_args(x, W)
        a.out, a.ldo, a.act = out.data_ptr(), out.shape[1], L.GLU_RELU
        a.bias = bias.data_ptr() if after == L.OUT_T else None
        ops.check(ops.lib.dv_mix_linear_wide(after, ops._ref(a), ops._stream()), "dv_mix_linear_wide")
        close(out, want, OP_LIMIT[BF16], f"{n}x{K}x{M}, after {after}")


def test_wide_products_through_the_ops():
    """A product on each side of the rule: 584 tiles of 1920 and 1922 rows, which ten and eleven tiles of 192 rows cover; the
    first go to the library, the others to the wide kernel, both with the same result."""
    from dejavu_amd import mixer_ops as ops

    g = torch.Generator(device="cuda").manual_seed(1)
    W = (torch.randn(18500, 4096, generator=g, device="cuda") / 64).to(BF16)
    x = torch.randn(1922, 4096, generator=g, device="cuda").to(BF16)
    assert not ops._wide(x[:1920], W) and ops._wide(x, W) and not ops._wide(x[:, :2048], W[:, :2048])
    for rows in (1920, 1922):
        want = x[:rows].float() @ W.float().t()
        got = ops.linear(x[:rows], W).float()
        assert (got - want).norm() / want.norm() < 3e-3  # one rounding to bf16
        unit = want[:, 0::2].clamp(min=0) * want[:, 1::2]
        got = ops.relu_glu(x[:rows], W).float()
        assert (got - unit).norm() / unit.norm() < 1e-2


@pytest.mark.parametrize("n,K,M,gated", [
    (129, 4096, 68, False), (192, 2048, 2048, False), (193, 4096, 2048, False), (256, 8200, 1026, False), (241, 4096, 4104, False),
    (200, 2048, 8192, False), (65, 520, 12288, True), (128, 264, 12296, True), (193, 4096, 12288, True), (256, 4104, 2050, True),
    (193, 2048, 8192, True),
    (131, 72, 12290, True), (210, 2048, 5122, False)])  # sizes that the launch behind the library's product refuses
def test_streamed_products_through_the_ops(n, K, M, gated):
    """The rows, columns and weights at which the rule ends, with each epilogue behind the tiles."""
    from dejavu_amd import mixer_ops as ops

    g = torch.Generator().manual_seed(n + M)
    x = torch.randn(n, K, generator=g).to(BF16).cuda()
    W = (torch.randn(M, K, generator=g) * K ** -0.5).to(BF16).cuda()
    assert ops._tiles(x, W, gated=gated) or (n * M // 2 if gated else M) % 4
    prod = host(x) @ host(W).T
    if gated:
        close(ops.relu_glu(x, W), np.maximum(prod[:, 0::2], 0) * prod[:, 1::2], OP_LIMIT[BF16], "gated unit")
        return
    close(ops.linear(x, W), prod, OP_LIMIT[BF16], "plain")
    (post, f_post), (pre, f_pre) = _norm(M, 1), _norm(M, 2)
    x0 = torch.randn(n, M, generator=g).cuda()
    stream = ops.ResidualStream(x0.clone(), None, BF16)
    h = ops.linear_residual(x, W, stream, post, pre)
    want = host(x0) + f_post(prod)
    close(stream.x, want, OP_LIMIT[BF16], "residual")
    close(h, f_pre(want), OP_LIMIT[BF16], "next norm")


def test_unaligned_operands():
    """What the streaming kernel refuses is still multiplied where several kernels could."""
    from dejavu_amd import mixer_ops as ops

    g = torch.Generator().manual_seed(3)
    x, W = torch.randn(70, 65, generator=g).to(BF16).cuda()[:, 1:], torch.randn(48, 64, generator=g).to(BF16).cuda()
    close(ops.linear(x, W), host(x) @ host(W).T, OP_LIMIT[BF16], "rows that start at odd places")


def test_odd_places_of_the_result():
    """Outputs whose rows do not start where four values can be stored at once."""
    from dejavu_amd import _lib_mixers as L
    from dejavu_amd import mixer_ops as ops

    n, K, M = 19, 512, 70
    g = torch.Generator().manual_seed(5)
    x, W = torch.randn(n, K, generator=g).to(BF16).cuda(), torch.randn(M, K, generator=g).to(BF16).cuda()
    prod = host(x) @ host(W).T
    for after, dtype, ldo in ((L.OUT_T, BF16, 71), (L.OUT_T, BF16, 72), (L.OUT_F32, torch.float32, 73), (L.OUT_GLU, BF16, 37)):
        out = torch.zeros(n * ldo + 1, dtype=dtype, device="cuda")
        a = ops._tile_args(x, W)
        a.out, a.ldo, a.act = out.data_ptr() + out.element_size(), ldo, L.GLU_RELU
        ops._tile_launch(after, a, x.device)
        got = out[1:].view(n, ldo)
        want = np.maximum(prod[:, 0::2], 0) * prod[:, 1::2] if after == L.OUT_GLU else prod
        close(got[:, :want.shape[1]], want, 1e-5 if dtype == torch.float32 else OP_LIMIT[BF16], f"after {after}, rows {ldo} apart")
        assert not got[:, want.shape[1]:].any(), "stored past the end of a row"


@pytest.mark.parametrize("n,K,M", [
    (2, 2048, 32768), (16, 4096, 11008), (47, 4096, 22016), (100, 4096, 32768),  # one split
    (24, 12288, 8192), (250, 4096, 11008),                                       # two
    (64, 4096, 4096), (100, 4096, 4096),                                         # four, and eight
])
def test_fp32_results_of_long_rows(n, K, M):
    """Sums of at most a quarter of K: the error in 64 bits is 2.9e-9 sqrt(K) of the result (1.9e-7 with 4096 columns), with
    sums of half of K 4.3e-9 and with one sum 6.1e-9.  The limit lies between, at 3.8e-9."""
    from dejavu_amd import mixer_ops as ops

    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n, K, generator=g, device="cuda").to(BF16)
    W = (torch.randn(M, K, generator=g, device="cuda") * K ** -0.5).to(BF16)
    want = x.double() @ W.double().t()
    assert (ops.linear(x, W, f32=True) - want).norm() / want.norm() < 3.8e-9 * K ** 0.5
