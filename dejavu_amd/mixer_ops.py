"""Tensor interface of libdejavu_mixers.so.

Weights and activations are bf16 or fp32 (one type per model); the residual stream, norms, scores and recurrent state
are fp32.  All ops enqueue on ``torch.cuda.current_stream()`` and refuse CPU tensors.  Products: one row goes to the
row kernel, up to 64 bf16 rows, and up to ``TILE_MAX_ROWS`` where it is the faster one (``_tile_rule``), to the matrix-core
kernel that streams the weight, longer portions where they fill it to the one with wide tiles (``_wide_rule``, ``_fill_rule``), all
with the operation that follows in the same launch; the other portions (and several fp32 rows) take the library GEMM and a
separate elementwise launch, as the dense products of long prompts do elsewhere in this package.
"""
from __future__ import annotations

import ctypes
from functools import lru_cache
from typing import Optional

import torch
import torch.nn.functional as F

from . import _lib_mixers as L
from ._binding import results_only
from ._lib_mixers import check, lib

# Beyond 64 rows the streaming kernel where it is ahead of the library GEMM and the launch that follows it, with weights that are
# not in the caches (us, library / kernel, or times the library's speed; its call costs the host 5 to 15 us less):
#   up to 192 rows weights of up to 12288 rows: the gated unit of 6144 x 4096 with 65 / 128 / 192 rows 1.25 / 1.32 / 1.45, of 11264 x 2048
#   1.07 / 1.01 / 1.13; norm and residual of 4096 x 4096 with 96 / 192 rows 26 / 20 and 38 / 27, 4096 x 11008 54 / 33 and 86 / 40, 2048 x 2048
#   14.6 / 11.5 and 16 / 14 (with 2048 columns also where it is behind, 4096 x 2048 with 130 rows 18 / 21: such models wait for the host).
#   Of taller weights the tiles make more than a round, and the library's larger ones read x less often (22016 x 4096 with 65 / 128 /
#   192 rows 0.88 / 0.89 / 1.00, plain 0.83 / 0.82 / 0.95; 50000 x 2048 0.9): it takes them, but gated units of 129 to 192 rows only: with fewer the
#   calls are the time, with more it is not ahead inside a model (a prompt of vimulorn-4k by itself with 65 / 100 / 128 / 160 tokens 1.71 /
#   1.77 / 1.83 / 2.04 ms with the kernel, 1.86 / 1.89 / 1.87 / 1.98 with the library; among others 200 / 256 tokens 2.00 / 2.09 and 2.02 / 2.13);
#   beyond 192: 4096 x 11008 52 / 44, 4096 x 8192 39 / 38, 3072 x 4096 26 / 24, 2048 x 5632 24 / 21, gated 4096 x 4096 1.02 and 11264 x 2048
#   1.06, 8192 x 4096 with 208 / 256 rows 0.94 / 1.29; but 2048 x 2048 with 256 rows 0.9 and 4096 x 2048 0.7.
TILE_MAX_ROWS = 256
TILE_MAX_WEIGHT_ROWS, TILE_TALL_ROWS = 12288, 128
TILE_ALL_ROWS = 192                # up to here whatever the weight's size
TILE_WEIGHT, TILE_COLUMNS = 1 << 23, 4096   # elements from which the rows may be more; twice as many where the columns are fewer

_DTYPES = {torch.bfloat16: L.BF16, torch.float32: L.F32}
_ref = ctypes.byref


def padded(size: int) -> int:
    """Sizes along vectorised dimensions are multiples of 8 in memory."""
    return (size + 7) // 8 * 8


def _code(t: torch.Tensor) -> int:
    if not t.is_cuda:
        raise RuntimeError("dejavu_amd ops run on the GPU only; got a CPU tensor (there is no CPU fallback)")
    return _DTYPES[t.dtype]


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def _stream() -> int:
    """``torch.cuda.current_stream().cuda_stream`` without the Stream object (0.3 instead of 4 us a launch)."""
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def _f32(*tensors):
    for t in tensors:
        assert t is None or (t.dtype == torch.float32 and t.is_cuda and t.is_contiguous()), "fp32 contiguous expected"


class ResidualStream:
    """The fp32 residual rows of a portion; ``start`` is a copy of the embedding output for models that add it again."""

    def __init__(self, x: torch.Tensor, start: Optional[torch.Tensor], dtype: torch.dtype):
        self.x, self.start, self.dtype = x, start, dtype

    def args(self, post, pre, add_start: bool, h: Optional[torch.Tensor]) -> L.Residual:
        r = L.Residual(self.x.data_ptr(), self.start.data_ptr() if add_start else None, None if h is None else h.data_ptr())
        if post is not None:
            r.post = post.struct()
        if pre is not None:
            r.pre = pre.struct()
        return r

    def new_h(self) -> torch.Tensor:
        return torch.empty(self.x.shape, dtype=self.dtype, device=self.x.device)


def embed(tokens: torch.Tensor, weight: torch.Tensor, norm, keep_start: bool):
    """tokens (n,) int64 -> (ResidualStream, norm(x))."""
    code = _code(weight)
    assert tokens.dtype == torch.int64 and tokens.is_cuda and tokens.is_contiguous() and weight.is_contiguous()
    n, width = tokens.numel(), weight.shape[1]
    x = torch.empty(n, width, dtype=torch.float32, device=weight.device)
    stream = ResidualStream(x, torch.empty_like(x) if keep_start else None, weight.dtype)
    h = stream.new_h()
    check(lib.dv_mix_embed(code, _ptr(tokens), weight.shape[0], _ptr(weight), n, width, _ptr(x), _ptr(stream.start),
                           _ref(norm.struct()), _ptr(h), _stream()), "dv_mix_embed")
    return stream, h


def residual(y: Optional[torch.Tensor], stream: ResidualStream, post, pre, add_start: bool = False):
    """x += post(y) (y may be None); x += start; returns pre(x) (None without ``pre``)."""
    h = None if pre is None else stream.new_h()
    assert y is None or (y.is_contiguous() and y.shape == stream.x.shape and y.dtype == stream.dtype)
    n, width = stream.x.shape
    check(lib.dv_mix_residual(_DTYPES[stream.dtype], _ptr(y), n, width, _ref(stream.args(post, pre, add_start, h)),
                              _stream()), "dv_mix_residual")
    return h


# Tiles of 256 weight rows (gemm_wide.hpp) against the library GEMM, weights out of the caches (the library's time over the
# kernel's).  The library also has tiles 192 wide; where the kernel's make three rounds of the compute units, and those of 192 by 256 four
# either way, its choice costs it most: 22016 x 4096 with 1700 / 1999 / 2048 rows 1.24 / 1.40 / 1.42, 18560 x 4096 1.22 / 1.38 / 1.29.  Outside of
# these lines a plain product of 4096 columns and more is ahead as often as it is behind (22016 x 4096 with 640 / 777 / 1000 / 1200 / 1435 rows 1.00 / 1.03 / 0.97 /
# 0.93 / 1.31, 12288 x 4096 with 257 / 777 / 1200 / 1435 / 1999 rows 0.91 / 1.03 / 0.95 / 1.12 / 0.95, 8192 x 4096 0.73 / 1.08 / 1.05 / 1.04 / 0.93, 4096 x 11008 with 777 / 2048
# rows 0.70 / 0.99).
WIDE_MAX_ROWS = 2048
WIDE_MAX_STRIDE = 1 << 25             # elements (the kernel counts 64 rows' bytes in 32 bits)
WIDE_COLUMNS = 4096, 5120
WIDE_MAX_WEIGHT_ROWS = 22528
WIDE_TILE, NARROW_TILE, WIDE_ROUND = 256, 192, 256
WIDE_TILES = 2 * WIDE_ROUND + 1, 3 * WIDE_ROUND - 10  # (a third round that is all but full is the library's again)


def _remembered(rule):
    """A rule's answers are kept by its sizes, but those of symbolic sizes, which have no hash (to look at the types first costs
    0.3 us a product, which is as much as a rule)."""
    known = lru_cache(maxsize=4096)(rule)

    def ask(n, M, K, *more):
        try:
            return known(n, M, K, *more)
        except TypeError:
            return rule(n, M, K, *more)

    return ask


def _tiles_of(n: int, M: int, rows: int, weight_rows: int) -> int:
    return -(-n // rows) * -(-M // weight_rows)


@_remembered
def _wide_rule(n: int, M: int, K: int) -> bool:
    if n > WIDE_MAX_ROWS or M > WIDE_MAX_WEIGHT_ROWS or M % NARROW_TILE == 0 or not WIDE_COLUMNS[0] <= K <= WIDE_COLUMNS[1]:
        return False
    narrow = min(_tiles_of(n, M, NARROW_TILE, WIDE_TILE), _tiles_of(n, M, WIDE_TILE, NARROW_TILE))
    return WIDE_TILES[0] <= _tiles_of(n, M, WIDE_TILE, WIDE_TILE) <= WIDE_TILES[1] and narrow > 3 * WIDE_ROUND


# Where the library's product is followed by a launch of its own for the gated unit, and for few columns, the kernel is ahead as
# soon as its tiles fill the chip (at least so many tiles of 128 rows by 256 weight rows, by columns).  The library's time over the kernel's, weights
# cold, of 37 numbers of rows from 257 to 2048 those that are taken:
#   gated, 4096 columns: 28672 / 22016 / 20480 / 18560 / 17920 / 16384 / 14336 / 12288 / 10240 / 8192 weight rows from 0.95 / 0.96 / 0.97 / 1.05 / 0.98 / 0.98 / 0.98 / 0.99 / 0.98 / 1.03 on,
#     up to 1.15 (8192) and 1.61; 18944 x 4608 0.97 to 1.51.  Left for their few tiles: 8192 weight rows with up to 768 rows 0.73 to 1.07.
#   gated, 2048 columns: 11264 / 9216 / 8192 / 6144 / 4368 weight rows from 1.05 / 1.09 / 1.05 / 1.06 / 1.12 on, up to 1.5; 16384 and 8192 x 1024 from 1.04 and 1.15 on.
#     Left: 6144 weight rows with up to 640 rows 0.92 to 1.02.
#   gated, more columns, where tiles of 256 x 256 leave little of their last round empty: 24576 x 5120 0.97 to 1.15 (else 0.79 to 1.00), 27648 x 5120 0.96 to 1.20 (0.87 to 0.99),
#     13696 x 5120 1.09 to 1.23 (0.77 to 1.02), 16384 x 8192 0.96 to 1.29, 22016 x 8192 1.26 to 1.31 (0.91 to 1.31).
#   plain, where rows and weight rows leave some of such a round empty, 2048 columns: 24576 / 12288 / 11264 / 9216 / 8192 / 6144 / 4368 weight rows from 0.93 / 1.00 / 0.94 / 1.04 / 1.04 / 1.04 /
#     1.17 on, up to 1.2 and 1.7; 5632 x 1536, 10240 x 1280, 16384 and 8192 x 1024 from 1.07, 1.03, 1.05 and 1.20 on.  Left, where the library's larger tiles fill their rounds:
#     2048 rows by 8192 x 2048 / 24576 x 2048 / 16384 x 1024 0.94 / 0.91 / 0.90.
# Gated units of 2049 to 8192 rows: 22016 / 18560 / 16384 / 14336 / 12288 x 4096 from 0.96 / 1.00 / 0.97 / 0.96 / 0.97 on, up to 1.54, 11264 x 2048 1.01 to 1.30, 16384 x 1024 from 1.02 on; 8192 x
# 4096, with fewer tiles, 0.96 to 1.15.
WIDE_FEW_COLUMNS, WIDE_GATED_COLUMNS = 2048, (4608, 8192)
WIDE_LONG_GATED = 8192, 11264, 4096    # rows at most, weight rows at least, columns at most
WIDE_FILL_GATED, WIDE_FILL_FEW_GATED, WIDE_FILL_FEW = 200, 144, 176
WIDE_FULL_GATED, WIDE_FULL_FEW = 0.84, 0.83  # of the rounds of 256 x 256 tiles: tiles at least, rows by weight rows below


@_remembered
def _fill_rule(n: int, M: int, K: int, gated: bool) -> bool:
    columns = WIDE_GATED_COLUMNS if gated else (WIDE_FEW_COLUMNS, WIDE_FEW_COLUMNS)
    if n <= TILE_MAX_ROWS or not 1024 <= K <= columns[1]:
        return False
    most, rows, few = WIDE_LONG_GATED
    if n > (most if gated and M >= rows and K <= few else WIDE_MAX_ROWS):
        return False
    fill = (WIDE_FILL_FEW_GATED if gated else WIDE_FILL_FEW) if K <= WIDE_FEW_COLUMNS else WIDE_FILL_GATED
    if _tiles_of(n, M, 128, WIDE_TILE) < fill:
        return False
    tiles = _tiles_of(n, M, WIDE_TILE, WIDE_TILE)
    places = -(-tiles // WIDE_ROUND) * WIDE_ROUND
    if not gated:
        return n * M < WIDE_FULL_FEW * WIDE_TILE * WIDE_TILE * places
    return K <= columns[0] or tiles >= WIDE_FULL_GATED * places


# Long rows whose tiles leave much of the chip idle: K in parts on the same tiles, the sums added up by the launch that follows (plan_wide_split),
# with the residual in it.  The library's time over the kernels', weights cold, 16 numbers of rows from 257 to 2048 each:
#   plain: 4096 x 11008 / 14336 1.00 to 1.17 and 1.03 to 2.09, 5120 x 13824 1.05 to 2.05, 3072 x 12288 1.14 to 1.34, 3072 / 2560 x 10240 from 385 rows on
#     1.01 to 1.17 and 1.06 to 1.31 (fewer 0.91 to 1.18); but 4096 x 8192 0.80 to 1.18, 2048 x 8192 0.89 to 1.13, 4096 x 4096 0.78 to 1.01;
#   with the residual: 4096 x 8192 1.06 to 1.26, 4096 x 11008 1.06 to 1.17, 4096 x 14336 1.06 to 1.95, 5120 x 13824 1.11 to 1.40, 3072 x 12288 1.14 to 1.40;
#     but 2048 x 5632 0.95 to 1.17, 3072 x 8192 0.96 to 1.17, 4096 x 4096 0.91 to 1.04.
#   Of more weight rows only in three parts and more: 8192 x 28672 in four 1.07 to 1.50, in two 0.87 to 1.10.
PARTS_COLUMNS, PARTS_RESIDUAL_COLUMNS = 10240, 8192
PARTS_WEIGHT, PARTS_LIGHT_WEIGHT, PARTS_LIGHT_ROWS = 1 << 25, 26_000_000, 385   # elements; a lighter one with so many rows at least
PARTS_TALL = 7168, 3                                                            # weight rows, parts at least of more of them


def _parts_rule(n: int, M: int, K: int, residual: bool) -> bool:
    if not TILE_MAX_ROWS < n <= WIDE_MAX_ROWS or M % 8:
        return False
    light = not residual and n >= PARTS_LIGHT_ROWS
    return K >= (PARTS_RESIDUAL_COLUMNS if residual else PARTS_COLUMNS) and M * K >= (PARTS_LIGHT_WEIGHT if light else PARTS_WEIGHT)


@lru_cache(maxsize=4096)
def _parts_workspace_bytes(device: int, n: int, M: int, K: int) -> int:
    """As ``_tile_workspace_bytes``; 0: the tiles are enough for the chip."""
    return lib.dv_mix_linear_wide_workspace_bytes(n, M, K)


def _parts_bytes(x: torch.Tensor, W: torch.Tensor, bias=None, residual: bool = False) -> int:
    """What the wide kernel's parts of the product need; 0: it is not one of its products."""
    n = x.shape[0]
    if x.shape[1] < PARTS_RESIDUAL_COLUMNS or not TILE_MAX_ROWS < n <= WIDE_MAX_ROWS:  # (before anything that costs the host more)
        return 0
    M, K = W.shape
    if not _parts_rule(n, M, K, residual) or not _wide_fits(x, W, bias):  # (tracers go no further)
        return 0
    nbytes = _parts_workspace_bytes(torch._C._cuda_getDevice(), n, M, K)
    return nbytes if nbytes >= (PARTS_TALL[1] if M > PARTS_TALL[0] else 2) * 4 * n * M else 0


def _parts_launch(after, a, nbytes, device) -> None:
    ws = torch.empty(nbytes, dtype=torch.uint8, device=device)
    check(lib.dv_mix_linear_wide_ws(after, _ref(a), _ptr(ws), nbytes, _stream()), "dv_mix_linear_wide_ws")


@_remembered
def _tile_rule(n: int, M: int, K: int, gated: bool) -> bool:
    if n > TILE_MAX_ROWS:
        return False
    if M > TILE_MAX_WEIGHT_ROWS:
        return gated and not TILE_TALL_ROWS < n <= TILE_ALL_ROWS
    return n <= TILE_ALL_ROWS or M * K >= (TILE_WEIGHT if K >= TILE_COLUMNS else 2 * TILE_WEIGHT)


def _aligned(x: torch.Tensor, W: torch.Tensor) -> bool:
    return all(t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0 for t in (x, W)) and x.shape[1] % 8 == 0 and W.shape[0] % 2 == 0


def _wide_fits(x: torch.Tensor, W: torch.Tensor, bias=None) -> bool:
    return (x.dtype == torch.bfloat16 and results_only(x, W, bias) and _aligned(x, W) and
            max(x.stride(0), W.stride(0)) < WIDE_MAX_STRIDE)


def _wide(x: torch.Tensor, W: torch.Tensor, bias=None) -> bool:
    """Whether the wide kernel takes the product whatever follows it."""
    return _wide_rule(x.shape[0], *W.shape) and _wide_fits(x, W, bias)


def _fills(x: torch.Tensor, W: torch.Tensor, bias=None, gated: bool = False) -> bool:
    """Whether the wide kernel takes it for what follows, or for its few columns."""
    return _fill_rule(x.shape[0], *W.shape, gated) and _wide_fits(x, W, bias)


def _tiles(x: torch.Tensor, W: torch.Tensor, bias=None, gated: bool = False, whole: bool = True) -> bool:
    """Whether the streaming kernel takes the product.  From 65 rows on the library takes what it would refuse; whole: a
    separate launch can follow the library (else what the streaming kernel can take is its own)."""
    n = x.shape[0]
    if x.dtype != torch.bfloat16 or n <= 64:
        return x.dtype == torch.bfloat16
    taken = _tile_rule(n, *W.shape, gated) if whole else n <= TILE_MAX_ROWS
    return taken and results_only(x, W, bias) and _aligned(x, W)


def _product_ok(x, W):
    assert x.dim() == 2 and W.dim() == 2 and x.dtype == W.dtype and x.shape[1] == W.shape[1], "product shapes"
    assert x.stride(1) == 1 and W.stride(1) == 1
    return _code(W)


# fp32 products by parts in bf16 (linear_split.hpp), which are as exact as fp32 products for values of any range, where what the launches take
# (``_split_us``: a round of tiles 2.2 us a chunk of columns, splits of K 4 us and 0.05 for each tile, all launches 8) is less than the
# library's fp32 GEMM does at 118 TFLOP/s; it ranges from 85 to 140.  Times the library's speed: 11264 x 2048 with 256 / 400 / 500 /
# 1000 / 2000 rows 1.30 / 1.28 / 1.56 / 1.41 / 1.50, 2048 x 5632 with 400 / 500 / 1000 1.18 / 1.15 / 1.22, 4368 x 2048 with 384 / 500 1.10 /
# 1.58, 22016 x 4096 with 200 / 500 / 1000 / 2048 1.32 / 1.42 / 1.61 / 1.46, 500 by 3072 x 2048 1.18, 300 by 8192 x 4096 1.20, 200 by 4096 x
# 11008 1.32, 4000 by 4096 x 512 1.31.  Left to the library: too little for the launches (500 by 2048 x 2048 0.91, 256 by 2048 x 5632 0.93, 200
# by 4368 x 2048 0.89, 2000 by 1024 x 1024 0.87), and where its own speed, which jumps with the sizes, decides (161 by 11264 x 2048 1.13, 161 by
# 22016 x 4096 1.08, 400 by 4368 x 2048 1.02).  On the line: 300 by 22016 x 4096 1.07, 300 by 4096 x 4096 1.07, 2000 by 2048 x 768 1.00.
SPLIT_MIN_ROWS, SPLIT_COLUMNS = 161, 512
SPLIT_RATE = 59_000_000        # products a us (118 TFLOP/s) that the tiles have to reach
SPLIT_VALUES = 1 << 27         # of x, whose parts take 6 bytes each: beyond, the library, which needs no memory for them
SPLIT_TILE, SPLIT_CHUNK, SPLIT_ROUND = (256, 128), 32, 256
SPLIT_MAX_STRIDE = 1 << 25     # 32 rows' bytes are counted in 32 bits


@lru_cache(maxsize=4096)
def _split_us(n: int, M: int, K: int) -> float:
    """What the launches take, as estimated for the choice of the splits of K."""
    tiles, chunks = _tiles_of(n, M, SPLIT_TILE[1], SPLIT_TILE[0]), -(-K // SPLIT_CHUNK)
    return 8 + min(2.2 * -(-tiles * s // SPLIT_ROUND) * -(-chunks // s) + (4 + 0.05 * s * tiles if s > 1 else 0)
                   for s in range(1, max(1, min(8, K // 256)) + 1))


def _split_rule(n: int, M: int, K: int) -> bool:
    return n >= SPLIT_MIN_ROWS and K >= SPLIT_COLUMNS and n * K <= SPLIT_VALUES and n * M * K >= SPLIT_RATE * _split_us(n, M, K)


@lru_cache(maxsize=4096)
def _split_workspace_bytes(device: int, n: int, M: int, K: int) -> int:
    """As ``_tile_workspace_bytes``."""
    return lib.dv_mix_linear_split_workspace_bytes(n, M, K)


def _split_product(x: torch.Tensor, W: torch.Tensor, bias=None) -> Optional[torch.Tensor]:
    """``F.linear`` of fp32 rows by the kernel that multiplies parts in bf16; None where the library takes them."""
    (n, K), M = x.shape, W.shape[0]
    if (x.dtype != torch.float32 or not _split_rule(n, M, K) or M % 4 or K % 4 or not results_only(x, W, bias) or
            W.stride(0) >= SPLIT_MAX_STRIDE or
            any(t.stride(0) % 4 or t.data_ptr() % 16 for t in (x, W)) or (bias is not None and bias.data_ptr() % 16)):
        return None
    out = torch.empty(n, M, dtype=torch.float32, device=x.device)
    nbytes = _split_workspace_bytes(torch._C._cuda_getDevice(), n, M, K)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
    check(lib.dv_mix_linear_split(_ptr(x), x.stride(0), _ptr(W), W.stride(0), _ptr(bias), n, M, K, _ptr(out), M, _ptr(ws), nbytes,
                                  _stream()), "dv_mix_linear_split")
    return out


def _library_or_split(x: torch.Tensor, W: torch.Tensor, bias=None) -> torch.Tensor:
    y = _split_product(x, W, bias)
    return F.linear(x, W, bias) if y is None else y


class RmsRow:
    """One fp32 row that still has to be RMS-normed and weighted; the products that read it do that themselves."""

    before = L.ROW_RMS

    def __init__(self, u: torch.Tensor, weight: torch.Tensor, dim: int, eps: float, dtype: torch.dtype):
        _f32(u, weight)
        assert u.shape == (1, weight.numel())
        self.u, self.weight, self.dim, self.eps, self.dtype = u, weight, dim, eps, dtype
        self.shape, self.device = u.shape, u.device

    def fill(self, a: L.RowArgs) -> None:
        a.xw, a.norm_dim, a.eps = self.weight.data_ptr(), self.dim, self.eps


class GroupedRow(RmsRow):
    """The same with ``groups`` equal parts of the first ``dim`` entries, each by its own root mean square."""

    before = L.ROW_GROUPS

    def __init__(self, u, weight, dim, groups, eps, dtype):
        super().__init__(u, weight, dim, eps, dtype)
        self.groups = groups

    def fill(self, a: L.RowArgs) -> None:
        a.xw, a.x_dim, a.norm_dim, a.eps = self.weight.data_ptr(), self.dim, self.dim // self.groups, self.eps


class SplitRow(RmsRow):
    """One row of attention whose splits ``part`` still have to be merged, with the heads' sinks and gate logits."""

    before = L.ROW_SPLITS

    def __init__(self, part, splits: int, heads: int, vdim_s: int, sink, gate, dtype: torch.dtype):
        self.u, self.splits, self.vdim_s, self.sink, self.gate, self.dtype = part, splits, vdim_s, sink, gate, dtype
        self.shape, self.device = torch.Size((1, heads * vdim_s)), part.device

    def fill(self, a: L.RowArgs) -> None:
        a.xw, a.gate, a.norm_dim, a.head_stride = _ptr(self.sink), _ptr(self.gate), self.splits, self.vdim_s


def _row_product(x, W):
    """(code, before, arguments) of the product of one row: a tensor in W's type, or an ``RmsRow``."""
    if not isinstance(x, RmsRow):
        return _product_ok(x, W), L.ROW_PLAIN, _row_args(x, W)
    assert x.shape == (1, W.shape[1]) and W.stride(1) == 1 and x.dtype == W.dtype, "product shapes"
    a = _row_args(x.u, W)
    x.fill(a)
    return _code(W), x.before, a


def _row_launch(code, before, after, a) -> None:
    check(lib.dv_mix_linear_row(code, before, after, _ref(a), _stream()), "dv_mix_linear_row")


def _row_args(x, W) -> L.RowArgs:
    M, K = W.shape
    return L.RowArgs(x.data_ptr(), W.data_ptr(), W.stride(0), M, K)


def _tile_args(x, W) -> L.TileArgs:
    M, K = W.shape
    return L.TileArgs(x.data_ptr(), x.stride(0), W.data_ptr(), W.stride(0), x.shape[0], M, K)  # (fields by place: half the time)


@lru_cache(maxsize=4096)
def _tile_workspace_bytes(device: int, n: int, M: int, K: int) -> int:
    """A function of the sizes and of the current device, whose compute units the splits are made for."""
    return lib.dv_mix_linear_tiles_workspace_bytes(n, M, K)


def _tile_launch(after, a, device) -> None:
    """The workspace is this call's own: calls on other streams have theirs, and a captured one is its graph's."""
    nbytes = _tile_workspace_bytes(torch._C._cuda_getDevice(), a.n, a.M, a.K)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=device) if nbytes else None
    check(lib.dv_mix_linear_tiles_ws(after, _ref(a), _ptr(ws), nbytes, _stream()), "dv_mix_linear_tiles_ws")


def linear(x, W: torch.Tensor, bias: Optional[torch.Tensor] = None, f32: bool = False) -> torch.Tensor:
    """x (n, K) W (M, K)^T + bias -> (n, M) in x's type, or fp32."""
    n, M = x.shape[0], W.shape[0]
    out_t = torch.float32 if f32 else x.dtype
    assert bias is None or (bias.dtype == W.dtype and bias.shape == (M,) and bias.is_contiguous())
    if n == 1:
        code, before, a = _row_product(x, W)
        out = torch.empty(1, M, dtype=out_t, device=x.device)
        a.out, a.bias = out.data_ptr(), _ptr(bias)
        _row_launch(code, before, L.OUT_F32 if f32 else L.OUT_T, a)
        return out
    code = _product_ok(x, W)
    if _tiles(x, W, bias) or (f32 and code == L.BF16):
        out = torch.empty(n, M, dtype=out_t, device=x.device)
        a = _tile_args(x, W)
        a.out, a.ldo, a.bias = out.data_ptr(), M, _ptr(bias)
        _tile_launch(L.OUT_F32 if f32 else L.OUT_T, a, x.device)
        return out
    nbytes = 0 if f32 else _parts_bytes(x, W, bias)
    if nbytes:
        out = torch.empty(n, M, dtype=out_t, device=x.device)
        a = _tile_args(x, W)
        a.out, a.ldo, a.bias = out.data_ptr(), M, _ptr(bias)
        _parts_launch(L.OUT_T, a, nbytes, x.device)
        return out
    # (rows of results off 16-byte boundaries are stored value by value: 400 / 1200 rows by 11266 x 2048 0.91 / 0.88 of the library's speed, where
    # 11264 x 2048 is 1.17 / 0.97; 2048 by 22020 x 4096 343 us, 274)
    if not f32 and M % 8 == 0 and (_wide(x, W, bias) or _fills(x, W, bias)):
        out = torch.empty(n, M, dtype=out_t, device=x.device)
        a = _tile_args(x, W)
        a.out, a.ldo, a.bias = out.data_ptr(), M, _ptr(bias)
        check(lib.dv_mix_linear_wide(L.OUT_T, _ref(a), _stream()), "dv_mix_linear_wide")
        return out
    return _library_or_split(x, W, bias)


def gated_unit(x, W: torch.Tensor, act: int, limit: float = 0.0) -> torch.Tensor:
    """W holds gate and up rows alternately; act: GLU_*.  Returns (n, M / 2)."""
    n, M = x.shape[0], W.shape[0]
    y = torch.empty(n, M // 2, dtype=x.dtype, device=x.device)
    if n == 1:
        code, before, a = _row_product(x, W)
        a.out, a.act, a.limit = y.data_ptr(), act, limit
        _row_launch(code, before, L.OUT_GLU, a)
        return y
    code = _product_ok(x, W)
    if _tiles(x, W, gated=True, whole=y.numel() % 4 == 0):
        a = _tile_args(x, W)
        a.out, a.ldo, a.act, a.limit = y.data_ptr(), M // 2, act, limit
        _tile_launch(L.OUT_GLU, a, x.device)
    elif _wide(x, W) or _fills(x, W, gated=True):
        a = _tile_args(x, W)
        a.out, a.ldo, a.act, a.limit = y.data_ptr(), M // 2, act, limit
        check(lib.dv_mix_linear_wide(L.OUT_GLU, _ref(a), _stream()), "dv_mix_linear_wide")
    else:
        gu = _library_or_split(x, W)
        check(lib.dv_mix_glu(code, _ptr(gu), y.numel(), act, limit, _ptr(y), _stream()), "dv_mix_glu")
    return y


def clamped_glu(x, W: torch.Tensor, limit: float) -> torch.Tensor:
    return gated_unit(x, W, L.GLU_CLAMPED, limit)


def relu_glu(x, W: torch.Tensor) -> torch.Tensor:
    return gated_unit(x, W, L.GLU_RELU)


def linear_residual(x: torch.Tensor, W: torch.Tensor, stream: ResidualStream, post, pre, add_start: bool = False):
    """``residual(x W^T, ...)``."""
    n = x.shape[0]
    if n != 1:
        _product_ok(x, W)
    assert stream.x.shape == (n, W.shape[0])
    if n != 1 and not _tiles(x, W, whole=W.shape[0] % 8 == 0):
        nbytes = _parts_bytes(x, W, residual=True)
        if not nbytes:
            return residual(_library_or_split(x, W), stream, post, pre, add_start)
        h = None if pre is None else stream.new_h()
        a = _tile_args(x, W)
        a.res = stream.args(post, pre, add_start, h)
        _parts_launch(L.OUT_RESIDUAL, a, nbytes, x.device)
        return h
    h = None if pre is None else stream.new_h()
    if n == 1:
        code, before, a = _row_product(x, W)
        a.res = stream.args(post, pre, add_start, h)
        _row_launch(code, before, L.OUT_RESIDUAL, a)
    else:
        a = _tile_args(x, W)
        a.res = stream.args(post, pre, add_start, h)
        _tile_launch(L.OUT_RESIDUAL, a, x.device)
    return h


class GatedHeads:
    """fp32 head outputs of one token that still have to be RMS-normed per head, weighted and gated."""

    def __init__(self, o, gate, weight, dim, eps):
        _f32(o, gate, weight)
        self.o, self.gate, self.weight, self.dim, self.eps = o, gate, weight, dim, eps

    def linear_residual(self, W, stream, post, pre, add_start=False):
        h = None if pre is None else stream.new_h()
        a = _row_args(self.o, W)
        a.xw, a.gate, a.eps = self.weight.data_ptr(), self.gate.data_ptr(), self.eps
        a.norm_dim, a.head_stride = self.dim, self.weight.numel()
        a.res = stream.args(post, pre, add_start, h)
        assert self.o.numel() == W.shape[1]
        _row_launch(_code(W), L.ROW_HEADS, L.OUT_RESIDUAL, a)
        return h


class StreamRead:
    """How a sublayer reads several residual streams: their sum weighted by ``weights`` (streams,), RMS-normed with
    ``norm`` (weight (width,), dim, eps)."""

    def __init__(self, norm, weights: torch.Tensor):
        self.norm, self.weights = norm, weights


class HyperStream:
    """Several fp32 residual streams of a portion, x (n, streams, width)."""

    def __init__(self, x: torch.Tensor, dtype: torch.dtype):
        _f32(x)
        assert x.dim() == 3 and x.shape[1] <= L.HYPER_MAX, "streams"
        self.x, self.dtype = x, dtype

    def total(self) -> torch.Tensor:
        return self.x.sum(1)

    def _structs(self, read: StreamRead, normed: bool):
        """Arguments, and the row(s) that ``read`` will hold: fp32 before its norm, or normed."""
        n, streams, width = self.x.shape
        norm = read.norm
        assert read.weights.shape == (streams,) and norm.weight.shape == (width,)
        _f32(read.weights, norm.weight)
        r = L.Hyper(x=self.x.data_ptr(), in_=read.weights.data_ptr(), streams=streams, width=width)
        o = L.RmsOut(w=norm.weight.data_ptr(), eps=norm.eps, dim=norm.dim)
        if normed:
            h = torch.empty(n, width, dtype=self.dtype, device=self.x.device)
            o.h = h.data_ptr()
        else:
            u = torch.empty(n, width, dtype=torch.float32, device=self.x.device)
            r.u = u.data_ptr()
            h = RmsRow(u, norm.weight, norm.dim, norm.eps, self.dtype)
        return r, o, h

    def read(self, read: StreamRead):
        """The input of a sublayer: an ``RmsRow`` for one token, the normed rows for several."""
        n = self.x.shape[0]
        r, o, h = self._structs(read, n > 1)
        check(lib.dv_mix_hyper_rows(_DTYPES[self.dtype], None, n, _ref(r), _ref(o), _stream()), "dv_mix_hyper_rows")
        return h

    def update(self, y, W: torch.Tensor, bias: Optional[torch.Tensor], write, read: StreamRead):
        """The sublayer's result y W^T + bias joins the streams through ``write`` (mix (from, to), out); returns
        ``read`` of them."""
        n, streams, width = self.x.shape
        assert y.shape[0] == n and W.shape[0] == width and write.mix.shape == (streams, streams)
        _f32(write.mix, write.out)
        fused = n == 1 and streams <= L.HYPER_ROW_MAX
        r, o, h = self._structs(read, not fused)
        r.mix, r.out = write.mix.data_ptr(), write.out.data_ptr()
        if fused:
            code, before, a = _row_product(y, W)
            a.hyper, a.bias = r, _ptr(bias)
            _row_launch(code, before, L.OUT_HYPER, a)
        else:
            y = linear(y, W, bias)
            check(lib.dv_mix_hyper_rows(_DTYPES[self.dtype], _ptr(y), n, _ref(r), _ref(o), _stream()),
                  "dv_mix_hyper_rows")
        return h


def hyper_embed(tokens: torch.Tensor, table: torch.Tensor, scale: float, bigram: Optional[torch.Tensor], mul_prev: int,
                mul_cur: int, history: torch.Tensor, pos_dev, pos: int, streams: int, read: StreamRead):
    """tokens (n,) int64 at positions pos ..; history (capacity,) int64 holds the sequence's earlier tokens and takes
    these.  Returns (HyperStream, ``read`` of it)."""
    code = _code(table)
    n, width = tokens.numel(), table.shape[1]
    for t in (tokens, history):
        assert t.dtype == torch.int64 and t.is_cuda and t.is_contiguous()
    assert table.is_contiguous() and (bigram is None or (bigram.is_contiguous() and bigram.dtype == table.dtype and
                                                         bigram.shape[1] == width))
    stream = HyperStream(torch.empty(n, streams, width, dtype=torch.float32, device=table.device), table.dtype)
    r, o, h = stream._structs(read, n > 1)
    e = L.EmbedArgs(tokens=tokens.data_ptr(), history=history.data_ptr(), capacity=history.numel(), vocab=table.shape[0],
                    embed=table.data_ptr(), scale=scale, pos_dev=_ptr(pos_dev), pos_host=pos, n=n)
    if bigram is not None:
        e.bigram, e.buckets, e.mul_prev, e.mul_cur = bigram.data_ptr(), bigram.shape[0] - 1, mul_prev, mul_cur
    check(lib.dv_mix_hyper_embed(code, _ref(e), _ref(r), _ref(o), _stream()), "dv_mix_hyper_embed")
    return stream, h


def head_rows(x: torch.Tensor, groups) -> None:
    """x (n, >= channels): the groups' heads one after the other, each group (heads, stride, dim, what, out) with out
    (n, heads * stride); what: (weight, eps) for an RMS norm per head, (other, lambda) for (1 - lambda) x + lambda
    other, None for a copy."""
    a = L.HeadArgs(in_=x.data_ptr(), ldi=x.stride(0), n=x.shape[0])
    for i, (heads, stride, dim, what, out) in enumerate(groups):
        assert out.shape == (x.shape[0], heads * stride) and out.stride(1) == 1 and out.dtype == x.dtype
        g = L.HeadGroup(heads=heads, stride=stride, dim=dim, out=out.data_ptr(), ld=out.stride(0))
        if what is not None and isinstance(what[1], float):
            _f32(what[0])
            g.w, g.eps = what[0].data_ptr(), what[1]
        elif what is not None:
            other, lam = what
            _f32(lam)
            assert other.shape == out.shape and other.dtype == x.dtype and other.stride(1) == 1
            g.other, g.ldo = other.data_ptr(), other.stride(0)
            setattr(g, "lambda", lam.data_ptr())
        a.g[i] = g
    check(lib.dv_mix_head_rows(_code(x), _ref(a), _stream()), "dv_mix_head_rows")


def gated_group_norm(y: torch.Tensor, z: torch.Tensor, weight: torch.Tensor, dim: int, groups: int, eps: float):
    """t = y silu(z); t / rms(t) * weight per group of dim / groups entries.  y fp32 (n, padded), z (n, padded)."""
    _f32(weight)
    n, padded_dim = z.shape
    assert y.shape == z.shape and y.dtype == torch.float32 and y.stride(1) == z.stride(1) == 1
    out = torch.empty(n, padded_dim, dtype=z.dtype, device=z.device)
    check(lib.dv_mix_gated_group_norm(_code(z), _ptr(y), y.stride(0), _ptr(z), z.stride(0), n, dim, groups, padded_dim,
                                      _ptr(weight), eps, _ptr(out), _stream()), "dv_mix_gated_group_norm")
    return out


def row_conv(x, W: torch.Tensor, conv_w: torch.Tensor, conv_state: torch.Tensor, silu: bool,
             conv_b: Optional[torch.Tensor] = None):
    """One token: the product in fp32; its first conv_w.shape[0] values pass the short convolution (state moved on)."""
    _f32(conv_w, conv_state, conv_b)
    code, before, a = _row_product(x, W)
    out = torch.empty(1, W.shape[0], dtype=torch.float32, device=x.device)
    a.out = out.data_ptr()
    a.conv_w, a.conv_b, a.conv_state = conv_w.data_ptr(), _ptr(conv_b), conv_state.data_ptr()
    a.conv_rows, a.taps, a.silu = conv_w.shape[0], conv_w.shape[1], int(silu)
    _row_launch(code, before, L.OUT_CONV, a)
    return out


def row_rms_linear(x, weight, dim, eps, W, side=None):
    """One token: fp32 (x / rms(x) * weight) W^T.  ``side``: (row, weight, dim, out, seq_pos, position), a second row
    that is normed the same way and stored as row ``position`` of ``out``."""
    _f32(x, weight)
    out = torch.empty(1, W.shape[0], dtype=torch.float32, device=x.device)
    a = _row_args(x, W)
    assert weight.numel() == W.shape[1]
    a.xw, a.norm_dim, a.eps, a.out = weight.data_ptr(), dim, eps, out.data_ptr()
    if side is not None:
        row, w, sdim, dst, pos_dev, pos = side
        a.side_x, a.side_w, a.side_dim, a.side_padded = row.data_ptr(), w.data_ptr(), sdim, w.numel()
        a.side_out, a.side_ld, a.pos_dev, a.pos_host = dst.data_ptr(), dst.stride(0), _ptr(pos_dev), pos
    _row_launch(_code(W), L.ROW_RMS, L.OUT_F32, a)
    return out


def rms_rows(x: torch.Tensor, weight: torch.Tensor, dim: int, eps: float, out: Optional[torch.Tensor] = None):
    code = _code(x)
    n = x.shape[0]
    if out is None:
        out = torch.empty(n, weight.numel(), dtype=x.dtype, device=x.device)
    assert out.dtype == x.dtype and x.stride(1) == out.stride(1) == 1 and out.shape == (n, weight.numel())
    check(lib.dv_mix_rms_rows(code, _ptr(x), x.stride(0), n, dim, weight.numel(), _ptr(weight), eps, _ptr(out),
                              out.stride(0), _stream()), "dv_mix_rms_rows")
    return out


def rms_rows_two(x: torch.Tensor, a, b, eps: float) -> None:
    """``rms_rows`` of two stretches of the rows of x in one launch.  a, b: (first entry, weight, dim, out)."""
    n, rows = x.shape[0], []
    for at, weight, dim, out in (a, b):
        assert out.dtype == x.dtype and x.stride(1) == out.stride(1) == 1 and out.shape == (n, weight.numel())
        assert at + weight.numel() <= x.shape[1]
        rows.append(L.RmsRows(x.data_ptr() + at * x.element_size(), dim, weight.numel(), weight.data_ptr(), out.data_ptr(), out.stride(0)))
    check(lib.dv_mix_rms_rows_two(_code(x), _ref(rows[0]), _ref(rows[1]), x.stride(0), n, eps, _stream()), "dv_mix_rms_rows_two")


def gated_head_norm(o: torch.Tensor, gate: torch.Tensor, weight: torch.Tensor, dim: int, eps: float):
    """o (n, heads, vdim_s) fp32, gate (n, heads * vdim_s) -> (n, heads * vdim_s)."""
    n, heads, vs = o.shape
    y = torch.empty(n, heads * vs, dtype=gate.dtype, device=o.device)
    check(lib.dv_mix_gated_head_norm(_code(gate), _ptr(o), _ptr(gate), gate.stride(0), n, heads, dim, vs, _ptr(weight),
                                     eps, _ptr(y), _stream()), "dv_mix_gated_head_norm")
    return y


NORM_NONE, NORM_RMS, NORM_UNIT = 0, 1, 2


def short_conv(x: torch.Tensor, conv_w: torch.Tensor, state: torch.Tensor, groups, silu: bool,
               conv_b: Optional[torch.Tensor] = None, move: bool = False) -> None:
    """x (n, >= channels): the groups' channels one after the other.  groups: (heads, stride, dim, norm, eps, scale,
    out) with out (n, heads * stride), all fp32 or all of x's type.  The state is read; with ``move`` it moves on by
    the rows of x as well (``conv_state``)."""
    _f32(conv_w, conv_b)
    a = L.ConvArgs(in_=x.data_ptr(), ldi=x.stride(0), n=x.shape[0], taps=conv_w.shape[1], silu=int(silu),
                   w=conv_w.data_ptr(), b=_ptr(conv_b), state=state.data_ptr())
    for i, (heads, stride, dim, norm, eps, scale, out) in enumerate(groups):
        assert out.shape == (x.shape[0], heads * stride) and out.stride(1) == 1
        a.g[i] = L.ConvGroup(heads, stride, dim, norm, eps, scale, out.data_ptr(), out.stride(0))
    code, f32 = _code(x), int(groups[0][6].dtype == torch.float32)
    if move:
        check(lib.dv_mix_short_conv_move(code, f32, _ref(a), a.state, _stream()), "dv_mix_short_conv_move")
    else:
        check(lib.dv_mix_short_conv(code, f32, _ref(a), _stream()), "dv_mix_short_conv")


def conv_state(x: torch.Tensor, channels: int, taps: int, state: torch.Tensor) -> None:
    """Moves the state on by the n rows of x."""
    check(lib.dv_mix_conv_state(_code(x), _ptr(x), x.stride(0), x.shape[0], channels, taps, _ptr(state), _stream()),
          "dv_mix_conv_state")


def _ring_rows(buf: torch.Tensor, ring: torch.Tensor) -> L.RingRows:
    assert buf.dtype == ring.dtype and buf.shape[1] == ring.shape[1]
    return L.RingRows(buf.data_ptr(), buf.stride(0), ring.data_ptr(), ring.stride(0), buf.shape[1])


def ring_copy_two(bufs, rings, first: int, to_ring: bool) -> None:
    """Rows of two buffers, tokens first, first + 1, .. in both, to two rings of as many rows, or from there, in one launch."""
    (a, b), (ra, rb) = bufs, rings
    assert a.shape[0] == b.shape[0] and ra.shape[0] == rb.shape[0] and a.dtype == b.dtype
    check(lib.dv_mix_ring_copy_two(_code(a), _ref(_ring_rows(a, ra)), _ref(_ring_rows(b, rb)), ra.shape[0], first, a.shape[0],
                                   int(to_ring), _stream()), "dv_mix_ring_copy_two")


# Up to so many keys that a decode row can ever see, one launch (a workgroup per head) takes it all in bf16; beyond, splits
# and a merge.  us, split / one, all of the keys seen: 16 heads on 4 key heads of 128 + 128, 81 / 256 / 320 / 384 / 400 / 448 / 512 / 768 keys 10.9 /
# 6.4, 11.0 / 7.7, 11.0 / 10.1, 11.1 / 10.2, 10.6 / 10.2, 11.0 / 10.4, 11.1 / 10.5, 11.2 / 13.0; 32 heads on 8, 320 to 512 keys 11.1 / 10.3, 11.1 / 10.9,
# 10.8 / 10.9, 11.1 / 11.0, 11.0 / 11.2; 64 heads on 8, 384 keys 14.9 / 11.0; 32 heads with keys of their own are behind from 300 on when
# all keys are seen (9.3 / 10.3, at 384 10.3 / 10.9) and ahead with five eighths of them (8.6 / 7.6, 8.4 / 7.9).  Latent attention of 16
# heads and rank 256, 81 / 256 / 384 / 400 / 448 / 512 keys 12.3 / 6.1, 12.9 / 7.8, 13.0 / 9.4, 13.0 / 12.5, 13.1 / 12.6, 13.0 / 12.8, of 32 heads and rank
# 512, 256 to 512 keys 18.9 / 13.9, 19.3 / 17.0, 19.4 / 19.2, 19.4 / 19.6, 19.4 / 20.0.
ONE_LAUNCH_KEYS = 384
ONE_LAUNCH_LATENTS = 400


def decode_splits(keys: int) -> int:
    """Workgroups that share the keys of a decode row.  ``keys`` is the most there can be: the value may not depend
    on the position, which captured steps only know on the device."""
    return max(1, min(16, (keys + 63) // 64), min(128, keys // 128))


# Small rows of many keys: the output projection merges the splits while it stages its row (eight at most: every workgroup reads them all, 66
# KB of 2048 entries), so neither the launch that merges nor the one workgroup per head is waited for.  us a token, otherwise and so: vimulorn-2k
# (16 heads of 128) at 100 / 170 / 270 / 350 / 460 / 740 / 1340 tokens 399.7 / 409.9, 414 / 423, 437 / 441, 450.6 / 446.5, 465 / 461, 468 / 462, 484 / 476, varolorn-2k at
# 270 / 350 / 460 / 740 / 1340 462 / 465, 471 / 472, 477 / 469, 482 / 483, 506 / 496; rows of 4096 880 / 884 at 350, 901 / 899 at 460, 928 / 933 at 740, 982 / 995 at 1340.
# Beyond eight tiles of 64 keys a workgroup walks over several, and more splits with a launch that merges them are ahead: with a window, which stays
# full, from there on, with a chunk or a whole sequence, of which half is seen on average, from twice as many.  us a token that the merge saves at 460 / 740 / 1000 /
# 1340 / 1900 tokens (three such layers, 16 heads on 4 key heads): windows of 512 3.2 / 4.9 / 5.2 / 5.5 / 5.8, 1024 4.6 / -1.8 / -2.8 / -2.8 / -2.1, 2048 5.0 / -1.6 /
# -1.9 / -1.7 / -9.7; chunks of 1024 5.8 / -0.3 / 1.8 / 4.1 / -1.6, 2048 4.3 / -1.3 / -2.7 / -2.0 / -9.0, 4096 6.2 / -0.5 / -1.2 / -1.6 / -10.1.  A row with its projection,
# all keys seen, so many keys possible, 2048 / 4096 / 8192 / 32768: 19.9 / 23.9, 20.5 / 34.5, 21.6 / 56, 36.8 / 201.
MERGE_KEYS, MERGE_ROW, MERGE_SPLITS = 320, 2048, 8
MERGE_WINDOW, MERGE_CHUNK = 512, 1024


def _merge_splits(keys: int) -> int:
    return min((keys + 63) // 64, MERGE_SPLITS)


def _merge_rule(heads: int, vdim_s: int, keys: int, dtype, full: bool) -> bool:
    """full: all of the keys are seen from some token on (a window's)."""
    most = MERGE_WINDOW if full else MERGE_CHUNK
    return dtype == torch.bfloat16 and MERGE_KEYS < keys <= most and heads * vdim_s <= MERGE_ROW


def _attn_args(q, k, v, n, H, G, dim_s, vdim_s, scale, sink, gate, window, ring, base, pos_dev, pos):
    a = L.AttnArgs(q=q.data_ptr(), ldq=q.stride(0), k=k.data_ptr(), ldk=k.stride(0), k_head=dim_s, v=v.data_ptr(),
                   ldv=v.stride(0), v_head=vdim_s, n=n, H=H, G=G, dim_s=dim_s, vdim_s=vdim_s, scale=scale,
                   sink=_ptr(sink), window=window or 0, ring=ring, base=base, pos_dev=_ptr(pos_dev), pos_host=pos,
                   splits=1)
    if gate is not None:
        a.gate, a.ldg = gate.data_ptr(), gate.stride(0)
    return a


def _mask_args(a, window, chunk, rel) -> None:
    a.window, a.chunk = window or 0, chunk or 0
    if rel is not None:
        _f32(rel)
        assert rel.dim() == 2 and rel.shape[0] == a.H
        a.rel, a.rel_len = rel.data_ptr(), rel.shape[1]


# fp32 queries (rows x heads) from which the matrix cores are the faster ones: heads of 128, 16 of them on 4, 256 rows after
# none / 300 tokens: 22 / 45 us, row by row 30 / 59; 128 rows: 14 / 37 and 13 / 29
F32_TILE_ROWS = 3072


def portion_attention(q, k, v, heads: int, kv_heads: int, scale: float, first_key: int, pos: int, sink=None, gate=None,
                      window=None, chunk=None, rel=None) -> torch.Tensor:
    """Causal attention of a portion: q (n, heads * dim) at positions pos .., k / v (keys, kv_heads * dim / vdim) from
    token ``first_key`` on.  window: the newest so many tokens are seen; chunk: the tokens of the query's own chunk,
    counted from position 0; rel (heads, distances): added to the scaled scores, its last entry beyond.  On the
    matrix cores: bf16 with heads of up to 256, fp32 with heads of up to 128 and enough rows; the rest row by row."""
    n, dim_s, vdim_s = q.shape[0], q.shape[1] // heads, v.shape[1] // kv_heads
    out = torch.empty(n, heads * vdim_s, dtype=q.dtype, device=q.device)
    a = _attn_args(q, k, v, n, heads, kv_heads, dim_s, vdim_s, scale, sink, gate, window, 0, first_key, None, pos)
    _mask_args(a, window, chunk, rel)
    a.out = out.data_ptr()
    assert gate is None or gate.dtype == q.dtype
    if q.dtype == torch.bfloat16 and dim_s <= 256 and vdim_s <= 256:
        check(lib.dv_mix_attn_tiles(_ref(a), k.shape[0], _stream()), "dv_mix_attn_tiles")
        return out
    step = 32768  # rows per launch
    for i in range(0, n, step):
        a.n, a.pos_host = min(step, n - i), pos + i
        a.q, a.out = q[i:].data_ptr(), out[i:].data_ptr()
        if gate is not None:
            a.gate = gate[i:].data_ptr()
        if (q.dtype == torch.float32 and a.n * heads >= F32_TILE_ROWS and dim_s <= 128 and vdim_s <= 128
                and a.ldq % 4 == 0):
            check(lib.dv_mix_attn_tiles_f32(_ref(a), k.shape[0], _stream()), "dv_mix_attn_tiles_f32")
        else:
            check(lib.dv_mix_attn_rows(_code(q), 0, _ref(a), _stream()), "dv_mix_attn_rows")
    return out


def ring_attention_row(row, k_ring, v_ring, heads, kv_heads, dim, scale, eps, pos_dev, pos, sink=None, window=None,
                       chunk=None, rel=None, q_weight=None, k_weight=None, mix_v=None, gate=None, defer=False):
    """One token of attention over rings of keys and values (cap, kv_heads * stride).  row: fp32 (q, k, v); q and k
    are RMS-normed (times their weights), v mixed with ``mix_v`` = (other fp32 values, lambda), this token's k and v
    stored.  gate: fp32 logits (heads,).  Masks and rel as in ``portion_attention``.  defer: the row goes to a product of this
    module, which may merge the splits itself (a ``SplitRow`` is returned then)."""
    _f32(row, sink, q_weight, k_weight)
    dim_s, vdim_s, cap = k_ring.shape[1] // kv_heads, v_ring.shape[1] // kv_heads, k_ring.shape[0]
    a = _attn_args(row, k_ring, v_ring, 1, heads, kv_heads, dim_s, vdim_s, scale, sink, None, window, cap, 0, pos_dev,
                   pos)
    _mask_args(a, window, chunk, rel)
    a.q_w, a.k_w = _ptr(q_weight), _ptr(k_weight)
    if mix_v is not None:
        _f32(*mix_v)
        assert mix_v[0].numel() == kv_heads * vdim_s
        a.other_v = mix_v[0].data_ptr()
        setattr(a, "lambda", mix_v[1].data_ptr())
    if gate is not None:
        _f32(gate)
        a.gate, a.ldg = gate.data_ptr(), heads
    a.norm_dim, a.eps = dim, eps
    a.fresh_k = row.data_ptr() + 4 * heads * dim_s
    a.fresh_v = row.data_ptr() + 4 * (heads + kv_heads) * dim_s
    keys = min(cap, window or cap, chunk or cap)
    if defer and _merge_rule(heads, vdim_s, keys, k_ring.dtype, keys == window):
        a.splits = _merge_splits(keys)
        part = torch.empty(heads * a.splits * (vdim_s + 2), dtype=torch.float32, device=row.device)
        a.part = part.data_ptr()
        check(lib.dv_mix_attn_splits(_code(k_ring), 1, _ref(a), _stream()), "dv_mix_attn_splits")
        return SplitRow(part, a.splits, heads, vdim_s, sink, gate, k_ring.dtype)
    out = torch.empty(1, heads * vdim_s, dtype=k_ring.dtype, device=row.device)
    a.out = out.data_ptr()
    if k_ring.dtype != torch.bfloat16 or dim_s > 128 or vdim_s > 128 or keys > ONE_LAUNCH_KEYS:
        a.splits = decode_splits(cap)
    part = None
    if a.splits > 1:
        part = torch.empty(heads * a.splits * (vdim_s + 2), dtype=torch.float32, device=row.device)
        a.part = part.data_ptr()
    check(lib.dv_mix_attn_rows(_code(k_ring), 1, _ref(a), _stream()), "dv_mix_attn_rows")
    return out


def window_attention_row(row, k_ring, v_ring, heads, kv_heads, dim, scale, eps, sink, window, pos_dev, pos, defer=False):
    return ring_attention_row(row, k_ring, v_ring, heads, kv_heads, dim, scale, eps, pos_dev, pos, sink=sink, window=window, defer=defer)


def latent_attention_row(q, k_up, v_up, cache, heads, scale, gate, pos_dev, pos):
    """One token of latent attention.  q fp32 (1, heads * dim), k_up (heads * dim, rank), v_up (heads * vdim, rank),
    cache (tokens, rank) whose row for this token is there, gate fp32 logits (heads,)."""
    _f32(q)
    rank, dim_s, vdim_s = cache.shape[1], k_up.shape[0] // heads, v_up.shape[0] // heads
    code = _code(cache)
    out = torch.empty(1, heads * vdim_s, dtype=cache.dtype, device=q.device)
    if cache.dtype == torch.bfloat16 and rank <= 512 and cache.shape[0] <= ONE_LAUNCH_LATENTS:
        a = _attn_args(q, cache, cache, 1, heads, 1, rank, rank, scale, None, None, None, 0, 0, pos_dev, pos)
        a.gate, a.ldg, a.out = gate.data_ptr(), heads, out.data_ptr()
        check(lib.dv_mix_latent_one(_ref(a), cache.shape[0], _ptr(k_up), dim_s, _ptr(v_up), vdim_s, _ptr(out), _stream()),
              "dv_mix_latent_one")
        return out
    ql = torch.empty(heads, rank, dtype=torch.float32, device=q.device)
    check(lib.dv_mix_latent_absorb(code, _ptr(q), _ptr(k_up), heads, dim_s, rank, _ptr(ql), _stream()),
          "dv_mix_latent_absorb")
    a = _attn_args(ql.view(1, -1), cache, cache, 1, heads, 1, rank, rank, scale, None, None, None, 0, 0, pos_dev, pos)
    a.gate, a.ldg = gate.data_ptr(), heads
    a.splits = max(2, min(128, (cache.shape[0] + 127) // 128))
    part = torch.empty(heads * a.splits * (rank + 2), dtype=torch.float32, device=q.device)
    a.part = part.data_ptr()
    check(lib.dv_mix_latent_attn(code, _ref(a), _ptr(v_up), vdim_s, _ptr(out), _stream()), "dv_mix_latent_attn")
    return out


def delta_gates(z, b, A_log, dt_bias, heads: int):
    """z (n, heads * dim_s) and b (n, >= heads) logits -> decays (n, heads * dim_s), beta (n, heads), fp32."""
    n, dim_s = z.shape[0], z.shape[1] // heads
    g = torch.empty(n, heads * dim_s, dtype=torch.float32, device=z.device)
    beta = torch.empty(n, heads, dtype=torch.float32, device=z.device)
    check(lib.dv_mix_delta_gates(_code(z), _ptr(z), z.stride(0), _ptr(b), b.stride(0), _ptr(A_log), _ptr(dt_bias), n,
                                 heads, dim_s, _ptr(g), _ptr(beta), _stream()), "dv_mix_delta_gates")
    return g, beta


def delta_scan(q, k, v, g, beta, S, heads: int, kv_heads: int) -> torch.Tensor:
    """The gated delta rule over n tokens; S (heads, vdim_s, dim_s) is updated.  Returns (n, heads, vdim_s) fp32."""
    _f32(q, k, v, g, beta, S)
    n, vs, ds = q.shape[0], S.shape[1], S.shape[2]
    o = torch.empty(n, heads, vs, dtype=torch.float32, device=q.device)
    assert q.shape == k.shape == (n, kv_heads * ds) and v.shape == (n, heads * vs) and g.shape == (n, heads * ds)
    tm = torch.empty((min(n, 4096) + 15) // 16 * heads * (49 * ((ds + 63) // 64 * 64) + 512), dtype=torch.float32,
                     device=q.device)
    a = L.DeltaArgs(q=q.data_ptr(), k=k.data_ptr(), v=v.data_ptr(), g=g.data_ptr(), beta=beta.data_ptr(),
                    S=S.data_ptr(), o=o.data_ptr(), tm=tm.data_ptr(), tm_floats=tm.numel(), n=n, heads=heads, kv_heads=kv_heads, dim_s=ds, vdim_s=vs)
    check(lib.dv_mix_delta_scan(_ref(a), _stream()), "dv_mix_delta_scan")
    return o


def delta_row(row, offsets, heads, kv_heads, dim, decay_up, gate_up, A_log, dt_bias, S):
    """One token of the gated delta rule from the fp32 projection row; returns (o, gate), fp32 (heads * vdim_s,)."""
    _f32(row, A_log, dt_bias, S)
    vs, ds = S.shape[1], S.shape[2]
    o = torch.empty(1, heads * vs, dtype=torch.float32, device=row.device)
    gate = torch.empty(heads * vs, dtype=torch.float32, device=row.device)
    off_k, off_v, off_b, off_a, off_g = offsets
    a = L.DeltaStepArgs(p=row.data_ptr(), off_k=off_k, off_v=off_v, off_b=off_b, off_a=off_a, off_g=off_g, heads=heads,
                        kv_heads=kv_heads, dim=dim, dim_s=ds, vdim_s=vs, Wa=decay_up.data_ptr(),
                        Wg=gate_up.data_ptr(), rank_a=decay_up.shape[1], rank_g=gate_up.shape[1],
                        A_log=A_log.data_ptr(), dt_bias=dt_bias.data_ptr(), S=S.data_ptr(), o=o.data_ptr(),
                        gate=gate.data_ptr())
    check(lib.dv_mix_delta_step(_code(decay_up), _ref(a), _stream()), "dv_mix_delta_step")
    return o, gate


SSD_CHUNK = 64


def ssd_rows(n: int, channels: int, device) -> torch.Tensor:
    """(n, channels) fp32 for ``ssd_scan``: zeros follow up to the end of the last chunk."""
    rows = torch.empty((n + SSD_CHUNK - 1) // SSD_CHUNK * SSD_CHUNK, channels, dtype=torch.float32, device=device)
    if rows.shape[0] > n:
        rows[n:].zero_()
    return rows[:n]


def ssd_scan(xbc, dt, A_log, dt_bias, D, S, groups: int, off_b: int, off_c: int, width: int) -> torch.Tensor:
    """The Mamba-2 recurrence over n tokens; xbc fp32 (n, channels) from ``ssd_rows``: x of all heads, B from column off_b and C from
    off_c on; dt (n, heads) logits of the step sizes.  S (heads, vdim, state) is updated.  Returns fp32 (n, width), of
    which the first heads * vdim columns are written."""
    _f32(xbc, A_log, dt_bias, D, S)
    n, (heads, vdim, state) = xbc.shape[0], S.shape
    chunks = (n + SSD_CHUNK - 1) // SSD_CHUNK
    assert xbc.untyped_storage().nbytes() >= 4 * (xbc.storage_offset() + chunks * SSD_CHUNK * xbc.stride(0)), "ssd_rows"
    assert dt.shape == (n, heads) and dt.stride(1) == 1 and heads * vdim <= width
    assert heads * vdim <= off_b and off_b + groups * state <= off_c and off_c + groups * state <= xbc.shape[1]
    y = torch.empty(n, width, dtype=torch.float32, device=xbc.device)
    tm = torch.empty(min(chunks, 64) * heads * 2688, dtype=torch.float32, device=xbc.device)
    a = L.SsdArgs(xbc=xbc.data_ptr(), ld=xbc.stride(0), off_b=off_b, off_c=off_c, dt=dt.data_ptr(), lddt=dt.stride(0),
                  A_log=A_log.data_ptr(), dt_bias=dt_bias.data_ptr(), D=D.data_ptr(), S=S.data_ptr(), y=y.data_ptr(),
                  ldy=width, tm=tm.data_ptr(), tm_floats=tm.numel(), n=n, heads=heads, groups=groups, vdim=vdim,
                  state_s=state)
    check(lib.dv_mix_ssd_scan(_code(dt), _ref(a), _stream()), "dv_mix_ssd_scan")
    return y


def ssd_step(row, A_log, dt_bias, D, S, groups: int, off_b: int, off_c: int, off_z: int, off_dt: int, width: int):
    """One token of it from the fp32 projection row, also multiplied by silu(z).  Returns fp32 (1, width)."""
    _f32(row, A_log, dt_bias, D, S)
    heads, vdim, state = S.shape
    assert heads * vdim <= width and off_dt + heads <= row.shape[1] and off_z + heads * vdim <= row.shape[1]
    assert max(off_b, off_c) + groups * state <= row.shape[1]
    y = torch.empty(1, width, dtype=torch.float32, device=row.device)
    a = L.SsdStepArgs(p=row.data_ptr(), off_b=off_b, off_c=off_c, off_z=off_z, off_dt=off_dt, A_log=A_log.data_ptr(),
                      dt_bias=dt_bias.data_ptr(), D=D.data_ptr(), S=S.data_ptr(), y=y.data_ptr(), heads=heads,
                      groups=groups, vdim=vdim, state_s=state)
    check(lib.dv_mix_ssd_step(_ref(a), _stream()), "dv_mix_ssd_step")
    return y


# From so many logits on two launches, many workgroups and then one wave, take less than one workgroup alone (us, one / two: 1000 / 4096 / 8192 / 16384 / 32768 /
# 131072 logits 4.8 / 5.7, 5.6 / 6.2, 6.3 / 6.3, 7.8 / 6.4, 10.3 / 6.5, 26.8 / 7.1).
GREEDY_PARTS = 8192


def greedy_advance(logits, token, position, seq_pos, sequences, out_index, scores=None, score_index=None) -> None:
    """``ops.greedy_advance`` for fp32 logits."""
    _f32(logits)
    assert logits.dim() == 1
    args = (_ptr(logits), logits.numel(), _ptr(token), _ptr(position), _ptr(seq_pos), _ptr(sequences), sequences.numel(), _ptr(out_index),
            _ptr(scores), 0 if scores is None else scores.stride(0), 0 if scores is None else scores.shape[0], _ptr(score_index))
    if logits.numel() < GREEDY_PARTS:
        check(lib.dv_mix_greedy_advance(*args, _stream()), "dv_mix_greedy_advance")
        return
    ws = torch.empty(lib.dv_mix_greedy_advance_workspace_bytes(logits.numel()), dtype=torch.uint8, device=logits.device)
    check(lib.dv_mix_greedy_advance_ws(*args, _ptr(ws), ws.numel(), _stream()), "dv_mix_greedy_advance_ws")
