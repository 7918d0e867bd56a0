"""gemm_wide.hpp: every width of its tiles at sizes where they end, the rule that sends products to it, and what the matrix
instructions written in assembly rely on, seen in the assembly that the compiler makes of every form."""
import os
import re
import subprocess

import pytest
import torch

from dejavu_amd.build import CSRC, HIPCC_FLAGS, hipcc_path
from test_ring_handover import registers, states_before_use

# (rows, weight rows) whose tiles are 128 / 160 / 192 / 224 / 256 rows wide on 256 compute units
SIZES = [(257, 1030), (300, 22016), (380, 32700), (777, 16380), (500, 22010)]
WIDTHS = [128, 160, 192, 224, 256]
SOURCE = """
#include <stdio.h>
#include "gemm_wide.hpp"
template <typename T>
struct Store {
  T* y;
  static constexpr int kOuts = 4;
  typedef T vec_t __attribute__((ext_vector_type(4)));
  __device__ T* base() const { return y; }
  __device__ int64_t ld() const { return 4096; }
  __device__ int columns() const { return 4090; }
  struct Row {};
  __device__ Row row(int m) const { return {}; }
  __device__ vec_t make(const Row&, const dv::float4_t& v) const { return vec_t{(T)v[0], (T)v[1], (T)v[2], (T)v[3]}; }
};
struct Launch {
  template <auto KERNEL, typename... A>
  int operator()(dim3 grid, dim3 threads, size_t lds, hipStream_t s, A... args) const {
    hipLaunchKernelGGL(KERNEL, grid, threads, lds, s, args...);
    return 0;
  }
};
int all(int nb, const dv::RingOperands<dv::half_t>& a, const dv::RingOperands<__bf16>& b) {
  return dv::gemm_wide(nb, a, Store<dv::half_t>{}, nullptr, Launch{}) + dv::gemm_wide(nb, b, Store<__bf16>{}, nullptr, Launch{});
}
"""


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    try:
        hipcc = hipcc_path()
    except RuntimeError as e:
        pytest.skip(str(e))
    where = tmp_path_factory.mktemp("wide")
    src, out = where / "wide.hip", where / "wide.s"
    src.write_text(SOURCE)
    flags = [f for f in HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([hipcc, *flags, "-w", "-S", "--cuda-device-only", "-I", CSRC, "-I", os.path.join(CSRC, "..", "..", "include"),
                    str(src), "-o", str(out)], check=True)
    found, name = {}, None
    for line in out.read_text().splitlines():
        line = line.split(";")[0].strip()
        if re.match(r"_ZN2dv16gemm_wide_kernel.*:$", line):
            name = line[:-1]
            found[name] = []
        elif line.startswith(".Lfunc_end"):
            name = None
        elif name and line and (not line.startswith(".") or line.endswith(":")):
            found[name].append(re.sub(r"\s+", " ", line))
    assert len(found) == 2 * len(WIDTHS)
    return found


def test_widths_that_are_chosen(tmp_path):
    """The sizes of the tests are of every width, and sizes for which other widths were measured to take up to a quarter longer."""
    try:
        hipcc = hipcc_path()
    except RuntimeError as e:
        pytest.skip(str(e))
    src, exe = tmp_path / "plan.hip", tmp_path / "plan"
    src.write_text('#include <cstdio>\n#include "gemm_wide.hpp"\nint main() { int n, M; while (scanf("%d %d", &n, &M) == 2) '
                   'printf("%d\\n", dv::plan_wide(n, M, 256)); }\n')
    subprocess.run([hipcc, "--offload-arch=gfx950", "-std=c++17", "-w", "-I", CSRC, "-I", os.path.join(CSRC, "..", "..", "include"),
                    str(src), "-o", str(exe)], check=True)
    measured = {(1024, 36864): 224, (2048, 28672): 256, (1152, 27648): 192, (2048, 22016): 256, (1999, 18560): 224, (777, 16384): 224, (400, 22016): 224,
                (777, 12288): 160, (2048, 11264): 192}
    asked = SIZES + list(measured)
    out = subprocess.run([str(exe)], input="\n".join("%d %d" % q for q in asked), text=True, check=True, capture_output=True).stdout
    assert list(map(int, out.split())) == WIDTHS + list(measured.values())


def test_matrix_instructions_in_assembly(kernels):
    """Nothing in the hardware waits for their sums (8 states) or for operands that a vector instruction has just written (2), and
    the compiler does not see what they are."""
    for name, lines in kernels.items():
        assert not any(line.startswith("scratch_") for line in lines), name
        matrix = [i for i, line in enumerate(lines) if line.startswith("v_mfma")]
        assert len(matrix) >= 2 * 2 * 8 * 4, name
        uses = [states_before_use(lines, i) for i in matrix]
        uses = [u for u in uses if u is not None]
        assert uses and min(uses) >= 8, (name, sorted(uses)[:4])
        for i in matrix:
            operands = set().union(*map(registers, lines[i].split(None, 1)[1].split(", ")))
            states = 0
            for line in reversed(lines[:i]):
                op = line.split()[0]
                if states >= 2 or op.endswith(":"):
                    break
                if op.startswith("v_") and not op.startswith("v_mfma"):
                    assert not registers(line.split(None, 1)[1].split(",")[0]) & operands, (name, line, lines[i])
                states += int(line.split()[1]) + 1 if op == "s_nop" else 1


def test_loop_keeps_its_sums_in_place(kernels):
    """The loop over the chunks: one barrier, behind everybody's reads and the next chunk's loads, and no copies of sums."""
    for name, lines in kernels.items():
        width = int(re.search(r"Li(\d+)E", name)[1])
        starts = [i for i, line in enumerate(lines) if line.endswith(":")] + [len(lines)]
        blocks = [lines[a:b] for a, b in zip(starts, starts[1:])]
        loop = [b for b in blocks if sum(line.startswith("v_mfma") for line in b) == width // 2 and any(line.startswith("buffer_load") for line in b)]
        assert len(loop) == 1, name
        assert not any(line.startswith("v_accvgpr") for line in loop[0]), name
        at = [i for i, line in enumerate(loop[0]) if line.startswith("s_barrier")]
        assert len(at) == 1 and re.search(r"vmcnt\(8\) lgkmcnt\(0\)", loop[0][at[0] - 1]), (name, loop[0][at[0] - 1])


def test_which_products_the_wide_kernel_takes():
    """Gated units and few columns on both sides of the lines; each was measured with its weights out of the caches."""
    from dejavu_amd.mixer_ops import _fill_rule

    for n, M, K in ((400, 22016, 4096), (2048, 22016, 4096), (1999, 18560, 4096), (640, 12288, 4096), (777, 8192, 4096),
                    (2049, 22016, 4096), (8192, 11264, 4096)):
        assert _fill_rule(n, M, K, True) and not _fill_rule(n, M, K, False), (n, M, K)
    for n, M, K in ((400, 11264, 2048), (2048, 11264, 2048), (1000, 9216, 2048), (1200, 6144, 2048), (1999, 4368, 2048)):
        assert _fill_rule(n, M, K, True) and _fill_rule(n, M, K, False), (n, M, K)
    for n, M, K in ((256, 22016, 4096), (512, 8192, 4096), (1200, 4096, 4096), (300, 11264, 2048), (640, 6144, 2048), (8193, 22016, 4096), (2049, 8192, 4096),
                    (2049, 22016, 8192), (1000, 22016, 16384)):
        assert not _fill_rule(n, M, K, True) and not _fill_rule(n, M, K, False), (n, M, K)
    # more columns: where the last round of 256 x 256 tiles is nearly full, few columns without a unit: where it is not
    for n, M, K, gated in ((1025, 24576, 5120, True), (777, 13696, 5120, True), (1800, 22016, 8192, True), (513, 18944, 4608, True),
                           (1600, 8192, 2048, False), (1100, 11264, 2048, False), (1792, 24576, 1024, True)):
        assert _fill_rule(n, M, K, gated), (n, M, K)
    for n, M, K, gated in ((513, 24576, 5120, True), (1152, 13696, 5120, True), (1152, 22016, 8192, True), (640, 27648, 5120, True),
                           (2048, 8192, 2048, False), (1800, 24576, 2048, False), (2048, 16384, 1024, False)):
        assert not _fill_rule(n, M, K, gated), (n, M, K)             # 0.79 to 0.94 of the library's speed


@pytest.mark.gpu
@pytest.mark.parametrize("K", [64, 136, 584])  # one chunk; two and a piece; nine and a piece
@pytest.mark.parametrize("n,M", SIZES)
def test_widths_of_the_tiles(n, M, K):
    """Against fp32 sums; rows of the results on and off 16-byte boundaries, and nothing beside them written."""
    from dejavu_amd import _lib_mixers as L
    from dejavu_amd import mixer_ops as ops

    g = torch.Generator(device="cuda").manual_seed(n + K)
    x = torch.randn(n, K + 16, generator=g, device="cuda").to(torch.bfloat16)[:, 8:8 + K]
    W = (torch.randn(M, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    bias = torch.randn(M, generator=g, device="cuda").to(torch.bfloat16)
    prod = x.double() @ W.double().t()
    for after, want in ((L.OUT_T, prod + bias.double()), (L.OUT_GLU, prod[:, 0::2].clamp(min=0) * prod[:, 1::2])):
        for pad in (8 - want.shape[1] % 8, 3):
            out = torch.full((n, want.shape[1] + pad), 77.0, dtype=torch.bfloat16, device="cuda")
            a = ops._tile_args(x, W)
            a.out, a.ldo, a.act = out.data_ptr(), out.shape[1], L.GLU_RELU
            a.bias = bias.data_ptr() if after == L.OUT_T else None
            ops.check(ops.lib.dv_mix_linear_wide(after, ops._ref(a), ops._stream()), "dv_mix_linear_wide")
            assert (out[:, want.shape[1]:] == 77.0).all()
            got = out[:, :want.shape[1]].double()
            # one rounding to bf16, 2 ** -9 at most, and fp32 sums of values of unit size
            assert ((got - want).abs() <= want.abs() * 2.0 ** -8 + 1e-5 * K ** 0.5).all(), (after, pad)


@pytest.mark.gpu
@pytest.mark.parametrize("n,M,K,x_far,w_far", [(300, 6, 136, False, True), (6, 1030, 72, True, False), (5, 12, 584, True, True),
                                               (2 ** 23 + 5, 4, 8, False, True)])  # (as many rows as one launch takes and more)
def test_rows_that_are_far_apart(n, M, K, x_far, w_far):
    """Strides beyond what 32 bits count the bytes of."""
    from dejavu_amd import _lib_mixers as L
    from dejavu_amd import mixer_ops as ops

    def far(t, yes):
        if not yes:
            return t
        room = torch.empty((t.shape[0] - 1) * 2 ** 25 + t.shape[1], dtype=t.dtype, device="cuda")
        return room.as_strided(t.shape, (2 ** 25, 1)).copy_(t)

    g = torch.Generator(device="cuda").manual_seed(n + K)
    x = torch.randn(n, K, generator=g, device="cuda").to(torch.bfloat16)
    W = (torch.randn(M, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    prod = x.double() @ W.double().t()
    x, W = far(x, x_far), far(W, w_far)
    for after, want in ((L.OUT_T, prod), (L.OUT_GLU, prod[:, 0::2].clamp(min=0) * prod[:, 1::2])):
        out = torch.full((n, want.shape[1]), 77.0, dtype=torch.bfloat16, device="cuda")
        a = ops._tile_args(x, W)
        a.out, a.ldo, a.act = out.data_ptr(), out.shape[1], L.GLU_RELU
        ops.check(ops.lib.dv_mix_linear_wide(after, ops._ref(a), ops._stream()), "dv_mix_linear_wide")
        # one rounding to bf16, 2 ** -9 at most, and fp32 sums of values of unit size
        assert ((out.double() - want).abs() <= want.abs() * 2.0 ** -8 + 1e-5 * K ** 0.5).all(), after


@pytest.mark.gpu
@pytest.mark.parametrize("M,ours", [(11264, True), (11268, False)])
def test_plain_products_whose_rows_leave_16_byte_boundaries(M, ours, monkeypatch):
    from dejavu_amd import mixer_ops as ops

    launches, kernel = [], ops.lib.dv_mix_linear_wide
    monkeypatch.setattr(ops.lib, "dv_mix_linear_wide", lambda *a: [launches.append(1), kernel(*a)][1])
    g = torch.Generator(device="cuda").manual_seed(M)
    x, W = (torch.randn(s, generator=g, device="cuda").to(torch.bfloat16) for s in ((400, 2048), (M, 2048)))
    got, want = ops.linear(x, W), x.float() @ W.float().t()
    assert bool(launches) == ours and (got - want).norm() < 1e-2 * want.norm()
    assert ops._fills(x, W, gated=True)
    ops.relu_glu(x, W)
    assert len(launches) == 1 + ours


@pytest.mark.gpu
def test_gated_units_through_the_ops():
    """A product on each side of the rule's line (144 tiles), both with the same result."""
    from dejavu_amd import mixer_ops as ops

    g = torch.Generator(device="cuda").manual_seed(1)
    W = (torch.randn(9200, 2048, generator=g, device="cuda") / 45).to(torch.bfloat16)
    x = torch.randn(385, 2048, generator=g, device="cuda").to(torch.bfloat16)
    assert ops._fills(x, W, gated=True) and not ops._fills(x[:384], W, gated=True) and not ops._wide(x, W)
    W2, x2 = W.repeat(2, 1)[:11264], x.repeat(22, 1)[:8193]
    assert ops._fills(x2[:8192], W2, gated=True) and not ops._fills(x2, W2, gated=True)
    for x, W, rows in ((x, W, 384), (x, W, 385), (x2, W2, 2049), (x2, W2, 8192), (x2, W2, 8193)):
        want = x[:rows].float() @ W.float().t()
        unit = want[:, 0::2].clamp(min=0) * want[:, 1::2]
        got = ops.relu_glu(x[:rows], W).float()
        assert (got - unit).norm() / unit.norm() < 1e-2


def test_which_products_of_a_prompt_the_wide_kernel_takes():
    from dejavu_amd.modules import _wide_rule as rule

    for rows, M, K in ((400, 8192, 2048), (777, 16384, 4096), (512, 20480, 5120), (2000, 16384, 4096), (8192, 20480, 5120)):
        assert rule(rows, M, K, "relu") and rule(rows, M, K, "squared_relu") and not rule(rows, M, K, "id") and not rule(rows, M, K, "gelu")
    for rows, M, K in ((256, 16384, 4096), (300, 16384, 4096), (257, 8192, 2048), (8193, 16384, 4096), (2049, 36864, 9216), (777, 3072, 768)):
        assert not rule(rows, M, K, "relu"), (rows, M, K)
    assert rule(777, 5120, 20480, "id") and not rule(767, 5120, 20480, "id") and not rule(1200, 4096, 16384, "id")
    # where the library is ahead at some sizes, and on both sides of the lines
    for rows, M, K in ((300, 36864, 9216), (1000, 36864, 9216), (640, 24576, 6144), (513, 12288, 3072), (768, 16384, 5128)):
        assert not rule(rows, M, K, "relu"), (rows, M, K)
    assert rule(641, 12288, 3072, "relu") and rule(257, 12288, 3064, "relu") and rule(1000, 20480, 5120, "relu")
    for rows, M, K in ((768, 5120, 20480), (1000, 5124, 20496), (2049, 5120, 20480), (1024, 4096, 20480), (1152, 5376, 21504), (1600, 9216, 36864)):
        assert not rule(rows, M, K, "id"), (rows, M, K)
    assert rule(769, 5120, 20480, "id") and rule(1025, 4096, 20480, "id") and rule(2048, 5120, 20480, "id")


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["id", "relu", "squared_relu"])
@pytest.mark.parametrize("n,M,K", [(257, 1030, 136), (300, 1001, 72), (777, 520, 584)])
def test_wide_products_in_fp16(n, M, K, act):
    """Rows of results on and off 16-byte boundaries, the bias past the end of a tile."""
    from dejavu_amd import ops

    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n, K, generator=g, device="cuda").half()
    W = (torch.randn(M, K, generator=g, device="cuda") * K ** -0.5).half()
    bias = torch.randn(M, generator=g, device="cuda").half()
    for b in (bias, None):
        want = x.double() @ W.double().t() + (0 if b is None else b.double())
        want = {"id": lambda t: t, "relu": lambda t: t.clamp(min=0), "squared_relu": lambda t: t.clamp(min=0) ** 2}[act](want)
        got = ops.dense_linear_wide(x, W, b, act).double()
        # one rounding to fp16, 2 ** -11 at most, and fp32 sums of values of unit size
        assert ((got - want).abs() <= want.abs() * 2.0 ** -10 + 1e-5 * K ** 0.5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["id", "relu", "squared_relu"])
@pytest.mark.parametrize("n,M", SIZES)
def test_widths_of_the_tiles_in_fp16(n, M, act):
    from dejavu_amd import ops

    K = 136
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n, K, generator=g, device="cuda").half()
    W = (torch.randn(M, K, generator=g, device="cuda") * K ** -0.5).half()
    bias = torch.randn(M, generator=g, device="cuda").half()
    want = x.double() @ W.double().t() + bias.double()
    want = {"id": lambda t: t, "relu": lambda t: t.clamp(min=0), "squared_relu": lambda t: t.clamp(min=0) ** 2}[act](want)
    got = ops.dense_linear_wide(x, W, bias, act).double()
    # one rounding to fp16, 2 ** -11 at most, and fp32 sums of values of unit size
    assert ((got - want).abs() <= want.abs() * 2.0 ** -10 + 1e-5 * K ** 0.5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("K", [8, 40, 56, 64])
def test_fewer_columns_than_a_chunk(K):
    """The last columns are all there are: no chunk goes before them."""
    from dejavu_amd import _lib_mixers as L
    from dejavu_amd import mixer_ops, ops

    g = torch.Generator(device="cuda").manual_seed(K)
    n, M = 300, 1030
    for dtype in (torch.float16, torch.bfloat16):
        room = torch.full((n + M, K + 16), float("nan"), dtype=dtype, device="cuda")  # what lies beside the rows does not get in
        x, W = room[:n, 8:K + 8], room[n:, 8:K + 8]
        x.copy_(torch.randn(n, K, generator=g, device="cuda"))
        W.copy_(torch.randn(M, K, generator=g, device="cuda") * K ** -0.5)
        want = x.double() @ W.double().t()
        if dtype == torch.float16:
            got = torch.empty(n, M, dtype=dtype, device="cuda")
            ops.check(ops.lib.dv_dense_linear_wide_f16(x.data_ptr(), x.stride(0), W.data_ptr(), W.stride(0), None, n, K, M, 0, got.data_ptr(), M,
                                                       ops._stream()), "dv_dense_linear_wide_f16")
        else:
            got = torch.empty(n, M, dtype=dtype, device="cuda")
            a = mixer_ops._tile_args(x, W)
            a.out, a.ldo = got.data_ptr(), M
            ops.check(mixer_ops.lib.dv_mix_linear_wide(L.OUT_T, mixer_ops._ref(a), ops._stream()), "dv_mix_linear_wide")
        # one rounding, half of a last place, and fp32 sums of values of unit size
        assert ((got.double() - want).abs() <= want.abs() * torch.finfo(dtype).eps + 1e-5 * K ** 0.5).all(), dtype


@pytest.mark.gpu
@torch.no_grad()
@pytest.mark.parametrize("positive", [False, True])
def test_longest_rows_through_the_layers(positive):
    """fc2 without an activation, whose sums are one chain over 20480 columns; of numbers of one sign they grow all the way."""
    from dejavu_amd import modules

    g = torch.Generator(device="cuda").manual_seed(3)
    n, M, K = 769, 5120, 20480
    layer = torch.nn.Linear(K, M, device="cuda", dtype=torch.float16)
    x, W = torch.randn(1, n, K, generator=g, device="cuda"), torch.randn(M, K, generator=g, device="cuda") * K ** -0.5
    if positive:
        x, W = x.abs(), W.abs() * K ** -0.5
    x = x.half()
    layer.weight.copy_(W)
    assert modules._wide_product(layer, x, "id") and not modules._wide_product(layer, x[:, :768], "id")
    got = modules.decode_linear(layer, x)[0].double()
    want = x[0].double() @ layer.weight.double().t() + layer.bias.double()
    # a rounding to fp16, half of 2 ** -10, and one of 2 ** -24 of a sum at each of 640 instructions: all of one sign together, or of sums
    # of unit size, a few times their root mean square
    limit = want.abs() * (2.0 ** -11 + 640 * 2.0 ** -24) if positive else want.abs() * 2.0 ** -11 + 8 * 640 ** 0.5 * 2.0 ** -24
    assert ((got - want).abs() <= limit).all()


@pytest.mark.gpu
@torch.no_grad()
@pytest.mark.parametrize("act", ["id", "relu", "squared_relu"])
def test_values_that_are_no_finite_numbers(act):
    """They are where the library and a launch for the activation have them: NaN and both infinities in rows, weight and bias."""
    from dejavu_amd import modules, ops

    inf, nan = float("inf"), float("nan")
    layer = torch.nn.Linear(2048, 8192, device="cuda", dtype=torch.float16)
    layer.bias[17:20] = torch.tensor([nan, inf, -inf], dtype=torch.float16)
    layer.weight[300, 5], layer.weight[301, 6], layer.weight[302, 7] = nan, inf, -inf
    x = torch.randn(1, 400, 2048, device="cuda").half()
    x[0, 3, 100], x[0, 130, 101], x[0, 399, 102] = nan, inf, -inf
    y = torch.nn.functional.linear(x, layer.weight, layer.bias)
    want = {"id": y, "relu": torch.relu(y), "squared_relu": torch.relu(y) ** 2}[act]
    results = [ops.dense_linear_wide(x, layer.weight, layer.bias, act)]
    if act != "id":
        assert modules._wide_product(layer, x, act)
        results.append(modules.decode_linear(layer, x, act))
    for got in results:
        assert want.isnan().sum() > 8192 and torch.equal(got.isnan(), want.isnan())
        assert want.isinf().any() and torch.equal(got.isinf(), want.isinf()) and torch.equal(got[want.isinf()], want[want.isinf()])


@pytest.mark.gpu
def test_long_prompts_through_the_layers():
    """fc1 with its activation on both sides of the rule's line, and what only the library does."""
    from dejavu_amd import modules

    layer = torch.nn.Linear(2048, 8192, device="cuda", dtype=torch.float16)
    x = torch.randn(1, 400, 2048, device="cuda").half()
    with torch.no_grad():
        for rows in (384, 385, 400):
            assert modules._wide_product(layer, x[:, :rows], "relu") == (rows > 384)
            want = torch.relu(layer(x[:, :rows]))
            got = modules.decode_linear(layer, x[:, :rows], "relu")
            assert got.shape == want.shape and (got - want).abs().max() <= 2.0 ** -9 * want.abs().max()
        long = x.repeat(1, 21, 1)[:, :8193]
        for rows in (2049, 8192, 8193):
            assert modules._wide_product(layer, long[:, :rows], "relu") == (rows < 8193)
            want, got = torch.relu(layer(long[:, :rows])), modules.decode_linear(layer, long[:, :rows], "relu")
            assert (got - want).abs().max() <= 2.0 ** -9 * want.abs().max()
        assert not modules._wide_product(layer, x[:, ::2].expand(1, 200, 2048), "relu")
        seen = []
        hook = layer.register_forward_hook(lambda *a: seen.append(1))
        assert not modules._wide_product(layer, x, "relu")
        modules.decode_linear(layer, x, "relu")
        hook.remove()
        assert seen == [1] and modules._wide_product(layer, x, "relu")
    assert not modules._wide_product(layer, x, "relu")  # gradients
    modules.decode_linear(layer, x, "relu").sum().backward()
    assert layer.weight.grad is not None


@pytest.mark.gpu
def test_window_reset():
    from dejavu_amd._lib import check, lib

    for heads in (1, 17, 40):
        tracker = torch.full((heads + 1, 16), -7, dtype=torch.int32, device="cuda")
        place = torch.full((2,), -7, dtype=torch.int32, device="cuda")
        check(lib.dv_window_reset(tracker.data_ptr(), heads, place.data_ptr(), 123, torch.cuda.current_stream().cuda_stream), "dv_window_reset")
        assert torch.equal(tracker[:heads], torch.arange(16, device="cuda", dtype=torch.int32).repeat(heads, 1))
        assert (tracker[heads] == -7).all() and place.tolist() == [123, -7]
    assert lib.dv_window_reset(None, 4, None, 0, None) == -1
