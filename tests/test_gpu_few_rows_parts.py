"""Up to 256 rows on one column of wide tiles with K in parts: widths of tiles, what ends within one, activations, what the modules send there."""
import pytest
import torch
import torch.nn as nn

from dejavu_amd import modules, ops

pytestmark = pytest.mark.gpu
ACT = {"id": lambda v: v, "relu": lambda v: v.clamp_min(0), "squared_relu": lambda v: v.clamp_min(0) ** 2}


@pytest.mark.parametrize("rows", [1, 65, 128, 129, 160, 161, 193, 225, 256])
@pytest.mark.parametrize("M,K,activation", [(15368, 2568, "relu"), (1032, 4104, "id"), (20480, 1536, "squared_relu")])
def test_few_rows_in_parts(rows, M, K, activation):
    g = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(1, rows, K, device="cuda", generator=g).half()
    W = (torch.randn(M, K, device="cuda", generator=g) * K ** -0.5).half()
    b = torch.randn(M, device="cuda", generator=g).half()
    assert ops.wide_parts(rows, K, M) > 1
    got = ops.dense_linear_wide_parts(x, W, b, activation)[0].double()
    sums = x[0].double() @ W.double().t() + b.double()
    want = ACT[activation](sums)
    # half a step of fp16, and the rounding of fp32 sums of K products of values of about one, which the square multiplies
    bound = 2.0 ** -11 * want.abs() + 2.0 ** -24 * K ** 0.5 * 8 * (1 + 2 * sums.abs()) + 2.0 ** -25
    assert bool(((got - want).abs() <= bound).all())


def test_what_the_modules_send_there():
    # (columns, and weight rows up to 16384, by what was measured on both sides of each line)
    taken = [(rows, M, K) for M, K in ((15368, 4096), (20480, 2560), (20488, 2560), (15360, 4096), (20480, 2552), (15368, 2560), (16384, 5120), (16392, 5120),
                                       (20480, 6144), (16384, 6144), (16384, 8192)) for rows in (128, 129, 192, 193)
             if modules._few_parts_product(nn.Linear(K, M, device="cuda", dtype=torch.float16).requires_grad_(False),
                                           torch.zeros(1, rows, K, device="cuda", dtype=torch.float16), "relu")]
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert taken == [(rows, M, K) for M, K in ((15368, 4096), (20480, 2560), (16392, 5120), (16384, 8192)) for rows in (129, 192)]
    lin = nn.Linear(2560, 16392, device="cuda", dtype=torch.float16).requires_grad_(False)
    x = torch.randn(1, 150, 2560, device="cuda").half()
    assert modules._few_parts_product(lin, x, "relu") or torch.cuda.get_device_properties(0).multi_processor_count != 256
    assert not modules._few_parts_product(lin, x, "gelu") and not modules._few_parts_product(lin, torch.cat([x, x])[:, ::2], "relu")
    y = modules.decode_linear(lin, x, "relu")
    want = torch.relu(x.double() @ lin.weight.double().t() + lin.bias.double())
    assert (y.double() - want).norm() <= 2 ** -10 * want.norm()
    lin.requires_grad_(True)
    assert not modules._few_parts_product(lin, x, "relu")  # (gradients are asked for)
