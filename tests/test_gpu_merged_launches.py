"""Launches that do what two did before: the convolution that moves its state on, two kinds of normed rows, two rings."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DTYPES = [torch.bfloat16, torch.float32]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5])                  # (five by the kernel for any number)
@pytest.mark.parametrize("n", [1, 2, 3, 7, 8, 9, 47])
def test_convolution_moves_its_state(n, taps, dtype):
    from dejavu_amd import mixer_ops as ops

    g = torch.Generator(device="cuda").manual_seed(n * 10 + taps)
    heads, stride, dim = 5, 24, 21
    x = torch.randn(n, heads * stride + 8, generator=g, device="cuda").to(dtype)
    w = torch.randn(heads * stride, taps, generator=g, device="cuda")
    state = torch.randn(heads * stride, max(1, taps - 1), generator=g, device="cuda")
    outs = []
    for move in (False, True):
        st, out = state.clone(), torch.zeros(n, heads * stride, dtype=dtype, device="cuda")
        ops.short_conv(x, w, st, [(heads, stride, dim, ops.NORM_RMS, 1e-5, 1.0, out)], silu=True, move=move)
        if not move:
            assert torch.equal(st, state)
            ops.conv_state(x, heads * stride, taps, st)
        outs.append((out, st))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    if taps > 1:
        rows = torch.cat([state.t(), x[:, :heads * stride].float()])[-(taps - 1):]
        assert torch.equal(outs[1][1], rows.t())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n", [2, 5, 47])
def test_two_kinds_of_normed_rows(n, dtype):
    from dejavu_amd import mixer_ops as ops

    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n, 24 + 2056 + 8, generator=g, device="cuda").to(dtype)
    wa, wb = torch.randn(24, generator=g, device="cuda"), torch.randn(2056, generator=g, device="cuda")
    cache = torch.full((n + 3, 2056), 7.0, dtype=dtype, device="cuda")
    a = torch.empty(n, 24, dtype=dtype, device="cuda")
    ops.rms_rows_two(x, (0, wa, 21, a), (24, wb, 2050, cache[1:n + 1]), 1e-5)
    assert torch.equal(a, ops.rms_rows(x[:, :24], wa, 21, 1e-5))
    assert torch.equal(cache[1:n + 1], ops.rms_rows(x[:, 24:2080], wb, 2050, 1e-5))
    assert (cache[0] == 7).all() and (cache[n + 1:] == 7).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("first,count", [(0, 1), (5, 9), (13, 20)])  # round the end of the ring, all of it
def test_two_rings(first, count, dtype):
    from dejavu_amd import mixer_ops as ops

    g = torch.Generator(device="cuda").manual_seed(first)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)  # noqa: E731
    bufs, rings = [rand(count + 2, 16), rand(count + 2, 1032)], [rand(20, 16), rand(20, 1032)]
    rows = [(first + i) % 20 for i in range(count)]
    want = [r.clone() for r in rings]
    for r, b in zip(want, bufs):
        r[rows] = b[2:]
    ops.ring_copy_two([b[2:] for b in bufs], rings, first, to_ring=True)
    assert all(torch.equal(r, w) for r, w in zip(rings, want))
    back = [torch.zeros_like(b) for b in bufs]
    ops.ring_copy_two([b[:count] for b in back], rings, first, to_ring=False)
    assert all(torch.equal(b[:count], w[rows]) and (b[count:] == 0).all() for b, w in zip(back, want))
