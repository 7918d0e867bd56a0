"""Prompt attention whose key tiles two groups of waves share: odd and even numbers of them, masks that begin inside one, groups without any."""
import pytest
import torch

from dejavu_amd import mixer_ops as ops

pytestmark = pytest.mark.gpu


def _reference(q, k, v, H, G, scale, pos, window, chunk, rel, sink, gate):
    n, keys = q.shape[0], k.shape[0]
    q, k, v = (t.double().view(t.shape[0], h, -1).transpose(0, 1) for t, h in ((q, H), (k, G), (v, G)))
    k, v = (t.repeat_interleave(H // G, 0) for t in (k, v))
    s = (q @ k.transpose(1, 2)) * scale
    i, j = torch.arange(pos, pos + n, device="cuda")[:, None], torch.arange(keys, device="cuda")[None]
    if rel is not None:
        s = s + rel.double()[:, (i - j).clamp(0, rel.shape[1] - 1)]
    low = i - window + 1 if window else i - i % chunk if chunk else i * 0
    s = s.masked_fill((j > i) | (j < low), float("-inf"))
    if sink is not None:
        s = torch.cat([s, sink.double()[:, None, None].expand(H, n, 1)], -1)
    p = s.softmax(-1)[..., :keys]
    o = (p @ v).transpose(0, 1)
    if gate is not None:
        o = o * gate.double().sigmoid()[..., None]
    return o.reshape(n, -1)


# (tokens, of which came before): below the line between one group and two, on it, one more tile, the last group's last tile short, rows past the end
@pytest.mark.parametrize("n,before", [(128, 0), (129, 0), (191, 0), (193, 0), (257, 0), (1, 200), (47, 130), (130, 511), (300, 85)])
@pytest.mark.parametrize("mask", ["causal", "window", "chunk"])
@pytest.mark.parametrize("dim,vdim", [(128, 128), (64, 32), (40, 104)])
def test_two_groups(n, before, mask, dim, vdim):
    H, G, keys = 4, 2, n + before
    g = torch.Generator(device="cuda").manual_seed(n + before)
    q, k, v = (torch.randn(r, h * d, device="cuda", generator=g).bfloat16() for r, h, d in ((n, H, dim), (keys, G, dim), (keys, G, vdim)))
    window, chunk = (65 if n < 200 else 150 if mask == "window" else None), None
    window = window if mask == "window" else None
    chunk = 140 if mask == "chunk" else None
    rel = torch.randn(H, 70, device="cuda", generator=g) if mask == "chunk" else None
    sink = torch.randn(H, device="cuda", generator=g) if mask == "window" else None
    gate = torch.randn(n, H, device="cuda", generator=g).bfloat16() if mask == "causal" else None
    got = ops.portion_attention(q, k, v, H, G, dim ** -0.5, 0, before, sink=sink, gate=gate, window=window, chunk=chunk, rel=rel)
    want = _reference(q, k, v, H, G, dim ** -0.5, before, window, chunk, rel, sink, gate)
    # weights and results are rounded to bf16: 2^-9 each
    assert (got.double() - want).norm() <= 2 ** -8 * want.norm()
    assert (got.double() - want).abs().max() <= 2 ** -6 * want.abs().max()


def test_large_scores_in_one_group_only():
    """Maxima that differ between the groups, and keys whose scores underflow in one."""
    n, H = 256, 2
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.randn(n, H * 128, device="cuda", generator=g).bfloat16() for _ in range(3))
    k[64:128] *= 12.0
    got = ops.portion_attention(q, k, v, H, H, 128 ** -0.5, 0, 0)
    want = _reference(q, k, v, H, H, 128 ** -0.5, 0, None, None, None, None, None)
    assert bool(torch.isfinite(got).all()) and (got.double() - want).norm() <= 2 ** -8 * want.norm()


# around one and two workgroups a compute unit (256 of them), key tiles a query tile on both sides of the lines
@pytest.mark.parametrize("H,n", [(64, 500), (72, 500), (128, 500), (136, 500), (40, 1500), (4, 400)])
@pytest.mark.parametrize("mask", [{}, {"window": 64}, {"window": 66}, {"window": 130}, {"chunk": 64}, {"chunk": 128}, {"chunk": 700}])
@pytest.mark.parametrize("dim,vdim", [(64, 64), (128, 128), (64, 72)])
def test_many_workgroups(H, n, mask, dim, vdim):
    G = 4
    g = torch.Generator(device="cuda").manual_seed(H + n)
    q, k, v = (torch.randn(n, h * d, device="cuda", generator=g).bfloat16() for h, d in ((H, dim), (G, dim), (G, vdim)))
    got = ops.portion_attention(q, k, v, H, G, dim ** -0.5, 0, 0, **mask).view(n, H, vdim)
    some = [0, H // 4, 3 * H // 4 - 1, H - 1]  # a head of each key head
    want = _reference(q.view(n, H, dim)[:, some].reshape(n, -1), k, v, G, G, dim ** -0.5, 0, mask.get("window"), mask.get("chunk"), None, None, None)
    got = got[:, some].reshape(n, -1).double()
    assert (got - want).norm() <= 2 ** -8 * want.norm() and (got - want).abs().max() <= 2 ** -6 * want.abs().max()
