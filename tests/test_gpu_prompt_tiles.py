"""Prompt attention in tiles of 128 queries: lengths around tiles of queries and keys, several sequences, caches and where they begin."""
import pytest
import torch

from dejavu_amd import ops

pytestmark = pytest.mark.gpu


# each with enough heads for the tiles; 32 queries a workgroup below them (the last)
@pytest.mark.parametrize("B,T,H,hd", [(1, 450, 72, 128), (1, 512, 64, 128), (1, 513, 64, 128), (1, 575, 56, 128), (2, 641, 25, 128), (1, 1023, 32, 128),
                                      (1, 256, 128, 128), (1, 450, 144, 64), (3, 577, 38, 64), (1, 400, 90, 128)])
@pytest.mark.parametrize("pos0,more", [(0, 0), (5, 9)])
def test_tiles(B, T, H, hd, pos0, more):
    g = torch.Generator(device="cuda").manual_seed(T)
    qkv = torch.randn(B, T, 3, H, hd, device="cuda", generator=g).half()
    qkv[:, 64:128, 1] *= 3  # a maximum that one group of the keys' tiles has
    S = pos0 + T + more
    kc, vc = torch.full((B, H, hd // 8, S, 8), 7.0, device="cuda").half(), torch.full((B, H, S, hd), 7.0, device="cuda").half()
    got = ops.prefill_attention(qkv, kc, vc, pos0)
    k = kc[:, :, :, pos0:pos0 + T].permute(0, 3, 1, 2, 4).reshape(B, T, H, hd)
    assert torch.equal(k, qkv[:, :, 1]) and torch.equal(vc[:, :, pos0:pos0 + T].transpose(1, 2), qkv[:, :, 2])
    for c, at in ((kc, 3), (vc, 2)):
        rest = torch.cat([c.narrow(at, 0, pos0), c.narrow(at, pos0 + T, more)], at)
        assert bool((rest == 7).all())
    q, k, v = (t.double().transpose(1, 2) for t in qkv[:, :, :, ::7].unbind(2))  # every seventh head
    s = (q @ k.transpose(2, 3).contiguous()) * hd ** -0.5
    s = s.masked_fill(torch.ones(T, T, device="cuda", dtype=torch.bool).triu(1), float("-inf"))
    want = (s.softmax(-1) @ v.contiguous()).transpose(1, 2)
    got = got.view(B, T, H, hd)[:, :, ::7].double()
    # weights and results are rounded to fp16, 2^-12 each
    assert (got - want).norm() <= 2 ** -10 * want.norm() and (got - want).abs().max() <= 2 ** -9 * want.abs().max()
    assert torch.equal(ops.prefill_attention(qkv).view(B, T, H, hd)[:, :, ::7].double(), got)  # without caches


# short prompts on both sides of the lines in full tiles and in workgroups (288, 384; 588, 600 of 256 compute units)
@pytest.mark.parametrize("B,T,H,hd", [(2, 224, 72, 128), (2, 224, 96, 128), (1, 256, 128, 128), (2, 308, 98, 128), (2, 308, 100, 128), (4, 307, 50, 128), (4, 410, 50, 64),
                                      (4, 448, 40, 64), (4, 447, 40, 64)])
def test_short_prompts(B, T, H, hd):
    test_tiles(B, T, H, hd, 0, 3)
