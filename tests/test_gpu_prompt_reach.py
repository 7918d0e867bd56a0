"""Prompt attention with a value that is not finite: which queries it reaches."""
import pytest
import torch

from dejavu_amd import ops

pytestmark = pytest.mark.gpu


# the last: 32 queries a workgroup, whose reach the tiles of 128 queries have too
@pytest.mark.parametrize("T,H,hd", [(512, 64, 128), (1000, 33, 128), (777, 83, 64), (512, 4, 128)])
@pytest.mark.parametrize("key", [0, 31, 32, 63, 64, 95, 100, 127, 128, 200, 511])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_reach_of_a_value(T, H, hd, key, bad):
    """A query multiplies its own 32 keys and those before them, the later ones of them with weight zero: nothing further on."""
    g = torch.Generator(device="cuda").manual_seed(key)
    qkv = torch.randn(1, T, 3, H, hd, device="cuda", generator=g).half()
    want = ops.prefill_attention(qkv).view(T, H, hd)
    qkv[0, key, 2, 1, 3] = bad
    got = ops.prefill_attention(qkv).view(T, H, hd)
    first = key // 32 * 32
    # before it, other heads, other channels: as they were, to the bit
    assert torch.equal(got[:first], want[:first])
    assert torch.equal(got[:, :1], want[:, :1]) and torch.equal(got[:, 2:], want[:, 2:])
    assert torch.equal(got[:, 1, :3], want[:, 1, :3]) and torch.equal(got[:, 1, 4:], want[:, 1, 4:])
    assert not bool(torch.isfinite(got[key:, 1, 3]).any())  # who sees it
