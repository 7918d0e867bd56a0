"""Decode rows whose splits the output projection merges: who is given one, and what the projections make of it."""
import pytest
import torch
import torch.nn as nn

from dejavu_amd import mixer_ops as ops
from dejavu_amd import mixers

pytestmark = pytest.mark.gpu
WIDTH, HEADS, DIM = 256, 4, 64


def _filled(m, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    with torch.no_grad():
        for name, p in m.named_parameters():
            p.copy_(torch.randn(p.shape, device="cuda", generator=g) * (p.shape[-1] ** -0.5 if p.dim() == 2 else 0.3))
            if name.endswith("norm"):
                p.add_(1.0)
    return m


def _window(keys=400):
    return _filled(mixers.WindowAttention(WIDTH, HEADS, 2, DIM, DIM, 4, keys, DIM ** -0.5, 1e-5, dtype=torch.bfloat16, device="cuda"))


def _chunk(keys=400, values=None):
    return _filled(mixers.ChunkAttention(WIDTH, HEADS, 2, DIM, DIM, keys, DIM ** -0.5, 16, 64, values, 1e-5, dtype=torch.bfloat16, device="cuda"))


def _state(m, seen, seed=1):
    """The state of a sequence that has ``seen`` tokens, as random as they are."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return {k: torch.randn(t.shape, device="cuda", generator=g).to(t.dtype) for k, t in m.new_state(2000).items()}


@pytest.mark.parametrize("make", [_window, _chunk])
@torch.no_grad()
def test_only_who_asks_gets_rows_in_splits(make):
    h = torch.randn(1, WIDTH, device="cuda").bfloat16()

    def row(m, call):
        return call(m, h, _state(m, 390), mixers.StepInfo(390))

    m = make()
    want = row(m, lambda m, *a: m(*a))
    assert isinstance(want, torch.Tensor) and want.shape == (1, HEADS * DIM)
    assert isinstance(row(m, mixers.apply_mixer), ops.SplitRow)

    class Scaled(type(m)):
        def forward(self, *args):
            return super().forward(*args) * 2

    class Wrapped(nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, *args):
            return self.inner(*args) * 2

        new_state = property(lambda self: self.inner.new_state)

    assert torch.equal(row(Wrapped(m), mixers.apply_mixer), want * 2)
    seen = []
    handle = m.register_forward_hook(lambda m, a, o: seen.append(o))
    assert torch.equal(row(m, mixers.apply_mixer), want) and torch.equal(seen[0], want)
    handle.remove()
    m.__class__ = Scaled
    assert torch.equal(row(m, mixers.apply_mixer), want * 2)
