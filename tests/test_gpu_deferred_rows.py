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


class _Norm:
    def __init__(self, width):
        self.w, self.b = torch.rand(width, device="cuda") + 0.5, torch.rand(width, device="cuda")

    def struct(self):
        return ops.L.DynTanh(self.w.data_ptr(), self.b.data_ptr(), 0.7)

    def __call__(self, x):
        return torch.tanh(0.7 * x) * self.w.double() + self.b.double()


def _row_in_splits(heads, vdim, splits, seed, gated=True):
    """What the splits' launch leaves, and the row of it in 64 bits."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rand(*shape, scale=1.0):
        return torch.randn(*shape, device="cuda", generator=g) * scale

    l = rand(heads, splits).abs() + 0.5
    sums, m = rand(heads, splits, vdim) * l[..., None], rand(heads, splits, scale=3.0)
    sums[-1, 0], m[-1, 0], l[-1, 0] = 0.0, -1e30, 0.0  # a split without keys
    part = torch.cat([sums.reshape(-1), torch.stack([m, l], -1).reshape(-1)])
    sink, gate = (None, rand(heads)) if gated else (rand(heads), None)
    top = m.double().amax(1, keepdim=True)
    if sink is not None:
        top = torch.maximum(top, sink.double()[:, None])
    w = (m.double() - top).exp()
    den = (w * l.double()).sum(1) + (0 if sink is None else (sink.double() - top[:, 0]).exp())
    o = (w[..., None] * sums.double()).sum(1) / den[:, None] * (1 if gate is None else gate.double().sigmoid()[:, None])
    return ops.SplitRow(part, splits, heads, vdim, sink, gate, torch.bfloat16), o.reshape(1, -1)


SIZES = [(1, 8, 2, 72), (4, 64, 7, 256), (5, 80, 9, 264), (16, 128, 8, 2048), (17, 128, 6, 2056)]  # the last two: rows that two waves share


# The row is rounded to bf16 before the product (2^-9 a value); what follows is fp32.
@pytest.mark.parametrize("heads,vdim,splits,M", SIZES)
@torch.no_grad()
def test_merge_before_a_residual(heads, vdim, splits, M):
    row, o = _row_in_splits(heads, vdim, splits, heads, gated=False)
    W = (torch.randn(M, o.shape[1], device="cuda") * o.shape[1] ** -0.5).bfloat16()
    stream = ops.ResidualStream(torch.randn(1, M, device="cuda"), torch.randn(1, M, device="cuda"), torch.bfloat16)
    post, pre, old = _Norm(M), _Norm(M), stream.x.double()
    h = ops.linear_residual(row, W, stream, post, pre, add_start=True)
    y = o @ W.double().t()
    step = 2.0 ** -8 * float(o.norm()) * float(W.double().norm(dim=1).max())  # of a sum of rounded values
    want = old + post(y) + stream.start.double()
    assert float((stream.x.double() - want).abs().max()) <= 1.5 * 0.7 * step + 1e-5
    h_want = pre(stream.x.double())
    assert float((h.double() - h_want).abs().max()) <= 2.0 ** -8 * float(h_want.abs().max())


@pytest.mark.parametrize("heads,vdim,splits,M", SIZES)
@pytest.mark.parametrize("streams", [1, 2, 4, 5])  # five: more than the row's launch takes
@torch.no_grad()
def test_merge_before_several_streams(heads, vdim, splits, M, streams):
    row, o = _row_in_splits(heads, vdim, splits, heads + streams)
    W = (torch.randn(M, o.shape[1], device="cuda") * o.shape[1] ** -0.5).bfloat16()
    bias = torch.randn(M, device="cuda").bfloat16()
    write, norm = mixers.HyperConnection(streams, device="cuda"), mixers.RMSNorm(M, 1e-5, device="cuda")
    for p in (write.mix, write.out, norm.weight):
        p.normal_()
    weights = torch.randn(streams, device="cuda")
    stream = ops.HyperStream(torch.randn(1, streams, M, device="cuda"), torch.bfloat16)
    old = stream.x.double()
    h = stream.update(row, W, bias, write, ops.StreamRead(norm, weights))
    y = o @ W.double().t() + bias.double()
    want = torch.einsum("st,nsw->ntw", write.mix.double(), old) + write.out.double()[None, :, None] * y[:, None]
    step = 2.0 ** -8 * (float(o.norm()) * float(W.double().norm(dim=1).max()) + float(y.abs().max()))  # (five: the result is rounded, too)
    assert float((stream.x.double() - want).abs().max()) <= float(write.out.abs().max()) * step + 1e-5 * float(want.abs().max())
    read = (stream.x.double() * weights.double()[None, :, None]).sum(1)
    if streams <= ops.L.HYPER_ROW_MAX:
        assert isinstance(h, ops.RmsRow) and float((h.u.double() - read).abs().max()) <= 1e-5 * (1 + float(read.abs().max()))
    else:
        normed = read / (read.square().mean() + 1e-5).sqrt() * norm.weight.double()
        assert float((h.double() - normed).abs().max()) <= 2.0 ** -8 * float(normed.abs().max())


@pytest.mark.parametrize("seen", [0, 63, 399, 400, 401, 1203])
@pytest.mark.parametrize("values", [None, "first", "mixed"])
@torch.no_grad()
def test_chunk_attention_deferred(seen, values):
    """Biases by distance, normed and mixed values, gates; before, at and behind the end of a chunk of 400."""
    m, h = _chunk(400, values), torch.randn(1, WIDTH, device="cuda").bfloat16()
    rows, rings = [], []
    for call in (mixers.apply_mixer, lambda m, *a: m(*a)):
        state, step = _state(m, seen), mixers.StepInfo(seen)
        step.first_values = torch.randn(1, 2 * DIM, device="cuda", generator=torch.Generator(device="cuda").manual_seed(2))
        rows.append(call(m, h, state, step))
        rings.append(state)
    assert isinstance(rows[0], ops.SplitRow) and isinstance(rows[1], torch.Tensor)
    assert all(torch.equal(rings[0][k], rings[1][k]) for k in rings[0])
    a, b = (ops.linear(r, m.out_proj, m.out_bias).double() for r in rows)
    assert float((a - b).norm()) <= 2.0 ** -8 * float(b.norm())


@pytest.mark.parametrize("kind", ["window", "chunk"])
@torch.no_grad()
def test_layers_of_a_model(kind, monkeypatch):
    """A block's decode steps with the merge in the projection and with its own launch, from before the ring's end to behind it."""
    from dejavu_amd.hybrid import HybridBlock, LayerSpec, StreamsBlock

    mixer = dict(heads=HEADS, kv_heads=2, dim=DIM, vdim=DIM, scale=DIM ** -0.5)
    if kind == "window":
        spec = LayerSpec("attention", dict(mixer, conv=4, mask={"size": 400}), {"ff": 512, "limit": 7.0})
        block = _filled(HybridBlock(spec, WIDTH, 1e-5, dtype=torch.bfloat16, device="cuda"))
    else:
        spec = LayerSpec("chunk_attention", dict(mixer, chunk=400, bias_rows=16, bias_max=64, values="first"), {"ff": 512})
        block = _filled(StreamsBlock(spec, WIDTH, 1e-5, 3, dtype=torch.bfloat16, device="cuda"))
    asked, rule = [], ops._merge_rule
    results = []
    for merged in (True, False):
        monkeypatch.setattr(ops, "_merge_rule", lambda *a: [asked.append(1), merged and rule(*a)][1])
        g = torch.Generator(device="cuda").manual_seed(5)
        state = _state(block.mixer, 395)
        for pos in range(396, 404):
            x = torch.randn(1, WIDTH, device="cuda", generator=g)
            if kind == "window":
                stream = ops.ResidualStream(x, None, torch.bfloat16)
                h = block((x * 0.5).bfloat16(), stream, state, mixers.StepInfo(pos), _Norm(WIDTH))
            else:
                stream = ops.HyperStream(torch.randn(1, 3, WIDTH, device="cuda", generator=g), torch.bfloat16)
                block(stream.read(block.entry), stream, state, mixers.StepInfo(pos), block.entry)
            results.append(stream.x.double())
    assert len(asked) == 16
    for a, b in zip(results[:8], results[8:]):
        # the row's rounding, 2^-9, through two products and the norms between them
        assert float((a - b).norm()) <= 2.0 ** -6 * float(b.norm())
