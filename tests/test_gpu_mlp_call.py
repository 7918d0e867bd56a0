"""The sparse MLP module's decode step as one call of the library gives what its ops give one by one, bit for bit."""
import pytest
import torch
from torch.nn.utils import prune

from dejavu_amd.modules import ParallelFusedMLPDejavu

pytestmark = pytest.mark.gpu


def _module(d, ffn, rank, K, bias=True, activation="relu", n_out=None):
    torch.manual_seed(d + ffn)
    m = ParallelFusedMLPDejavu(d, ffn, {"embed_dim": d, "low_rank_dim": rank, "out_dim": ffn, "K": K}, out_features=n_out,
                               activation=activation, bias1=bias, bias2=bias, layer_idx=0, sequence_parallel=False, device="cuda",
                               dtype=torch.float16)
    with torch.no_grad():
        for p in m.parameters():
            p.normal_(0.0, 0.05)
    return m


def _ops(monkeypatch, m, *args):
    with monkeypatch.context() as c:
        c.setattr(ParallelFusedMLPDejavu, "_one_call", lambda *a: None)
        return m(*args)


@pytest.mark.parametrize("d,ffn,rank,K,n_out", [(8, 16, 8, 1, None), (768, 3072, 128, 1024, None), (1024, 2056, 1024, 65, 264),
                                                (1032, 4104, 1032, 129, None), (4096, 8192, 1000, 4097, 520)])
@pytest.mark.parametrize("batch", [1, 2, 3, 9, 33])
@torch.no_grad()
def test_one_call_equals_ops(monkeypatch, d, ffn, rank, K, n_out, batch):
    for bias, activation, dtype in ((True, "relu", torch.int64), (False, "gelu_approx", torch.int32)):
        m = _module(d, ffn, rank, K, bias, activation, n_out)
        x, residual = (torch.randn(batch, 1, d, device="cuda").half() for _ in range(2))
        idx = torch.randperm(ffn, device="cuda")[:K].sort().values.to(dtype)
        idx[-1] = ffn  # out of range: a row of zeros
        assert m._one_call(x, residual, idx) is not None
        got, want = m(x, residual, idx), _ops(monkeypatch, m, x, residual, idx)
        assert got[0].shape == want[0].shape and got[1].shape == want[1].shape
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@torch.no_grad()
def test_other_forms_stay_with_the_ops(monkeypatch):
    m = _module(256, 1024, 64, 128)
    x, residual = (torch.randn(2, 1, 256, device="cuda").half() for _ in range(2))
    idx = torch.arange(128, device="cuda")
    want = m(x, residual, idx)
    calls = []
    hook = m.sp.register_forward_hook(lambda *a: calls.append(1))
    got = m(x, residual, idx)
    hook.remove()
    assert calls and all(torch.equal(a, b) for a, b in zip(got, want))
    wide = torch.zeros(2, 1, 512, device="cuda").half()
    wide[..., ::2] = x
    got = m(wide[..., ::2], residual, idx)
    assert torch.equal(got[0], want[0])
    m.sp.logits_out = torch.empty(2, 1024, device="cuda", dtype=torch.float16)
    assert m(x, residual, idx)[1].data_ptr() == m.sp.logits_out.data_ptr() and torch.equal(m.sp.logits_out, want[1])
    with pytest.raises(AssertionError):
        m(x.float(), residual, idx)
    with pytest.raises(AssertionError):
        m(x[..., :128].contiguous(), residual, idx)


@torch.no_grad()
def test_replayed_from_a_graph():
    m = _module(512, 2048, 128, 300)
    x, residual = (torch.randn(1, 1, 512, device="cuda").half() for _ in range(2))
    idx = torch.arange(300, device="cuda") * 5
    m(x, residual, idx)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = m(x, residual, idx)
    for _ in range(3):
        x.normal_()
        residual.normal_()
        graph.replay()
        want = m(x, residual, idx)
        assert torch.equal(out[0], want[0]) and torch.equal(out[1], want[1])


@pytest.mark.parametrize("name", ["fc1", "fc2"])
@pytest.mark.parametrize("parameter", ["bias", "weight"])
@torch.no_grad()
def test_pruned_layers(monkeypatch, name, parameter):
    """Pruning leaves the values in use as a plain attribute of the layer, not as its parameter."""
    m = _module(256, 1024, 64, 128)
    x, residual = (torch.randn(1, 1, 256, device="cuda").half() for _ in range(2))
    idx = torch.arange(128, device="cuda")
    whole = m(x, residual, idx)[0]
    prune.random_unstructured(getattr(m, name), parameter, 0.5)
    got = m(x, residual, idx)[0]
    assert torch.equal(got, _ops(monkeypatch, m, x, residual, idx)[0]) and not torch.equal(got, whole)


@pytest.mark.parametrize("batch,K,one", [(1, 512, True), (2, 512, True), (2, 513, False), (32, 32, True), (33, 32, False)])
@torch.no_grad()
def test_long_steps_use_the_side_stream(monkeypatch, batch, K, one):
    """Both sides of the line, laid where small sizes reach it; one sequence has no side stream."""
    m = _module(256, 1024, 64, 128)
    x, residual = (torch.randn(batch, 1, 256, device="cuda").half() for _ in range(2))
    idx = torch.arange(K, device="cuda")
    monkeypatch.setattr("dejavu_amd.modules.ONE_CALL_PRODUCTS", 2 * 2 * 256 * 512 if batch <= 2 else 2 * 32 * 256 * 32)
    calls, call = [], ParallelFusedMLPDejavu._one_call
    monkeypatch.setattr(ParallelFusedMLPDejavu, "_one_call", lambda *a: [calls.append(1), call(*a)][1])
    got = m(x, residual, idx)
    assert bool(calls) == one
    monkeypatch.undo()
    assert all(torch.equal(a, b) for a, b in zip(got, _ops(monkeypatch, m, x, residual, idx)))


def test_the_line_by_its_sizes():
    """9216 wide with 32 / 64 sequences, 12288 wide with 32 / 64, the same with four times the neurons and 8 / 16."""
    from dejavu_amd import modules

    sizes = ((9216, 4096, 32, 64), (12288, 4096, 32, 64), (12288, 16384, 8, 16))
    for d, K, below, above in sizes:
        assert 2 * d * K * below <= modules.ONE_CALL_PRODUCTS < 2 * d * K * above
