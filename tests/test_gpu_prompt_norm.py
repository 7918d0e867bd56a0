"""Products of a prompt whose last step rides in the add + LayerNorm that follows, against fp32 and against the launches one by one."""
import pytest
import torch

from dejavu_amd import modules, ops
from dejavu_amd.block import create_sparse_block

pytestmark = pytest.mark.gpu


def _operands(rows, M, K, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(1, rows, K, device="cuda", generator=g).half()
    W = (torch.randn(M, K, device="cuda", generator=g) * K ** -0.5).half()
    b, gamma, beta = (torch.randn(M, device="cuda", generator=g).half() for _ in range(3))
    return x, W, b, gamma, beta, torch.randn(1, rows, M, device="cuda", generator=g).half()


# rows at the edges of the row tiles, weight rows that end inside a tile, columns that end inside a chunk; the last two: wide parts
@pytest.mark.parametrize("rows,M,K,wide", [
    (2, 1024, 4096, False), (17, 1032, 2048, False), (33, 4096, 11008, False), (64, 5120, 5120, False), (65, 4104, 4096, False),
    (128, 5120, 20480, False), (129, 1032, 4104, False), (192, 5120, 5120, False), (256, 4096, 16384, False), (384, 4096, 16384, False),
    (257, 4096, 16384, True), (777, 4104, 16392, True)])
def test_pending_product_and_norm(rows, M, K, wide):
    x, W, b, gamma, beta, res = _operands(rows, M, K, rows)
    pending = ops.dense_linear_pending(x, W, b, wide=wide)
    assert pending is not None and pending.shape == (1, rows, M) and pending.groups > 1
    y, r = ops.add_layer_norm(pending, res, gamma, beta, 1e-5)
    h = (x.float().double() @ W.double().t() + b.double()).half().double()
    r_ref = (h + res.double())
    # one step of fp16 in h and one in the sum: values up to 8
    assert y.shape == r.shape == res.shape and (r.double() - r_ref).abs().max() <= 2 * 2 ** -8
    y_ref = torch.nn.functional.layer_norm(r.float(), (M,), gamma.float(), beta.float(), 1e-5)
    assert (y.float() - y_ref).abs().max() <= 2 ** -10 * (1 + y_ref.abs().max())
    alone = pending.materialize()
    assert torch.equal(alone + res, r)
    if not wide:
        assert torch.equal(alone, ops.dense_linear(x, W, b))
    else:
        assert torch.equal(alone, ops.dense_linear_wide_parts(x, W, b))
    assert all(torch.equal(p, q) for p, q in zip(ops.add_layer_norm(alone, res, gamma, beta, 1e-5), (y, r)))


def test_no_parts_no_pending():
    x, W, b, *_ = _operands(128, 32768, 512, 1)
    assert ops.dense_linear_pending(x, W, b) is None  # one split
    assert ops.dense_linear_pending(x[:, ::2], W, b) is None  # rows apart
    x, W, b, *_ = _operands(100, 1028, 4096, 1)
    assert ops.dense_linear_pending(x, W, b) is None  # M % 8


@pytest.mark.parametrize("s,att_sparse", [(2, True), (100, True), (100, False), (300, True)])
def test_block_prompt_with_and_without_the_fold(s, att_sparse, monkeypatch):
    d, ffn, H = 1024, 10240, 8
    block = create_sparse_block(d, ffn, H, 128, 1024, 128, 4, layer_idx=0, device="cuda", att_sparse=att_sparse).eval()
    with torch.no_grad():
        g = torch.Generator(device="cuda").manual_seed(3)
        for p in block.parameters():
            p.copy_(torch.randn(p.shape, device="cuda", generator=g) * (0.02 if p.dim() == 2 else 0.1))
    x = torch.randn(1, s, d, device="cuda", generator=g).half()
    out = []
    for fold in (True, False):
        monkeypatch.setattr("dejavu_amd.block.FOLD_NORM2", fold)
        ip = modules.InferenceParams(max_sequence_len=s + 16, max_batch_size=1)
        with torch.no_grad():
            hidden, residual = block(x, x, mixer_kwargs={"inference_params": ip})[:2]
        assert isinstance(hidden, torch.Tensor)  # nobody said that the next step is an add + LayerNorm
        out.append((hidden.float(), residual.float()))
    for a, b in zip(*out):
        assert torch.equal(a, b)  # the splits' sums are added up in the same order


def test_hooked_blocks_get_tensors():
    from dejavu_amd.gpt import GPTLMHeadModel, SparseGPTConfig

    conf = SparseGPTConfig(hidden_size=1024, num_attention_heads=8, num_hidden_layers=3, vocab_size=512, n_inner=4096,
                           max_position_embeddings=128, mlp_K=512, mlp_sp_dim=128, att_K=[4, 4], att_sp_dim=128, pad_vocab_size_multiple=8)
    model = GPTLMHeadModel(conf, device="cuda", dtype=torch.float16).eval()
    ids = torch.arange(100, device="cuda")[None]
    seen = []

    def logits():
        with torch.no_grad():
            return model(ids, inference_params=modules.InferenceParams(max_sequence_len=128, max_batch_size=1), last_token_only=True).logits

    plain = logits()
    layers = model.transformer.layers
    handles = [layers[2].register_forward_pre_hook(lambda m, a: seen.append(a[0])), layers[0].register_forward_hook(lambda m, a, o: seen.append(o[0])),
               layers[1].mixer.register_forward_hook(lambda m, a, o: seen.append(o[0]))]
    hooked = logits()
    for h in handles:
        h.remove()
    assert len(seen) == 3 and all(isinstance(t, torch.Tensor) and t.shape == (1, 100, 1024) for t in seen)
    assert torch.equal(plain, hooked)


@pytest.mark.parametrize("rows,M,K", [(2, 1024, 4096), (128, 5120, 5120), (150, 16384, 4096), (150, 16384, 2560), (192, 20480, 5120), (193, 4096, 16384), (300, 4096, 16384), (777, 5120, 20480)])
@torch.no_grad()
def test_pending_linear_is_decode_linear(rows, M, K):
    """Which kernel takes a product, and so its bits, does not depend on what follows."""
    lin = torch.nn.Linear(K, M, device="cuda", dtype=torch.float16).requires_grad_(False)
    x = torch.randn(1, rows, K, device="cuda").half()
    pending = modules.pending_linear(lin, x)
    assert pending is not None and torch.equal(pending.materialize(), modules.decode_linear(lin, x))
