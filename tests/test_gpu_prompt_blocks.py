"""Prompts through a model's blocks and what callers make of them: own loops, wrappers, subclasses and mixers get tensors, and the same values."""
import pytest
import torch
import torch.nn as nn

from dejavu_amd import block as dv_block
from dejavu_amd import modules
from dejavu_amd.gpt import GPTLMHeadModel, SparseGPTConfig

IDS = 100


def _model(att_sparse=True):
    conf = SparseGPTConfig(hidden_size=1024, num_attention_heads=8, num_hidden_layers=3, vocab_size=512, n_inner=4096, max_position_embeddings=128,
                           mlp_K=512, mlp_sp_dim=128, att_sparse=att_sparse, att_K=[4, 4], att_sp_dim=128, pad_vocab_size_multiple=8)
    torch.manual_seed(0)
    return GPTLMHeadModel(conf, device="cuda", dtype=torch.float16).eval()


def _state():
    return modules.InferenceParams(max_sequence_len=128, max_batch_size=1)


@torch.no_grad()
def _logits(model):
    return model(torch.arange(IDS, device="cuda")[None], inference_params=_state()).logits


@pytest.mark.gpu
@torch.no_grad()
def test_own_loop_over_a_models_blocks():
    model = _model()
    want, body = _logits(model), model.transformer
    h, residual = body.embeddings(torch.arange(IDS, device="cuda")[None]), None
    for layer in body.layers:
        h, residual, *_ = layer(h, residual, mixer_kwargs={"inference_params": _state()})
        assert isinstance(h, torch.Tensor)
        h = h * 1.0
    h = body.ln_f(residual + h)
    # LayerNorm in this package's kernel and in the library: one step of fp16 in its results, through a product of 1024 of them
    assert float((model.lm_head(h).float() - want.float()).norm()) <= 2.0 ** -9 * float(want.float().norm())


class _Wrapped(nn.Module):
    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, *args, **kwargs):
        h, *rest = self.inner(*args, **kwargs)
        return (h * 1.0, *rest)


class _Block(dv_block.BlockMlpAttSparse):
    def forward(self, hidden_states, residual=None, mixer_subset=None, mixer_kwargs=None, head_idx=None, mlp_sp_logit=None):
        h, *rest = super().forward(hidden_states * 1.0, residual, mixer_subset, mixer_kwargs, head_idx, mlp_sp_logit)
        return (h * 1.0, *rest)


class _Mlp(modules.ParallelFusedMLPDejavu):
    def forward(self, *args, **kwargs):
        out, logit = super().forward(*args, **kwargs)
        return out * 1.0, logit


@pytest.mark.gpu
@pytest.mark.parametrize("place", [0, 1, 2])
@pytest.mark.parametrize("what", ["wrapper", "block", "mlp"])
def test_what_is_not_plain_gets_tensors(what, place):
    model = _model()
    want, layers = _logits(model), model.transformer.layers
    if what == "wrapper":
        layers[place] = _Wrapped(layers[place])
    elif what == "block":
        layers[place].__class__ = _Block
    else:
        layers[place].mlp.__class__ = _Mlp
    assert torch.equal(_logits(model), want)


class _Attention(modules.ParallelMHADejavu):
    def forward(self, *args, **kwargs):
        out, idx = super().forward(*args, **kwargs)
        return out * 1.0, idx


class _SparseAttention(modules.ParallelMHASparseAttMlp):
    def forward(self, *args, **kwargs):
        out, *rest = super().forward(*args, **kwargs)
        return (out * 1.0, *rest)


@pytest.mark.gpu
@pytest.mark.parametrize("att_sparse", [True, False])
def test_mixers_of_a_callers_own_get_to_see_the_projection(att_sparse):
    model = _model(att_sparse)
    want = _logits(model)
    model.transformer.layers[1].mixer.__class__ = _SparseAttention if att_sparse else _Attention
    assert torch.equal(_logits(model), want)


@pytest.mark.parametrize("tokens", [1, 5])
def test_a_mixer_takes_the_arguments_that_it_always_took(tokens):
    class Mixer(nn.Module):
        def forward(self, x, mlp_sp_logit=None, defer_join=False, inference_params=None):
            return x * 2, None

        def join_side(self):
            pass

    class Mlp(nn.Module):
        def forward(self, x, residual, idx=None, defer_join=False):
            return x + residual, None

    block = dv_block.BlockDejavu(8, lambda d: Mixer(), lambda d: Mlp())
    h, residual, logit = block(torch.ones(1, tokens, 8), mixer_kwargs={"inference_params": None})
    assert h.shape == residual.shape == (1, tokens, 8) and logit is None
