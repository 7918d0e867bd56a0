"""Drop-in sparse MLP / sparse attention modules.

Same constructor arguments, submodule names (``fc1``, ``fc2``, ``Wqkv``,
``out_proj``, ``sp.fc0``, ``sp.fc1``) and ``forward`` signatures as the
reference's modules, with the decode step running on the HIP kernels:

  ParallelSP                Dejavu/src/ops/fused_dense_sparse_dejavu.py:33-76
  ParallelFusedMLPDejavu    Dejavu/src/ops/fused_dense_sparse_dejavu.py:821-951
  ParallelMHADejavu         Dejavu/src/models/modules/mha_dejavu.py:910-1075
  ParallelMHASparseAttMlp   Dejavu/src/models/modules/mha_dejavu.py:1152-1511

Single GPU: a process group of size 1 (or None) is accepted and the tensor
parallel all-reduces of the reference are the identity.  The prompt phase
(sequence length > 1) and layers that receive no prediction run dense through
the library GEMM / attention of PyTorch, as the reference's do through cuBLAS.
"""
from __future__ import annotations

from functools import lru_cache
from typing import Optional

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import ops
from ._binding import results_only
from ._lib import check, lib
from .inference import InferenceParams  # noqa: F401  (part of this module's interface)


# Side-stream overlap of predictor / top-k work with the main kernels (the reference's
# sp_stream).  Off = everything is enqueued on the current stream in program order.  Off by
# default: on one GPU there is no all-reduce to hide the predictors behind, the kernels are
# bandwidth-bound either way, and a fork / join inside a captured decode step slows the whole
# graph down (greedy decode of the 40-layer OPT-13B shape, only the dense first block on the
# module path: 322 tokens/s with the side stream, 357 without; eager 792 -> 765 ms).
USE_SIDE_STREAM = False
# From this many sequences on the side stream is used regardless: a batched layer step goes module by
# module, its predictors and top-ks are a dozen short launches beside kernels of 50-170 us, and
# overlapping them pays (OPT-175B shape: 279.9 -> 255.3 us/layer at batch 8, 425.1 -> 385.0 us at
# batch 32).  None: never.  (The sparse MLP called by itself, without a graph, first up to ``ONE_CALL_PRODUCTS``: the host is what it waits for.)
SIDE_STREAM_MIN_BATCH = 2
# A decode step of the sparse MLP alone is one call of the library, with everything on the current stream, up to so many products of the neurons' two
# rows; beyond, where a side stream is used, the kernels are longer than the host's part and the predictor runs beside them.  us a step among others / waited for, op by
# op with the side stream and in one call: 16 / 32 / 64 sequences, 4096 wide and 4096 neurons 76.7, 44.5 / 93.5, 68.6, 94.4, 52.8 / 105.8, 78.5, 104, 83 / 126, 110; 7168
# wide 64 sequences (3.8e9 products) 114, 104 / 134, 130; 9216 wide 32 (2.4e9) 95, 80 / 117, 106, 64 (4.8e9) 115, 122 / 146, 147; 12288 wide 8 / 32 (3.2e9) / 64 (6.4e9) 97.7, 92.6 /
# 117.1, 116.9, 103, 95 / 127, 121, 134, 140 / 162, 166; 12288 wide and 16384 neurons 8 (3.2e9) / 16 (6.4e9) / 32 / 64 206, 202 / 238, 228, 206, 204 / 227, 230, 196, 205 / 224, 231, 222, 241 / 250, 268.
ONE_CALL_PRODUCTS = 1 << 32

# Prompt phase on this package's own kernels (dense products: dv_dense_linear_f16; causal attention
# + cache fill: dv_prefill_attention_f16).  False: PyTorch's library GEMM and attention.
USE_HIP_PROMPT = True
# The dense products of a prompt are plain GEMMs.  Up to this many rows of X the package's kernel is at least as fast as
# the library (it is bound by the weight stream: 5120 x 5120 with 128 / 190 rows 22 / 26 against 32 / 29 us, 15360 x 5120
# with 190 rows 53 against 51 and a launch for the activation); beyond it the product is compute-bound and the library's
# GEMM is taken.
HIP_PROMPT_MAX_ROWS = 192
# But where the weight's rows are four times as long as they are many (fc2), the library leaves much of the chip idle for some
# hundred rows more: up to 256 from 2^23 elements on (us, this kernel against the library, 256 rows: 1024 x 8192 20.8 / 21.0, 2048 x
# 8192 24 / 28, 5120 x 20480 79 / 225, 12288 x 49152 396 / 478; but 768 x 3072 12.7 / 9.2, 4096 x 5120 31 / 29), up to 384 from 4096
# weight rows on (300 rows: 4096 x 16384 70 / 88, 5120 x 20480 103 / 129, 9216 x 36864 301 / 375; but 3072 x 12288 62 / 57) and up to
# 512 to 8192 of them (4096 x 16384 86 / 108, 8192 x 32768 292 / 347; but 9216 x 36864 506 / 403).
HIP_PROMPT_LONG_MAX_ROWS = 512
HIP_PROMPT_LONG_ROWS = 256, 384
HIP_PROMPT_LONG_WEIGHT = 1 << 23
HIP_PROMPT_LONG_WEIGHT_ROWS = 4096, 8192
# From 257 rows on the kernel of wide tiles (gemm_wide.hpp) takes fc1 with its activation, for which the library needs a launch more, where its tiles
# of 128 rows by 256 weight rows are so many (below 3072 columns / from there on) and the columns up to 5120, up to 8192 rows.  The library's time over
# the kernel's, weights cold, 385 to 2048 rows: 8192 x 2048 1.04 to 1.34, 10240 x 2560 1.05 to 1.66, 12288 x 3072 (641 rows and more) 1.04 to 1.28, 16384 x 4096
# 1.00 to 1.25, 18432 x 4608 0.98 to 1.20, 20480 x 5120 0.98 to 1.45, 16384 x 5120 0.96 to 1.20; beyond 2048 rows the first, fourth and sixth 0.99 to 1.45.  Left to the
# library: 22528 x 5632 0.94 to 1.46, 24576 x 6144 0.83 to 1.12, 28672 x 7168 0.93 to 1.15, 36864 x 9216 0.85 to 1.14, 12288 x 3072 with 257 to 512 rows 0.94 to 1.00 (513 to 640 1.01 to 1.11).
# And fc2 whose rows are the longest but for those that go on from 21504 columns, of more than 768 rows and where the tiles are so many: 5120 x 20480 0.98 to
# 1.79, 4096 x 20480 1.03 to 1.52.  Of longer rows the library has its good choices at other sizes for each weight: 5376 x 21504 0.88 to 1.76, 6144 x 24576 0.92 to 1.61, 7168 x
# 28672 0.89 to 1.61, 9216 x 36864 0.92 to 1.61; of shorter ones mostly: 4608 x 18432 0.77 to 1.75, 4096 x 16384 0.73 to 2.01; 768 rows and fewer 0.56 to 0.87.
HIP_PROMPT_WIDE_ROWS = 257, 2048
HIP_PROMPT_WIDE_LONGEST = 8192, 5120   # rows, columns (with an activation)
HIP_PROMPT_WIDE_COLUMNS, HIP_PROMPT_WIDE_FILL = (2048, 3072), (128, 256)
HIP_PROMPT_WIDE_LONG = 769, (20480, 21504), 136  # rows, columns (from, to), tiles
HIP_PROMPT_WIDE_STRIDE = 1 << 25
# Long rows whose tiles leave much of the chip idle: the columns in parts, the sums added up by a second launch (plan_wide_split).  What took them before (the
# library, from 769 rows on by 20480 columns the wide tiles) over this, weights cold, 257 to 2048 rows: 2560 x 10240 1.06 to 1.30, 3072 x 12288 0.99 to 1.34,
# 4096 x 16384 1.00 to 2.09, 4608 x 18432 1.05 to 1.92, 5120 x 20480 1.14 to 1.72, 5632 x 22528 1.32 to 1.61, 7168 x 28672 1.38 to 1.62, 9216 x 36864 1.38
# to 1.39 (777 by 4096 x 16384 146 -> 103 us).  Of more weight rows only in three parts and more: in two 8192 x 28672 0.89 to 1.01, 12288 x 49152 0.90 to 1.00.
# Fewer rows where one column of such tiles makes three parts (15361 to 20480 weight rows on 256 compute units).  The streaming kernel over these, alone, 129 / 160 / 192
# rows: above 16384 weight rows (17408 to 20480), where the streaming kernel's tiles leave some of its round empty, 2560 columns 1.06 to 1.09 / 1.00 to 1.12 / 0.99 to 1.03, 2816 to 3584
# 1.09 to 1.18 / 1.04 to 1.12 / 1.00 to 1.08, 4096 1.15 to 1.20 / 1.11 to 1.15 / 1.07 to 1.10, 4608 and 5120 1.03 to 1.08 / 1.01 to 1.05 / 0.98 to 1.03, 5632 to 8192 1.10 to 1.23 / 1.06 to 1.19 / 1.01 to
# 1.13, 10240 and 12288 1.05 to 1.07 / 1.02 to 1.05 / 0.97 to 1.04, but 6144 0.94 to 0.98 / 0.93 to 0.95 / 0.89 to 0.93; of 16384 and fewer, which it has in a round, those whose rows lie a power of
# two apart: 4096 1.09 to 1.15 / 1.09 to 1.14 / 1.02 to 1.09, 8192 1.19 / 1.15 to 1.17 / 1.13 to 1.15, but 2560 to 3584 0.93 to 1.03 / 0.88 to 1.01 / 0.88 to 0.97, 4608 to 12288 0.84 to 1.03 / 0.82 to 1.00 /
# 0.80 to 0.97.  16384 x 2048 0.91 to 1.01, in two parts 24576 x 6144 0.94 to 1.00, in four and five 14336 / 12288 x 4096 0.93 to 1.10.  The line in rows is by whole prompts of eight blocks
# (us, streaming kernel or library / these), 6.7B shape 128 / 150 / 192 / 224 tokens 1309 / 1306, 1534 / 1504, 1586 / 1567, 1683 / 1695, 13B shape 1720 / 1775, 1993 /
# 1967, 2064 / 2048, 2351 / 2366: fewer rows are as fast alone, but not beside the launches around them.
HIP_PROMPT_FEW_PARTS, HIP_PROMPT_FEW_COLUMNS, HIP_PROMPT_FEW_ROWS = 3, (2560, 12288), (129, 192)
HIP_PROMPT_FEW_WEIGHT_ROWS, HIP_PROMPT_FEW_BUT = 16384, 6144   # weight rows above which any columns but these
HIP_PROMPT_PARTS_COLUMNS, HIP_PROMPT_PARTS_WEIGHT = 10240, 26_000_000
HIP_PROMPT_PARTS_TALL = 7168, 3
# The package's causal-attention kernel (cache fill in the same launch) is ahead of the library's attention with the
# permuted cache copies (40 heads of 128 and 128 / 1024 tokens: 7.5 / 47 us against 25 / 100; 32 heads and
# 777 / 2000 / 4000 tokens: 30 / 110 / 385 against 75 / 310 / 566; 16 sequences of 1024: 547 against 768).  Prompts of more than so
# many tokens leave gradients, functional transforms and the like to the library.
HIP_PROMPT_ATTN_MAX_TOKENS = 192
# Each workgroup reads the keys and values before its 32 queries, so the L2 bounds long prompts and the library, whose tiles
# were larger, overtook: with 40 heads of 128 from 8192 tokens on (1759 against 1691 us; 6000 tokens 961 against 1155, 16 sequences of
# 4096 and 32 heads 5875 against 6316), with 96 heads above 2048 (four sequences of 2048 1329 against 1404, of 4096 5184 against 4784).  (Its tiles of
# 128 queries, prefill.hpp, which take prompts of a thousand tokens and more since, are ahead beyond these lines alone: 40 heads and 8192 tokens 1051 against
# 1738, 96 heads and 4096 690 against 1305.  The lines are the older kernel's still: whole prompts of such lengths have not been measured on both sides.)
HIP_PROMPT_ATTN_LONGEST = 6144
HIP_PROMPT_ATTN_WIDE = 5120            # heads * head_dim above which it is
HIP_PROMPT_ATTN_WIDE_LONGEST = 2048

_side_streams: dict = {}
_side_pending = False  # work was enqueued on the side stream since the last join_side_stream()


def side_stream_enabled(batch: int = 1) -> bool:
    return bool(USE_SIDE_STREAM) or (SIDE_STREAM_MIN_BATCH is not None and batch >= SIDE_STREAM_MIN_BATCH)


def side_stream(device=None) -> "torch.cuda.Stream":
    """The one side stream (default priority) that all modules on a device share: predictors
    and top-ks are enqueued on it in program order, so work handed from one module to the
    next on that stream needs no event."""
    dev = torch.cuda.current_device() if device is None else torch.device(device).index
    if dev is None:
        dev = torch.cuda.current_device()
    st = _side_streams.get(dev)
    if st is None:
        st = torch.cuda.Stream(device=dev)
        _side_streams[dev] = st
    return st


_heads_event = None  # head selection of the last block that left it pending on a side stream


def mark_side_pending(heads_event=None) -> None:
    """Work was left on the side stream (and this event covers the head selection among it)."""
    global _side_pending, _heads_event
    _side_pending = True
    if heads_event is not None:
        _heads_event = heads_event


def join_heads() -> None:
    """Makes the current stream wait for the head selection a block left pending on a side stream."""
    global _heads_event
    if _heads_event is not None:
        torch.cuda.current_stream().wait_event(_heads_event)
        _heads_event = None


def join_side_stream() -> None:
    """Makes the current stream wait for everything enqueued on the side stream so far
    (e.g. before a graph capture that used the side stream ends)."""
    global _side_pending, _heads_event
    if _side_pending and _side_streams:
        _side_pending = False
        _heads_event = None
        ev = torch.cuda.Event(enable_timing=False, blocking=False)
        st = side_stream()
        st.record_event(ev)
        torch.cuda.current_stream().wait_event(ev)


def _transposed_copy(module, attr: str, weight: torch.Tensor) -> torch.Tensor:
    """``weight.t().contiguous()`` kept in ``module.<attr>`` and rebuilt when the weight has been
    written since (load_state_dict, an in-place update) or replaced.  A tensor the caller put
    there itself is taken as matching the weight at that moment."""
    stamp = (weight.data_ptr(), weight._version, tuple(weight.shape))
    cur = getattr(module, attr)
    if cur is None or (getattr(module, attr + "_stamp", None) not in (None, stamp)) or \
            cur.shape != (weight.shape[1], weight.shape[0]):
        cur = weight.t().contiguous()
        setattr(module, attr, cur)
    if getattr(module, attr + "_stamp", None) != stamp:
        setattr(module, attr + "_stamp", stamp)
    return cur


def _world_size(process_group) -> int:
    if process_group is None:
        return 1
    size = process_group.size() if callable(getattr(process_group, "size", None)) else int(process_group)
    if size != 1:
        raise NotImplementedError("this build runs the sparse decode path on one GPU (tensor parallel size 1)")
    return size


class ParallelSP(nn.Module):
    """Low-rank sparsity predictor ``fc1(fc0(x))``, both linears bias-free."""

    def __init__(self, layer_idx=None, embed_dim=None, low_rank_dim=None, out_dim=None, K=None,
                 process_group=None, sequence_parallel=False, device=None, dtype=None) -> None:
        super().__init__()
        size = _world_size(process_group)
        self.process_group = process_group
        self.layer_idx = layer_idx
        self.embed_dim = embed_dim
        self.fc0 = nn.Linear(embed_dim, low_rank_dim, bias=False, device=device, dtype=dtype)
        self.out = out_dim // size
        self.fc1 = nn.Linear(low_rank_dim, out_dim, bias=False, device=device, dtype=dtype)
        self.K = K // size
        # optional caller-owned result buffer (fixed addresses for graph capture)
        self.logits_out = None

    def forward(self, x):
        """x: anything viewable as (embed_dim,) -> (out_dim,) logits, as the
        reference; a (B, 1, embed_dim) batch gives (B, out_dim)."""
        single = x.numel() == self.embed_dim
        logits = ops.predictor_logits(x.reshape(-1, self.embed_dim), self.fc0.weight, self.fc1.weight,
                                      out=self.logits_out)
        return logits.view(-1) if single else logits

    def topk(self, logits, k=None, dtype=torch.int64):
        return ops.topk_indices(logits, self.K if k is None else k, dtype=dtype)


class ParallelFusedMLPDejavu(nn.Module):
    def __init__(self, in_features, hidden_features, sp_kwargs, out_features=None, activation="gelu_approx",
                 layer_idx=None, process_group=None, bias1=True, bias2=True, sequence_parallel=True,
                 checkpoint_lvl=0, heuristic="auto", device=None, dtype=None):
        assert checkpoint_lvl in [0, 1, 2]
        assert activation in ["gelu_approx", "relu"]
        assert sp_kwargs != None, "sparse predictor parameters are not passed in."
        super().__init__()
        _world_size(process_group)
        if out_features is None:
            out_features = in_features
        self.activation = activation
        self.process_group = process_group
        self.sequence_parallel = sequence_parallel
        self.checkpoint_lvl = checkpoint_lvl
        self.heuristic = heuristic
        self.fc1 = nn.Linear(in_features, hidden_features, bias=bias1, device=device, dtype=dtype)
        self.fc2 = nn.Linear(hidden_features, out_features, bias=bias2, device=device, dtype=dtype)
        self.layer_idx = layer_idx
        # fc2.weight transposed to (hidden, out) so that active neurons are contiguous rows;
        # built on first sparse use, as the reference does
        self.fc2_weight_t = None
        self.sp = ParallelSP(layer_idx=layer_idx, device=device, dtype=dtype, process_group=process_group,
                             sequence_parallel=sequence_parallel, **sp_kwargs)
        self.sp_stream = None
        self.event_mlp = None
        self.event_mlp_sp = None

    def _streams(self):
        if self.sp_stream is None:
            self.sp_stream = side_stream(self.fc1.weight.device)
            self.event_mlp = torch.cuda.Event(enable_timing=False, blocking=False)
            self.event_mlp_sp = torch.cuda.Event(enable_timing=False, blocking=False)

    def transposed_fc2(self) -> torch.Tensor:
        """fc2.weight as (hidden, out), contiguous; follows updates of fc2.weight."""
        return _transposed_copy(self, "fc2_weight_t", self.fc2.weight)

    def _one_call(self, x, residual, idx):
        """``forward`` of a decode step with everything in its plain form in one call of the library; None where something is not
        (what then runs op by op converts it or says what is wrong).  The host's part of a step is what takes long: op by op, with the
        selection before it, 55 us at d = 768 and 60 at 4096 for one sequence, 80 to 110 for 2 to 32 (the events of the side stream);
        in one call 33, 38 and 44 to 71, whereof launches 8 to 20."""
        # (the dictionaries, not the attributes: nn.Module looks a name up in three places, half a microsecond each)
        fc1, fc2, sp = (self._modules.get(k) for k in ("fc1", "fc2", "sp"))
        if type(sp) is not ParallelSP or type(fc1) is not nn.Linear or type(fc2) is not nn.Linear or _hooked(sp):
            return None
        if "bias" not in fc1._parameters or "bias" not in fc2._parameters:  # a plain tensor, as pruning leaves it
            return None
        W1, b1, b2 = fc1._parameters.get("weight"), fc1._parameters.get("bias"), fc2._parameters.get("bias")
        Wa, Wb = (sp._modules[k]._parameters.get("weight") for k in ("fc0", "fc1"))
        for t in (x, residual, W1, Wa, Wb):
            if t is None or t.dtype != torch.float16 or not t.is_cuda or not t.is_contiguous():
                return None
        B, d = x.shape[0], x.shape[-1]
        if (W1.dim() != 2 or Wa.dim() != 2 or Wb.dim() != 2 or x.dim() != 3 or not 1 <= B <= 64 or idx.dim() != 1 or
                not idx.is_contiguous() or not idx.is_cuda or idx.dtype not in (torch.int64, torch.int32)):
            return None
        (ffn, d1), (r, d2), (n_logits, r2), K = W1.shape, Wa.shape, Wb.shape, idx.shape[0]
        W2t = self.transposed_fc2()
        n_out = W2t.shape[1]
        if (d1 != d or d2 != d or sp.embed_dim != d or r2 != r or n_logits != ffn or W2t.shape[0] != ffn or K < 1 or W2t.dtype != torch.float16 or
                not W2t.is_contiguous() or residual.numel() != B * d):
            return None
        for b, n in ((b1, ffn), (b2, n_out)):
            if b is not None and (b.dtype != torch.float16 or not b.is_cuda or b.shape != (n,) or not b.is_contiguous()):
                return None
        logits = sp.logits_out
        if logits is None:
            logits = torch.empty(B, ffn, dtype=torch.float16, device=x.device)
        elif logits.numel() != B * ffn or logits.dtype != torch.float16 or not logits.is_contiguous():
            return None
        out = torch.empty(B, 1, n_out, dtype=torch.float16, device=x.device)
        nbytes = _one_call_bytes(torch._C._cuda_getDevice(), B, d, n_out, ffn, K, r)
        ws = ops._workspace(x.device, nbytes)
        if lib.dv_sparse_mlp_f16(x.data_ptr(), residual.data_ptr(), W1.data_ptr(), d, None if b1 is None else b1.data_ptr(), W2t.data_ptr(),
                                 n_out, None if b2 is None else b2.data_ptr(), idx.data_ptr(), 8 if idx.dtype == torch.int64 else 4, B, d,
                                 n_out, ffn, K, ops._ACT[self.activation], Wa.data_ptr(), d, Wb.data_ptr(), r, r, out.data_ptr(),
                                 logits.data_ptr(), ws.data_ptr(), ws.numel(), ops._stream()):
            return None
        return out, logits.view(-1) if B == 1 else logits.view(B, ffn)

    def forward(self, x, residual, idx=None, defer_join=False, defer_reduce=False):
        """x, residual: (B, 1, d) at decode (or (B, s, d) for the prompt).
        idx: (K,) active neurons or None for the dense MLP.
        defer_reduce: the caller's next step is an ``ops.add_layer_norm`` / ``add_layer_norm_window`` of
        ``out``; for 3..64 sequences, and for prompts whose fc2 ends in such a step, ``out`` is then ``ops.PendingRows`` (the
        split reduction of fc2 runs inside that LayerNorm launch).
        Returns (out, mlp_logit); mlp_logit, the predictor output for the next
        layer's MLP, only when decoding one token.  defer_join: when the predictor runs on the side
        stream, the current stream does not wait for it: mlp_logit is then only good for work
        enqueued on the side stream (the next layer's top-k is) or after ``join_side_stream()``."""
        do_token_generation = x.size(1) == 1
        # The predictor only needs `residual`, so it streams its weights on the side
        # stream while fc1 / fc2 run (the reference starts it after the MLP, to
        # overlap the tensor-parallel all-reduce that one GPU does not have).
        # The side work is ENQUEUED AFTER the main work of the phase (it still starts from the event
        # recorded here).  In a captured graph the first-captured successor of a node stays on its
        # hardware queue and the others move to another one; a hand-over between queues costs about
        # 10 us when the consumer is waiting for it, so the chain that is waited for -- fc1, fc2 --
        # must be the one captured first (batch 8, OPT-175B shape: four such hand-overs per layer step).
        mlp_logit = None
        side = do_token_generation and side_stream_enabled(x.shape[0])
        # (from a graph the products and the predictor of several sequences side by side, as below: there the host takes no part)
        if idx is not None and do_token_generation and not (defer_reduce or USE_SIDE_STREAM or (side and (
                defer_join or 2 * x.numel() * idx.numel() > ONE_CALL_PRODUCTS or torch.cuda.is_current_stream_capturing()))):
            done = self._one_call(x, residual, idx)
            if done is not None:
                return done
        if side:
            self._streams()
            curr_stream = torch.cuda.current_stream()
            curr_stream.record_event(self.event_mlp)
        if idx is not None:
            assert x.size(1) == 1
            h = ops.gather_gemv(x.squeeze(1), self.fc1.weight, idx, self.fc1.bias, activation=self.activation)
        else:
            h = decode_linear(self.fc1, x, self.activation)
        if side:  # behind fc1: the main chain's first launch of the phase is captured, the rest follows
            global _side_pending
            _side_pending = True
            with torch.cuda.stream(self.sp_stream):
                self.sp_stream.wait_event(self.event_mlp)
                mlp_logit = self.sp(residual)
                self.sp_stream.record_event(self.event_mlp_sp)
        if idx is not None:
            out = ops.gather_transposed_gemv(h, self.transposed_fc2(), idx, self.fc2.bias, defer_reduce=defer_reduce)
            if not isinstance(out, ops.PendingRows):
                out = out.unsqueeze(1)
        else:
            out = pending_linear(self.fc2, h) if defer_reduce else None
            if out is None:
                out = decode_linear(self.fc2, h)
        # (tensor parallel all-reduce of `out` is the identity on one GPU)
        if side:
            if defer_join:
                # The predictor may still be reading `residual` when the caller lets go of it: the
                # tensor stays referenced here until this module's next forward.  By then the current
                # stream has waited for side work that was enqueued behind this predictor (the top-k
                # that consumes mlp_logit), so its memory is not handed out again too early.
                self._side_keep = residual
            else:
                curr_stream.wait_event(self.event_mlp_sp)
        elif do_token_generation:
            mlp_logit = self.sp(residual)
        return out, mlp_logit


def _hooked(module) -> bool:
    return bool("forward" in module.__dict__ or module._forward_hooks or module._forward_pre_hooks or
                nn.modules.module._global_forward_hooks or nn.modules.module._global_forward_pre_hooks)


@lru_cache(maxsize=4096)
def _one_call_bytes(device: int, B: int, d: int, n_out: int, ffn: int, K: int, r: int) -> int:
    """A function of the sizes and of the current device, whose compute units the splits are made for."""
    return lib.dv_sparse_mlp_workspace_bytes(B, d, n_out, ffn, K, r)


def _long_rule(rows: int, M: int, K: int) -> bool:
    if K < 4 * M or M * K < HIP_PROMPT_LONG_WEIGHT:
        return False
    (few, more), (low, high) = HIP_PROMPT_LONG_ROWS, HIP_PROMPT_LONG_WEIGHT_ROWS
    return rows <= few or (M >= low and (rows <= more or (rows <= HIP_PROMPT_LONG_MAX_ROWS and M <= high)))


def _wide_rule(rows: int, M: int, K: int, activation: str) -> bool:
    if activation not in ("id", "relu", "squared_relu"):
        return False
    tiles = -(-M // 256) * -(-rows // 128)
    if activation == "id":
        least, columns, fill = HIP_PROMPT_WIDE_LONG
        # (rows of results off 16-byte boundaries are stored value by value: 780 to 1200 rows by 5124 x 20496 0.84 to 0.89)
        return M % 8 == 0 and least <= rows <= HIP_PROMPT_WIDE_ROWS[1] and max(4 * M, columns[0]) <= K < columns[1] and tiles >= fill
    most, columns = HIP_PROMPT_WIDE_LONGEST
    few = K < HIP_PROMPT_WIDE_COLUMNS[1]
    return (HIP_PROMPT_WIDE_ROWS[0] <= rows <= most and HIP_PROMPT_WIDE_COLUMNS[0] <= K <= columns and
            tiles >= HIP_PROMPT_WIDE_FILL[0 if few else 1])


def _plain_layer(linear, x: torch.Tensor) -> bool:
    """Whether a kernel does what ``linear(x)`` would: a layer that is nothing but its weight and bias, operands that the kernel
    takes where they are, only results asked for."""
    W, b = linear.weight, linear.bias
    return (type(linear) is nn.Linear and W.dim() == 2 and x.shape[-1] == W.shape[1] and
            not _hooked(linear) and
            results_only(x, W, b) and W.stride(1) == 1 and W.stride(0) >= W.shape[1] and W.stride(0) % 8 == 0 and W.data_ptr() % 16 == 0 and
            x.data_ptr() % 16 == 0 and (b is None or (b.dtype == W.dtype and b.shape == W.shape[:1])))


def _long_product(linear, x: torch.Tensor) -> bool:
    """Whether ``dense_linear`` is the faster one for more than ``HIP_PROMPT_MAX_ROWS`` rows and does what ``linear(x)`` would."""
    W = linear.weight
    return W.dim() == 2 and _long_rule(x.numel() // x.shape[-1], *W.shape) and _plain_layer(linear, x)


def _wide_fits(linear, x: torch.Tensor) -> bool:
    W, b = linear.weight, linear.bias
    return x.is_contiguous() and W.stride(0) < HIP_PROMPT_WIDE_STRIDE and (b is None or b.is_contiguous()) and _plain_layer(linear, x)


def _wide_product(linear, x: torch.Tensor, activation: str) -> bool:
    """The same of ``dense_linear_wide``."""
    W = linear.weight
    return W.dim() == 2 and _wide_rule(x.numel() // x.shape[-1], *W.shape, activation) and _wide_fits(linear, x)


def _parts_rule(rows: int, M: int, K: int) -> bool:
    return (HIP_PROMPT_WIDE_ROWS[0] <= rows <= HIP_PROMPT_WIDE_ROWS[1] and K >= HIP_PROMPT_PARTS_COLUMNS and
            M * K >= HIP_PROMPT_PARTS_WEIGHT and M % 8 == 0)


def _long_parts(linear, x: torch.Tensor) -> bool:
    """Whether ``dense_linear_wide_parts`` is the faster one and does what ``linear(x)`` would."""
    W = linear.weight
    rows = x.numel() // x.shape[-1]
    # (the number of parts is asked for last: tracers, which only the library's product is for, do not get that far)
    if W.dim() != 2 or not _parts_rule(rows, *W.shape) or not _wide_fits(linear, x):
        return False
    M, K = W.shape
    many, least = HIP_PROMPT_PARTS_TALL
    return ops.wide_parts(rows, K, M) >= (least if M > many else 2)


def _few_rule(M: int, K: int) -> bool:
    least, most = HIP_PROMPT_FEW_COLUMNS
    return (least <= K <= most and M % 8 == 0 and
            (K & (K - 1) == 0 if M <= HIP_PROMPT_FEW_WEIGHT_ROWS else K != HIP_PROMPT_FEW_BUT))


def _few_parts_product(linear, x: torch.Tensor, activation: str) -> bool:
    """The same for a prompt of few rows, with an activation too."""
    W = linear.weight
    rows = x.numel() // x.shape[-1]
    if not HIP_PROMPT_FEW_ROWS[0] <= rows <= HIP_PROMPT_FEW_ROWS[1] or W.dim() != 2 or activation not in ("id", "relu", "squared_relu"):
        return False
    M, K = W.shape
    return _few_rule(M, K) and ops.wide_parts(rows, K, M) == HIP_PROMPT_FEW_PARTS and _wide_fits(linear, x)


def _parts_product(linear, x: torch.Tensor) -> Optional[torch.Tensor]:
    return ops.dense_linear_wide_parts(x, linear.weight, linear.bias) if _long_parts(linear, x) else None


def _prompt_on_hip(linear, x: torch.Tensor) -> bool:
    return (USE_HIP_PROMPT and x.is_cuda and x.dtype == torch.float16 and linear.weight.dtype == torch.float16 and x.shape[-1] % 8 == 0)


def pending_linear(linear: nn.Linear, x: torch.Tensor) -> Optional[ops.PendingRows]:
    """``decode_linear(linear, x)`` of a prompt with its last step left to the add + LayerNorm that follows, where there is such a step.
    One launch instead of two, and the rows are not written and read between them: prompts of eight blocks of the 6.7B shape with 70 / 128 /
    192 tokens 1222 / 1336 / 1604 -> 1165 / 1309 / 1586 us, of the 13B shape 1558 / 1774 / 2075 -> 1508 / 1720 / 2064."""
    if not _prompt_on_hip(linear, x) or x.shape[1] == 1:
        return None
    rows = x.numel() // x.shape[-1]
    if _few_parts_product(linear, x, "id"):  # (in decode_linear's order: the same kernels, the same sums)
        return ops.dense_linear_pending(x, linear.weight, linear.bias, wide=True)
    if rows <= HIP_PROMPT_MAX_ROWS or (rows <= HIP_PROMPT_LONG_MAX_ROWS and _long_product(linear, x)):
        return ops.dense_linear_pending(x, linear.weight, linear.bias)
    return ops.dense_linear_pending(x, linear.weight, linear.bias, wide=True) if _long_parts(linear, x) else None


def decode_linear(linear: nn.Linear, x: torch.Tensor, activation: str = "id") -> torch.Tensor:
    """``activation(linear(x))``.  The rows of a decode step (x: (B, 1, d) with B <= 64, fp16, on the GPU)
    always go to this package's row kernels (vector ALUs for one or two rows, matrix cores above).  The
    rows of a prompt go to the matrix-core kernels that stream the weight while it is the bound (``USE_HIP_PROMPT``, up
    to ``HIP_PROMPT_MAX_ROWS`` rows, and more of them for long-rowed weights: ``_long_product``), with an activation or long
    rows to the one with wide tiles (``_wide_product``, ``_parts_product``, ``_few_parts_product``), else to the library GEMM."""
    on_hip = x.is_cuda and x.dtype == torch.float16 and linear.weight.dtype == torch.float16 and x.shape[-1] % 8 == 0
    if on_hip and x.dim() == 3 and x.shape[1] == 1 and x.shape[0] <= 64:
        return ops.dense_decode_linear(x, linear.weight, linear.bias, activation)
    if on_hip and USE_HIP_PROMPT:
        rows = x.numel() // x.shape[-1]
        if _few_parts_product(linear, x, activation):
            return ops.dense_linear_wide_parts(x, linear.weight, linear.bias, activation)
        if rows <= HIP_PROMPT_MAX_ROWS or (rows <= HIP_PROMPT_LONG_MAX_ROWS and _long_product(linear, x)):
            return ops.dense_linear(x, linear.weight, linear.bias, activation)
        parts = _parts_product(linear, x) if activation == "id" else None
        if parts is not None:
            return parts
        if _wide_product(linear, x, activation):
            return ops.dense_linear_wide(x, linear.weight, linear.bias, activation)
    y = linear(x)
    if activation == "relu":
        return F.relu(y)
    if activation == "gelu_approx":
        return F.gelu(y, approximate="tanh")
    if activation == "gelu":
        return F.gelu(y)
    if activation == "squared_relu":
        return F.relu(y) ** 2
    return y


def _project_norm(linear: nn.Linear, x: torch.Tensor, post_norm):
    """``decode_linear(linear, x)``, or with post_norm = (LayerNorm module, residual) the pair (normed, residual_out) where the reduction
    of the projection rides in that launch."""
    pending = pending_linear(linear, x) if post_norm is not None else None
    if pending is None:
        return decode_linear(linear, x)
    norm, residual = post_norm
    return ops.add_layer_norm(pending, residual, norm.weight, norm.bias, norm.eps)


def _kv_caches(inference_params, layer_idx, H, hd, dtype, device):
    """The layer's (k_cache, v_cache), created on first use: packed keys (B, H, hd/8, S, 8) and values
    (B, H, S, hd) (Dejavu/src/models/modules/mha_dejavu.py:404-446, fused_ft_kernel layout)."""
    if layer_idx not in inference_params.key_value_memory_dict:
        k_cache = torch.zeros(inference_params.max_batch_size, H, hd // 8, inference_params.max_sequence_len, 8,
                              dtype=dtype, device=device)
        v_cache = torch.zeros(inference_params.max_batch_size, H, inference_params.max_sequence_len, hd,
                              dtype=dtype, device=device)
        inference_params.key_value_memory_dict[layer_idx] = (k_cache, v_cache)
    return inference_params.key_value_memory_dict[layer_idx]


def _update_kv_cache(kv, inference_params, layer_idx):
    """Prompt-phase cache fill.  kv: (B, s, 2, H, hd).  Creates / fills the
    packed key cache (B, H, hd/8, S, 8) and the value cache (B, H, S, hd)
    (Dejavu/src/models/modules/mha_dejavu.py:385-447, fused_ft_kernel layout)."""
    B, s, _, H, hd = kv.shape
    assert kv.dtype == torch.float16
    if layer_idx not in inference_params.key_value_memory_dict:
        k_cache = torch.zeros(inference_params.max_batch_size, H, hd // 8, inference_params.max_sequence_len, 8,
                              dtype=kv.dtype, device=kv.device)
        v_cache = torch.zeros(inference_params.max_batch_size, H, inference_params.max_sequence_len, hd,
                              dtype=kv.dtype, device=kv.device)
        inference_params.key_value_memory_dict[layer_idx] = (k_cache, v_cache)
    k_cache, v_cache = inference_params.key_value_memory_dict[layer_idx]
    b0 = inference_params.batch_size_offset
    s0 = inference_params.sequence_len_offset
    assert b0 + B <= v_cache.shape[0] and s0 + s <= v_cache.shape[2]
    k_cache[b0:b0 + B, :, :, s0:s0 + s, :] = kv[:, :, 0].reshape(B, s, H, hd // 8, 8).permute(0, 2, 3, 1, 4)
    v_cache[b0:b0 + B, :, s0:s0 + s, :] = kv[:, :, 1].permute(0, 2, 1, 3)
    return kv


def _longest_prompt(width: int) -> int:
    """The most tokens of a prompt whose attention, heads * head_dim wide, this package's kernel computes."""
    return HIP_PROMPT_ATTN_LONGEST if width <= HIP_PROMPT_ATTN_WIDE else HIP_PROMPT_ATTN_WIDE_LONGEST


def _kernel_takes(*tensors) -> bool:
    """Whether the prompt attention takes these where they are: the copies fill a caller's own caches of any type, stride and
    place, and the library's attention reads from anywhere."""
    return results_only(*tensors) and all(
        t is None or (t.dtype == torch.float16 and t.is_contiguous() and t.data_ptr() % 16 == 0) for t in tensors)


class _MHABase(nn.Module):
    """Shared dense / prompt machinery of the two attention modules."""

    def _init_common(self, embed_dim, num_heads, process_group, bias, softmax_scale, causal, layer_idx,
                     rotary_emb_dim, device, dtype):
        _world_size(process_group)
        ops.require_no_rotary(rotary_emb_dim)
        self.embed_dim = embed_dim
        self.causal = causal
        self.layer_idx = layer_idx
        self.rotary_emb_dim = rotary_emb_dim
        self.num_heads = num_heads
        assert self.embed_dim % num_heads == 0, "self.kdim must be divisible by num_heads"
        self.head_dim = self.embed_dim // num_heads
        self.softmax_scale = softmax_scale
        self.num_head_per_node = self.num_heads
        self.Wqkv = nn.Linear(embed_dim, 3 * embed_dim, bias=bias, device=device, dtype=dtype)
        self.out_proj = nn.Linear(embed_dim, embed_dim, device=device, dtype=dtype)
        self.process_group = process_group
        self.mlp_k = None
        self.sp_stream = None
        self._side_used = False
        self._forked = False
        self._side_keep = None
        self._mlp_idx_event = False
        self._joined = False

    def _streams(self):
        if self.sp_stream is None:
            self.sp_stream = side_stream(self.Wqkv.weight.device)
            self.event_in = torch.cuda.Event(enable_timing=False, blocking=False)
            self.event_side = torch.cuda.Event(enable_timing=False, blocking=False)
            self.event_mlp_idx = torch.cuda.Event(enable_timing=False, blocking=False)

    def _dense_context(self, qkv, inference_params):
        """qkv: (B, s, 3, H, hd) -> context (B, s, H*hd) for the prompt or a dense decode step."""
        B, s = qkv.shape[0], qkv.shape[1]
        scale = self.softmax_scale
        if inference_params is None or inference_params.sequence_len_offset == 0:
            causal = self.causal if inference_params is None else True
            if USE_HIP_PROMPT and qkv.is_cuda and qkv.dtype == torch.float16 and qkv.shape[-1] in (64, 128) \
                    and (causal or s == 1) and (s <= HIP_PROMPT_ATTN_MAX_TOKENS or (
                        s <= _longest_prompt(qkv.shape[3] * qkv.shape[4]) and results_only(qkv))):
                # causal attention and the cache fill in one launch (no permuted copy of K / V)
                kc = vc = None
                if inference_params is not None:
                    assert self.layer_idx is not None, "Generation requires layer_idx in the constructor"
                    k_cache, v_cache = _kv_caches(inference_params, self.layer_idx, self.num_heads, self.head_dim,
                                                  qkv.dtype, qkv.device)
                    b0 = inference_params.batch_size_offset
                    kc, vc = k_cache[b0:b0 + B], v_cache[b0:b0 + B]
                rows = qkv.contiguous()
                if s <= HIP_PROMPT_ATTN_MAX_TOKENS or (_kernel_takes(rows, kc, vc) and (kc is None or kc.shape[3] == vc.shape[2])):
                    return ops.prefill_attention(rows, kc, vc, 0, scale)
            if inference_params is not None:
                assert self.layer_idx is not None, "Generation requires layer_idx in the constructor"
                _update_kv_cache(qkv[:, :, 1:], inference_params, self.layer_idx)
            q, k, v = (t.transpose(1, 2) for t in qkv.unbind(dim=2))  # (B, H, s, hd)
            ctx = F.scaled_dot_product_attention(q, k, v, is_causal=causal and s > 1, scale=scale)
            return ctx.transpose(1, 2).reshape(B, s, -1)
        assert s == 1, "decode processes one token at a time"
        k_cache, v_cache = inference_params.key_value_memory_dict[self.layer_idx]
        b0 = inference_params.batch_size_offset
        q, k, v = qkv[:, 0].unbind(dim=1)  # (B, H, hd) views
        ctx = ops.single_query_attention(q, k, v, k_cache[b0:b0 + B], v_cache[b0:b0 + B],
                                         inference_params.lengths_per_sample, inference_params.sequence_len_offset,
                                         self.rotary_emb_dim, softmax_scale=scale)
        return ctx.reshape(B, 1, -1)

    def _side_fork(self, batch):
        """Marks, at the start of the forward, the point from which the side work may run."""
        self._forked = side_stream_enabled(batch)
        if self._forked:
            torch.cuda.current_stream().record_event(self.event_in)

    def _side_work(self, mlp_sp_logit, residual=None, att_sp=None, att_k=None, att_idx_out=None):
        """Everything that does not depend on this layer's attention runs on the
        side stream from the point ``_side_fork`` marked: the head predictor + top-k for
        the next layer (from the residual stream) and the MLP top-k for this layer
        (from the previous layer's logits).  The forward enqueues it AFTER its own launches
        (see ParallelFusedMLPDejavu.forward: the chain that is waited for must be captured first)
        and joins with ``_join_side`` before returning."""
        mlp_idx, att_idx = None, None
        self._side_used = False
        if mlp_sp_logit is None and att_sp is None:
            return mlp_idx, att_idx
        batch = residual.shape[0] if residual is not None else (mlp_sp_logit.shape[0] if mlp_sp_logit.dim() > 1 else 1)
        if not (side_stream_enabled(batch) and self._forked):
            if att_sp is not None:
                att_idx = ops.topk_indices(att_sp(residual), att_k, dtype=torch.int32, out=att_idx_out)
            if mlp_sp_logit is not None:
                mlp_idx = ops.topk_indices(mlp_sp_logit, self.mlp_k)
            return mlp_idx, att_idx
        self._side_used = True
        global _side_pending
        _side_pending = True
        with torch.cuda.stream(self.sp_stream):
            self.sp_stream.wait_event(self.event_in)
            # the neuron selection first: fc1 of this layer waits for it, the head selection is for
            # the next layer
            if mlp_sp_logit is not None:
                mlp_idx = ops.topk_indices(mlp_sp_logit, self.mlp_k)
                self.sp_stream.record_event(self.event_mlp_idx)
            if att_sp is not None:
                att_idx = ops.topk_indices(att_sp(residual), att_k, dtype=torch.int32, out=att_idx_out)
            self.sp_stream.record_event(self.event_side)
        self._mlp_idx_event = mlp_sp_logit is not None
        return mlp_idx, att_idx

    def _join_side(self):
        if self._side_used:
            torch.cuda.current_stream().wait_event(self.event_side)

    def join_side(self):
        """For a caller that passed ``defer_join=True`` to ``forward``: makes the current stream wait for
        the neuron selection of that forward.  The head selection (for the next layer) stays pending:
        whoever uses it calls ``join_heads()`` first (the blocks do at their start;
        ``join_side_stream()`` covers it too)."""
        if not self._side_used or self._joined:
            return
        if self._mlp_idx_event:
            torch.cuda.current_stream().wait_event(self.event_mlp_idx)
            mark_side_pending(self.event_side)
        else:
            torch.cuda.current_stream().wait_event(self.event_side)


class ParallelMHADejavu(_MHABase):
    """Dense attention + the MLP top-k (MLP-sparse-only model)."""

    def __init__(self, embed_dim, num_heads, process_group=None, sp_kwargs=None, bias=True, dropout=0.0,
                 softmax_scale=None, causal=False, layer_idx=None, rotary_emb_dim=0, rotary_emb_scale_base=0,
                 use_flash_attn=False, checkpointing=False, sequence_parallel=True, device=None, dtype=None) -> None:
        super().__init__()
        self._init_common(embed_dim, num_heads, process_group, bias, softmax_scale, causal, layer_idx,
                          rotary_emb_dim, device, dtype)

    def forward(self, x, mlp_sp_logit=None, seqlen=None, inference_params=None, defer_join=False, post_norm=None, **kwargs):
        """x: (B, s, d).  Returns (out, mlp_idx).  defer_join: the caller calls ``join_side()`` itself
        before it uses mlp_idx.  post_norm: as ``ParallelMHASparseAttMlp``'s, for prompts."""
        assert seqlen is None, "sequence-parallel input layout is not used for generation"
        self._streams()
        self._side_fork(x.shape[0])
        qkv = decode_linear(self.Wqkv, x)
        qkv = qkv.view(x.shape[0], x.shape[1], 3, self.num_heads, self.head_dim)
        context = self._dense_context(qkv, inference_params)
        out = _project_norm(self.out_proj, context, post_norm)
        mlp_idx, _ = self._side_work(mlp_sp_logit)
        if defer_join:
            self._side_keep = mlp_sp_logit
        else:
            self._join_side()
        return out, mlp_idx


class ParallelMHASparseAttMlp(_MHABase):
    """Head-sparse attention; also runs both top-ks (this layer's MLP neurons,
    next layer's heads) beside the main stream."""

    WINDOW = 16

    def __init__(self, embed_dim, num_heads, process_group=None, sp_kwargs=None, bias=True, dropout=0.0,
                 softmax_scale=None, causal=False, layer_idx=None, rotary_emb_dim=0, rotary_emb_scale_base=0,
                 use_flash_attn=False, checkpointing=False, sequence_parallel=True, device=None, dtype=None) -> None:
        super().__init__()
        assert sp_kwargs != None, "sparse predictor parameters are not passed in."
        self._init_common(embed_dim, num_heads, process_group, bias, softmax_scale, causal, layer_idx,
                          rotary_emb_dim, device, dtype)
        self.sp_kwargs = sp_kwargs
        self.sp = ParallelSP(layer_idx=layer_idx, device=device, dtype=dtype, process_group=process_group,
                             sequence_parallel=sequence_parallel, **sp_kwargs)
        self.att_k = self.sp.K
        # LayerNorm outputs of the current 16-token window, to recompute K/V of skipped heads
        self.x_cache = torch.zeros((self.WINDOW, embed_dim), dtype=torch.float16, device=device)
        self.x_cache_batch = None  # (16, B * embed_dim): the same for B > 1 sequences, made on first use
        # tracker[h, s] == s while window token s has no K/V for head h, else -1
        self.tracker = torch.arange(self.WINDOW, dtype=torch.int32, device=device).repeat(num_heads, 1)
        self.counter = 0
        self.cache_offset = None  # device int32[1]: cache position of window token 0
        # True keeps the window at its cache position after a flush (benchmarks that replay one window)
        self.hold_window = False
        self.out_proj_weight_t = None
        self._all_heads = None
        # optional caller-owned buffer for the predicted heads (fixed address for graph capture)
        self.att_idx_out = None

    def transposed_out_proj(self) -> torch.Tensor:
        """out_proj.weight as (H * hd, d), contiguous; follows updates of out_proj.weight."""
        return _transposed_copy(self, "out_proj_weight_t", self.out_proj.weight)

    def _set_cache_offset(self, value: int, device) -> None:
        """Updated in place once it exists: captured launch sequences hold its address."""
        if self.cache_offset is None:
            self.cache_offset = torch.tensor([value], dtype=torch.int32, device=device)
        else:
            self.cache_offset.fill_(value)

    def reset_window(self, cache_offset: Optional[int] = None, device=None):
        """A new window; cache_offset: where it lies in the caches, kept on ``device`` (the tracker's)."""
        self.counter = 0
        t, place = self.tracker, self.cache_offset
        device = t.device if device is None else device
        # callers may have put tensors of their own in both places
        plain = (results_only(t, place) and device == t.device and t.dtype == torch.int32 and t.is_contiguous() and
                 t.shape == (self.num_heads, self.WINDOW) and (place is None or (place.dtype == torch.int32 and place.numel() == 1)))
        if not plain:
            if cache_offset is not None:
                self._set_cache_offset(cache_offset, device)
            t.copy_(torch.arange(self.WINDOW, dtype=torch.int32, device=t.device).repeat(self.num_heads, 1))
            return
        if cache_offset is not None and place is None:
            place = self.cache_offset = torch.empty(1, dtype=torch.int32, device=device)
        # one launch (two fills, an arange and a copy: 15 to 20 us a block of a prompt)
        check(lib.dv_window_reset(t.data_ptr(), self.num_heads, None if cache_offset is None else place.data_ptr(),
                                  cache_offset or 0, ops._stream()), "dv_window_reset")

    def _sparse_decode(self, x, head_idx, inference_params):
        """x: (1, 1, d).  Window step, then QKV for the active heads and the window
        tokens they miss; the K / V rows go straight into the caches."""
        dev = x.device
        assert x.dtype == torch.float16 and x.is_contiguous()
        H, hd = self.num_heads, self.head_dim
        flush = self.counter == self.WINDOW - 1
        if flush:  # every 16th token all heads catch up
            if self._all_heads is None:
                self._all_heads = torch.arange(H, dtype=torch.int32, device=dev)
            head_idx = self._all_heads
        nnz = head_idx.shape[0]
        nb = self.counter + 1
        batch_idx = torch.empty(nnz, nb, dtype=torch.int32, device=dev)
        stream = ops._stream()
        check(lib.dv_window_step_f16(x.data_ptr(), self.x_cache.data_ptr(), self.embed_dim, self.tracker.data_ptr(),
                                     head_idx.data_ptr(), nnz, H, self.counter, int(flush), batch_idx.data_ptr(),
                                     stream), "dv_window_step_f16")
        k_cache, v_cache = inference_params.key_value_memory_dict[self.layer_idx]
        b0 = inference_params.batch_size_offset
        kc, vc = k_cache[b0:b0 + 1], v_cache[b0:b0 + 1]
        if self.cache_offset is None:
            self._set_cache_offset(inference_params.sequence_len_offset - self.counter, dev)
        qkv = ops.qkv_proj_sparse(self.x_cache[:nb], self.Wqkv.weight.view(3, H, hd, self.embed_dim), head_idx,
                                  batch_idx, None if self.Wqkv.bias is None else self.Wqkv.bias.view(3, H, hd),
                                  k_cache=kc, v_cache=vc, padding=self.cache_offset)
        self.counter += 1
        return qkv, head_idx, kc, vc

    def begin_window_step(self, B, head_idx, dev):
        """What the block needs to fold this step's window write and tracker step into its
        LayerNorm 1 launch (``ops.add_layer_norm_window``) for B > 1 sequences: the window buffer's
        row of this position, the tracker, the head set of the step (all heads at the flush
        position) and the slot list to fill.  The result goes back in as ``window=`` of ``forward``."""
        d, H = self.embed_dim, self.num_heads
        if self.x_cache_batch is None or self.x_cache_batch.shape[1] != B * d:
            assert self.counter == 0, "the batch size cannot change inside a back-fill window"
            self.x_cache_batch = torch.zeros((self.WINDOW, B * d), dtype=torch.float16, device=dev)
        flush = self.counter == self.WINDOW - 1
        if flush:
            if self._all_heads is None:
                self._all_heads = torch.arange(H, dtype=torch.int32, device=dev)
            head_idx = self._all_heads
        batch_idx = torch.empty(head_idx.shape[0], self.counter + 1, dtype=torch.int32, device=dev)
        return {"x_cache_row": self.x_cache_batch[self.counter], "tracker": self.tracker, "head_idx": head_idx,
                "counter": self.counter, "flush": flush, "batch_idx": batch_idx}

    def _sparse_decode_batched(self, x, head_idx, inference_params, window=None):
        """x: (B, 1, d), B > 1 sequences that decode in lockstep and share the head set and the
        back-fill window (the reference's sparse attention is single-sequence, mha_dejavu.py:1469;
        this is its batch extension).  The window buffer holds the B LayerNorm rows of each of
        the 16 window tokens; the tracker is the one of the single-sequence path.  At the first
        window position the QKV is one pass over the active heads' weights for the B rows; later
        positions multiply all window tokens of all sequences (up to 16 B rows) in one pass and
        store, per head, the tokens that head still misses (the flush step: every head, 16 B rows)."""
        dev = x.device
        assert x.dtype == torch.float16 and x.is_contiguous()
        B, d, H, hd = x.shape[0], self.embed_dim, self.num_heads, self.head_dim
        if self.x_cache_batch is None or self.x_cache_batch.shape[1] != B * d:
            assert self.counter == 0, "the batch size cannot change inside a back-fill window"
            self.x_cache_batch = torch.zeros((self.WINDOW, B * d), dtype=torch.float16, device=dev)
        nb = self.counter + 1
        if window is not None:  # the block's LayerNorm launch has written the window row and run the tracker
            assert window["counter"] == self.counter and window["x_cache_row"].data_ptr() == \
                self.x_cache_batch[self.counter].data_ptr()
            head_idx, batch_idx = window["head_idx"], window["batch_idx"]
        else:
            flush = self.counter == self.WINDOW - 1
            if flush:
                if self._all_heads is None:
                    self._all_heads = torch.arange(H, dtype=torch.int32, device=dev)
                head_idx = self._all_heads
            nnz = head_idx.shape[0]
            batch_idx = torch.empty(nnz, nb, dtype=torch.int32, device=dev)
            check(lib.dv_window_step_f16(x.data_ptr(), self.x_cache_batch.data_ptr(), B * d, self.tracker.data_ptr(),
                                         head_idx.data_ptr(), nnz, H, self.counter, int(flush), batch_idx.data_ptr(),
                                         ops._stream()), "dv_window_step_f16")
        k_cache, v_cache = inference_params.key_value_memory_dict[self.layer_idx]
        b0 = inference_params.batch_size_offset
        kc, vc = k_cache[b0:b0 + B], v_cache[b0:b0 + B]
        if self.cache_offset is None:
            self._set_cache_offset(inference_params.sequence_len_offset - self.counter, dev)
        lengths = inference_params.lengths_per_sample
        weight = self.Wqkv.weight.view(3, H, hd, d)
        bias = None if self.Wqkv.bias is None else self.Wqkv.bias.view(3, H, hd)
        qkv = torch.empty(B, 3, H, hd, dtype=torch.float16, device=dev)
        # window token s goes to cache position cache_offset + s, or lengths[b] - (counter - s)
        positions = self.cache_offset if lengths is None else lengths
        if nb == 1:
            ops.qkv_proj_batch(self.x_cache_batch[0].view(B, d), weight, head_idx, bias, out=qkv, k_cache=kc,
                               v_cache=vc, positions=positions, pos_add=0, live=batch_idx[:, 0])
        else:  # all window tokens of all sequences in one pass over the weights
            ops.qkv_window_batch(self.x_cache_batch, weight, head_idx, batch_idx, B, bias, out=qkv, k_cache=kc,
                                 v_cache=vc, positions=positions, pos_add=0 if lengths is None else -self.counter)
        self.counter += 1
        return qkv, head_idx, kc, vc

    def forward(self, x, residual, head_idx=None, mlp_sp_logit=None, seqlen=None, inference_params=None, window=None,
                defer_join=False, post_norm=None, **kwargs):
        """x, residual: (B, s, d).  head_idx: (Hk,) int32 heads to compute, or None
        for dense attention.  mlp_sp_logit: predictor logits for this layer's MLP.  window: the
        result of ``begin_window_step`` when the caller's LayerNorm launch has already done the
        window step.  defer_join: the caller calls ``join_side()`` itself before it uses mlp_idx / att_idx
        (the block does).  post_norm = (LayerNorm module, its residual input): the caller's residual add + LayerNorm
        of `out`, done here when it can ride in the projection's reduction launch (batched sparse decode, five
        rows and more; prompts whose projection ends in one); `out` is then the pair (normed, residual_out) instead of the projection.
        Returns (out, mlp_idx, att_idx)."""
        assert seqlen is None, "sequence-parallel input layout is not used for generation"
        self._streams()
        do_token_generation = x.size(1) == 1
        if x.size(1) != 1:  # prompt: remember where the decode window starts
            self.reset_window(x.size(1), x.device)
        sparse = inference_params is not None and inference_params.sequence_len_offset > 0 and head_idx is not None
        self._side_fork(x.shape[0])
        side_done = None
        joined_early = False
        self._joined = False
        if sparse:
            assert x.size(1) == 1
            self.transposed_out_proj()
            if x.size(0) == 1:
                qkv, head_idx, kc, vc = self._sparse_decode(x, head_idx, inference_params)
                # the caches now hold the newest token for the active heads
                out = ops.attention_out_proj(qkv[-1:, 0], kc, vc, head_idx, inference_params.sequence_len_offset,
                                             self.out_proj_weight_t, self.out_proj.bias,
                                             inference_params.lengths_per_sample, self.softmax_scale).unsqueeze(1)
            else:
                qkv, head_idx, kc, vc = self._sparse_decode_batched(x, head_idx, inference_params, window)
                # the side work right behind the QKV launch (the main chain's first launch of the module is
                # captured, and the selections can be waited for in front of out_proj)
                side_done = self._side_work(mlp_sp_logit, residual, self.sp if do_token_generation else None,
                                            self.att_k, self.att_idx_out)
                ctx = ops.single_query_attention(qkv[:, 0], None, None, kc, vc, inference_params.lengths_per_sample,
                                                 inference_params.sequence_len_offset, self.rotary_emb_dim,
                                                 head_idx=head_idx, softmax_scale=self.softmax_scale)
                if post_norm is not None and x.size(0) >= ops.OUT_PROJ_LN_MIN_ROWS:
                    # the caller's residual add + LayerNorm ride in the projection's reduction launch; the
                    # wait for the neuron selection, which the caller would place in front of its LayerNorm,
                    # goes in front of the projection
                    if defer_join:
                        self.join_side()
                        joined_early = True
                    norm, norm_residual = post_norm
                    out = ops.out_proj_sparse_t_add_layer_norm(ctx, self.out_proj_weight_t, head_idx,
                                                               self.out_proj.bias, norm_residual, norm.weight,
                                                               norm.bias, norm.eps)
                    out = (out[0].unsqueeze(1), out[1].view_as(norm_residual))
                else:
                    out = ops.out_proj_sparse_t(ctx, self.out_proj_weight_t, head_idx,
                                                self.out_proj.bias).unsqueeze(1)
            if self.counter == self.WINDOW:  # window complete: start the next one
                self.counter = 0
                if not self.hold_window:
                    self.cache_offset += self.WINDOW
        else:
            qkv = decode_linear(self.Wqkv, x)
            qkv = qkv.view(x.shape[0], x.shape[1], 3, self.num_heads, self.head_dim)
            context = self._dense_context(qkv, inference_params)
            out = _project_norm(self.out_proj, context, post_norm)
        if side_done is None:
            side_done = self._side_work(mlp_sp_logit, residual, self.sp if do_token_generation else None,
                                        self.att_k, self.att_idx_out)
        mlp_idx, att_idx = side_done
        if defer_join:
            self._side_keep = (residual, mlp_sp_logit)  # read by the side work until the next step
            self._joined = joined_early  # the caller's join_side() then has nothing left to do
        else:
            self._join_side()
        return out, mlp_idx, att_idx
