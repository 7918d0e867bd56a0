"""GPU parity of the dense products of the prompt phase (dv_dense_linear_f16): blocks of up to 128
rows shared through LDS, split over the columns for short matrices."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def assert_close(got, want, what="", max_abs_tol=2e-2, rel_tol=1e-3):
    got = np.asarray(got, dtype=np.float64)
    want = np.asarray(want, dtype=np.float64)
    max_abs = np.max(np.abs(got - want)) if got.size else 0.0
    rel = np.linalg.norm(got - want) / max(np.linalg.norm(want), 1e-30)
    if (max_abs_tol, rel_tol) != (2e-2, 1e-3):  # a bound other than the per-operator one: say what was measured
        print(f"measured {what}: max_abs={max_abs:.3e} rel_l2={rel:.3e} (bounds {max_abs_tol:g} / {rel_tol:g})", flush=True)
    assert max_abs <= max_abs_tol and rel <= rel_tol, f"{what}: max_abs={max_abs:.3e} rel_l2={rel:.3e}"


@pytest.mark.parametrize("rows,N,M,act", [(1, 768, 2304, "id"), (7, 520, 1001, "relu"), (16, 1024, 4096, "id"),
                                          (33, 776, 300, "relu"), (64, 2048, 640, "id"), (128, 1024, 4096, "relu"),
                                          (130, 520, 2050, "id"), (300, 768, 3072, "relu"), (128, 5120, 15360, "id"),
                                          (520, 1024, 1000, "id"), (200, 256, 130, "relu"), (1030, 512, 2304, "id")])
def test_dense_linear_matches_fp32_reference(rows, N, M, act):
    """Against the fp32-accumulated product of the same fp16 operands (max-abs 2e-2, relative L2 1e-3).
    Ragged cases: a last column chunk that is not full, output widths that are not multiples of 4 or
    of a wavefront's 16 rows, more rows than one 128-row block, row-strided input and output."""
    from dejavu_amd import ops

    g = torch.Generator().manual_seed(rows * 7 + M)
    xbig = torch.randn(rows, N + 16, generator=g).half().cuda()
    x = xbig[:, :N]
    W = (torch.randn(M, N, generator=g) * 0.04).half().cuda()
    b = (torch.randn(M, generator=g) * 0.1).half().cuda()
    print(f"case dense linear rows={rows} N={N} M={M} {act}", flush=True)
    y = ops.dense_linear(x, W, b, act)
    ybig = torch.full((rows, M + 8), 3.0, dtype=torch.float16, device="cuda")
    ops.dense_linear(x, W, None, act, out=ybig[:, :M])
    y2 = ops.dense_linear(x, W, b, act)
    torch.cuda.synchronize()
    ref = x.float() @ W.float().t()
    want, want_nb = ref + b.float(), ref
    if act == "relu":
        want, want_nb = want.relu(), want_nb.relu()
    assert y.shape == (rows, M)
    assert_close(y.cpu().numpy(), want.cpu().numpy(), "dense linear + bias")
    assert_close(ybig[:, :M].cpu().numpy(), want_nb.cpu().numpy(), "dense linear into a strided output")
    assert torch.all(ybig[:, M:] == 3.0), "columns beyond the output width were written"
    assert torch.equal(y, y2), "two runs differ (the split reduction must be deterministic)"


# Both sides of the rules that choose a kernel and a tile (rows 64 | 65, 128 | 129, 192 | 193, 256 | 257, 384 | 385, 512 | 513;
# weights of 2^23, 21 and 52 million elements; 7680, 32768 and 40960 rows of W; fewer than 32 tiles of 128 rows; one round of
# tiles of 64; rows of W too short to split), last tiles of one to four rows.
@pytest.mark.parametrize("rows,N,M,act", [(9, 264, 70, "gelu"), (30, 4096, 4884, "id"), (20, 4096, 4100, "relu"),
                                          (50, 12288, 4097, "id"), (65, 264, 70, "relu"), (128, 2056, 4099, "id"),
                                          (100, 4104, 12290, "gelu_approx"), (129, 1032, 4101, "squared_relu"),
                                          (192, 2048, 5121, "id"), (140, 4096, 18433, "id"),
                                          (128, 2048, 14340, "id"), (100, 4096, 16383, "id"), (193, 8, 33, "relu"),
                                          (256, 2056, 4098, "relu"), (257, 520, 71, "id"), (384, 2056, 5442, "id"), (385, 2056, 130, "id"),
                                          (512, 2056, 130, "relu"),
                                          (513, 520, 70, "id"), (300, 256, 16390, "id"),
                                          (32, 2048, 4096, "id"), (32, 2048, 4104, "id"), (40, 5120, 4104, "relu"),
                                          (64, 6656, 7680, "id"), (64, 6656, 7688, "id"), (64, 264, 32770, "id"),
                                          (65, 264, 32768, "id"), (65, 264, 32770, "id"), (129, 264, 32770, "id"),
                                          (300, 264, 40970, "id"), (300, 256, 40970, "relu"),
                                          # activations that the wide tiles leave to gemm_big.hpp: 192, 256 and 128 weight rows a tile
                                          (520, 256, 9790, "gelu"), (520, 512, 13050, "gelu_approx"), (300, 256, 40970, "gelu"), (1030, 256, 2306, "gelu")])
def test_dense_linear_at_the_edges_of_its_rules(rows, N, M, act):
    from dejavu_amd import ops

    g = torch.Generator(device="cuda").manual_seed(rows + M)
    x = torch.randn(rows, N + 8, generator=g, device="cuda").half()[:, 8:]
    W = (torch.randn(M, N, generator=g, device="cuda") * N ** -0.5).half()
    b = torch.randn(M, generator=g, device="cuda").half()
    print(f"case dense linear rows={rows} N={N} M={M} {act}", flush=True)
    y = ops.dense_linear(x, W, b, act)
    want = x.float() @ W.float().t() + b.float()
    F = torch.nn.functional
    want = {"id": want, "relu": want.relu(), "gelu": F.gelu(want), "gelu_approx": F.gelu(want, approximate="tanh"),
            "squared_relu": want.relu() ** 2}[act]
    assert_close(y.cpu().numpy(), want.cpu().numpy(), "dense linear", max_abs_tol=4e-2)  # half an ulp at 64: 0.031


@pytest.mark.parametrize("rows", [40, 64])
def test_gathered_rows_out_of_range(rows):
    """An index outside the weight gives act(0), whichever kernel runs."""
    from dejavu_amd import ops

    g = torch.Generator(device="cuda").manual_seed(rows)
    x, W = torch.randn(rows, 520, generator=g, device="cuda").half(), torch.randn(90, 520, generator=g, device="cuda").half()
    b = torch.randn(90, generator=g, device="cuda").half()
    idx = torch.tensor([3, -1, 89, 90, 0, 7, 1 << 40], device="cuda")
    ok = (idx >= 0) & (idx < 90)
    want = torch.zeros(rows, idx.numel(), device="cuda")
    want[:, ok] = (x.float() @ W[idx[ok]].float().t() + b[idx[ok]].float()).relu()
    got = ops.gather_gemv(x, W, idx, b, activation="relu")
    assert_close(got.float().cpu().numpy(), want.cpu().numpy(), "gathered rows", max_abs_tol=8e-2)  # half an ulp at 128


@pytest.mark.parametrize("rows,N,M", [(33, 1024, 12288), (64, 2048, 10240), (48, 264, 16390)])
def test_gathered_rows_that_need_no_workspace(rows, N, M):
    """Weights with tiles enough for the chip are not split, and go to the same kernel as the dense product: the same bits."""
    from dejavu_amd import ops
    from dejavu_amd._lib import lib

    assert lib.dv_gather_gemv_workspace_bytes(rows, N, M) == 0
    g = torch.Generator(device="cuda").manual_seed(rows)
    x, W = torch.randn(rows, N, generator=g, device="cuda").half(), (torch.randn(M, N, generator=g, device="cuda") * N ** -0.5).half()
    want = ops.dense_linear(x, W)
    assert torch.equal(ops.gather_gemv(x, W, None), want)
    idx = torch.randperm(M, generator=g, device="cuda")
    assert torch.equal(ops.gather_gemv(x, W, idx), want[:, idx])


def test_dense_linear_three_dimensional_input():
    from dejavu_amd import ops

    g = torch.Generator().manual_seed(5)
    x = torch.randn(2, 9, 256, generator=g).half().cuda()
    W = (torch.randn(512, 256, generator=g) * 0.05).half().cuda()
    y = ops.dense_linear(x, W)
    torch.cuda.synchronize()
    assert y.shape == (2, 9, 512)
    assert_close(y.cpu().numpy(), (x.float() @ W.float().t()).cpu().numpy(), "3-d input")


@pytest.mark.parametrize("B,T,H,hd", [(1, 1, 2, 64), (1, 7, 3, 64), (2, 37, 4, 128), (1, 64, 2, 128), (1, 128, 5, 128),
                                      (1, 130, 2, 64), (3, 200, 2, 128),
                                      (2, 37, 128, 64), (4, 100, 33, 64), (4, 128, 32, 128), (3, 1, 171, 128)])  # 512 workgroups: two wavefronts
def test_prefill_attention_matches_oracle(B, T, H, hd):
    """Causal attention over the prompt against the oracle's prompt_attention, and the K / V rows in the
    packed caches bit for bit (they are copies); prompt lengths that are not multiples of 16 / 32 / 64."""
    from dejavu_amd import ops
    from oracle import dejavu_oracle as O

    g = torch.Generator().manual_seed(T * 10 + H)
    qkv = torch.randn(B, T, 3, H, hd, generator=g).half()
    S, pos0 = T + 9, 4
    k_cache = torch.full((B, H, hd // 8, S, 8), 5.0, dtype=torch.float16, device="cuda")
    v_cache = torch.full((B, H, S, hd), 5.0, dtype=torch.float16, device="cuda")
    print(f"case prefill attention B={B} T={T} H={H} hd={hd}", flush=True)
    ctx = ops.prefill_attention(qkv.cuda(), k_cache, v_cache, pos0)
    ctx_nc = ops.prefill_attention(qkv.cuda())
    torch.cuda.synchronize()
    assert ctx.shape == (B, T, H * hd) and torch.equal(ctx, ctx_nc)
    for b in range(B):
        kn = np.full((H, hd // 8, S, 8), 5.0, np.float16)
        vn = np.full((H, S, hd), 5.0, np.float16)
        want = O.prompt_attention(qkv[b].numpy(), kn, vn, pos0=pos0)
        assert_close(ctx[b].cpu().numpy().reshape(T, H, hd), want, f"context of sequence {b}", max_abs_tol=5e-3,
                     rel_tol=1e-3)
        assert np.array_equal(k_cache[b].cpu().numpy(), kn) and np.array_equal(v_cache[b].cpu().numpy(), vn)


@pytest.mark.parametrize("T", [45, 230])
def test_prompt_runs_on_the_hip_kernels_and_matches_the_library_path(T):
    """The prompt phase of a small model through dv_dense_linear_f16 / dv_prefill_attention_f16
    (USE_HIP_PROMPT) against PyTorch's library GEMM and attention on the same weights, and against
    the oracle's model_prompt; the caches the two paths leave behind agree within fp16 rounding.
    The 230-token prompt is past both lengths (HIP_PROMPT_MAX_ROWS, HIP_PROMPT_ATTN_MAX_TOKENS) from which
    on the library may be taken: its products are the library's, its attention and cache fill the kernel's
    as long as only results are asked for."""
    import dejavu_amd.modules as M
    from dejavu_amd.gpt import GPTLMHeadModel, SparseGPTConfig
    from dejavu_amd.modules import InferenceParams
    from oracle import dejavu_oracle as O
    from tests.model_utils import load_model_params, make_model_params

    L, d, H, ffn, r, V, P = 2, 256, 4, 1024, 32, 512, 256
    params = make_model_params(L, d, H, ffn, r, V, P, 256, [2, 2], seed=5)
    cfg = SparseGPTConfig(hidden_size=d, num_attention_heads=H, num_hidden_layers=L, vocab_size=V, n_inner=ffn,
                          max_position_embeddings=P, mlp_K=256, mlp_sp_dim=r, att_K=[2, 2], att_sp_dim=r)
    model = GPTLMHeadModel(cfg, device="cuda", dtype=torch.float16).eval()
    load_model_params(model, params)
    assert (T <= M.HIP_PROMPT_ATTN_MAX_TOKENS) == (T == 45)
    prompt = [int(v) for v in torch.randint(0, V, (T,), generator=torch.Generator().manual_seed(1))]
    ids = torch.tensor([prompt], device="cuda")
    outs, caches = [], []
    assert M.USE_HIP_PROMPT
    try:
        for flag in (True, False):
            M.USE_HIP_PROMPT = flag
            ip = InferenceParams(max_sequence_len=256, max_batch_size=1)
            print(f"case prompt phase of {T} tokens, hip kernels={flag}", flush=True)
            with torch.no_grad():
                logits = model(ids, inference_params=ip, last_token_only=True).logits[0, -1]
            torch.cuda.synchronize()
            outs.append(logits.float().cpu().numpy())
            caches.append([(k.float().cpu().numpy(), v.float().cpu().numpy()) for k, v in
                           (ip.key_value_memory_dict[l] for l in range(L))])
    finally:
        M.USE_HIP_PROMPT = True
    state = O.new_decode_state(params, 256)
    want = O.model_prompt(params, state, prompt).astype(np.float32)
    assert_close(outs[0], want, "prompt logits, hip kernels vs oracle", rel_tol=1.3e-3)
    assert_close(outs[1], want, "prompt logits, library path vs oracle", rel_tol=1.3e-3)
    for l in range(L):
        for got, ref, o in zip(caches[0][l], caches[1][l], state["caches"][l]):
            assert_close(got, o.astype(np.float32), f"layer {l} cache vs oracle")
            assert_close(got, ref, f"layer {l} cache, hip vs library path")


# the weights of a row are fp16 values of 2^-12 relative rounding at most, as the result: 5e-4 of values below 5
@pytest.mark.parametrize("B,T,H,hd", [(1, 31, 2, 64), (2, 32, 3, 128), (1, 33, 2, 128), (1, 129, 8, 64), (1, 257, 2, 128)])
def test_prefill_attention_at_the_edges_of_its_blocks(B, T, H, hd):
    """Prompts that end a block of 32 queries or keys, or begin one; a context that is not on 16 bytes; the results do
    not depend on later tokens."""
    from dejavu_amd._lib import check, lib

    g = torch.Generator(device="cuda").manual_seed(T)
    qkv = (torch.randn(B, T, 3, H, hd, generator=g, device="cuda") * 2).half()
    print(f"case prefill attention B={B} T={T} H={H} hd={hd}", flush=True)
    q, k, v = (t.transpose(1, 2).cpu().double() for t in qkv.unbind(2))
    s = (q @ k.transpose(2, 3) * hd ** -0.5).masked_fill(torch.ones(T, T).triu(1).bool(), -1e300)
    want = (s.softmax(-1) @ v).transpose(1, 2).reshape(B, T, H * hd)
    got = {}
    for offset, rows in ((0, T), (1, T), (0, T - 1)):
        room = torch.zeros(B * rows * H * hd + 8, dtype=torch.float16, device="cuda")
        part = qkv[:, :rows].contiguous()
        ctx = room[offset:offset + B * rows * H * hd]
        check(lib.dv_prefill_attention_f16(part.data_ptr(), B, rows, H, hd, hd ** -0.5, ctx.data_ptr(), None, None, 0, 0,
                                           torch.cuda.current_stream().cuda_stream), "dv_prefill_attention_f16")
        assert not room[:offset].any() and not room[offset + ctx.numel():].any()
        got[offset, rows] = ctx.view(B, rows, H * hd).cpu()
    torch.testing.assert_close(got[0, T].double(), want, rtol=1e-3, atol=5e-3)
    assert torch.equal(got[1, T], got[0, T]) and torch.equal(got[0, T - 1], got[0, T][:, :T - 1])


def test_gradients_of_a_long_prompts_attention():
    from dejavu_amd.modules import HIP_PROMPT_ATTN_MAX_TOKENS, ParallelMHADejavu

    T = HIP_PROMPT_ATTN_MAX_TOKENS + 8
    mha = ParallelMHADejavu(128, 2, causal=True, device="cuda", dtype=torch.float16)
    qkv = torch.randn(1, T, 3, 2, 64, device="cuda").half().requires_grad_()
    ctx = mha._dense_context(qkv, None)
    ctx.sum().backward()
    assert qkv.grad.abs().sum() > 0
    with torch.no_grad():
        torch.testing.assert_close(mha._dense_context(qkv, None), ctx.detach(), rtol=2e-3, atol=5e-3)
