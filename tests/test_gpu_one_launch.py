"""Decode rows whose keys one launch takes, at the edges of its turns and of the rule, against float64 softmax attention of the
same bf16 inputs."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# bf16 results: half an ulp is 2^-9 of a value; products and sums are fp32
LIMIT = 2.0 ** -8


def rounded(rng, *shape, std=1.0):
    t = torch.tensor(rng.normal(size=shape) * std, device="cuda").bfloat16()
    return t, t.double().cpu().numpy()


def attend(q, k, v, scale, extra=None, sink=None):
    s = k @ q * scale + (0.0 if extra is None else extra)
    top = max(s.max(), -np.inf if sink is None else sink)
    p = np.exp(s - top)
    return p @ v / (p.sum() + (0.0 if sink is None else np.exp(sink - top)))


def close(got, want):
    got = got.double().cpu().numpy().reshape(want.shape)
    assert np.linalg.norm(got - want) <= LIMIT * np.linalg.norm(want)


@pytest.mark.parametrize("H,G,dim,vdim", [(4, 2, 128, 128), (3, 1, 72, 40), (2, 2, 8, 120)])
@pytest.mark.parametrize("cap,pos", [(1, 0), (64, 63), (65, 64), (128, 100), (129, 300), (256, 255), (257, 256), (384, 383), (384, 1000),
                                     (385, 384)])
@pytest.mark.parametrize("biased", [False, True])
def test_ring_row(H, G, dim, vdim, cap, pos, biased):
    from dejavu_amd import mixer_ops as ops

    rng = np.random.default_rng(cap + dim)
    k, kd = rounded(rng, cap, G, dim)
    v, vd = rounded(rng, cap, G, vdim)
    row = torch.tensor(rng.normal(size=(1, H * dim + G * (dim + vdim))), dtype=torch.float32, device="cuda")
    gate = torch.tensor(rng.normal(size=H), dtype=torch.float32, device="cuda")
    rel = torch.tensor(rng.normal(size=(H, 50)), dtype=torch.float32, device="cuda") if biased else None
    sink = None if biased else gate + 1.0
    # a chunk ends the ring's use at its edge; a window keeps all of the ring
    start = pos // cap * cap if biased else max(0, pos - cap + 1)
    args = dict(chunk=cap, rel=rel) if biased else dict(window=cap, sink=sink)
    got = ops.ring_attention_row(row, k.view(cap, -1), v.view(cap, -1), H, G, dim, 0.1, 1e-5,
                                 torch.tensor([pos], dtype=torch.int32, device="cuda"), 0, gate=gate, **args)
    r = row[0].double().cpu().numpy()
    norm = lambda x: x / np.sqrt((x * x).mean(-1, keepdims=True) + 1e-5)  # noqa: E731
    q = norm(r[:H * dim].reshape(H, dim))
    own = [torch.tensor(x).bfloat16().double().numpy() for x in (norm(r[H * dim:(H + G) * dim].reshape(G, dim)),
                                                                  r[(H + G) * dim:].reshape(G, vdim))]
    kd[pos % cap], vd[pos % cap] = own
    seen = [j % cap for j in range(start, pos + 1)]
    want = np.empty((H, vdim))
    for h in range(H):
        g = h * G // H
        extra = rel[h].double().cpu().numpy()[np.minimum(pos - np.arange(start, pos + 1), 49)] if biased else None
        o = attend(q[h], kd[seen, g], vd[seen, g], 0.1, extra, None if biased else sink[h].item())
        want[h] = o / (1.0 + np.exp(-gate[h].item()))
    close(got, want)
    close(k[pos % cap], own[0]), close(v[pos % cap], own[1])


@pytest.mark.parametrize("rank,vdim", [(256, 128), (200, 72), (512, 128), (264, 40)])
@pytest.mark.parametrize("cap,pos", [(1, 0), (64, 63), (65, 64), (128, 127), (129, 128), (257, 256), (385, 384), (400, 399), (401, 400)])
def test_latent_row(rank, vdim, cap, pos):
    from dejavu_amd import mixer_ops as ops

    H, dim, rng = 3, 136, np.random.default_rng(cap + rank)
    c, cd = rounded(rng, cap, rank)
    ku, kd = rounded(rng, H * dim, rank, std=(rank * dim) ** -0.5)
    vu, vd = rounded(rng, H * vdim, rank, std=rank ** -0.5)
    q = torch.tensor(rng.normal(size=(1, H * dim)), dtype=torch.float32, device="cuda")
    gate = torch.tensor(rng.normal(size=H), dtype=torch.float32, device="cuda")
    got = ops.latent_attention_row(q, ku, vu, c, H, 2.0, gate, torch.tensor([pos], dtype=torch.int32, device="cuda"), 0)
    want = np.empty((H, vdim))
    for h in range(H):
        ql = q[0].double().cpu().numpy()[h * dim:(h + 1) * dim] @ kd[h * dim:(h + 1) * dim]
        lat = attend(ql, cd[:pos + 1], cd[:pos + 1], 2.0) / (1.0 + np.exp(-gate[h].item()))
        want[h] = vd[h * vdim:(h + 1) * vdim] @ lat
    close(got, want)


@pytest.mark.parametrize("n", [1032, 2048, 8184, 8192, 8200])
def test_top_k_of_one_row(n):
    """Both sides of the line up to which one workgroup selects: ties, few values, all kinds of k."""
    from dejavu_amd import ops
    from oracle import dejavu_oracle as O

    rng = np.random.default_rng(n)
    mixed = np.round(rng.normal(size=n) * 2).astype(np.float16)
    mixed[[0, n // 2, n - 1]] = np.inf, np.nan, -np.inf
    for x in (rng.normal(size=n).astype(np.float16), mixed, np.full(n, -1.5, dtype=np.float16)):
        for k in (1, n // 3, n - 1, n):
            want = O.topk_lower_index(x, k)
            for dtype in (torch.int32, torch.int64):
                got = ops.topk_indices(torch.from_numpy(x).cuda(), k, dtype=dtype)
                assert np.array_equal(got.cpu().numpy().astype(np.int64), want)
