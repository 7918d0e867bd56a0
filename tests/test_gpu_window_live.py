"""QKV of a back-fill window of several sequences by the rows that are live (qkv_window.hpp): as many rows as end a tile and one
more, one to all sixteen tokens, heads that share a tile, with and without splits of the columns."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nseq,hd,d,counts", [
    (32, 128, 1024, [2, 3, 4, 5, 8, 9, 16, 1]),   # 64, 96, 128, 160, 256, 288, 512 and 32 rows
    (17, 128, 2048, [4, 7, 8, 15, 16]),           # 68, 119, 136, 255, 272
    (13, 64, 264, [1, 5, 9, 10, 16]),             # two heads a tile; 33 pieces, no splits
    (5, 32, 520, [16, 1, 0, 13, 2, 3]),           # four heads a tile, 80 rows in all, one head without any
    (32, 128, 264, [2, 3, 4, 5, 8, 9, 16, 1, 7, 12, 10]),   # by the rows that are live: 64, 96, 128, 160, 256, 288, 512, 32 .. rows, no splits
    (13, 128, 2048, [4, 5, 9, 10, 16, 0, 15, 1, 2, 13, 8]),  # 52, 65, 117, 130, 208, no rows .., in splits
    (12, 128, 2048, [4, 5, 9, 10, 16, 0, 15, 1, 2, 13, 8]),  # the last that multiplies all rows
])
def test_live_rows(nseq, hd, d, counts):
    from dejavu_amd import ops

    H, T, S = len(counts) + 1, 16, 40
    g = torch.Generator().manual_seed(nseq * hd)
    rand = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).half()  # noqa: E731
    xw, W, bias = rand(T, nseq * d), rand(3, H, hd, d, std=d ** -0.5), rand(3, H, hd, std=0.1)
    heads = torch.arange(1, H).int()
    live = torch.full((H - 1, T), -1, dtype=torch.int32)
    for i, n in enumerate(counts):
        s = torch.cat([torch.tensor([T - 1]), torch.randperm(T - 1, generator=g)])[:n]  # the newest token whenever there is any
        live[i, s] = s.int()
    k0, v0 = torch.full((nseq, H, hd // 8, S, 8), 5.0).half(), torch.full((nseq, H, S, hd), 5.0).half()
    k, v, out = k0.clone().cuda(), v0.clone().cuda(), torch.full((nseq, 3, H, hd), 5.0, dtype=torch.float16, device="cuda")
    pos = torch.tensor([7], dtype=torch.int32)
    ops.qkv_window_batch(xw.cuda(), W.cuda(), heads.cuda(), live.cuda(), nseq, bias.cuda(), out=out, k_cache=k, v_cache=v,
                         positions=pos.cuda(), pos_add=1)
    want = (xw.view(T * nseq, d).double() @ W.view(-1, d).double().t()).view(T, nseq, 3, H, hd) + bias.double()
    k = k.cpu().permute(0, 1, 3, 2, 4).reshape(nseq, H, S, hd)
    checked = 0
    for h in range(H):
        for t in range(T):
            pairs = [(k[:, h, 8 + t], 1), (v.cpu()[:, h, 8 + t], 2)] + ([(out.cpu()[:, j, h], j) for j in range(3)] if t == T - 1 else [])
            for got, j in pairs:
                if h == 0 or live[h - 1, t] < 0:
                    assert (got == 5.0).all(), (h, t, j)
                else:
                    # one rounding to fp16 of sums of unit size
                    assert np.allclose(got.double(), want[t, :, j, h], rtol=2.0 ** -10, atol=2e-4), (h, t, j)
                    checked += 1
    assert checked == 2 * sum(counts) + 3 * sum(n > 0 for n in counts)
    assert (k[:, :, :8] == 5.0).all() and (v.cpu()[:, :, :8] == 5.0).all()
