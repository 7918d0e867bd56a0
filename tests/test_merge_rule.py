"""Which decode rows leave the merge of their splits to the output projection: both sides of each line."""
import pytest
import torch

from dejavu_amd import mixer_ops as ops


def test_rule():
    for keys, window, chunk in ((320, False, False), (321, True, True), (512, True, True), (513, False, True), (1024, False, True), (1025, False, False),
                                (16384, False, False)):
        assert ops._merge_rule(16, 128, keys, torch.bfloat16, True) == window, keys
        assert ops._merge_rule(16, 128, keys, torch.bfloat16, False) == chunk, keys
    assert ops._merge_rule(32, 64, 400, torch.bfloat16, True) and not ops._merge_rule(17, 128, 400, torch.bfloat16, True)
    assert not ops._merge_rule(16, 128, 400, torch.float32, True)


@pytest.mark.gpu
@pytest.mark.parametrize("mask,cap,merged", [("window", 512, True), ("window", 520, False), ("chunk", 520, True), ("chunk", 1024, True), ("chunk", 1032, False),
                                             (None, 1024, True), (None, 1032, False), (None, 4096, False)])
def test_what_rows_do(mask, cap, merged, monkeypatch):
    H, G, dim, pos = 4, 2, 64, cap - 1
    g = torch.Generator(device="cuda").manual_seed(cap)
    kr, vr = (torch.randn(cap, G * dim, device="cuda", generator=g).bfloat16() for _ in range(2))
    row = torch.randn(1, (H + 2 * G) * dim, device="cuda", generator=g)
    W = (torch.randn(72, H * dim, device="cuda", generator=g) * 0.06).bfloat16()
    masks = {mask: cap} if mask else {}
    got = [ops.ring_attention_row(row, kr.clone(), vr.clone(), H, G, dim, 0.125, 1e-5, None, pos, defer=d, **masks) for d in (True, False)]
    assert isinstance(got[0], ops.SplitRow) == merged and isinstance(got[1], torch.Tensor)
    a, b = (ops.linear(x, W).double() for x in got)
    assert (a - b).norm() <= 2 ** -8 * b.norm()
    if not merged:
        assert torch.equal(a, b)
