"""Argmax and bookkeeping of a generation step in two launches: ends of workgroups, ties, NaN, rows off 16-byte boundaries, full buffers."""
import pytest
import torch

from dejavu_amd import mixer_ops as ops

pytestmark = pytest.mark.gpu
LINE = ops.GREEDY_PARTS


@pytest.fixture(params=[1, 1 << 30], ids=["two launches", "one launch"], autouse=True)
def launches(request, monkeypatch):
    """Both forms at every size, whichever the line between them would choose."""
    monkeypatch.setattr(ops, "GREEDY_PARTS", request.param)


@pytest.mark.parametrize("vocab", [1, 3, 1023, 1024, 1025, 4099, 32768, 70001])
@pytest.mark.parametrize("kind", ["one", "tie", "nan", "lowest"])
@pytest.mark.parametrize("off", [0, 1])
def test_step(vocab, kind, off):
    g = torch.Generator(device="cuda").manual_seed(vocab)
    logits = torch.randn(vocab + 8, device="cuda", generator=g)[off:off + vocab]
    want = int(logits.argmax())
    if kind == "tie":
        top = logits.max() + 1
        for i in (vocab // 3, vocab // 2, vocab - 1):
            logits[i] = top
        want = vocab // 3
    elif kind == "nan":
        logits[vocab // 2], logits[vocab - 1], want = float("nan"), float("nan"), vocab // 2
    elif kind == "lowest":
        logits.fill_(float("-inf"))
        want = 0
    ones = [torch.full((1,), v, dtype=t, device="cuda") for v, t in ((7, torch.int64), (8, torch.int64), (9, torch.int32), (2, torch.int64), (1, torch.int64))]
    token, position, seq_pos, out_index, score_index = ones
    sequences = torch.full((1, 4), -1, dtype=torch.int64, device="cuda")
    scores = torch.full((3, vocab), 5.0, device="cuda")
    for step in range(3):  # the third token and the third row of scores have no place
        ops.greedy_advance(logits, token, position, seq_pos, sequences, out_index, scores, score_index)
        assert [int(t) for t in ones] == [want, 9 + step, 10 + step, 3 + step, 2 + step]
    assert sequences.tolist() == [[-1, -1, want, want]]
    assert bool((scores[0] == 5).all()) and all(torch.equal(scores[i], logits) or kind == "nan" for i in (1, 2))
    if kind == "nan":
        assert torch.equal(scores[1].nan_to_num(3.0), logits.nan_to_num(3.0))
    ops.greedy_advance(logits, token, position, seq_pos, sequences, out_index)
    assert int(score_index) == 4 and int(token) == want and int(out_index) == 6


@pytest.mark.parametrize("vocab", [1, 7, 1025, 32768, 50272])
@pytest.mark.parametrize("off", [0, 1])
def test_entry_without_scratch(vocab, off):
    """The one launch that callers of the C library without scratch have does the same."""
    g = torch.Generator(device="cuda").manual_seed(vocab)
    logits = torch.randn(vocab + 8, device="cuda", generator=g)[off:off + vocab]
    logits[vocab // 2] = logits.max() + 1
    logits[vocab - 1] = logits[vocab // 2]  # a tie: the first
    got = []
    for scratch in (True, False):
        ones = [torch.full((1,), v, dtype=t, device="cuda") for v, t in ((7, torch.int64), (8, torch.int64), (9, torch.int32), (2, torch.int64), (1, torch.int64))]
        token, position, seq_pos, out_index, score_index = ones
        sequences, scores = torch.full((1, 4), -1, dtype=torch.int64, device="cuda"), torch.full((3, vocab), 5.0, device="cuda")
        for _ in range(3):
            if scratch:
                ops.greedy_advance(logits, token, position, seq_pos, sequences, out_index, scores, score_index)
            else:
                assert ops.lib.dv_mix_greedy_advance(logits.data_ptr(), vocab, token.data_ptr(), position.data_ptr(), seq_pos.data_ptr(),
                                                     sequences.data_ptr(), 4, out_index.data_ptr(), scores.data_ptr(), vocab, 3, score_index.data_ptr(),
                                                     ops._stream()) == 0
        got.append([t.clone() for t in (*ones, sequences, scores)])
    assert int(got[0][0]) == vocab // 2 and all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("vocab,count", [(5, 1), (8191, 1), (8192, 2), (50272, 2)])
def test_few_logits_take_one_launch(vocab, count, monkeypatch):
    called = []
    monkeypatch.setattr(ops, "GREEDY_PARTS", LINE)
    for name, n in (("dv_mix_greedy_advance", 1), ("dv_mix_greedy_advance_ws", 2)):
        entry = getattr(ops.lib, name)
        monkeypatch.setattr(ops.lib, name, lambda *a, entry=entry, n=n: [called.append(n), entry(*a)][1])
    logits = torch.randn(vocab, device="cuda")
    logits[vocab - 2] = 9.0
    token, position, out_index = (torch.zeros(1, dtype=torch.int64, device="cuda") for _ in range(3))
    seq_pos, sequences = torch.zeros(1, dtype=torch.int32, device="cuda"), torch.zeros(1, 4, dtype=torch.int64, device="cuda")
    ops.greedy_advance(logits, token, position, seq_pos, sequences, out_index)
    assert called == [count] and int(token) == int(sequences[0, 0]) == vocab - 2
    assert int(position) == int(seq_pos) == int(out_index) == 1
