"""What the gradient of the embedding table is prepared with: order of the ids, gradient rows, zeros, in one launch."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck
import cpm_kernels_amd.torch as ct
from util import stream

pytestmark = pytest.mark.gpu


# (whole pieces on both sides, on one, on none; tiles of part of their rows and columns; a table of part of a piece; no tokens, no table)
@pytest.mark.parametrize("batch,hidden,seq,vocab", [(1, 8, 8, 1), (3, 264, 72, 50), (2, 64, 512, 9000), (17, 72, 64, 3), (2, 100, 72, 33), (2, 72, 100, 33), (5, 257, 63, 61),
                                                    (1, 3, 2, 5), (1, 4096, 40, 300), (0, 16, 8, 7), (2, 16, 8, 0)])
@pytest.mark.parametrize("ordered", [False, True])
def test_prepare(batch, hidden, seq, vocab, ordered):
    g = torch.Generator(device="cuda").manual_seed(hidden + seq)
    tokens = batch * seq
    ids = torch.randint(0, max(vocab, 1), (tokens,), generator=g, device="cuda", dtype=torch.int32)
    dy = torch.randn((batch, hidden, seq), generator=g, device="cuda").half()
    order, values = torch.full((2, tokens), -9, device="cuda", dtype=torch.int32)
    rows = torch.full((tokens + 1, hidden), float("nan"), device="cuda", dtype=torch.half)
    table = torch.full((vocab * hidden + 8,), float("nan"), device="cuda", dtype=torch.half)
    ck.embedding_backward_prepare(batch, hidden, seq, vocab, None if ordered else ids.data_ptr(), order.data_ptr(), values.data_ptr(), dy.data_ptr(), rows.data_ptr(),
                                  table.data_ptr(), stream())
    assert torch.equal(rows[:tokens], dy.transpose(1, 2).reshape(tokens, hidden)) and rows[tokens:].isnan().all()
    assert (table[:vocab * hidden] == 0).all() and table[vocab * hidden:].isnan().all()
    want = ids.sort(stable=True)
    if ordered:
        assert (order == -9).all() and (values == -9).all()
    else:
        assert torch.equal(order.long(), want.indices) and torch.equal(values, want.values)


def test_more_tiles_than_a_launch_holds():
    """262144 sequences of one token: 2^24 tiles, four a workgroup of 1024 threads"""
    batch, hidden, vocab = 1 << 18, 4096, 50
    g = torch.Generator(device="cuda").manual_seed(5)
    ids = torch.randint(0, vocab, (batch, 1), generator=g, device="cuda", dtype=torch.int32)
    dy = torch.empty((batch, hidden, 1), device="cuda", dtype=torch.half).normal_(generator=g)
    order, values = torch.full((2, batch), -9, device="cuda", dtype=torch.int32)
    rows = torch.full((batch, hidden), float("nan"), device="cuda", dtype=torch.half)
    table = torch.full((vocab * hidden,), float("nan"), device="cuda", dtype=torch.half)
    ck.embedding_backward_prepare(batch, hidden, 1, vocab, ids.data_ptr(), order.data_ptr(), values.data_ptr(), dy.data_ptr(), rows.data_ptr(), table.data_ptr(), stream())
    want = ids.view(-1).sort(stable=True)
    assert torch.equal(order.long(), want.indices) and torch.equal(values, want.values)
    assert torch.equal(rows, dy.view(batch, hidden)) and (table == 0).all()
    del rows, table
    emb = ct.Embedding(vocab, hidden).cuda()
    with torch.no_grad():
        emb.weight.normal_(generator=g)
    got = torch.autograd.grad(emb(ids), emb.weight, dy)[0].double()
    for v in (0, 1, vocab - 1):
        of = dy[(ids == v).view(-1)].view(-1, hidden).double()
        ref, size = of.sum(0), of.abs().sum(0)
        # some 5000 additions in fp32, one rounding to fp16
        assert ((got[v] - ref).abs() <= size * of.size(0) * 2.0 ** -24 + ref.abs() * 2.0 ** -11 + 2.0 ** -25).all()
