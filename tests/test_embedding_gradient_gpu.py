"""The gradient of the embedding table against float64: runs of equal ids inside, at and across the pieces of 32 sorted tokens,
hidden sizes off 16-byte pieces, and the gather at the edges of its tiles."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck
import cpm_kernels_amd.torch as ct
from cpm_kernels_amd.torch import embedding as module

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [1, 2, 63, 64, 65, 1000, 4099])
@pytest.mark.parametrize("vocab", [1, 3, 5000])
def test_order_of_ids(gpu, tokens, vocab):
    print("order of ids", tokens, vocab, flush=True)
    ids = torch.randint(-vocab, vocab, (tokens,), generator=torch.Generator().manual_seed(tokens), dtype=torch.int32).cuda()
    order, values = torch.full((2, tokens), -9, device="cuda", dtype=torch.int32)
    ck.embedding_order_ids(tokens, ids.data_ptr(), order.data_ptr(), values.data_ptr(), torch.cuda.current_stream().cuda_stream)
    want = ids.sort(stable=True)
    assert torch.equal(order.long(), want.indices) and torch.equal(values, want.values)


# (batch, seq, hidden, vocab): one token; one id only (a run over many pieces, over exactly two, ending at an edge); few ids; mostly single ones;
# hidden sizes of 8j and others, one above a workgroup's columns
@pytest.mark.parametrize("shape", [(1, 1, 8, 4), (1, 33, 7, 1), (2, 32, 16, 1), (1, 2100, 24, 1), (3, 37, 100, 3), (2, 500, 264, 40), (4, 129, 2056, 3000),
                                   (5, 64, 257, 60)])
@pytest.mark.parametrize("ranked", [True, False])
def test_embedding_gradient(gpu, monkeypatch, shape, ranked):
    batch, seq, hidden, vocab = shape
    print("embedding gradient", shape, ranked, flush=True)
    if not ranked:
        monkeypatch.setattr(module, "MAX_RANKED", 0)
    g = torch.Generator().manual_seed(seq + hidden)
    emb = ct.Embedding(vocab, hidden).cuda()
    with torch.no_grad():
        emb.weight.copy_(torch.randn(vocab, hidden, generator=g))
    ids = torch.randint(0, vocab, (batch, seq), generator=g, dtype=torch.int32).cuda()
    dy = torch.randn(batch, hidden, seq, generator=g).half().cuda()
    out = emb(ids)
    assert torch.equal(out, emb.weight[ids.long()].transpose(1, 2))
    (grad,) = torch.autograd.grad(out, [emb.weight], dy)
    rows = dy.transpose(1, 2).reshape(-1, hidden).double()
    zero = torch.zeros((vocab, hidden), device="cuda", dtype=torch.float64)
    want, size = zero.index_add(0, ids.view(-1).long(), rows), zero.index_add(0, ids.view(-1).long(), rows.abs())
    # rounded once to fp16 (2^-11), and fp32 sums in chains of at most 32 + tokens / 32 additions of 2^-24 of the magnitudes
    bound = want.abs() * 2.0 ** -11 + size * (32 + batch * seq / 32) * 2.0 ** -24 + 2.0 ** -25
    assert bool(((grad.double() - want).abs() <= bound).all())
