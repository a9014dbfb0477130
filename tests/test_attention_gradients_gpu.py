"""Gradients of the softmax and of the position bias over sequences of any length: tiles of 128 to 1024 rows, teams beyond, pieces across the
end of a row."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck
import oracle
from util import stream, to_gpu

pytestmark = pytest.mark.gpu


def _softmax_backward(b, n, m, shift=0):
    g = torch.Generator(device="cuda").manual_seed(n + m)
    p = torch.softmax(torch.randn((b, n, m), generator=g, device="cuda") * 2, dim=1).half()
    y = torch.randn((b, n, m), generator=g, device="cuda").half()
    bufs = [torch.zeros(t.numel() + 16, dtype=torch.half, device="cuda")[shift:shift + t.numel()] for t in (p, y, p)]
    bufs[0].copy_(p.view(-1))
    bufs[1].copy_(y.view(-1))
    bufs[2].fill_(float("nan"))
    ck.softmax_backward(b, n, m, bufs[0].data_ptr(), bufs[1].data_ptr(), bufs[2].data_ptr(), stream())
    got, pd, yd = bufs[2].view(b, n, m).double(), p.double(), y.double()
    s = (pd * yd).sum(1, keepdim=True)
    want = pd * (yd - s)
    # n products added in fp32, a difference, a product and one rounding to fp16 (or half a subnormal step)
    bound = pd * ((pd * yd).abs().sum(1, keepdim=True) * n * 2.0 ** -24 + (yd.abs() + s.abs()) * 2.0 ** -23) + want.abs() * 2.0 ** -10.9 + 2.0 ** -25
    assert ((got - want).abs() <= bound).all()


@pytest.mark.parametrize("n", [1, 2, 64, 65, 127, 128, 129, 256, 257, 512, 513, 900, 1024, 1025, 1600])
@pytest.mark.parametrize("m", [7, 64, 72, 130])
def test_softmax_backward_rows(n, m):
    _softmax_backward(3, n, m)


@pytest.mark.parametrize("n", [100, 200, 500, 1000])
def test_softmax_backward_any_address(n):
    _softmax_backward(2, n, 128, shift=3)


def test_softmax_backward_teams_in_several_launches():
    """2800 x 3 team parts exceed the packet slots of one launch."""
    _softmax_backward(2800, 1040, 64)


@pytest.mark.parametrize("bidirectional", [True, False])
@pytest.mark.parametrize("ql,kl,heads", [(1, 1, 3), (7, 5, 4), (1344, 1, 5), (102, 10, 3), (102, 20, 3), (96, 6, 4), (96, 8, 4), (50, 64, 32), (64, 64, 2), (36, 27, 770), (8, 13, 304), (100, 65, 12), (333, 130, 5), (250, 250, 40), (1022, 1022, 15), (2050, 40, 3), (2050, 2050, 2)])
@pytest.mark.parametrize("shift", [0, 1])
def test_position_bias_gradient(bidirectional, ql, kl, heads, shift):
    buckets, far = 32, 128
    mapping = to_gpu(oracle.position_embedding_init(buckets, far, bidirectional))
    gen = torch.Generator(device="cuda").manual_seed(ql + kl)
    g = torch.randn((heads, kl, ql), generator=gen, device="cuda").half()
    buf = torch.zeros(g.numel() + 16, dtype=torch.half, device="cuda")[shift:shift + g.numel()]
    buf.copy_(g.view(-1))
    grad = torch.full((heads, buckets), float("nan"), dtype=torch.half, device="cuda")
    ck.position_embedding_backward(ql, kl, buckets, far, heads, mapping.data_ptr(), buf.data_ptr(), grad.data_ptr(), bidirectional, stream())
    rel = torch.arange(ql, device="cuda")[None, :] - torch.arange(kl, device="cuda")[:, None]
    bucket = mapping.long()[(rel.abs() if bidirectional else rel.clamp(min=0)).clamp(max=far - 1)]
    if bidirectional:
        bucket = bucket + (rel < 0) * (buckets // 2)
    at = bucket.view(1, -1).expand(heads, -1)
    want = torch.zeros((heads, buckets), dtype=torch.float64, device="cuda").scatter_add_(1, at, g.view(heads, -1).double())
    size = torch.zeros_like(want).scatter_add_(1, at, g.view(heads, -1).double().abs())
    # fp32 sums in chains of at most one addition a row, a query and a part, one rounding to fp16
    assert ((grad.double() - want).abs() <= size * (ql + kl + 64) * 2.0 ** -24 + want.abs() * 2.0 ** -10.9 + 2.0 ** -25).all()
