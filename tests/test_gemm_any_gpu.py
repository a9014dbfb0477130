"""fp16 products of few rows or columns or of rows that are not whole pieces: edges of tiles and slabs, pieces across the end of a row, odd addresses."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck
import cpm_kernels_amd.torch as ct
from util import stream

pytestmark = pytest.mark.gpu


def _check(A, aT, B, bT, out):
    """out (batch, n, m) of A (., k, m) [(., m, k) if aT] and B (., n, k) [(., k, n) if bT]"""
    k = A.size(2 if aT else 1)
    last = out.size(0) - 1
    for i in sorted({0, 1, 2, last // 2, last - 1, last} & set(range(last + 1))):
        a, b = A[i % A.size(0)].double(), B[i % B.size(0)].double()
        a, b = (a.t() if aT else a).contiguous(), (b.t() if bT else b).contiguous()
        ref, size = b @ a, b.abs() @ a.abs()
        # k additions in fp32, one rounding to fp16 (or half a subnormal step)
        assert ((out[i].double() - ref).abs() <= size * k * 2.0 ** -24 + ref.abs() * 2.0 ** -10.9 + 2.0 ** -25).all()


def _product(batch_a, batch_b, m, k, n, aT, bT, shift=0):
    g = torch.Generator(device="cuda").manual_seed(m * 3 + n + k)
    A = torch.randn((batch_a, m, k) if aT else (batch_a, k, m), generator=g, device="cuda").half()
    B = torch.randn((batch_b, k, n) if bT else (batch_b, n, k), generator=g, device="cuda").half()
    batch = max(batch_a, batch_b)
    sizes = (A.numel(), B.numel(), batch * n * m)
    pa, pb, po = (torch.full((t + 16,), float("nan"), dtype=torch.half, device="cuda") for t in sizes)
    ua, ub, uo = (p[shift:shift + t] for p, t in zip((pa, pb, po), sizes))
    ua.copy_(A.view(-1))
    ub.copy_(B.view(-1))
    ck.gemm_fp16(m, k, n, batch_a, batch_b, aT, bT, ua.data_ptr(), ub.data_ptr(), uo.data_ptr(), stream())
    _check(A, aT, B, bT, uo.view(batch, n, m))
    assert po[:shift].isnan().all() and po[shift + sizes[2]:].isnan().all()


@pytest.mark.parametrize("aT,bT", [(True, False), (False, False), (True, True), (False, True)])
@pytest.mark.parametrize("m,n", [(2, 2), (6, 64), (62, 66), (64, 128), (66, 126), (126, 80), (128, 34), (130, 100), (200, 128), (258, 66)])
@pytest.mark.parametrize("k", [2, 30, 64, 66, 100, 192])
@pytest.mark.parametrize("batch", [3, 140])        # (tiles of 64 x 64, larger ones from where those are more than one a compute unit)
def test_edges(aT, bT, m, n, k, batch):
    _product(batch, batch, m, k, n, aT, bT)


# values that are not finite stay in their own rows and columns: pieces across a row's end are read with what lies behind it
@pytest.mark.parametrize("aT,bT", [(True, False), (False, False), (True, True), (False, True)])
@pytest.mark.parametrize("m,n,k,batch", [(70, 66, 30, 2), (190, 70, 100, 2), (66, 126, 200, 140), (130, 66, 72, 140), (2, 2, 2, 3)])
def test_values_that_are_not_finite(aT, bT, m, n, k, batch):
    g = torch.Generator(device="cuda").manual_seed(m + k)
    A = torch.randn((batch, m, k) if aT else (batch, k, m), generator=g, device="cuda").half()
    B = torch.randn((batch, k, n) if bT else (batch, n, k), generator=g, device="cuda").half()
    outs = []
    for spoilt in (False, True):
        if spoilt:
            A.select(1 if aT else 2, 0).fill_(float("nan"))
            B.select(2 if bT else 1, 0).fill_(float("inf"))
        out = torch.full((batch, n, m), 7.0, dtype=torch.half, device="cuda")
        ck.gemm_fp16(m, k, n, batch, batch, aT, bT, A.data_ptr(), B.data_ptr(), out.data_ptr(), stream())
        outs.append(out)
    clean, spoilt = outs
    assert not clean.isnan().any() and torch.equal(clean[:, 1:, 1:], spoilt[:, 1:, 1:])
    assert spoilt[:, :, 0].isnan().all() and not spoilt[:, 0, 1:].isfinite().any()


@pytest.mark.parametrize("aT,bT", [(True, False), (False, False), (True, True), (False, True)])
@pytest.mark.parametrize("shift", [1, 2, 7])
def test_any_address(aT, bT, shift):
    _product(2, 2, 190, 70, 100, aT, bT, shift)
    _product(1, 4, 60, 250, 130, aT, bT, shift)
    _product(4, 1, 130, 250, 60, aT, bT, shift)


@pytest.mark.parametrize("aT", [True, False])
@pytest.mark.parametrize("m,n,k,batch", [(500, 64, 500, 130), (512, 128, 512, 120), (700, 80, 700, 80), (400, 96, 400, 4)])
def test_many_small_tiles(aT, m, n, k, batch):
    _product(batch, batch, m, k, n, aT, False)


# the columns of several entries side by side: depths of 64- and 128-byte slabs and with a rest, P K-major and stored (K, rows), few and many tiles
@pytest.mark.parametrize("m,batch,n", [(4, 33, 136), (36, 7, 304), (100, 5, 128), (132, 3, 264), (252, 16, 4112)])
@pytest.mark.parametrize("k", [34, 64, 96, 130, 136, 512, 1000])
@pytest.mark.parametrize("bT", [False, True])
def test_joined_columns(m, batch, n, k, bT):
    _product(batch, 1, m, k, n, True, bT)


@pytest.mark.parametrize("aT", [False, True])
@pytest.mark.parametrize("tokens,batch,din,dout", [(36, 1, 4096, 1024), (100, 16, 1024, 4608), (52, 3, 1500, 640), (188, 1, 4096, 1024), (44, 5, 600, 600)])
def test_copied_operand(aT, tokens, batch, din, dout):
    g = torch.Generator(device="cuda").manual_seed(tokens)
    w = torch.randn((1, din, dout) if aT else (1, dout, din), generator=g, device="cuda").half()
    x = torch.randn((batch, din, tokens), generator=g, device="cuda").half()
    _check(x, False, w, aT, ct.bmm(w, aT, x, False, int8=False))


# depths that are not whole slabs beyond a few of them: large tiles, one and two small ones a compute unit and several, whole pieces and dwords
@pytest.mark.parametrize("m,n,batch,k", [(4100, 4112, 1, 708), (4100, 4112, 1, 1000), (4100, 4112, 1, 1504), (1500, 1200, 1, 1286), (640, 640, 1, 2824), (4004, 1200, 1, 324),
                                         (4004, 1200, 1, 1000), (300, 300, 70, 450), (300, 300, 70, 1000), (130, 1300, 9, 1500)])
def test_long_ragged_depths(m, n, batch, k):
    _product(batch, 1 if m == 130 else batch, m, k, n, True, False)
