"""fp16 products of a depth up to 128 with both operands stored (K, rows): tile edges, depths of part of a slab and of two, operands shared
by the batch, unaligned buffers, outputs that are stored with and without the hint, and sizes just outside."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck
import cpm_kernels_amd.torch as ct

pytestmark = pytest.mark.gpu


def _operands(batch_a, batch_b, k, m, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn((batch_a, k, m), generator=g, device="cuda").half(), torch.randn((batch_b, k, n), generator=g, device="cuda").half())


def _check(a, b, out):
    ad, bd = a.double().transpose(1, 2).contiguous(), b.double()
    ref = torch.stack([ad[i % ad.size(0)] @ bd[i % bd.size(0)] for i in range(out.size(0))])
    size = torch.stack([ad[i % ad.size(0)].abs() @ bd[i % bd.size(0)].abs() for i in range(out.size(0))])
    # K additions in fp32, one rounding to fp16 (or half a subnormal step)
    bound = size * a.size(1) * 2.0 ** -24 + ref.abs() * (2.0 ** -11 + 2.0 ** -20) + 2.0 ** -25
    assert ((out.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("m,n", [(128, 128), (130, 128), (128, 254), (256, 384), (258, 130), (500, 500), (126, 256), (256, 126)])
@pytest.mark.parametrize("k", [2, 62, 64, 66, 80, 126, 128, 130])
def test_depths_and_edges(m, n, k):
    a, b = _operands(3, 3, k, m, n, m + n + k)
    _check(a, b, ct.bmm(a, True, b, False, int8=False))


@pytest.mark.parametrize("batch_a,batch_b", [(1, 4), (4, 1)])
@pytest.mark.parametrize("k", [64, 100])
def test_shared_operand(batch_a, batch_b, k):
    a, b = _operands(batch_a, batch_b, k, 200, 300, k)
    _check(a, b, ct.bmm(a, True, b, False, int8=False))


@pytest.mark.parametrize("shift", [1, 2, 4])
def test_unaligned_buffers(shift):
    batch, k, m, n = 2, 72, 192, 256
    a, b = _operands(batch, batch, k, m, n, shift)
    pa, pb, po = (torch.zeros(t + 8, dtype=torch.half, device="cuda") for t in (a.numel(), b.numel(), batch * m * n))
    ua, ub, uo = pa[shift:shift + a.numel()], pb[shift:shift + b.numel()], po[shift:shift + batch * m * n]
    ua.copy_(a.view(-1))
    ub.copy_(b.view(-1))
    ck.gemm_fp16(n, k, m, batch, batch, False, True, ub.data_ptr(), ua.data_ptr(), uo.data_ptr(), torch.cuda.current_stream().cuda_stream)
    _check(a, b, uo.view(batch, m, n))
    assert (po[:shift] == 0).all() and (po[shift + batch * m * n:] == 0).all()


@pytest.mark.parametrize("batch,m,n,k", [(385, 512, 512, 64), (300, 500, 504, 64), (260, 500, 500, 80), (800, 300, 300, 64)])
def test_large_outputs(batch, m, n, k):
    a, b = _operands(batch, batch, k, m, n, batch)
    out = ct.bmm(a, True, b, False, int8=False)
    for i in (0, batch // 2, batch - 1):
        _check(a[i:i + 1], b[i:i + 1], out[i:i + 1])
