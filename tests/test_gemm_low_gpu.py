"""fp16 products of up to 64 rows beside an operand stored (K, rows): tile edges, depths of part of a slab and of several, operands shared by
the batch, unaligned buffers, and sizes at both sides of where the kernel or its loads change."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck
import cpm_kernels_amd.torch as ct

pytestmark = pytest.mark.gpu


def _operands(batch_a, batch_b, n, k, m, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn((batch_a, n, k), generator=g, device="cuda").half(), torch.rand((batch_b, k, m), generator=g, device="cuda").half()


def _check(a, b, out):
    ad, bd = a.double(), b.double()
    ref = torch.stack([ad[i % ad.size(0)] @ bd[i % bd.size(0)] for i in range(out.size(0))])
    size = torch.stack([ad[i % ad.size(0)].abs() @ bd[i % bd.size(0)].abs() for i in range(out.size(0))])
    # K additions in fp32, one rounding to fp16 (or half a subnormal step)
    bound = size * a.size(2) * 2.0 ** -24 + ref.abs() * (2.0 ** -11 + 2.0 ** -20) + 2.0 ** -25
    assert ((out.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("n,m", [(64, 128), (64, 130), (62, 254), (2, 256), (32, 500), (34, 130), (66, 128), (64, 126)])
@pytest.mark.parametrize("k", [2, 6, 62, 64, 66, 128, 500, 1024, 1026])
def test_depths_and_edges(n, m, k):
    a, b = _operands(3, 3, n, k, m, n + m + k)
    _check(a, b, ct.bmm(a, False, b, False, int8=False))


@pytest.mark.parametrize("batch_a,batch_b", [(1, 4), (4, 1)])
@pytest.mark.parametrize("k", [64, 100])
def test_shared_operand(batch_a, batch_b, k):
    a, b = _operands(batch_a, batch_b, 40, k, 300, k)
    _check(a, b, ct.bmm(a, False, b, False, int8=False))


@pytest.mark.parametrize("shift", [1, 2, 4])
def test_unaligned_buffers(shift):
    batch, n, k, m = 2, 48, 90, 192
    a, b = _operands(batch, batch, n, k, m, shift)
    pa, pb, po = (torch.zeros(t + 8, dtype=torch.half, device="cuda") for t in (a.numel(), b.numel(), batch * m * n))
    ua, ub, uo = pa[shift:shift + a.numel()], pb[shift:shift + b.numel()], po[shift:shift + batch * m * n]
    ua.copy_(a.view(-1))
    ub.copy_(b.view(-1))
    ck.gemm_fp16(m, k, n, batch, batch, False, False, ub.data_ptr(), ua.data_ptr(), uo.data_ptr(), torch.cuda.current_stream().cuda_stream)
    _check(a, b, uo.view(batch, n, m))
    assert (po[:shift] == 0).all() and (po[shift + batch * m * n:] == 0).all()


@pytest.mark.parametrize("batch,k,m", [(383, 512, 512), (385, 512, 512), (770, 512, 512), (400, 500, 500), (1000, 300, 300)])
def test_large_operands(batch, k, m):
    a, b = _operands(batch, batch, 64, k, m, batch)
    out = ct.bmm(a, False, b, False, int8=False)
    for i in (0, batch // 2, batch - 1):
        _check(a[i:i + 1], b[i:i + 1], out[i:i + 1])


# off cache lines, around the depth and the rounds of the device where the tile kernel takes over (256 tiles of 64 x 256 at a time)
@pytest.mark.parametrize("batch,n,k,m", [(400, 64, 1000, 200), (150, 64, 1000, 200), (80, 64, 1000, 200), (400, 30, 600, 200), (300, 64, 600, 200),
                                         (400, 64, 510, 200), (234, 64, 700, 500), (171, 64, 700, 500), (400, 64, 700, 198), (58, 2, 700, 2002)])
def test_deep_products_choose_the_kernel(batch, n, k, m):
    a, b = _operands(batch, batch, n, k, m, batch + k)
    out = torch.full((batch, n, m), float("nan"), dtype=torch.half, device="cuda")
    ck.gemm_fp16(m, k, n, batch, batch, False, False, b.data_ptr(), a.data_ptr(), out.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert torch.isfinite(out).all()
    for i in (0, batch // 2, batch - 1):
        _check(a[i:i + 1], b[i:i + 1], out[i:i + 1])
