"""fp16 products of a depth up to 128 with both operands stored (K, rows): tile edges, depths of part of a slab and of two, operands shared
by the batch, unaligned buffers, outputs that are stored with and without the hint, and sizes just outside."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck
import cpm_kernels_amd.torch as ct
from util import quickest, stream

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


@pytest.mark.parametrize("m,n", [(128, 130), (192, 136), (200, 384), (254, 250), (500, 130), (262, 300)])
@pytest.mark.parametrize("k", [40, 64, 128])
def test_overlapping_tiles_leave_no_gap(m, n, k):
    """The last tiles store what the ones before them do not: every element of an output full of NaN is written."""
    a, b = _operands(3, 3, k, m, n, m * n + k)
    out = torch.full((3, n, m), float("nan"), dtype=torch.half, device="cuda")
    ck.gemm_fp16(m, k, n, 3, 3, False, True, a.data_ptr(), b.data_ptr(), out.data_ptr(), stream())
    _check(b, a, out)


def test_overlapping_tiles_store_once():
    """6510 of 160 x 192 beside as many outputs in whole tiles, 3051 of 256 x 256: 201 and 84 us where the overlaps were stored again, 148 and
    86 now (the tiles of the first cover 2.1 times its area, all of which is still computed).  The bound lies between the ratios of 2.4 and 1.7."""
    def product(batch, n, m, k=64):
        a, b = _operands(batch, batch, k, m, n, n)
        out = torch.empty((batch, n, m), dtype=torch.half, device="cuda")
        return lambda: ck.gemm_fp16(m, k, n, batch, batch, False, True, a.data_ptr(), b.data_ptr(), out.data_ptr(), stream())
    t = quickest([product(3051, 256, 256), product(6510, 160, 192)], reps=10)
    print("whole tiles %.1f us, overlapping ones %.1f us" % tuple(t), flush=True)
    assert t[1] <= 2.05 * t[0], t


@pytest.mark.parametrize("batch_a,batch_b,m,n,k", [
    # both sides of a quarter of the last-level cache, where overlapping tiles give way to the large ones: two slabs, a shared operand
    (1285, 1285, 192, 136, 128), (1286, 1286, 192, 136, 128), (1286, 1286, 192, 136, 112),
    (1285, 1, 192, 136, 64), (1286, 1, 192, 136, 64), (1, 1286, 192, 136, 64), (1, 1286, 192, 136, 120), (340, 1, 512, 200, 64), (1, 340, 512, 200, 64),
    # rows that are not whole pieces, in and beyond a tile
    (190, 1, 400, 450, 128), (600, 1, 400, 250, 128), (1, 1300, 198, 136, 64),
])
def test_overlap_and_depth_choose_the_kernel(batch_a, batch_b, m, n, k):
    a, b = _operands(batch_a, batch_b, k, m, n, m + n)
    batch = max(batch_a, batch_b)
    out = torch.full((batch, n, m), float("nan"), dtype=torch.half, device="cuda")
    ck.gemm_fp16(m, k, n, batch_a, batch_b, False, True, a.data_ptr(), b.data_ptr(), out.data_ptr(), stream())
    assert torch.isfinite(out).all()
    for i in (0, batch // 2, batch - 1):
        _check(b[i % batch_b:][:1], a[i % batch_a:][:1], out[i:i + 1])
