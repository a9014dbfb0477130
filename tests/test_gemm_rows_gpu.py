"""fp16 products of a depth up to 80, both operands stored (K, rows), whose many rows are off cache lines: blocks of rows and columns that end
inside the matrix, lines that begin in one block and end in the next, depths of one to three k-steps, operands shared by the batch, the memory around
the output."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck
from util import stream

pytestmark = pytest.mark.gpu

LARGE = 3 << 23         # outputs from which such products have a kernel of their own


def _operands(batch, n, m, k, shared=""):
    g = torch.Generator(device="cuda").manual_seed(n * 3 + m + k)
    A = torch.randn((1 if "A" in shared else batch, k, m), generator=g, device="cuda").half()
    return A, torch.randn((1 if "B" in shared else batch, k, n), generator=g, device="cuda").half()


def _run(A, B):
    batch, k, m, n = max(A.size(0), B.size(0)), A.size(1), A.size(2), B.size(2)
    total, front = batch * n * m, 8
    padded = torch.full((total + 2 * front,), float("nan"), dtype=torch.half, device="cuda")
    ck.gemm_fp16(m, k, n, A.size(0), B.size(0), False, True, A.data_ptr(), B.data_ptr(), padded[front:].data_ptr(), stream())
    assert padded[:front].isnan().all() and padded[front + total:].isnan().all()
    return padded[front:front + total].view(batch, n, m)


def _product(batch, n, m, k, shared=""):
    A, B = _operands(batch, n, m, k, shared)
    out = _run(A, B)
    assert not out.isnan().any()
    for i in sorted({0, 1, 2, batch // 2, batch - 2, batch - 1} & set(range(batch))):
        a, b = A[i % A.size(0)].double(), B[i % B.size(0)].double().t().contiguous()
        ref, size = b @ a, b.abs() @ a.abs()
        # k additions in fp32, one rounding to fp16 (or half a subnormal step)
        assert ((out[i].double() - ref).abs() <= size * k * 2.0 ** -24 + ref.abs() * 2.0 ** -10.9 + 2.0 ** -25).all()


# rows that start on 16, 8 and 4 bytes; one wave of columns to eight; blocks of 16 rows and parts of them, workgroups of 16 rows to 560 and shorter last ones
@pytest.mark.parametrize("n,m,k", [(8, 130, 64), (10, 134, 64), (66, 130, 64), (64, 254, 2), (500, 500, 64), (500, 500, 80), (62, 136, 32), (72, 362, 34), (130, 502, 66),
                                   (300, 300, 48), (18, 1022, 78), (1000, 1000, 64), (80, 900, 62), (200, 260, 30), (8, 1000, 64), (1030, 140, 62), (254, 154, 80), (560, 162, 28)])
def test_large(n, m, k):
    _product(LARGE // (n * m) + 1, n, m, k)


@pytest.mark.parametrize("batch,n,m,k", [(1, 26000, 970, 64), (3, 9000, 1002, 80), (27, 1018, 922, 40)])
def test_few_entries(batch, n, m, k):
    _product(batch, n, m, k)


@pytest.mark.parametrize("n,m", [(66, 66), (66, 126), (112, 68), (100, 100), (98, 74)])
@pytest.mark.parametrize("batch", [1, 5, 600])
@pytest.mark.parametrize("k", [2, 64, 80])
def test_little(n, m, batch, k):
    _product(batch, n, m, k)


# workgroups as tall as their share of LDS holds them: short depths, from as many entries on as fill the device with one each
@pytest.mark.parametrize("n,m,k,batch", [(1200, 130, 32, 2000), (800, 140, 16, 1600), (592, 130, 64, 2560)])
def test_tallest_workgroups(n, m, k, batch):
    _product(batch, n, m, k)


# values that are not finite stay in their own rows and columns
@pytest.mark.parametrize("n,m,k,batch", [(500, 500, 64, 110), (130, 502, 66, LARGE // (130 * 502) + 1), (100, 100, 30, 5), (66, 74, 2, 3)])
def test_values_that_are_not_finite(n, m, k, batch):
    A, B = _operands(batch, n, m, k)
    clean = _run(A, B)
    A[:, :, 0], A[:, :, m - 1], B[:, :, 0], B[:, :, n - 1] = float("nan"), float("nan"), float("inf"), float("nan")
    spoilt = _run(A, B)
    assert not clean.isnan().any() and torch.equal(clean[:, 1:n - 1, 1:m - 1], spoilt[:, 1:n - 1, 1:m - 1])
    assert spoilt[:, :, 0].isnan().all() and spoilt[:, :, m - 1].isnan().all() and spoilt[:, n - 1].isnan().all() and not spoilt[:, 0].isfinite().any()


@pytest.mark.parametrize("shared", ["A", "B"])
def test_shared_operand(shared):
    _product(110, 500, 500, 64, shared)
