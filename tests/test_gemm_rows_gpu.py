"""fp16 products of a depth up to 80, both operands stored (K, rows), whose many rows are off cache lines: blocks of rows and columns that end
inside the matrix, lines that begin in one block and end in the next, depths of one to three k-steps, operands shared by the batch, the memory around
the output."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck
from util import stream

pytestmark = pytest.mark.gpu

LARGE = 3 << 23         # outputs from which such products have a kernel of their own


def _product(batch, n, m, k, shared=""):
    g = torch.Generator(device="cuda").manual_seed(n * 3 + m + k)
    A = torch.randn((1 if "A" in shared else batch, k, m), generator=g, device="cuda").half()
    B = torch.randn((1 if "B" in shared else batch, k, n), generator=g, device="cuda").half()
    total, front = batch * n * m, 8
    padded = torch.full((total + 2 * front,), float("nan"), dtype=torch.half, device="cuda")
    ck.gemm_fp16(m, k, n, A.size(0), B.size(0), False, True, A.data_ptr(), B.data_ptr(), padded[front:].data_ptr(), stream())
    out = padded[front:front + total].view(batch, n, m)
    assert padded[:front].isnan().all() and padded[front + total:].isnan().all() and not out.isnan().any()
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


@pytest.mark.parametrize("shared", ["A", "B"])
def test_shared_operand(shared):
    _product(110, 500, 500, 64, shared)
