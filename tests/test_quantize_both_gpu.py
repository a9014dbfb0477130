"""The two operands of a product quantised in one launch, one along its columns and one along its rows, against a launch for each."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck
from util import stream

pytestmark = pytest.mark.gpu


def _ld(k):
    return (k + 127) // 128 * 128


# (depths around what a wave's and a workgroup's lanes hold, of one part and of several; K % 8 != 0 takes two launches)
@pytest.mark.parametrize("k", [8, 504, 512, 1032, 2056, 4096, 4104, 8200, 12296, 16384, 1028])
@pytest.mark.parametrize("batch,m,rows,both", [(1, 4, 1, False), (3, 72, 9, True), (2, 500, 700, False), (2, 128, 257, True)])
def test_one_launch_equals_two(k, batch, m, rows, both):
    g = torch.Generator(device="cuda").manual_seed(k + m)
    x = torch.randn((batch, k, m), generator=g, device="cuda").half()
    w = torch.randn((rows, k), generator=g, device="cuda").half()
    x[0, :, 0] = 0.0
    x[-1, 3, m - 1], w[0, 2] = float("nan"), float("nan")
    w[rows // 2] = 0.0
    w[rows - 1] = 3e-8                                   # (a subnormal scale)
    ld, ld_n = _ld(k), _ld(m)
    outs = []
    for joint in (False, True):
        scale = torch.full((batch, m), 7.0, dtype=torch.half, device="cuda")
        out_t = torch.full((batch, m, ld), 77, dtype=torch.int8, device="cuda")
        out_n = torch.full((batch, k, ld_n), 77, dtype=torch.int8, device="cuda")
        row_scale = torch.full((rows,), 7.0, dtype=torch.half, device="cuda")
        row_out = torch.full((rows, ld), 77, dtype=torch.int8, device="cuda")
        n_ptr = out_n.data_ptr() if both else None
        if joint:
            ck.gemm_quantize_cols_rows(batch, k, m, x.data_ptr(), scale.data_ptr(), out_t.data_ptr(), ld, n_ptr, ld_n if both else 0,
                                       rows, w.data_ptr(), row_scale.data_ptr(), row_out.data_ptr(), stream())
        else:
            ck.gemm_quantize_cols_ld(batch, k, m, x.data_ptr(), None, False, scale.data_ptr(), out_t.data_ptr(), ld, n_ptr, ld_n if both else 0, stream())
            ck.gemm_quantize_pair_ld(rows, w.data_ptr(), row_scale.data_ptr(), row_out.data_ptr(), 0, None, None, None, k, ld, stream())
        outs.append((scale.view(torch.int16), out_t, out_n, row_scale.view(torch.int16), row_out))
    for one, two in zip(*outs):
        assert torch.equal(one, two)


# (rows of one to four pieces a lane and beyond them, of whole pieces or not; columns of one part and of several; scales shared by the batch or not)
@pytest.mark.parametrize("m", [4, 72, 500, 512, 516, 1024, 1500, 2048, 2052, 2056])
@pytest.mark.parametrize("batch,n,bc_row,bc_col", [(1, 4, True, True), (3, 70, True, False), (2, 516, False, True), (2, 1200, False, False)])
def test_gradient_in_one_launch_equals_two(m, batch, n, bc_row, bc_col):
    g = torch.Generator(device="cuda").manual_seed(m + n)
    x = torch.randn((batch, n, m), generator=g, device="cuda").half()
    rs = (torch.rand((1 if bc_row else batch, n), generator=g, device="cuda") * 0.1).half()
    cs = (torch.rand((1 if bc_col else batch, m), generator=g, device="cuda") * 0.1).half()
    x[0, 1], x[-1, :, 2] = 0.0, 0.0
    x[0, 0, 1] = float("nan")
    x[-1, 3] *= 1e-4
    ld, ld_t = _ld(m), _ld(n)
    outs = []
    for joint in (False, True):
        scale = torch.full((batch, m), 7.0, dtype=torch.half, device="cuda")
        out_t = torch.full((batch, m, ld_t), 77, dtype=torch.int8, device="cuda")
        row_scale = torch.full((batch, n), 7.0, dtype=torch.half, device="cuda")
        out = torch.full((batch, n, ld), 77, dtype=torch.int8, device="cuda")
        if joint:
            ck.gemm_backward_quantize_both(batch, n, m, x.data_ptr(), rs.data_ptr(), bc_row, scale.data_ptr(), out_t.data_ptr(), ld_t,
                                           cs.data_ptr(), bc_col, out.data_ptr(), ld, row_scale.data_ptr(), stream())
        else:
            ck.gemm_quantize_cols_ld(batch, n, m, x.data_ptr(), rs.data_ptr(), bc_row, scale.data_ptr(), out_t.data_ptr(), ld_t, None, 0, stream())
            ck.gemm_backward_round_scale_ld(batch, n, m, x.data_ptr(), cs.data_ptr(), out.data_ptr(), ld, row_scale.data_ptr(), bc_col, stream())
        outs.append((scale.view(torch.int16), out_t, row_scale.view(torch.int16), out))
    for one, two in zip(*outs):
        assert torch.equal(one, two)
