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
