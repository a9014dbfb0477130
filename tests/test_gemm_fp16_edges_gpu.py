"""fp16 products whose output rows are 4j + 2 elements, in all four layouts and at depths of whole slabs and not, against
float64; nothing is written past the output."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("k", [34, 64, 66, 80, 96, 128, 250, 320])
@pytest.mark.parametrize("shape", [(3, 64, 194), (2, 66, 258), (2, 130, 190), (2, 258, 198), (70, 260, 258), (1, 4, 1026)])
def test_rows_of_4j_plus_2(gpu, layout, k, shape):
    aT, bT = layout          # of the launcher: A (k, m) unless aT, B (n, k) unless bT
    batch, n, m = shape
    print("fp16 edges", layout, k, shape, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n * 3 + m + k)
    A = torch.randn((batch, m, k), generator=g, device="cuda").half()
    B = torch.randn((batch, n, k), generator=g, device="cuda").half()
    As, Bs = A if aT else A.transpose(1, 2).contiguous(), B.transpose(1, 2).contiguous() if bT else B
    buf = torch.full((batch * n * m + 64,), 7.0, device="cuda", dtype=torch.half)
    ck.gemm_fp16(m, k, n, batch, batch, aT, bT, As.data_ptr(), Bs.data_ptr(), buf.data_ptr(), torch.cuda.current_stream().cuda_stream)
    out = buf[:batch * n * m].view(batch, n, m).double()
    want = torch.bmm(B.double(), A.double().transpose(1, 2).contiguous())
    mag = torch.bmm(B.double().abs(), A.double().abs().transpose(1, 2).contiguous())
    assert bool((buf[batch * n * m:] == 7.0).all())
    assert bool(((out - want).abs() <= mag * k * 2.0 ** -24 + want.abs() * 2.0 ** -11 + 2.0 ** -25).all()), (layout, k, shape)
