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


# (K, rows) operands: between one and two 128x128 tiles a compute unit (two workgroups share one), more and fewer of them; edges of rows
# that are not whole 16-byte pieces; depths of one slab, several and a rest; one round of large tiles, and large tiles that would leave most
# of a second round idle
@pytest.mark.parametrize("layout", [(True, True), (False, False), (True, False)])
@pytest.mark.parametrize("k", [64, 128, 320, 328])
@pytest.mark.parametrize("shape", [(1280, 1280, 3), (1284, 1156, 3), (384, 384, 50), (384, 388, 60), (640, 640, 12), (260, 260, 30)])
def test_rounds_of_operands_stored_k_first(gpu, shape, k, layout):
    M, N, batch = shape
    aT, bT = layout
    print("k-first rounds", shape, k, layout, flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + k)
    A = torch.randn((batch, k, M) if aT else (batch, M, k), generator=g, device="cuda").half()
    B = torch.randn((batch, N, k) if bT else (batch, k, N), generator=g, device="cuda").half()
    out = torch.full((batch * M * N + 64,), 77.0, device="cuda", dtype=torch.half)
    ck.gemm_fp16(N, k, M, batch, batch, bT, aT, B.data_ptr(), A.data_ptr(), out.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert bool((out[batch * M * N:] == 77.0).all())
    got = out[:batch * M * N].view(batch, M, N)
    for e in (0, batch // 2, batch - 1):
        a, b = (A[e].t() if aT else A[e]).double(), (B[e].t() if bT else B[e]).double()
        want, mag = a @ b, a.abs() @ b.abs()
        bound = mag * k * 2.0 ** -24 + want.abs() * 2.0 ** -11 + 2.0 ** -25      # fp32 sums in any order, one rounding to fp16
        assert bool(((got[e].double() - want).abs() <= bound).all()), e
