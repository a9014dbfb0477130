"""Products summed over the batch (cpmk_gemm_int8_scale_sum, cpmk_gemm_fp16_sum) against float64, at the sizes where their
tiles, slabs and groups change."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck

pytestmark = pytest.mark.gpu

# batch, groups, n, m, k: one entry; partial tiles; one slab per entry; several groups; 16 entries; 256x128 tiles (the last three)
SHAPES = [(1, 1, 4, 4, 128), (3, 1, 132, 260, 128), (4, 2, 128, 128, 256), (16, 1, 36, 200, 384), (6, 3, 300, 124, 640),
          (2, 1, 4100, 2052, 128), (5, 1, 3080, 3072, 256), (8, 4, 1024, 1028, 512)]


def _st():
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("shape", SHAPES)
def test_int8_sum(gpu, shape):
    batch, groups, n, m, k = shape
    print("int8 sum", shape, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n * 7 + m + k)
    A = torch.randint(-128, 128, (batch, m, k), generator=g, device="cuda", dtype=torch.int8)
    B = torch.randint(-128, 128, (batch, n, k), generator=g, device="cuda", dtype=torch.int8)
    s = (torch.rand((batch, n), generator=g, device="cuda") * 1e-3 + 1e-4).half()
    out = torch.full((groups, n, m), float("nan"), device="cuda", dtype=torch.half)
    ck.gemm_int8_scale_sum(m, k, n, batch, groups, A.data_ptr(), B.data_ptr(), s.data_ptr(), out.data_ptr(), _st())
    for q in range(groups):
        want = torch.zeros((n, m), device="cuda", dtype=torch.float64)
        mag = torch.zeros_like(want)
        for e in range(q * batch // groups, (q + 1) * batch // groups):
            acc = (B[e].double() @ A[e].double().t()) * s[e].double()[:, None]      # exact integers (|acc| < 2^53) times the scale
            want += acc
            mag += acc.abs()
        # one fp32 rounding per entry (the fused multiply-add) and one of the conversion of a 24-bit integer, then one to fp16
        bound = mag * (batch + 1) * 2.0 ** -24 + want.abs() * 2.0 ** -11 + 2.0 ** -25
        assert bool(((out[q].double() - want).abs() <= bound).all()), shape


@pytest.mark.parametrize("k", [34, 64, 66, 72, 96, 128, 320, 500])
@pytest.mark.parametrize("shape", [(1, 1, 4, 4), (4, 2, 132, 260), (3, 1, 128, 512), (2, 1, 3588, 3584)])
def test_fp16_sum(gpu, shape, k):
    batch, groups, n, m = shape
    print("fp16 sum", shape, k, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n * 7 + m + k)
    A = torch.randn((batch, m, k), generator=g, device="cuda").half()
    B = torch.randn((batch, n, k), generator=g, device="cuda").half()
    out = torch.full((groups, n, m), float("nan"), device="cuda", dtype=torch.half)
    ck.gemm_fp16_sum(m, k, n, batch, groups, A.data_ptr(), B.data_ptr(), out.data_ptr(), _st())
    per = batch // groups
    for q in range(groups):
        want = torch.zeros((n, m), device="cuda", dtype=torch.float64)
        mag = torch.zeros_like(want)
        for e in range(q * per, (q + 1) * per):
            want += B[e].double() @ A[e].double().t()
            mag += B[e].double().abs() @ A[e].double().abs().t()
        bound = mag * (per * k) * 2.0 ** -24 + want.abs() * 2.0 ** -11 + 2.0 ** -25      # fp32 sums in any order, one rounding to fp16
        assert bool(((out[q].double() - want).abs() <= bound).all()), (shape, k)


def test_groups(gpu):
    for m, n, batch in ((4, 4, 1), (512, 512, 8), (4096, 10240, 8), (4096, 4096, 13), (64, 64, 7), (8192, 8192, 64)):
        groups = ck.gemm_sum_groups(m, n, batch)
        assert 1 <= groups <= batch and batch % groups == 0 and (groups == batch or batch // groups <= 16)
