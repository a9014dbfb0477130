"""Products with a dimension of size zero: an empty result, or zeros where nothing is summed, and gradients of the same kind."""
import pytest
import torch

import cpm_kernels_amd.torch as ct

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("int8", [True, False])
@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("batches", [(1, 3), (2, 2), (3, 1)])
@pytest.mark.parametrize("sizes", [(64, 128, 0), (0, 128, 64), (128, 0, 64), (0, 0, 64), (0, 128, 0)])       # M, K, N
def test_empty_product(gpu, sizes, batches, layout, int8):
    M, K, N = sizes
    aT, bT = layout
    print("empty product", sizes, batches, layout, int8, flush=True)
    A = torch.randn((batches[0],) + ((K, M) if aT else (M, K)), device=gpu).half().requires_grad_()
    B = torch.randn((batches[1],) + ((N, K) if bT else (K, N)), device=gpu).half().requires_grad_()
    # memory that a forgotten result would be taken from
    poison = [torch.full((n,), float("nan"), device=gpu, dtype=torch.half) for n in (64, 256, 1024, 8192, 32768)]
    del poison
    out = ct.bmm(A, aT, B, bT, int8=int8)
    assert out.shape == (max(batches), M, N) and bool((out == 0).all())
    grads = torch.autograd.grad(out, [A, B], torch.randn_like(out))
    for x, g in zip((A, B), grads):
        assert g.shape == x.shape and g.dtype == torch.half and bool((g == 0).all())
