"""Results stored for the next kernel to find in the last-level cache, at both ends of the range of sizes that rule takes."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck
from util import stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(10, 4096, 1024), (9, 4096, 1024), (80, 1024, 512), (40, 1000, 1088), (20, 4096, 1024), (21, 4096, 1024)])
@pytest.mark.parametrize("bias", [True, False])
def test_layernorm(gpu, shape, bias):
    """The fused form against the norm (which never keeps its result) followed by the affine kernel, bit for bit."""
    b, n, m = shape
    print("kept layernorm", shape, bias, flush=True)
    g = torch.Generator(device=gpu).manual_seed(n)
    x = torch.randn(shape, generator=g, device=gpu).half()
    gamma, beta = (1 + 0.1 * torch.randn(n, generator=g, device=gpu)).half(), (0.1 * torch.randn(n, generator=g, device=gpu)).half()
    two, one = torch.full_like(x, 77.0), torch.full_like(x, 77.0)
    ck.layernorm_forward(b, n, m, x.data_ptr(), two.data_ptr(), 1e-5, bias, stream())
    if bias:
        ck.arith_ln_mul_add(b, n, m, two.data_ptr(), gamma.data_ptr(), beta.data_ptr(), two.data_ptr(), stream())
    else:
        ck.arith_ln_mul(b, n, m, two.data_ptr(), gamma.data_ptr(), two.data_ptr(), stream())
    ck.layernorm_affine_forward(b, n, m, x.data_ptr(), gamma.data_ptr(), beta.data_ptr() if bias else None, one.data_ptr(), 1e-5, bias, stream())
    assert torch.equal(one, two)


@pytest.mark.parametrize("total", [3 << 20, (3 << 20) + 8, (24 << 20) - 8, 24 << 20, (24 << 20) + 5, 44 << 20, (44 << 20) + 3])
@pytest.mark.parametrize("shift", [0, 1])
def test_gelu(gpu, total, shift):
    """One call against pieces of another choice, bit for bit; off 16-byte boundaries too."""
    print("kept gelu", total, shift, flush=True)
    g = torch.Generator(device=gpu).manual_seed(total)
    x = torch.randn(total + 8, generator=g, device=gpu).half()[shift:shift + total]
    out, pieces = torch.full((total + 16,), 77.0, dtype=torch.half, device=gpu), torch.empty(total, dtype=torch.half, device=gpu)
    ck.gelu_forward(1, total, x.data_ptr(), out[shift:].data_ptr(), stream())
    step = 1 << (22 if total > 1 << 24 else 20)
    for i in range(0, total, step):
        ck.gelu_forward(1, min(step, total - i), x[i:].data_ptr(), pieces[i:].data_ptr(), stream())
    assert torch.equal(out[shift:shift + total], pieces)
    assert bool((out[shift + total:] == 77.0).all())
