"""The batch_* elementwise ops at sizes where a thread takes several rows (rows 2, 3 and more, remainders, any width and
alignment), bit for bit against numpy's fp16 arithmetic; in place too."""
import numpy as np
import pytest
import torch

import cpm_kernels_amd.kernels as ck
from util import assert_bits_equal, rand_half, to_gpu, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 9])
@pytest.mark.parametrize("cols", [16384 * 512, 16384 * 512 + 6])
@pytest.mark.parametrize("shift", [0, 1])
def test_batch_add_and_multiply(gpu, rows, cols, shift):
    print("batch rows", rows, cols, shift, flush=True)
    rng = np.random.default_rng(cols + rows)
    x, a, b = rand_half(rng, (rows, cols)), rand_half(rng, cols), rand_half(rng, cols)
    st = torch.cuda.current_stream().cuda_stream
    dx = torch.empty(rows * cols + 8, dtype=torch.half, device="cuda")[shift:shift + rows * cols].view(rows, cols)
    dx.copy_(to_gpu(x))
    da, db, out = to_gpu(a), to_gpu(b), torch.zeros_like(dx)
    ck.arith_batch_mul(rows, cols, dx.data_ptr(), da.data_ptr(), out.data_ptr(), st)
    assert_bits_equal(to_np(out), x * a[None], "mul")
    ck.arith_batch_add_forward(rows, cols, dx.data_ptr(), db.data_ptr(), dx.data_ptr(), st)
    assert_bits_equal(to_np(dx), x + b[None], "add in place")
