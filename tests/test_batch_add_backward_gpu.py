"""Sums over the batch: rows that end inside a piece, fewer columns than a piece, rows dealt to groups of lanes and not, numbers of rows around what is requested at a
time, the size from which they are read past the caches."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck
from util import stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 7, 8, 9, 14, 2046, 2050, 100000, (1 << 20) + 6, (1 << 20) + 8])
@pytest.mark.parametrize("batch", [1, 2, 3, 4, 5, 8, 9, 17, 70])
def test_sums(batch, n):
    _sums(batch, n)


@pytest.mark.parametrize("batch,n", [(16, 1 << 24), (17, (1 << 24) - 8), (17, (1 << 24) - 4)])
def test_beyond_the_cache(batch, n):
    _sums(batch, n)


def _sums(batch, n):
    g = torch.Generator(device="cuda").manual_seed(batch + n)
    x = torch.randn((batch, n), generator=g, device="cuda").half()
    out = torch.full((n + 16,), float("nan"), dtype=torch.half, device="cuda")
    ck.arith_batch_add_backward(batch, n, x.data_ptr(), out[8:].data_ptr(), stream())
    got = out[8:8 + n].double()
    assert out[:8].isnan().all() and out[8 + n:].isnan().all()
    ref, size = x.sum(0, dtype=torch.float64), x.abs().sum(0, dtype=torch.float64)
    # batch additions in fp32, one rounding to fp16
    assert ((got - ref).abs() <= size * batch * 2.0 ** -24 + ref.abs() * 2.0 ** -10.9 + 2.0 ** -25).all()
