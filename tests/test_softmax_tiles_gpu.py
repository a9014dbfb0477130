"""Softmax over dim 1 on the tile kernels: each form of a tile (rows on cache lines, on 16-byte pieces, anywhere), heights at both sides of
where it changes, and numbers of tiles at both sides of what the device holds at once."""
import pytest
import torch

import cpm_kernels_amd.torch as ct

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,n,m", [
    (2, 256, 100), (2, 257, 100), (3, 512, 65), (2, 513, 66), (130, 300, 500), (2, 1, 70),
    (2, 257, 72), (64, 300, 504), (65, 300, 504), (65, 512, 504), (520, 257, 72), (65, 256, 504),
    (2, 300, 128), (3, 512, 192), (300, 257, 128),
    # both sides of the last-level cache's line, where lanes work for themselves beyond it
    (915, 200, 504), (916, 200, 504), (1135, 161, 505), (205, 225, 2001), (180, 257, 2002), (144, 320, 2001), (716, 256, 504),
])
def test_softmax_tiles(batch, n, m):
    g = torch.Generator(device="cuda").manual_seed(batch * 7 + n + m)
    x = (torch.randn((batch, n, m), generator=g, device="cuda") * 4).half()
    if n > 1:
        x[:, n - n // 4:, :] = float("-inf")        # whole rows masked out
        x[:, :, 3] = float("-inf")                  # a column of nothing but -inf: zeros
        x[0, n // 2, 5] = float("nan")
        x[0, 0, 6] = 60000.0
    out = ct.softmax(x)
    inplace = x.clone()
    ct.softmax_inplace(inplace)
    xd = x.double()
    top = xd.amax(1, keepdim=True).clamp(min=-1e6)
    e = torch.exp(xd - top)
    ref = e / (e.sum(1, keepdim=True) + 1e-10)
    if n > 1:
        assert torch.isnan(out[0, :, 5]).all()
        ref[0, :, 5] = 0
        out[0, :, 5] = 0
        assert (out[:, :, 3] == 0).all()
    # one rounding to fp16 (2^-11, or half a subnormal step), exponents of up to 40 that differ from one another in fp32 and n additions in fp32
    bound = ref * (2.0 ** -11 + 40 * 2.0 ** -23 + n * 2.0 ** -24) + 2.0 ** -25
    assert ((out.double() - ref).abs() <= bound).all()
    if n > 1:
        inplace[0, :, 5] = 0
    assert torch.equal(inplace, out)
