"""fp16 products whose depth is not whole slabs, beside operands stored either way: every kind of remainder, fewer slabs than ring
stages, one tile and several tiles a workgroup, and infinities just before and just behind the end of the depth."""
import pytest
import torch

import cpm_kernels_amd.torch as ct

pytestmark = pytest.mark.gpu


# (batch, rows, columns): 64-row tiles; tiles moved inside the matrix; more tiles than compute units
@pytest.mark.parametrize("shape", [(2, 64, 256), (3, 50, 260), (2, 130, 140), (600, 64, 300), (2, 300, 520), (40, 264, 770)])
@pytest.mark.parametrize("k", [66, 70, 72, 100, 126, 130, 190, 200])
@pytest.mark.parametrize("a_t", [False, True])
@pytest.mark.parametrize("b_t", [False, True])
def test_rest_of_the_depth(gpu, shape, k, a_t, b_t):
    b, m, n = shape
    print("rest of the depth", shape, k, a_t, b_t, flush=True)
    g = torch.Generator(device="cuda").manual_seed(k + m)
    x = torch.randn((b, k, m) if a_t else (b, m, k), generator=g, device="cuda").half()
    y = torch.randn((b, n, k) if b_t else (b, k, n), generator=g, device="cuda").half()
    xd, yd = (x.transpose(1, 2) if a_t else x), (y.transpose(1, 2) if b_t else y)
    with torch.no_grad():
        out = ct.bmm(x, a_t, y, b_t, int8=False)
        want = torch.matmul(xd.double().contiguous(), yd.double().contiguous())
        size = torch.matmul(xd.double().abs().contiguous(), yd.double().abs().contiguous())
        # one rounding to fp16, and fp32 sums of k products, each addition off by at most 2^-23 of the magnitudes
        assert bool(((out.double() - want).abs() <= want.abs() * 2.0 ** -11 + size * k * 2.0 ** -23 + 2.0 ** -25).all())
        # the second entry starts with infinities: the first one's depth ends before them
        xd[1, 0, 0] = float("inf")
        yd[1, 0, 0] = float("inf")
        again = ct.bmm(x, a_t, y, b_t, int8=False)
        assert torch.equal(again[0], out[0])
        # an infinity at the very end of the depth counts once, and multiplies no zero behind it
        yd[0, k - 1, 5] = float("inf")
        last = ct.bmm(x, a_t, y, b_t, int8=False)[0, :, 5].double()
        inf = xd[0, :, k - 1].double() * float("inf")
        assert torch.equal(torch.nan_to_num(last, nan=7.0), torch.nan_to_num(inf, nan=7.0))
