"""The one-pass backward of the affine layernorm against float64, at the edges of its tiles and teams."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck

pytestmark = pytest.mark.gpu


# one row, one column; a part's edge (256 rows) on either side; ragged widths; teams of 32 and the taller parts; past a team's reach
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 7, 64), (3, 256, 66), (2, 257, 128), (1, 1030, 61), (4, 1024, 192), (1, 8192, 8), (1, 8200, 72),
                                   (1, 16388, 3)])
@pytest.mark.parametrize("mean", [True, False])
def test_layernorm_backward(gpu, shape, mean):
    b, n, m = shape
    print("layernorm backward", shape, mean, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + m)
    x = (torch.randn(shape, generator=g, device="cuda") + 0.5).half()
    dy = (torch.randn(shape, generator=g, device="cuda") * 0.1).half()
    w = (1 + 0.1 * torch.randn(n, generator=g, device="cuda")).half()
    beta = torch.randn(n, generator=g, device="cuda").half()
    st = torch.cuda.current_stream().cuda_stream
    out, want_out, dx = torch.empty_like(x), torch.empty_like(x), torch.full_like(x, float("nan"))
    stats = torch.full((b, 2, m), float("nan"), device="cuda")
    dw, db = (torch.full((n,), float("nan"), device="cuda", dtype=torch.half) for _ in range(2))
    part = torch.full((b * ((m + 63) // 64), 2, n), float("nan"), device="cuda")
    ck.layernorm_affine_forward_stats(b, n, m, x.data_ptr(), w.data_ptr(), beta.data_ptr() if mean else None, out.data_ptr(), stats.data_ptr(),
                                      1e-5, mean, st)
    ck.layernorm_affine_forward(b, n, m, x.data_ptr(), w.data_ptr(), beta.data_ptr() if mean else None, want_out.data_ptr(), 1e-5, mean, st)
    assert torch.equal(out, want_out)
    ck.layernorm_affine_backward(b, n, m, x.data_ptr(), dy.data_ptr(), w.data_ptr(), stats.data_ptr(), dx.data_ptr(), dw.data_ptr(),
                                 db.data_ptr() if mean else None, part.data_ptr(), st)
    xd, gd, wd = x.double(), dy.double(), w.double()[None, :, None]
    mu = xd.mean(1, keepdim=True) if mean else torch.zeros((b, 1, m), device="cuda", dtype=torch.float64)
    rstd = 1 / torch.sqrt((xd * xd).mean(1, keepdim=True) - mu * mu + 1e-5)
    # fp32 sums in chains of at most n / 4 + 64 terms, each addition off by 2^-24 of the magnitudes; the deviation sees half of the
    # relative error of E[x^2] - mean^2
    chain = (n / 4 + 64) * 2.0 ** -24
    ex2 = (xd * xd).mean(1, keepdim=True)
    assert bool(((stats[:, 0].double() - mu[:, 0]).abs() <= chain * xd.abs().mean(1)).all())
    assert bool(((stats[:, 1].double() - rstd[:, 0]).abs() <= (0.5 * chain * (ex2 + 2 * mu.abs() * xd.abs().mean(1, keepdim=True)) * rstd ** 2 + 2.0 ** -21)[:, 0] * rstd[:, 0]).all())
    rstd, mu = stats[:, 1:].double(), stats[:, :1].double()           # the backward pass starts from these
    xh = (xd - mu) * rstd
    gw = gd * wd
    want = rstd * (gw - (gw.mean(1, keepdim=True) if mean else 0) - xh * (gw * xh).mean(1, keepdim=True))
    # fp32 terms and sums, then one rounding to fp16 (2^-11 relative, 2^-25 where it is subnormal)
    mag = rstd * (gw.abs() + gw.abs().mean(1, keepdim=True) + (1 + mu.abs() * rstd + xh.abs()) * (gw * xh).abs().mean(1, keepdim=True))
    assert bool(((dx.double() - want).abs() <= want.abs() * 2.0 ** -11 + 2.0 ** -24 + chain * mag).all())
    terms = gd * xh
    rows = (b * m / 256 + 64) * 2.0 ** -24          # (64 columns in a tree, the tiles in four chains)
    assert bool(((dw.double() - terms.sum((0, 2))).abs() <= terms.sum((0, 2)).abs() * 2.0 ** -11 + 2.0 ** -24 +
                 rows * (gd.abs() * (xh.abs() + mu.abs() * rstd)).sum((0, 2))).all())
    if mean:
        assert bool(((db.double() - gd.sum((0, 2))).abs() <= gd.sum((0, 2)).abs() * 2.0 ** -11 + 2.0 ** -24 + rows * gd.abs().sum((0, 2))).all())


@pytest.mark.parametrize("shape", [(2, 64, 0), (0, 64, 8)])
@pytest.mark.parametrize("bias", [True, False])
def test_layernorm_of_no_tokens(gpu, shape, bias):
    import cpm_kernels_amd.torch as ct
    print("empty layernorm", shape, bias, flush=True)
    ln = ct.LayerNorm(shape[1], bias=bias).half().cuda()
    x = torch.empty(shape, device="cuda", dtype=torch.half, requires_grad=True)
    out = ln(x)
    assert out.shape == x.shape
    grads = torch.autograd.grad(out, [x, ln.weight] + ([ln.bias] if bias else []), torch.empty_like(out))
    assert grads[0].shape == x.shape and all(bool((g == 0).all()) for g in grads[1:])
