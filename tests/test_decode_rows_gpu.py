"""The decode step's row kernels where they hold a row in registers: widths around every register count and off 16-byte pieces,
rows that start anywhere, one row and more rows than workgroups of one wave are used for."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck

pytestmark = pytest.mark.gpu

WIDTHS = [1, 7, 8, 9, 511, 512, 513, 1000, 1025, 2047, 2048, 2049, 4096, 4104, 8192, 8200]


def _rows(rows, n, shift, seed):
    x = (torch.randn((rows, n), generator=torch.Generator().manual_seed(seed)) * 3).half().cuda()
    buf = torch.full((rows * n + 16,), 7.0, dtype=torch.half, device="cuda")
    buf[shift:shift + rows * n] = x.view(-1)
    return x.double(), buf, buf[shift:shift + rows * n].view(rows, n)


@pytest.mark.parametrize("n", WIDTHS)
@pytest.mark.parametrize("rows,shift", [(1, 0), (5, 1), (2100, 0)])
def test_softmax_rows(gpu, n, rows, shift):
    print("softmax rows", rows, n, shift, flush=True)
    x, buf, view = _rows(rows, n, shift, n)
    if rows > 2:
        view[1] = x[1] = -float("inf")
        view[2, n // 2:] = -float("inf")
        x[2, n // 2:] = -float("inf")
    ck.softmax_step_inplace(rows, n, view.data_ptr(), torch.cuda.current_stream().cuda_stream)
    top = x.amax(1, keepdim=True).clamp(min=-1e6)
    e = torch.exp(x - top)
    want = e / (e.sum(1, keepdim=True) + 1e-10)
    # one rounding to fp16 (2^-11, 2^-25 below its normal range); the exponent's argument x log2(e) - M log2(e) off by 2^-23 of |M| log2(e) <= 2^5
    assert bool(((view.double() - want).abs() <= want * (2.0 ** -11 + 2.0 ** -17) + 2.0 ** -25).all())
    assert bool((buf[:shift] == 7).all()) and bool((buf[shift + rows * n:] == 7).all())


@pytest.mark.parametrize("n", WIDTHS)
@pytest.mark.parametrize("rows,shift,mean", [(1, 0, True), (5, 1, False), (40, 0, False), (40, 8, True)])
def test_layernorm_rows(gpu, n, rows, shift, mean):
    print("layernorm rows", rows, n, shift, mean, flush=True)
    x, buf, view = _rows(rows, n, shift, n + 1)
    ck.layernorm_step_inplace(rows, n, view.data_ptr(), 1e-3, mean, torch.cuda.current_stream().cuda_stream)
    ex2, mu = (x * x).mean(1, keepdim=True), x.mean(1, keepdim=True) * mean
    rstd = 1 / torch.sqrt(ex2 - mu * mu + 1e-3)
    want = (x - mu) * rstd
    # fp32 sums in chains of at most n / 256 + 16 additions, relative to E[x^2] and E|x|; then one rounding to fp16
    chain = (n / 256 + 16) * 2.0 ** -24
    rel = 0.5 * chain * (ex2 + 2 * mu.abs() * x.abs().mean(1, keepdim=True)) * rstd ** 2 + 2.0 ** -21
    bound = want.abs() * (2.0 ** -11 + rel) + chain * x.abs().mean(1, keepdim=True) * rstd + 2.0 ** -25
    assert bool(((view.double() - want).abs() <= bound).all())
    assert bool((buf[:shift] == 7).all()) and bool((buf[shift + rows * n:] == 7).all())


@pytest.mark.parametrize("keys,heads,pos", [(1, 1, 0), (300, 3, 299), (70, 65537, 20)])
@pytest.mark.parametrize("bidirectional", [True, False])
def test_position_step(gpu, keys, heads, pos, bidirectional):
    print("position step", keys, heads, pos, bidirectional, flush=True)
    st = torch.cuda.current_stream().cuda_stream
    mapping = torch.empty(128, dtype=torch.int32, device="cuda")
    ck.position_embedding_init(32, 128, mapping.data_ptr(), bidirectional, st)
    table = torch.randn((heads, 32), generator=torch.Generator().manual_seed(keys)).half().cuda()
    out = torch.empty((heads, keys), dtype=torch.half, device="cuda")
    ck.position_embedding_step(pos, keys, 32, 128, heads, mapping.data_ptr(), table.data_ptr(), out.data_ptr(), bidirectional, st)
    rel = pos - torch.arange(keys, device="cuda")
    below = (rel < 0).long() * (16 if bidirectional else 0)
    rel = torch.where(rel < 0, -rel if bidirectional else torch.zeros_like(rel), rel).clamp(max=127)
    assert torch.equal(out, table[:, mapping[rel].long() + below])
