"""Pieces across the end of a row are read with what lies behind it: columns of NaN next to it, in the following row, stay out of the others, also in the last row and in
matrices of less than a piece."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck
from util import stream

pytestmark = pytest.mark.gpu

SIZES = [(1, 2), (1, 6), (2, 2), (3, 4), (1, 10), (2, 12), (50, 70), (100, 100), (130, 66), (300, 30), (240, 236), (500, 500), (520, 20), (1000, 134),
         # tiles with rows nearly throughout (seven eighths) and just not, rows of whole pieces
         (55, 66), (56, 66), (111, 70), (112, 70), (224, 66), (446, 70), (448, 70), (898, 66), (50, 72), (120, 72), (70, 136), (230, 80)]


def _pair(batch, n, m, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((batch, n, m), generator=g, device="cuda").half()
    y = x.clone()
    y[:, :, 0] = float("nan")
    return x, y


def _same(outs, axis):
    for one, two in zip(*outs):
        keep = torch.arange(1, one.size(axis), device="cuda")
        a, b = one.index_select(axis, keep), two.index_select(axis, keep)
        assert torch.equal(a.view(torch.int16) if a.dtype == torch.half else a, b.view(torch.int16) if b.dtype == torch.half else b)
        if one.dtype == torch.half:
            assert not a.isnan().any()


@pytest.mark.parametrize("n,m", SIZES)
def test_softmax_columns(n, m):
    x, y = _pair(3, n, m, n + m)
    grad = _pair(3, n, m, n)[0]
    outs = []
    for v in (x, y):
        out, back = torch.empty_like(v), torch.empty_like(v)
        ck.softmax_forward(3, n, m, v.data_ptr(), out.data_ptr(), stream())
        probs = out.clone()
        probs[:, :, 0] = v[:, :, 0]
        ck.softmax_backward(3, n, m, probs.data_ptr(), grad.data_ptr(), back.data_ptr(), stream())
        outs.append((out, back))
    _same(outs, 2)
    ref = torch.softmax(x.double(), 1)
    assert ((outs[0][0].double() - ref).abs() <= ref * 2.0 ** -10 + 2.0 ** -24).all()


# (from 100 million elements on: the form of lanes for themselves, its rows and columns at the edges of where it is taken)
@pytest.mark.parametrize("n,m", [(257, 300), (330, 501), (384, 310), (386, 500), (448, 700), (450, 640), (512, 388)])
def test_softmax_columns_of_large_batches(n, m):
    batch = -(-(3 << 25) // (n * m)) + 1
    x, y = _pair(batch, n, m, n + m)
    out, out_nan = torch.empty_like(x), torch.empty_like(x)
    for v, o in ((x, out), (y, out_nan)):
        ck.softmax_forward(batch, n, m, v.data_ptr(), o.data_ptr(), stream())
    assert torch.equal(out[:, :, 1:].contiguous().view(torch.int16), out_nan[:, :, 1:].contiguous().view(torch.int16))
    for i in (0, batch // 2, batch - 1):
        ref = torch.softmax(x[i].double(), 0)
        assert ((out[i].double() - ref).abs() <= ref * 2.0 ** -10 + 2.0 ** -24).all()


@pytest.mark.parametrize("n,m", SIZES)
def test_normalised_columns(n, m):
    x, y = _pair(3, n, m, n + m)
    grad = _pair(3, n, m, n)[0]
    outs = []
    for v in (x, y):
        out, back = torch.empty_like(v), torch.empty_like(v)
        mean, var, most = torch.empty((3, 3, m), dtype=torch.half, device="cuda")
        ck.layernorm_forward_mv(3, n, m, v.data_ptr(), out.data_ptr(), mean.data_ptr(), var.data_ptr(), 1e-2, stream())
        ck.layernorm_backward_v(3, n, m, v.data_ptr(), grad.data_ptr(), var.data_ptr(), back.data_ptr(), stream())
        ck.gemm_calc_scale_transpose(3, n, m, v.data_ptr(), most.data_ptr(), stream())
        outs.append((out, back, mean.unsqueeze(1), var.unsqueeze(1), most.unsqueeze(1)))
    _same(outs, 2)
    xd = x.double()
    ref = (xd - xd.mean(1, keepdim=True)) / (xd.var(1, unbiased=False, keepdim=True) + 1e-2).sqrt()
    # (variances as a difference of fp32 sums: 2^-20 of the mean square, of which the smallest here is a hundredth)
    assert ((outs[0][0].double() - ref).abs() <= (ref.abs() + 1) * 2.0 ** -10).all()
    assert torch.equal(outs[0][4].squeeze(1), (x.float().abs().amax(1).double() / 127.0).half())


@pytest.mark.parametrize("n,m", SIZES)
@pytest.mark.parametrize("scaled", [False, True])
def test_quantised_columns(n, m, scaled):
    rows = torch.rand((3, n), device="cuda").half()
    ld = (n + 127) // 128 * 128
    outs = []
    for v in _pair(3, n, m, n * 3 + m):
        scale, out = torch.empty((3, m), dtype=torch.half, device="cuda"), torch.empty((3, m, ld), dtype=torch.int8, device="cuda")
        ck.gemm_quantize_cols_ld(3, n, m, v.data_ptr(), rows.data_ptr() if scaled else None, False, scale.data_ptr(), out.data_ptr(), ld, None, 0, stream())
        outs.append((scale, out))
    _same(outs, 1)
    assert (outs[0][1][:, :, n:] == 0).all()


# (the maximum of a row skips NaN, so it has a row of values of its own in front: what a row's end must not take from the next row)
# (the last one: beyond 48 MB, rows of whole pieces)
@pytest.mark.parametrize("m,n", [(m, 70) for m in (2, 6, 10, 70, 172, 500, 516, 1030, 2044)] + [(520, 24600)])
def test_scaled_rows(m, n):
    ld = (m + 127) // 128 * 128
    x = _pair(2, n, m, m)[0]
    x[:, 1::2] *= 1000.0
    cols = torch.rand((2, m), device="cuda").half() + 0.5
    scale, out = torch.empty((2, n), dtype=torch.half, device="cuda"), torch.empty((2, n, ld), dtype=torch.int8, device="cuda")
    ck.gemm_backward_round_scale_ld(2, n, m, x.data_ptr(), cols.data_ptr(), out.data_ptr(), ld, scale.data_ptr(), False, stream())
    p = x.float() * cols.float()[:, None, :]
    s = (p.abs().amax(2).double() / 127.0).float()
    assert torch.equal(scale, s.half())
    assert torch.equal(out[:, :, :m].float(), torch.round(p / s[:, :, None])) and (out[:, :, m:] == 0).all()


# rows that a wave holds, beside a second matrix of other values
@pytest.mark.parametrize("m", [2, 6, 10, 70, 504, 508, 516, 1030, 1538, 2044, 4090])
def test_quantised_rows(m):
    n, ld = 37, (m + 127) // 128 * 128
    outs = []
    x, y = _pair(1, n, m, m)
    other = torch.full((n, m), float("inf"), device="cuda").half()
    for v in (x, y):
        scale, out = torch.empty((2, n), dtype=torch.half, device="cuda"), torch.empty((2, n, ld), dtype=torch.int8, device="cuda")
        ck.gemm_quantize_pair_ld(n, v.data_ptr(), scale[0].data_ptr(), out[0].data_ptr(), n, other.data_ptr(), scale[1].data_ptr(), out[1].data_ptr(), m, ld, stream())
        outs.append((scale, out))
    s = (x[0].float().abs().amax(1).double() / 127.0).half()
    assert torch.equal(outs[0][0][0], s)
    assert torch.equal(outs[0][1][0, :, :m].float(), torch.round(x[0].float() / s.float()[:, None])) and (outs[0][1][0, :, m:] == 0).all()
    skipped = (x[0, :, 1:].float().abs().amax(1).double() / 127.0).half() if m > 1 else s
    assert torch.equal(outs[1][0][0], skipped) and (outs[1][1][0, :, m:] == 0).all()


# many ragged sequences: lanes that work for themselves
@pytest.mark.parametrize("batch,n,m", [(1024, 386, 266), (420, 512, 470), (400, 500, 502), (1540, 450, 146)])
def test_softmax_of_many_sequences(batch, n, m):
    x = _pair(batch, n, m, batch)[0]
    out = torch.empty_like(x)
    ck.softmax_forward(batch, n, m, x.data_ptr(), out.data_ptr(), stream())
    for i in (0, 1, batch // 2, batch - 1):
        ref = torch.softmax(x[i].double(), 0)
        assert ((out[i].double() - ref).abs() <= ref * 2.0 ** -10 + 2.0 ** -24).all()
