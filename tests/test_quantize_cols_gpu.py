"""The column quantiser's two ways of rounding: what sends a tile of 64 columns to the longer one, and what that may cost."""
import numpy as np
import pytest
import torch

import cpm_kernels_amd.kernels as ck
import oracle
from oracle import training as ot
from util import assert_bits_equal, quickest, to_gpu, to_np

pytestmark = pytest.mark.gpu


def _quantise(x, row_scale=None):
    b, n, m = x.shape
    s = torch.full((b, m), -1.0, dtype=torch.half, device=x.device)
    q = torch.full((b, m, n), 77, dtype=torch.int8, device=x.device)

    def call():
        ck.gemm_quantize_cols_ld(b, n, m, x.data_ptr(), None if row_scale is None else row_scale.data_ptr(), False, s.data_ptr(),
                                 q.data_ptr(), n, None, 0, torch.cuda.current_stream().cuda_stream)
    return call, s, q


@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("n", [512, 1536])
def test_empty_columns(gpu, n, scaled):
    """Columns of zeros, of negative zeros, of zeros and NaN and of nothing but NaN beside ordinary ones: scale 0, all 0."""
    g = torch.Generator(device=gpu).manual_seed(n)
    x = torch.randn((2, n, 128), generator=g, device=gpu).half()
    rs = (torch.rand((2, n), generator=g, device=gpu) + 0.5).half() if scaled else None
    ordinary, s_ordinary, q_ordinary = _quantise(x, rs)
    ordinary()
    y = x.clone()
    y[:, :, 1] = 0
    y[:, :, 20] = -0.0
    y[:, :, 63] = 0
    y[:, n // 2:, 63] = float("nan")
    y[:, :, 64] = float("nan")
    y[:, 5, 70] = float("nan")         # an ordinary column with a NaN element
    call, s, q = _quantise(y, rs)
    call()
    empty = [1, 20, 63, 64]
    assert (s[:, empty] == 0).all() and (q[:, empty] == 0).all()
    rest = [i for i in range(128) if i not in empty + [70]]
    assert torch.equal(s[:, rest], s_ordinary[:, rest]) and torch.equal(q[:, rest], q_ordinary[:, rest])
    assert (q[:, 70, 5] == 0).all()


@pytest.mark.parametrize("scaled", [False, True])
def test_empty_columns_cost_nothing(gpu, scaled):
    """A padded token in every tile: 23.7 us against 15.7 (25.0 against 18.7 with row scales) when such a column sent its tile through
    the longer rounding, 16.0 and 18.5 now.  The bound lies between, well over what two runs of the same call differ by (1 %)."""
    b, n, m = 8, 4096, 512
    x = torch.randn((b, n, m), device=gpu).half()
    y = x.clone()
    y[:, :, ::64] = 0
    rs = (torch.rand((b, n), device=gpu) + 0.5).half() if scaled else None
    t = quickest([_quantise(x, rs)[0], _quantise(y, rs)[0]])
    print("ordinary %.1f us, with empty columns %.1f us" % tuple(t), flush=True)
    assert t[1] <= 1.15 * t[0], t


@pytest.mark.parametrize("n", [40, 1030])
def test_every_scale_below_the_normal_numbers(gpu, n):
    """One column for each largest magnitude whose scale is subnormal or 0, one with an infinity among them: the oracle's divisions."""
    rng = np.random.default_rng(n)
    top = np.arange(1, 8192, dtype=np.uint16)          # up to 127 * 2^-14 and a little more
    x = (rng.integers(0, 65536, (1, n, top.size)) % (top.astype(np.int64) + 1)).astype(np.uint16)
    x[0, 0] = top
    x |= (rng.integers(0, 2, x.shape) << 15).astype(np.uint16)
    x = x.view(np.float16)
    x[0, n // 2, 77] = np.inf
    d = to_gpu(x)
    want = oracle.gemm_calc_scale_transpose(x)
    q_want = oracle.gemm_round_transpose(x, want)
    for tr in (False, True):
        s2 = torch.full((1, top.size), -1.0, dtype=torch.half, device=gpu)
        q2 = torch.full((1, top.size, n) if tr else x.shape, 77, dtype=torch.int8, device=gpu)
        ck.gemm_quantize_cols(1, n, top.size, d.data_ptr(), s2.data_ptr(), q2.data_ptr(), tr, torch.cuda.current_stream().cuda_stream)
        assert_bits_equal(to_np(s2), want, "scales")
        assert_bits_equal(to_np(q2), np.ascontiguousarray(q_want.transpose(0, 2, 1)) if tr else q_want, "int8 (transposed=%s)" % tr)


def test_scales_below_the_normal_numbers_cost_little(gpu):
    """One such column in every tile: 23.9 us against 15.7 when the longer rounding divided element by element, 18.7 through the reciprocal."""
    b, n, m = 8, 4096, 512
    x = torch.randn((b, n, m), device=gpu).half()
    y = x.clone()
    y[:, :, ::64] *= 1e-4
    t = quickest([_quantise(x)[0], _quantise(y)[0]])
    print("ordinary %.1f us, with columns of a subnormal scale %.1f us" % tuple(t), flush=True)
    assert t[1] <= 1.3 * t[0], t


@pytest.mark.parametrize("n", [40, 512, 1030, 16384])
@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("m", [128, 100])
def test_short_rounding_of_whole_tiles(gpu, n, scaled, m):
    """Tiles in which every column has a normal scale, so that all of them take the shorter rounding: exact ties between all neighbouring
    integers, the largest magnitudes of either sign, quiet and signalling NaN.  One part of a team and several, both output layouts."""
    rng = np.random.default_rng(n + m)
    x = rng.standard_normal((1, n, m)).astype(np.float16)
    for c in range(0, m, 3):       # scale 2^e exactly: k + 1/2 of it is a tie
        e = np.float16(2.0 ** rng.integers(-4, 6))
        x[0, :, c] = ((np.arange(n) * 7 % 252 - 126) + 0.5).astype(np.float16) * e
        x[0, rng.integers(n), c] = np.float16(127) * e * (-1) ** c
    for c in range(1, m, 3):
        x[0, rng.integers(n), c] = np.float16(-60000 if c % 2 else 60000)
    bits = x.view(np.uint16)
    for c in range(2, m, 3):
        bits[0, rng.integers(n), c] = (0x7e00, 0x7c01, 0xfe01, 0xfdff)[c % 4]
    rs = np.ones((1, n), np.float16) * np.float16(0.5) if scaled else None
    clean = np.where(np.isnan(x.astype(np.float32)), np.float16(0), x)         # a NaN element takes no part in the maximum and rounds to 0
    if scaled:
        want_q, want = ot.gemm_backward_scale_round(clean, rs, False)
    else:
        want = oracle.gemm_calc_scale_transpose(clean)
        want_q = oracle.gemm_round_transpose(clean, want)
    assert (want >= np.float16(2.0 ** -14)).all()
    d = to_gpu(x)
    drs = to_gpu(rs) if scaled else None
    ld = (n + 15) // 16 * 16
    s = torch.full((1, m), -1.0, dtype=torch.half, device=gpu)
    qt = torch.full((1, m, ld), 77, dtype=torch.int8, device=gpu)
    qn = torch.full((1, n, m), 77, dtype=torch.int8, device=gpu)
    for t, nat in ((True, False), (False, True)) if scaled else ((True, True), (True, False), (False, True)):
        s.fill_(-1); qt.fill_(77); qn.fill_(77)
        ck.gemm_quantize_cols_ld(1, n, m, d.data_ptr(), drs.data_ptr() if scaled else None, False, s.data_ptr(), qt.data_ptr() if t else None,
                                 ld if t else 0, qn.data_ptr() if nat else None, m if nat else 0, torch.cuda.current_stream().cuda_stream)
        assert_bits_equal(to_np(s), want, "scales")
        if t:
            assert_bits_equal(to_np(qt)[:, :, :n], np.ascontiguousarray(want_q.transpose(0, 2, 1)), "transposed")
        if nat:
            assert_bits_equal(to_np(qn), want_q, "in place")
