"""The quantisers with padded rows (`_ld` launchers) against the oracle, at the edges of their tiles, teams and register
rows; the surplus bytes must be zero whatever the buffer held."""
import numpy as np
import pytest
import torch

import cpm_kernels_amd.kernels as ck
import oracle
from oracle import training as ot
from util import assert_bits_equal, rand_half, to_gpu, to_np

pytestmark = pytest.mark.gpu


def _st():
    return torch.cuda.current_stream().cuda_stream


def _up(k, to):
    return (k + to - 1) // to * to


def _pad(q, ld):
    return np.pad(q, [(0, 0)] * (q.ndim - 1) + [(0, ld - q.shape[-1])])


# rows held by a wave (up to 4096 columns), by a workgroup (up to 16384), pieces across the end, no surplus
@pytest.mark.parametrize("m", [1, 4, 100, 128, 500, 2052, 4096, 4100, 6148, 8196, 10240, 12001, 16384])
@pytest.mark.parametrize("rows", [(1, 0), (5, 3), (0, 7)])
def test_rows(gpu, m, rows):
    print("rows", m, rows, flush=True)
    rng = np.random.default_rng(m)
    ld = _up(m, 128) if m % 2 or m % 128 else m
    mats = [rand_half(rng, (max(r, 1), m)) for r in rows]
    mats[0][0, :] = 0                                   # a row of zeros, a NaN element, a subnormal scale
    mats[1][-1, m // 2] = np.nan
    mats[0][-1] *= np.float16(1e-6) if rows[0] > 1 else np.float16(1)
    d = [to_gpu(x) for x in mats]
    s = [torch.full((max(r, 1),), -1.0, dtype=torch.half, device="cuda") for r in rows]
    q = [torch.full((max(r, 1), ld), 77, dtype=torch.int8, device="cuda") for r in rows]
    ck.gemm_quantize_pair_ld(rows[0], d[0].data_ptr(), s[0].data_ptr(), q[0].data_ptr(), rows[1], d[1].data_ptr(), s[1].data_ptr(),
                             q[1].data_ptr(), m, ld, _st())
    for i in (0, 1):
        if rows[i]:
            want = oracle.gemm_calc_scale(mats[i][None])
            assert_bits_equal(to_np(s[i]), want[0], "scale")
            assert_bits_equal(to_np(q[i]), _pad(oracle.gemm_round(mats[i][None], want), ld)[0], "rows")


@pytest.mark.parametrize("shape", [(2, 1, 4), (1, 7, 60), (3, 8, 64), (1, 500, 100), (2, 513, 129), (1, 1030, 72), (1, 4096, 128), (1, 16400, 3)])
@pytest.mark.parametrize("form", ["t", "n", "both", "t scaled", "n scaled", "t shared"])
def test_cols(gpu, shape, form):
    b, n, m = shape
    print("cols", shape, form, flush=True)
    rng = np.random.default_rng(n + m)
    mat = rand_half(rng, shape)
    mat[0, :, 0] = 0
    want_t, want_n = form[0] in "tb", form[0] in "nb"
    ld_t, ld_n = _up(n, 128), _up(m, 128)
    scaled = "scaled" in form or "shared" in form
    sx = np.abs(rand_half(rng, (1 if "shared" in form else b, n), 0.01))
    dm, dsx = to_gpu(mat), to_gpu(sx)
    s = torch.full((b, m), -1.0, dtype=torch.half, device="cuda")
    qt = torch.full((b, m, ld_t), 77, dtype=torch.int8, device="cuda")
    qn = torch.full((b, n, ld_n), 77, dtype=torch.int8, device="cuda")
    ck.gemm_quantize_cols_ld(b, n, m, dm.data_ptr(), dsx.data_ptr() if scaled else None, "shared" in form, s.data_ptr(),
                             qt.data_ptr() if want_t else None, ld_t, qn.data_ptr() if want_n else None, ld_n, _st())
    if scaled:
        q, scale = ot.gemm_backward_scale_round(mat, sx[0] if "shared" in form else sx, "shared" in form)
    else:
        scale = oracle.gemm_calc_scale_transpose(mat)
        q = oracle.gemm_round_transpose(mat, scale)
    assert_bits_equal(to_np(s), scale, "scale")
    if want_t:
        assert_bits_equal(to_np(qt), _pad(np.ascontiguousarray(q.transpose(0, 2, 1)), ld_t), "transposed")
    if want_n:
        assert_bits_equal(to_np(qn), _pad(q, ld_n), "in place")


@pytest.mark.parametrize("m", [4, 100, 512, 700, 1500, 2048, 2052, 3001])
def test_scaled_rows(gpu, m):
    print("scaled rows", m, flush=True)
    rng = np.random.default_rng(m)
    b, n, ld = 2, 5, _up(m, 128)
    mat, sy = rand_half(rng, (b, n, m)), np.abs(rand_half(rng, (b, m), 0.01))
    mat[1, 2] = 0
    dm, dsy = to_gpu(mat), to_gpu(sy)
    s = torch.full((b, n), -1.0, dtype=torch.half, device="cuda")
    q = torch.full((b, n, ld), 77, dtype=torch.int8, device="cuda")
    ck.gemm_backward_round_scale_ld(b, n, m, dm.data_ptr(), dsy.data_ptr(), q.data_ptr(), ld, s.data_ptr(), False, _st())
    want, scale = ot.gemm_backward_round_scale(mat, sy, False)
    assert_bits_equal(to_np(s), scale, "scale")
    assert_bits_equal(to_np(q), _pad(want, ld), "rows")


def test_scaled_rounding_is_the_division(gpu):
    """Eight million quotients x * sx / s by fp32 scales of every magnitude against the IEEE division, on rows and on columns."""
    rng = np.random.default_rng(11)
    n = 2048
    mat = (rng.standard_normal((1, n, n)) * np.exp2(rng.integers(-12, 6, (1, n, 1)))).astype(np.float16)
    sx = np.abs(rng.standard_normal((1, n)) * np.exp2(rng.integers(-14, 4, (1, n)))).astype(np.float16)
    dm, dsx = to_gpu(mat), to_gpu(sx)
    for cols in (False, True):
        s = torch.empty((1, n), dtype=torch.half, device="cuda")
        q = torch.empty((1, n, n), dtype=torch.int8, device="cuda")
        fn = ck.gemm_backward_scale_round if cols else ck.gemm_backward_round_scale
        fn(1, n, n, dm.data_ptr(), dsx.data_ptr(), q.data_ptr(), s.data_ptr(), False, _st())
        want, scale = (ot.gemm_backward_scale_round if cols else ot.gemm_backward_round_scale)(mat, sx, False)
        assert_bits_equal(to_np(s), scale, "scale")
        assert_bits_equal(to_np(q), want, "int8")


@pytest.mark.parametrize("shape", [(1, 4, 4), (2, 15, 17), (1, 16, 64), (3, 100, 130), (1, 129, 256)])
def test_transpose(gpu, shape):
    b, n, m = shape
    print("transpose", shape, flush=True)
    rng = np.random.default_rng(n)
    ldi, ldo = _up(m, 128), _up(n, 128)
    src = rng.integers(-128, 128, (b, n, ldi)).astype(np.int8)
    d = to_gpu(src)
    out = torch.full((b, m, ldo), 77, dtype=torch.int8, device="cuda")
    ck.transpose_i8_ld(b, n, m, d.data_ptr(), ldi, out.data_ptr(), ldo, _st())
    assert_bits_equal(to_np(out), _pad(np.ascontiguousarray(src[:, :, :m].transpose(0, 2, 1)), ldo), "transposed")


# 17 x 17 tiles of 256x256: a last round of 33 tiles, issued as row halves, beside operands stored (K, rows)
@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, True)])
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("n", [4352, 4208])
def test_half_tiles_of_operands_stored_k_first(gpu, layout, f16, n):
    aT, bT = layout          # of the launcher: A (k, m) if not aT, B (k, n) if bT
    print("half tiles", layout, f16, n, flush=True)
    m, k = 4352, 384 if not f16 else 320
    g = torch.Generator(device="cuda").manual_seed(n)
    if f16:
        A, B = (torch.randint(-8, 9, (r, k), generator=g, device="cuda").half() for r in (m, n))       # products and sums exact in fp16 / fp32
        out = torch.zeros((n, m), dtype=torch.half, device="cuda")
    else:
        A, B = (torch.randint(-128, 128, (r, k), generator=g, device="cuda", dtype=torch.int8) for r in (m, n))
        out = torch.zeros((n, m), dtype=torch.int32, device="cuda")
    As, Bs = A if aT else A.t().contiguous(), B.t().contiguous() if bT else B
    (ck.gemm_fp16 if f16 else ck.gemm_int8)(m, k, n, 1, 1, aT, bT, As.data_ptr(), Bs.data_ptr(), out.data_ptr(), _st())
    want = B.float() @ A.float().t() if not f16 else B.double() @ A.double().t()
    if f16:
        assert torch.equal(out, want.half())
    else:
        assert torch.equal(out.double(), B.double() @ A.double().t())
