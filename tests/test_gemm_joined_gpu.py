"""Products of a batch and an operand that it shares, as one product over the joined rows or columns, and products whose depth is divided."""
import pytest
import torch

import cpm_kernels_amd.kernels as ck
import cpm_kernels_amd.torch as ct
from util import stream

pytestmark = pytest.mark.gpu


def _int8(batch_a, batch_b, m, k, n, bT, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def ints(*shape):
        return torch.randint(-127, 128, shape, generator=g, device="cuda", dtype=torch.int8)

    def scales(*shape):
        return (torch.rand(shape, generator=g, device="cuda") * 0.01 + 0.001).half()
    return ints(batch_a, m, k), ints(*((batch_b, k, n) if bT else (batch_b, n, k))), scales(batch_b, n), scales(batch_a, m)


def _reference(A, B, bT, s_row, s_col):
    """(batch, n, m): exact sums, scaled as the epilogue does it"""
    out = []
    for i in range(max(A.size(0), B.size(0))):
        ia, ib = i % A.size(0), i % B.size(0)
        b = B[ib].double()
        acc = (b.t() if bT else b).contiguous() @ A[ia].double().t().contiguous()
        out.append(((acc.float() * s_row[ib].float()[:, None]) * s_col[ia].float()[None, :]).half())
    return torch.stack(out)


def _whole(A, B, bT, s_row, s_col, k, parts=0):
    batch, m, n = max(A.size(0), B.size(0)), A.size(1), s_row.size(1)
    out = torch.full((batch, n, m), float("nan"), dtype=torch.half, device="cuda")
    args = (m, k, n, A.size(0), B.size(0), True, bT, A.data_ptr(), B.data_ptr(), s_row.data_ptr(), s_col.data_ptr(), B.size(0) == 1, A.size(0) == 1, out.data_ptr())
    if parts:
        ws = torch.full((parts, batch, n, m), -1, dtype=torch.int32, device="cuda")
        ck.gemm_int8_scale_split(*args, parts, ws.data_ptr(), stream())
    else:
        ck.gemm_int8_scale_one(*args, stream())
    return out


# (depths of 64-byte and 128-byte slabs; entries of whole pieces, of half pieces, shorter than a piece, and around a tile; few and many tiles)
@pytest.mark.parametrize("m,batch,n", [(4, 33, 132), (36, 7, 300), (100, 5, 128), (132, 3, 260), (64, 7, 272), (252, 16, 4112)])
@pytest.mark.parametrize("k,bT", [(64, False), (192, False), (128, False), (1152, False), (128, True), (640, True)])
def test_shared_row_operand(m, batch, n, k, bT):
    if bT:
        n = (n + 15) // 16 * 16
    A, B, s_row, s_col = _int8(batch, 1, m, k, n, bT, m + k)
    assert torch.equal(_whole(A, B, bT, s_row, s_col, k), _reference(A, B, bT, s_row, s_col))


@pytest.mark.parametrize("n,batch,m", [(4, 33, 132), (36, 7, 300), (132, 3, 260), (252, 16, 4112)])
@pytest.mark.parametrize("k", [4, 68, 128, 640])
def test_shared_column_operand(n, batch, m, k):
    A, B, s_row, s_col = _int8(1, batch, m, k, n, False, n + k)
    assert torch.equal(_whole(A, B, False, s_row, s_col, k), _reference(A, B, False, s_row, s_col))


# (entries that are joined because that saves rounds of tiles: shorter than a piece, off pieces, past a tile, and of large tiles; depths as above)
MANY = [(4, 300, 132), (36, 130, 300), (132, 140, 260), (300, 40, 2000)]


@pytest.mark.parametrize("m,batch,n", MANY)
@pytest.mark.parametrize("k,bT", [(64, False), (192, False), (128, False), (384, True)])
def test_shared_row_operand_of_many_entries(m, batch, n, k, bT):
    if bT:
        n = (n + 15) // 16 * 16
    A, B, s_row, s_col = _int8(batch, 1, m, k, n, bT, m + k)
    assert torch.equal(_whole(A, B, bT, s_row, s_col, k), _reference(A, B, bT, s_row, s_col))


@pytest.mark.parametrize("n,batch,m", MANY)
@pytest.mark.parametrize("k", [4, 68, 128, 192])
def test_shared_column_operand_of_many_entries(n, batch, m, k):
    A, B, s_row, s_col = _int8(1, batch, m, k, n, False, n + k)
    assert torch.equal(_whole(A, B, False, s_row, s_col, k), _reference(A, B, False, s_row, s_col))


@pytest.mark.parametrize("a_shared", [False, True])
@pytest.mark.parametrize("edge,batch,other", MANY)
@pytest.mark.parametrize("k", [66, 128, 520])
@pytest.mark.parametrize("stored_other", [False, True])        # the shared operand stored (K, rows or columns)
def test_fp16_of_many_entries(a_shared, edge, batch, other, k, stored_other):
    m, n, batch_a, batch_b = (other, edge, 1, batch) if a_shared else (edge, other, batch, 1)
    aT, bT = (not stored_other, False) if a_shared else (True, stored_other)
    g = torch.Generator(device="cuda").manual_seed(edge + k)
    A = torch.randn((batch_a, m, k) if aT else (batch_a, k, m), generator=g, device="cuda").half()
    B = torch.randn((batch_b, k, n) if bT else (batch_b, n, k), generator=g, device="cuda").half()
    out = torch.full((batch, n, m), float("nan"), dtype=torch.half, device="cuda")
    ck.gemm_fp16(m, k, n, batch_a, batch_b, aT, bT, A.data_ptr(), B.data_ptr(), out.data_ptr(), stream())
    for i in range(0, batch, 1 if batch < 64 else 7):
        a, b = A[i % batch_a].double(), B[i % batch_b].double()
        a, b = (a.t() if aT else a).contiguous(), (b.t() if bT else b).contiguous()        # (k, m), (n, k)
        ref, size = b @ a, b.abs() @ a.abs()
        # k additions in fp32, one rounding to fp16 (or half a subnormal step)
        assert ((out[i].double() - ref).abs() <= size * k * 2.0 ** -24 + ref.abs() * 2.0 ** -10.9 + 2.0 ** -25).all()


# (as many rounds of fewer tiles: 128 x 64, 128 x 128 in two rounds, 256 x 256)
@pytest.mark.parametrize("shared,edge,batch", [(432, 164, 7), (2176, 196, 12), (2048, 192, 24)])
@pytest.mark.parametrize("k", [384, 704, 1536])
def test_fewer_tiles(shared, edge, batch, k):
    A, B, s_row, s_col = _int8(batch, 1, edge, k, shared, False, edge + k)
    assert torch.equal(_whole(A, B, False, s_row, s_col, k), _reference(A, B, False, s_row, s_col))
    A, B, s_row, s_col = _int8(1, batch, shared, k, edge, False, edge + k)
    assert torch.equal(_whole(A, B, False, s_row, s_col, k), _reference(A, B, False, s_row, s_col))
    for a_shared in (False, True):
        test_fp16_of_many_entries(a_shared, edge, batch, shared, k, False)
    test_fp16_of_many_entries(False, edge, batch, shared, k, True)


# (tiles of 128 x 64, two a compute unit, up to a depth of 768, of 128 x 128 beyond; whole and over the joined columns of many entries)
@pytest.mark.parametrize("m,batch,n", [(5000, 1, 500), (1100, 1, 2164), (36, 500, 128), (68, 130, 252)])
@pytest.mark.parametrize("k", [128, 768, 896])
def test_narrow_tiles(m, batch, n, k):
    A, B, s_row, s_col = _int8(batch, 1, m, k, n, False, m + k)
    assert torch.equal(_whole(A, B, False, s_row, s_col, k), _reference(A, B, False, s_row, s_col))


# (parts of one slab, of several, a shorter last part, more parts than slabs)
@pytest.mark.parametrize("batch_a,batch_b,m,n,bT", [(1, 1, 64, 128, False), (3, 1, 44, 260, False), (1, 5, 132, 60, False), (2, 2, 132, 132, False),
                                                    (3, 1, 100, 272, True), (3, 1, 20, 16, True)])
@pytest.mark.parametrize("slabs,parts", [(2, 2), (7, 3), (33, 16), (5, 9)])
def test_int8_in_parts(batch_a, batch_b, m, n, bT, slabs, parts):
    k = slabs * 128
    A, B, s_row, s_col = _int8(batch_a, batch_b, m, k, n, bT, slabs)
    assert torch.equal(_whole(A, B, bT, s_row, s_col, k, parts), _reference(A, B, bT, s_row, s_col))


@pytest.mark.parametrize("aT,bT", [(True, False), (False, False), (True, True), (False, True)])
@pytest.mark.parametrize("batch_a,batch_b,m,n", [(1, 1, 56, 136), (3, 1, 40, 264), (1, 5, 136, 64), (2, 2, 136, 136)])
@pytest.mark.parametrize("slabs,parts", [(2, 2), (7, 3), (33, 16)])
def test_fp16_in_parts(aT, bT, batch_a, batch_b, m, n, slabs, parts):
    k = slabs * 64
    g = torch.Generator(device="cuda").manual_seed(slabs)
    A = torch.randn((batch_a, m, k) if aT else (batch_a, k, m), generator=g, device="cuda").half()
    B = torch.randn((batch_b, k, n) if bT else (batch_b, n, k), generator=g, device="cuda").half()
    batch = max(batch_a, batch_b)
    out = torch.full((batch, n, m), float("nan"), dtype=torch.half, device="cuda")
    ws = torch.full((parts, batch, n, m), float("nan"), dtype=torch.float32, device="cuda")
    ck.gemm_fp16_split(m, k, n, batch_a, batch_b, aT, bT, A.data_ptr(), B.data_ptr(), out.data_ptr(), parts, ws.data_ptr(), stream())
    for i in range(batch):
        a, b = A[i % batch_a].double(), B[i % batch_b].double()
        a, b = (a.t() if aT else a).contiguous(), (b.t() if bT else b).contiguous()        # (k, m), (n, k)
        ref, size = b @ a, b.abs() @ a.abs()
        # k additions in fp32, one rounding to fp16 (or half a subnormal step)
        assert ((out[i].double() - ref).abs() <= size * k * 2.0 ** -24 + ref.abs() * 2.0 ** -10.9 + 2.0 ** -25).all()


# (more parts of tiles than workgroups that are resident at once, two a compute unit, of 128 x 64 outputs and of 128 x 128; sixteen even parts, eleven of which the last is shorter)
@pytest.mark.parametrize("m,n", [(64, 16256), (1280, 1664)])
def test_more_parts_than_workgroups(m, n):
    A, B, s_row, s_col = _int8(1, 1, m, 32 * 128, n, False, m)
    assert torch.equal(_whole(A, B, False, s_row, s_col, 32 * 128, 16), _reference(A, B, False, s_row, s_col))
    test_fp16_in_parts(True, False, 1, 1, m, n, 32, 11)
    test_fp16_in_parts(False, True, 1, 1, m, n, 32, 11)


@pytest.mark.parametrize("at_a,at_b,at_scale", [(4, 0, 0), (0, 1, 0), (0, 0, 2), (0, 0, 0)])
def test_operands_off_whole_pieces(at_a, at_b, at_scale):
    """A product whose depth would be divided, from operands and scales at any address"""
    from cpm_kernels_amd.torch.gemm import gemm_and_scale
    M, K, N = 120, 8192, 512
    assert ck.gemm_depth_parts(False, N, K, M, 1, 1, True, False) > 1
    B, A, s_row, s_col = _int8(1, 1, N, K, M, False, 3)

    def moved(t, at):
        flat = torch.empty(t.numel() + at, dtype=t.dtype, device="cuda")
        return flat[at:].view(t.shape).copy_(t)
    out = gemm_and_scale(moved(A, at_a), s_row, moved(B, at_b), moved(s_col, at_scale), False, True)
    assert torch.equal(out, _reference(B, A, False, s_row, s_col))


def test_parts_are_refused_elsewhere():
    A, B, s_row, s_col = _int8(1, 1, 64, 320, 128, False, 0)       # (a depth of whole 64-byte slabs only)
    assert ck.gemm_depth_parts(False, 64, 320, 128, 1, 1, True, False) == 1
    with pytest.raises(RuntimeError):
        _whole(A, B, False, s_row, s_col, 320, 2)


@pytest.mark.parametrize("rows", [True, False])
@pytest.mark.parametrize("batch,tokens,din,dout", [(2, 4, 128, 132), (13, 64, 832, 260), (5, 192, 132, 1024), (16, 68, 640, 640), (3, 512, 512, 2304)])
def test_weight_gradient_of_few_tiles(rows, batch, tokens, din, dout):
    """int8: against the separate launches, whose entries are rounded to fp16 before they are added (and once more behind that); fp16: in 64 bits"""
    g = torch.Generator(device="cuda").manual_seed(tokens)
    x = torch.randn((batch, tokens, din) if rows else (batch, din, tokens), generator=g, device="cuda").half()
    w = (torch.randn((1, dout, din), generator=g, device="cuda") * 0.02).half().requires_grad_()
    grad = (torch.randn((batch, tokens, dout) if rows else (batch, dout, tokens), generator=g, device="cuda") * 0.05).half()

    def product(w, x, grad, **how):
        out = ct.bmm(x, False, w, True, **how) if rows else ct.bmm(w, False, x, False, **how)
        return torch.autograd.grad(out, w, grad)[0]
    ours = product(w, x, grad, int8=True).double()
    apart = [product(w, x[i:i + 1].contiguous(), grad[i:i + 1].contiguous(), int8=True, fused=False).double() for i in range(batch)]
    bound = sum(a.abs() * 2.0 ** -11 + 2.0 ** -25 for a in apart) * (1 + batch * 2.0 ** -12)
    want = sum(apart)
    assert ((ours - want).abs() <= bound + want.abs() * 2.0 ** -11 + 2.0 ** -25).all()
    xd, gd = (t.double() if rows else t.double().transpose(1, 2).contiguous() for t in (x, grad))
    want = sum(gd[i].t().contiguous() @ xd[i] for i in range(batch))
    size = sum(gd[i].abs().t().contiguous() @ xd[i].abs() for i in range(batch))
    ours = product(w, x, grad, int8=False).double()[0]
    rounded = sum((gd[i].t().contiguous() @ xd[i]).abs() for i in range(batch)) * 2.0 ** -11        # (where entries are formed one by one)
    assert ((ours - want).abs() <= rounded + size * (batch * tokens) * 2.0 ** -24 + want.abs() * 2.0 ** -10.9 + batch * 2.0 ** -25).all()
