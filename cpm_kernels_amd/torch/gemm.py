"""``bmm(A, aT, B, bT, int8)`` with the interface of cpm_kernels/torch/gemm.py:233-239.

int8=True is the hot path: row-wise absmax quantisation of both operands, int8 GEMM with
int32 accumulation, fp16 dequantisation (GEMMInt8.forward, torch/gemm.py:84-113).  The
reference does that in six launches with an int32 round trip; here the default is three
(two fused quantise launches and one GEMM with the dequantising epilogue), bit-identical to
the six-launch sequence, which ``fused=False`` still runs through the kernel-level API.
"""
import torch
from ..kernels import gemm_calc_scale, gemm_calc_scale_transpose, gemm_round, gemm_round_transpose, \
    gemm_scale, gemm_scale_x, gemm_scale_y, gemm_int8, gemm_int8_scale_one, gemm_quantize, \
    gemm_quantize_cols_ld, gemm_quantize_cols_rows, gemm_quantize_pair_ld, gemm_fp16, gemm_sum_groups_timed, gemm_sum_krows_groups, gemm_int8_scale_sum, gemm_fp16_sum, \
    gemm_int8_scale_parts, gemm_fp16_parts, gemm_add_parts, gemm_depth_parts, gemm_fp16_copy_pays, gemm_int8_scale_split, gemm_fp16_split, \
    arith_batch_add_backward, gemm_backward_round_scale, gemm_backward_round_scale_ld, gemm_backward_quantize_both, gemm_backward_scale_round, transpose, \
    transpose_i8_ld
from ._common import cur_stream


def calc_scale(mat: torch.Tensor, transpose: bool) -> torch.Tensor:
    """reference: torch/gemm.py:5-19"""
    assert mat.is_contiguous() and mat.is_cuda
    b, n, m = mat.size()
    out = torch.empty((b, m if transpose else n), dtype=torch.half, device=mat.device)
    fn = gemm_calc_scale_transpose if transpose else gemm_calc_scale
    fn(b, n, m, mat.data_ptr(), out.data_ptr(), cur_stream())
    return out


def round_i8(mat: torch.Tensor, scale: torch.Tensor, transpose: bool) -> torch.Tensor:
    """reference: torch/gemm.py:21-38"""
    assert mat.is_contiguous() and mat.is_cuda
    assert scale.is_contiguous() and scale.is_cuda
    b, n, m = mat.size()
    out = torch.empty(mat.size(), dtype=torch.int8, device=mat.device)
    fn = gemm_round_transpose if transpose else gemm_round
    fn(b, n, m, mat.data_ptr(), scale.data_ptr(), out.data_ptr(), cur_stream())
    return out


def quantize(mat: torch.Tensor, transpose: bool):
    """calc_scale + round_i8 in one launch; returns (scale, int8 tensor)."""
    assert mat.is_contiguous() and mat.is_cuda and mat.dtype == torch.half
    b, n, m = mat.size()
    scale = torch.empty((b, m if transpose else n), dtype=torch.half, device=mat.device)
    out = torch.empty(mat.size(), dtype=torch.int8, device=mat.device)
    gemm_quantize(b, n, m, mat.data_ptr(), scale.data_ptr(), out.data_ptr(), transpose, cur_stream())
    return scale, out


def _row_bytes(k: int) -> int:
    """Bytes from one row of a quantised operand to the next when it is contracted over its k columns: whole 128-byte slabs
    of the tile kernel, the surplus zeros, which add nothing (NS shape with K = 4100: 150 us, 233-250 with the rest of each
    row taken on its own; K = 4032 also ran 5-10 % behind on 64-byte slabs).  Short rows of whole 64-byte slabs stay as they are."""
    return k if k % 128 == 0 or k > 16384 or (k % 64 == 0 and k < 1024) else (k + 127) // 128 * 128


def _sum_row_bytes(k: int) -> int:
    """The same where the product is summed over the batch (gemm_and_scale_sum): whole slabs always."""
    return _row_bytes(k) if k > 16384 else (k + 127) // 128 * 128


def _quantize_rows(*mats):
    """One or two (b, rows, K) operands quantised along K in one launch: [(scale (b, rows), int8 (b, rows, _row_bytes(K)))]"""
    K = mats[0].size(2)
    ld = _row_bytes(K)
    if K > 16384:
        return [quantize(x, False) for x in mats]
    out = [(torch.empty(x.shape[:2], dtype=torch.half, device=x.device),
            torch.empty((x.size(0), x.size(1), ld), dtype=torch.int8, device=x.device)) for x in mats]
    args = []
    for x, (s, q) in zip(mats, out):
        args += [x.size(0) * x.size(1), x.data_ptr(), s.data_ptr(), q.data_ptr()]
    if len(mats) == 1:
        args += [0, 0, 0, 0]
    gemm_quantize_pair_ld(*args, K, ld, cur_stream())
    return out


def _cols_row_bytes(n: int, summed: bool) -> int:
    return (n + 15) // 16 * 16 if n > 16384 else _sum_row_bytes(n) if summed else _row_bytes(n)


def _quantize_cols(x, both: bool, row_scale=None, summed: bool = False):
    """A (b, n, m) operand quantised along n: scale (b, m), int8 (b, m, _row_bytes(n)) -- _sum_row_bytes(n) if `summed` -- and, with
    `both`, the same values where they were, (b, n, _sum_row_bytes(m)) (else None).  row_scale: of the values multiplied by it, see
    gemm_backward_scale_round."""
    b, n, m = x.size()
    scale = torch.empty((b, m), dtype=torch.half, device=x.device)
    ld_t = _cols_row_bytes(n, summed)
    ld_n = _sum_row_bytes(m) if both else 0
    out_t = torch.empty((b, m, ld_t), dtype=torch.int8, device=x.device)
    out_n = torch.empty((b, n, ld_n), dtype=torch.int8, device=x.device) if both else None
    gemm_quantize_cols_ld(b, n, m, x.data_ptr(), None if row_scale is None else row_scale.data_ptr(),
                          row_scale is not None and row_scale.size(0) == 1, scale.data_ptr(), out_t.data_ptr(), ld_t,
                          out_n.data_ptr() if both else None, ld_n, cur_stream())
    return scale, out_t, out_n


# Outputs of a product that may be worth dividing along its depth (gemm_depth_parts): a larger one has a tile for every compute unit.
_PARTS_MOST = 1 << 22


def _quantize_cols_rows(x, both: bool, w):
    """_quantize_cols of x (b, K, m) and _quantize_rows of w (b', rows, K) in one launch, whose streaming of the rows fills the
    waits of the columns' workgroups."""
    b, n, m = x.size()
    if n > 16384:
        return _quantize_cols(x, both), _quantize_rows(w)[0]
    ld, ld_n = _row_bytes(n), _sum_row_bytes(m) if both else 0
    scale = torch.empty((b, m), dtype=torch.half, device=x.device)
    out_t = torch.empty((b, m, ld), dtype=torch.int8, device=x.device)
    out_n = torch.empty((b, n, ld_n), dtype=torch.int8, device=x.device) if both else None
    row_scale = torch.empty(w.shape[:2], dtype=torch.half, device=x.device)
    row_out = torch.empty((w.size(0), w.size(1), ld), dtype=torch.int8, device=x.device)
    gemm_quantize_cols_rows(b, n, m, x.data_ptr(), scale.data_ptr(), out_t.data_ptr(), ld, out_n.data_ptr() if both else None, ld_n,
                            w.size(0) * w.size(1), w.data_ptr(), row_scale.data_ptr(), row_out.data_ptr(), cur_stream())
    return (scale, out_t, out_n), (row_scale, row_out)


def _dims(quantA, quantB, aT, bT):
    _, M, K = quantA.shape
    if aT:
        M, K = K, M
    N = quantB.shape[1 if bT else 2]
    return M, K, N


def gemm_and_scale(quantA, scaleA, quantB, scaleB, aT, bT, fused=True) -> torch.Tensor:
    """reference: torch/gemm.py:40-82.  The operands are swapped in the kernel call exactly as
    there (:45-52) so the (M, N) product comes out row-major.  One of the scales may be None
    (the backward products): the accumulator is then scaled along the other side only."""
    M, K, N = _dims(quantA, quantB, aT, bT)
    batch = max(quantA.size(0), quantB.size(0))
    result_fp = torch.empty((batch, M, N), dtype=torch.float16, device=quantA.device)
    if fused:
        parts = 1
        # (whole 16-byte pieces: a caller's operands may lie anywhere)
        if K >= 2048 and result_fp.numel() < _PARTS_MOST and (quantA.data_ptr() | quantB.data_ptr()) % 16 == 0 and (scaleB is None or scaleB.data_ptr() % 8 == 0):
            parts = gemm_depth_parts(False, N, K, M, quantB.size(0), quantA.size(0), bT, aT)
        if parts > 1:
            workspace = torch.empty((parts, result_fp.numel()), dtype=torch.int32, device=quantA.device)
            gemm_int8_scale_split(N, K, M, quantB.size(0), quantA.size(0), bT, aT, quantB.data_ptr(), quantA.data_ptr(),
                                  None if scaleA is None else scaleA.data_ptr(), None if scaleB is None else scaleB.data_ptr(),
                                  scaleA is None or scaleA.size(0) == 1, scaleB is None or scaleB.size(0) == 1,
                                  result_fp.data_ptr(), parts, workspace.data_ptr(), cur_stream())
            return result_fp
        gemm_int8_scale_one(N, K, M, quantB.size(0), quantA.size(0), bT, aT,
                            quantB.data_ptr(), quantA.data_ptr(),
                            None if scaleA is None else scaleA.data_ptr(), None if scaleB is None else scaleB.data_ptr(),
                            scaleA is None or scaleA.size(0) == 1, scaleB is None or scaleB.size(0) == 1,
                            result_fp.data_ptr(), cur_stream())
        return result_fp
    result_i32 = torch.empty((batch, M, N), dtype=torch.int32, device=quantA.device)
    gemm_int8(N, K, M, quantB.size(0), quantA.size(0), bT, aT,
              quantB.data_ptr(), quantA.data_ptr(), result_i32.data_ptr(), cur_stream())
    if scaleA is not None and scaleB is not None:
        gemm_scale(batch, M, N, result_i32.data_ptr(), scaleA.data_ptr(), scaleB.data_ptr(),
                   result_fp.data_ptr(), quantA.size(0) == 1, quantB.size(0) == 1, cur_stream())
    elif scaleA is not None:
        gemm_scale_x(batch, M, N, result_i32.data_ptr(), scaleA.data_ptr(), result_fp.data_ptr(), cur_stream())
    else:
        assert scaleB is not None
        gemm_scale_y(batch, M, N, result_i32.data_ptr(), scaleB.data_ptr(), result_fp.data_ptr(), cur_stream())
    return result_fp


def _sum_entries(parts: torch.Tensor) -> torch.Tensor:
    """(g, r, c) -> (1, r, c), fp32 sums rounded once"""
    if parts.size(0) == 1:
        return parts
    out = torch.empty((1,) + parts.shape[1:], dtype=torch.half, device=parts.device)
    arith_batch_add_backward(parts.size(0), out.numel(), parts.data_ptr(), out.data_ptr(), cur_stream())
    return out


def _add_parts(parts: torch.Tensor) -> torch.Tensor:
    """(groups, r, c) fp32 sums -> (1, r, c) fp16"""
    out = torch.empty((1,) + parts.shape[1:], dtype=torch.half, device=parts.device)
    gemm_add_parts(parts.size(0), out.numel(), parts.data_ptr(), out.data_ptr(), cur_stream())
    return out


def gemm_and_scale_sum(quantA, scaleA, quantB) -> torch.Tensor:
    """(1, M, N): the sum over the batch of scaleA * (quantA x quantB^T), quantA (b, M, K) and quantB (b, N, K)."""
    batch, M, K = quantA.size()
    N = quantB.size(1)
    groups = gemm_sum_groups_timed(0, N, K, M, batch)
    if groups == batch or quantB.size(0) != batch or K == 0 or K % 128 != 0 or max(M, N) * K >= 2 ** 31 or batch * K >= 2 ** 22:
        return _sum_entries(gemm_and_scale(quantA, scaleA, quantB, None, False, True))
    parts = torch.empty((groups, M, N), dtype=torch.half if groups == 1 else torch.float32, device=quantA.device)
    launch = gemm_int8_scale_sum if groups == 1 else gemm_int8_scale_parts
    launch(N, K, M, batch, groups, quantB.data_ptr(), quantA.data_ptr(), scaleA.data_ptr(), parts.data_ptr(), cur_stream())
    return parts if groups == 1 else _add_parts(parts)


class GEMMInt8(torch.autograd.Function):
    @staticmethod
    def forward(ctx, A: torch.Tensor, aT: bool, B: torch.Tensor, bT: bool, fused: bool = True, train: bool = True):
        """A: (batchA, M, K) [(batchA, K, M) if aT], B: (batchB, K, N) [(batchB, N, K) if bT]
        -> (batch, M, N) fp16.  reference: torch/gemm.py:84-113"""
        assert A.is_cuda and B.is_cuda and A.device == B.device
        assert A.is_contiguous() and B.is_contiguous()
        assert A.dtype == torch.half and B.dtype == torch.half
        ctx.layout = (aT, bT)
        ctx.fused = fused
        if not fused:
            scale_A = calc_scale(A, aT)
            scale_B = calc_scale(B, not bT)
            quantized_A = round_i8(A, scale_A, aT)
            quantized_B = round_i8(B, scale_B, not bT)
            ctx.save_for_backward(scale_A, quantized_A, scale_B, quantized_B)
            return gemm_and_scale(quantized_A, scale_A, quantized_B, scale_B, aT, bT, False)
        # Both operands are brought to K-major int8 while they are quantised, so every layout runs on the fast GEMM kernel:
        # A (bA, M, ld) and B (bB, N, ld).  An operand that is quantised along its columns and whose partner wants a gradient
        # also leaves its int8 values where they were: that product is contracted over its other dimension.
        M, K, N = _dims(A, B, aT, bT)
        assert M % 4 == 0 and K % 4 == 0 and N % 4 == 0
        want_A, want_B = train and ctx.needs_input_grad[0], train and ctx.needs_input_grad[2]
        own_A = own_B = None
        if not aT and bT:
            (scale_A, quant_A), (scale_B, quant_B) = _quantize_rows(A, B)
        elif aT and bT:
            (scale_A, quant_A, own_A), (scale_B, quant_B) = _quantize_cols_rows(A, want_B, B)
        elif not aT:
            (scale_B, quant_B, own_B), (scale_A, quant_A) = _quantize_cols_rows(B, want_A, A)
        else:
            scale_A, quant_A, own_A = _quantize_cols(A, want_B)
            scale_B, quant_B, own_B = _quantize_cols(B, want_A)
        if quant_A.size(2) != quant_B.size(2):      # (contractions beyond what the row quantiser holds in registers)
            quant_A, quant_B = (x[:, :, :K].contiguous() for x in (quant_A, quant_B))
        if train:
            ctx.dims = (M, K, N)
            ctx.own = (own_A is not None, own_B is not None)
            ctx.save_for_backward(scale_A, quant_A if own_A is None else own_A, scale_B, quant_B if own_B is None else own_B)
        return gemm_and_scale(quant_A, scale_A, quant_B, scale_B, False, True)

    @staticmethod
    def backward(ctx, grad_f: torch.Tensor):
        """reference: torch/gemm.py:115-186.  grad_A = int8(grad * scale_B, row scales) x quantized_B and
        grad_B = int8(grad * scale_A, column scales)^T x quantized_A, each dequantised by the new
        scales only (the other operand's scales went into the gradient before rounding)."""
        assert grad_f.is_contiguous() and grad_f.is_cuda and grad_f.dtype == torch.float16
        scale_A, quantized_A, scale_B, quantized_B = ctx.saved_tensors
        aT, bT = ctx.layout
        batch, m, n = grad_f.size()
        st = cur_stream()
        if ctx.fused:
            # Each gradient is formed directly in the layout its operand came in, summed inside the product where the operand was
            # broadcast over the batch.
            M, K, N = ctx.dims
            own_A, own_B = ctx.own
            grad_A = grad_B = None
            want_A, want_B = ctx.needs_input_grad[0], ctx.needs_input_grad[2]
            quant_B_side = None
            if want_A:                                                      # contracted over N
                summed = scale_A.size(0) == 1 and batch > 1 and not aT
                ld = quantized_B.size(2) if own_B else _sum_row_bytes(N) if summed else _row_bytes(N)
                scale_G = torch.empty((batch, M), dtype=torch.half, device=grad_f.device)
                quant_G = torch.empty((batch, M, ld), dtype=torch.int8, device=grad_f.device)
                if want_B:
                    # (both operands made from the gradient in one launch)
                    summed_B = scale_B.size(0) == 1 and batch > 1 and bT
                    ld_t = _cols_row_bytes(M, summed_B or own_A)
                    quant_B_side = (torch.empty((batch, N), dtype=torch.half, device=grad_f.device),
                                    torch.empty((batch, N, ld_t), dtype=torch.int8, device=grad_f.device))
                    gemm_backward_quantize_both(batch, M, N, grad_f.data_ptr(), scale_A.data_ptr(), scale_A.size(0) == 1, quant_B_side[0].data_ptr(),
                                                quant_B_side[1].data_ptr(), ld_t, scale_B.data_ptr(), scale_B.size(0) == 1, quant_G.data_ptr(), ld,
                                                scale_G.data_ptr(), st)
                else:
                    gemm_backward_round_scale_ld(batch, M, N, grad_f.data_ptr(), scale_B.data_ptr(), quant_G.data_ptr(), ld,
                                                 scale_G.data_ptr(), scale_B.size(0) == 1, st)
                other, lies = _contracted(quantized_B, K, N, ld, own_B, summed)
                if aT:              # grad_A (b, K, M), scaled per column m
                    grad_A = gemm_and_scale(other, None, quant_G, scale_G, lies, True)
                elif summed:
                    grad_A = gemm_and_scale_sum(quant_G, scale_G, other)
                else:               # grad_A (b, M, K), scaled per row m
                    grad_A = gemm_and_scale(quant_G, scale_G, other, None, False, not lies)
                del quant_G, other
                if scale_A.size(0) == 1 and grad_A.size(0) > 1:
                    grad_A = grad_A.sum(dim=0, keepdim=True)
            if want_B:                                                      # contracted over M
                summed = scale_B.size(0) == 1 and batch > 1 and bT
                scale_G, quant_G = quant_B_side if quant_B_side is not None else _quantize_cols(grad_f, False, scale_A, summed or own_A)[:2]
                other, lies = _contracted(quantized_A, K, M, quant_G.size(2), own_A, summed)
                if summed:
                    grad_B = gemm_and_scale_sum(quant_G, scale_G, other)
                elif bT:            # grad_B (b, N, K), scaled per row n
                    grad_B = gemm_and_scale(quant_G, scale_G, other, None, False, not lies)
                else:               # grad_B (b, K, N), scaled per column n
                    grad_B = gemm_and_scale(other, None, quant_G, scale_G, lies, True)
                if scale_B.size(0) == 1 and grad_B.size(0) > 1:
                    grad_B = grad_B.sum(dim=0, keepdim=True)
            return grad_A, None, grad_B, None, None, None
        scale_G_a = torch.empty((batch, m), dtype=torch.half, device=grad_f.device)
        quant_G_a = torch.empty((batch, m, n), dtype=torch.int8, device=grad_f.device)
        gemm_backward_round_scale(batch, m, n, grad_f.data_ptr(), scale_B.data_ptr(), quant_G_a.data_ptr(),
                                  scale_G_a.data_ptr(), scale_B.size(0) == 1, st)
        if aT:
            grad_A = gemm_and_scale(quantized_B, None, quant_G_a, scale_G_a, bT, True)
        else:
            grad_A = gemm_and_scale(quant_G_a, scale_G_a, quantized_B, None, False, not bT)
        del scale_G_a, quant_G_a

        scale_G_b = torch.empty((batch, n), dtype=torch.half, device=grad_f.device)
        quant_G_b = torch.empty((batch, m, n), dtype=torch.int8, device=grad_f.device)
        gemm_backward_scale_round(batch, m, n, grad_f.data_ptr(), scale_A.data_ptr(), quant_G_b.data_ptr(),
                                  scale_G_b.data_ptr(), scale_A.size(0) == 1, st)
        if bT:
            grad_B = gemm_and_scale(quant_G_b, scale_G_b, quantized_A, None, True, aT)
        else:
            grad_B = gemm_and_scale(quantized_A, None, quant_G_b, scale_G_b, not aT, False)

        if scale_A.size(0) == 1 and grad_A.size(0) > 1:
            grad_A = grad_A.sum(dim=0, keepdim=True)
        if scale_B.size(0) == 1 and grad_B.size(0) > 1:
            grad_B = grad_B.sum(dim=0, keepdim=True)
        return grad_A, None, grad_B, None, None, None


def _contracted(q, K, length, ld, own, must_copy):
    """The saved int8 values of an operand -- (b, length, K-major rows), or with `own` (b, K, length padded) -- for a product
    contracted over `length`: (operand, whether it lies as (b, length, K)).  The tile kernel reads it as it lies where rows and
    length are whole pieces and slabs, 8 % slower than from (b, K, ld), which is less than the transposition costs."""
    if own and q.size(2) == ld:
        return q, False
    if own:
        q, own = q[:, :, :length].transpose(1, 2).contiguous(), False       # (a padding of another length: only past 16384)
    if not must_copy and q.size(2) == K and length == ld and length % 128 == 0 and K % 16 == 0:
        return q, True
    out = torch.empty((q.size(0), K, ld), dtype=torch.int8, device=q.device)
    transpose_i8_ld(q.size(0), length, K, q.data_ptr(), q.size(2), out.data_ptr(), ld, cur_stream())
    return out, False


def _transposed_copy(x: torch.Tensor) -> torch.Tensor:
    out = torch.empty((x.size(0), x.size(2), x.size(1)), dtype=torch.half, device=x.device)
    transpose(x.size(0), x.size(1), x.size(2), x.data_ptr(), out.data_ptr(), cur_stream())
    return out


def gemm_pth_fp16(A: torch.Tensor, aT: bool, B: torch.Tensor, bT: bool) -> torch.Tensor:
    """reference: torch/gemm.py:189-203; operands are passed swapped to the kernel so that the
    (M, N) result comes out row-major.  The MFMA tile kernel reads an operand stored (K, rows) as it lies, at 2-8 % more time
    than K-major ones: a transposed copy pays only for products very large next to the operand.  Measured (direct / with a copy):
    8 x 4096 x 4096 x 512, B transposed 108 / 121 us, A 109 / 118; 4 x 1024 x 4096 x 512 34 / 40-44; 8192 x 4096 x 4096 204 / 208;
    8 x 10240 x 4096 x 512, B transposed 298 / 279; 4096 x 4096 x 10240, A transposed 298 / 275.  Or for results beyond the
    last-level cache of few slabs, where the two compete for memory: 2032 x 4096 over 32 entries of A, K = 256 223 / 203 us, 2048 x 8064
    x 32 434 / 398 (512 MB and more; 2048 x 2048 x 32 and K = 1024 about even); or for few columns an entry (gemm_fp16_copy_pays).  Rows of A that are not whole 16-byte pieces are
    copied always."""
    M, K, N = _dims(A, B, aT, bT)
    bA, bB = A.shape[0], B.shape[0]
    if K % 64 == 0 and N % 8 == 0 and M * K < 2 ** 31 and N * K < 2 ** 31:
        large = 128 < K <= 512 and M * N * max(bA, bB) > 2 ** 27
        # (short K: the product is bound by writing its output)
        if aT and ((N * max(bB // bA, 1) > 8192 and K > 128) or large and N > 512 or M % 8 != 0):
            A, aT = _transposed_copy(A), False
        if not bT and (M > 8192 and K > 128 or large and M > 2048):
            B, bT = _transposed_copy(B), True
    if bA == 1 and not bT and N < 512 and K >= 256 and gemm_fp16_copy_pays(N, K, M, bB, aT):
        B, bT = _transposed_copy(B), True
    out = torch.empty((max(bA, bB), M, N), dtype=torch.half, device=A.device)
    parts = gemm_depth_parts(True, N, K, M, bB, bA, bT, aT) if K >= 1024 and out.numel() < _PARTS_MOST and (A.data_ptr() | B.data_ptr()) % 16 == 0 else 1
    if parts > 1:
        workspace = torch.empty((parts, out.numel()), dtype=torch.float32, device=A.device)
        gemm_fp16_split(N, K, M, bB, bA, bT, aT, B.data_ptr(), A.data_ptr(), out.data_ptr(), parts, workspace.data_ptr(), cur_stream())
        return out
    gemm_fp16(N, K, M, bB, bA, bT, aT, B.data_ptr(), A.data_ptr(), out.data_ptr(), cur_stream())
    return out


def _entry_groups(M: int, K: int, N: int, batch: int, joined: bool) -> int:
    """Groups that an fp16 product summed over the batch is formed in.  `joined`: both operands stored (K, rows), so that a group's
    entries are one contraction."""
    return gemm_sum_groups_timed(2 if joined else 1, N, K, M, batch)


def gemm_pth_fp16_sum(A: torch.Tensor, aT: bool, B: torch.Tensor, bT: bool) -> torch.Tensor:
    """The same product summed over the batch, (1, M, N)."""
    M, K, N = _dims(A, B, aT, bT)
    batch = A.size(0)
    joined = aT and not bT
    groups = batch if batch != B.size(0) else gemm_sum_krows_groups(N, K, M, batch) if joined else _entry_groups(M, K, N, batch, False)
    if joined and groups and batch == B.size(0):
        # both operands stored (K, rows): the entries of a group are one longer contraction as they lie
        if groups == 1:
            return gemm_pth_fp16(A.view(1, batch * K, M), True, B.view(1, batch * K, N), False)
        parts = torch.empty((groups, M, N), dtype=torch.float32, device=A.device)
        gemm_fp16_parts(N, K, M, batch, groups, 2, B.data_ptr(), A.data_ptr(), parts.data_ptr(), cur_stream())
        return _add_parts(parts)
    if groups < batch and not aT and bT and M % 4 == 0 and N % 4 == 0 and K > 32 and max(M, N) * K < 2 ** 31 and \
            batch * K < 2 ** 21 and (A.data_ptr() | B.data_ptr()) % 4 == 0:
        if groups == 1:
            out = torch.empty((1, M, N), dtype=torch.half, device=A.device)
            gemm_fp16_sum(N, K, M, batch, 1, B.data_ptr(), A.data_ptr(), out.data_ptr(), cur_stream())
            return out
        parts = torch.empty((groups, M, N), dtype=torch.float32, device=A.device)
        gemm_fp16_parts(N, K, M, batch, groups, False, B.data_ptr(), A.data_ptr(), parts.data_ptr(), cur_stream())
        return _add_parts(parts)
    return _sum_entries(gemm_pth_fp16(A, aT, B, bT))


class GEMMFloat(torch.autograd.Function):
    @staticmethod
    def forward(ctx, A: torch.Tensor, aT: bool, B: torch.Tensor, bT: bool):
        """fp16 product with fp32 accumulation.  reference: torch/gemm.py:205-217 (cuBLASLt there)."""
        assert A.is_cuda and B.is_cuda and A.device == B.device
        assert A.is_contiguous() and B.is_contiguous()
        assert A.dtype == torch.half and B.dtype == torch.half
        ctx.save_for_backward(A, B)
        ctx.aT = aT
        ctx.bT = bT
        return gemm_pth_fp16(A, aT, B, bT)

    @staticmethod
    def backward(ctx, grad_f):
        """reference: torch/gemm.py:219-239"""
        assert grad_f.is_cuda and grad_f.is_contiguous() and grad_f.dtype == torch.float16
        aT, bT = ctx.aT, ctx.bT
        A, B = ctx.saved_tensors
        product_A = gemm_pth_fp16_sum if A.size(0) == 1 else gemm_pth_fp16
        product_B = gemm_pth_fp16_sum if B.size(0) == 1 else gemm_pth_fp16
        grad_A = product_A(B, bT, grad_f, True) if aT else product_A(grad_f, False, B, not bT)
        grad_B = product_B(grad_f, True, A, aT) if bT else product_B(A, not aT, grad_f, False)
        return grad_A, None, grad_B, None


def bmm(A: torch.Tensor, aT: bool, B: torch.Tensor, bT: bool, int8: bool = False, fused: bool = True) -> torch.Tensor:
    size_A, size_B = A.shape, B.shape
    assert len(size_A) == 3
    assert len(size_B) == 3
    assert size_A[1 if aT else 2] == size_B[2 if bT else 1], "operands of different contraction lengths"      # (B would be read past its end)
    if int8:
        return GEMMInt8.apply(A, aT, B, bT, fused, torch.is_grad_enabled())
    return GEMMFloat.apply(A, aT, B, bT)
