"""Quantisation, int8 GEMM and dequantisation launchers with the signatures of
cpm_kernels/kernels/gemm.py.  Arithmetic contracts are stated in include/cpmk.h."""
from ..library import cpmk
from .base import DevicePointer, CUDAStream


def gemm_round(batch: int, n: int, m: int,
               mat: DevicePointer,      # (b, n, m)  fp16
               scale: DevicePointer,    # (b, n)     fp16
               out: DevicePointer,      # (b, n, m)  int8
               stream: CUDAStream):
    """reference: kernels/gemm.py:21-41"""
    cpmk.gemm_round(batch, n, m, mat, scale, out, stream)


def gemm_round_transpose(batch: int, n: int, m: int,
                         mat: DevicePointer,    # (b, n, m)  fp16
                         scale: DevicePointer,  # (b, m)     fp16
                         out: DevicePointer,    # (b, n, m)  int8
                         stream: CUDAStream):
    """reference: kernels/gemm.py:43-63"""
    cpmk.gemm_round_transpose(batch, n, m, mat, scale, out, stream)


def gemm_scale(batch: int, n: int, m: int,
               mat: DevicePointer,        # (b, n, m)  int32
               scale_x: DevicePointer,    # (b, n)     fp16
               scale_y: DevicePointer,    # (b, m)     fp16
               out: DevicePointer,        # (b, n, m)  fp16
               broad_cast_x: bool, broad_cast_y: bool,
               stream: CUDAStream):
    """reference: kernels/gemm.py:65-89"""
    cpmk.gemm_scale(batch, n, m, mat, scale_x, scale_y, out, int(bool(broad_cast_x)),
                    int(bool(broad_cast_y)), stream)


def gemm_calc_scale(batch: int, n: int, m: int,
                    mat: DevicePointer,    # (b, n, m) fp16
                    out: DevicePointer,    # (b, n)    fp16
                    stream: CUDAStream):
    """reference: kernels/gemm.py:91-107"""
    cpmk.gemm_calc_scale(batch, n, m, mat, out, stream)


def gemm_calc_scale_transpose(batch: int, n: int, m: int,
                              inp: DevicePointer,    # (b, n, m) fp16
                              out: DevicePointer,    # (b, m)    fp16
                              stream: CUDAStream):
    """reference: kernels/gemm.py:109-125"""
    cpmk.gemm_calc_scale_transpose(batch, n, m, inp, out, stream)


def gemm_int8(m: int, k: int, n: int,
              batchA: int, batchB: int,
              aT: bool, bT: bool,
              A: DevicePointer,      # (bA, k, m) int8   [(bA, m, k) if aT]
              B: DevicePointer,      # (bB, n, k) int8   [(bB, k, n) if bT]
              out: DevicePointer,    # (max(bA, bB), n, m) int32
              stream: CUDAStream):
    """reference: kernels/gemm.py:127-186 (cuBLASLt); same asserts (:139-140)."""
    assert m % 4 == 0 and n % 4 == 0 and k % 4 == 0
    assert batchA == batchB or batchA == 1 or batchB == 1
    cpmk.gemm_int8(m, k, n, batchA, batchB, int(bool(aT)), int(bool(bT)), A, B, out, stream)


def gemm_int8_scale(m: int, k: int, n: int,
                    batchA: int, batchB: int,
                    aT: bool, bT: bool,
                    A: DevicePointer, B: DevicePointer,
                    scale_row: DevicePointer,   # fp16 per output row j:  (n) or (batch, n)
                    scale_col: DevicePointer,   # fp16 per output col i:  (m) or (batch, m)
                    broad_cast_row: bool, broad_cast_col: bool,
                    out: DevicePointer,         # (max(bA, bB), n, m) fp16
                    stream: CUDAStream):
    """gemm_int8 with the gemm_scale epilogue fused (no counterpart launcher in the reference;
    it fuses kernels/gemm.py:127-186 and :65-89 as torch/gemm.py:40-64 chains them)."""
    assert m % 4 == 0 and n % 4 == 0 and k % 4 == 0
    assert batchA == batchB or batchA == 1 or batchB == 1
    cpmk.gemm_int8_scale(m, k, n, batchA, batchB, int(bool(aT)), int(bool(bT)), A, B, scale_row, scale_col,
                         int(bool(broad_cast_row)), int(bool(broad_cast_col)), out, stream)


def gemm_quantize(batch: int, n: int, m: int,
                  mat: DevicePointer,      # (b, n, m) fp16
                  scale: DevicePointer,    # (b, n) or, transposed, (b, m) fp16
                  out: DevicePointer,      # (b, n, m) int8
                  transpose: bool,
                  stream: CUDAStream):
    """gemm_calc_scale[_transpose] + gemm_round[_transpose] in one call (fuses
    torch/gemm.py:5-38)."""
    cpmk.gemm_quantize(batch, n, m, mat, scale, out, int(bool(transpose)), stream)


def gemm_quantize_pair(rows0: int, mat0: DevicePointer, scale0: DevicePointer, out0: DevicePointer,
                       rows1: int, mat1: DevicePointer, scale1: DevicePointer, out1: DevicePointer,
                       m: int, stream: CUDAStream):
    """gemm_quantize(transpose=False) of two tensors with rows of length m (rows0 x m fp16 at
    mat0, rows1 x m at mat1) in one launch."""
    cpmk.gemm_quantize_pair(rows0, mat0, scale0, out0, rows1, mat1, scale1, out1, m, stream)


def gemm_quantize_cols(batch: int, n: int, m: int,
                       mat: DevicePointer,      # (b, n, m) fp16
                       scale: DevicePointer,    # (b, m) fp16
                       out: DevicePointer,      # (b, n, m) int8, or (b, m, n) if out_transposed
                       out_transposed: bool,
                       stream: CUDAStream):
    """gemm_calc_scale_transpose + gemm_round_transpose in one pass (fuses torch/gemm.py:5-38 for
    an operand quantised along dim 1), optionally writing the int8 tensor transposed so that it
    is K-major for gemm_int8."""
    cpmk.gemm_quantize_cols(batch, n, m, mat, scale, out, int(bool(out_transposed)), stream)


def gemm_scale_x(batch: int, n: int, m: int,
                 mat: DevicePointer,        # (b, n, m)  int32
                 scale_x: DevicePointer,    # (b, n)     fp16
                 out: DevicePointer,        # (b, n, m)  fp16
                 stream: CUDAStream):
    """reference: kernels/gemm.py:309-327"""
    cpmk.gemm_scale_x(batch, n, m, mat, scale_x, out, stream)


def gemm_scale_y(batch: int, n: int, m: int,
                 mat: DevicePointer,        # (b, n, m)  int32
                 scale_y: DevicePointer,    # (b, m)     fp16
                 out: DevicePointer,        # (b, n, m)  fp16
                 stream: CUDAStream):
    """reference: kernels/gemm.py:329-347"""
    cpmk.gemm_scale_y(batch, n, m, mat, scale_y, out, stream)


def gemm_int8_scale_one(m: int, k: int, n: int, batchA: int, batchB: int, aT: bool, bT: bool,
                        A: DevicePointer, B: DevicePointer,
                        scale_row: DevicePointer,   # as in gemm_int8_scale; one of the two may be None
                        scale_col: DevicePointer,
                        broad_cast_row: bool, broad_cast_col: bool,
                        out: DevicePointer,         # (batch, n, m)  fp16
                        stream: CUDAStream):
    """gemm_int8 + gemm_scale_x / gemm_scale_y (kernels/gemm.py:309-347) in one launch."""
    assert m % 4 == 0 and n % 4 == 0 and k % 4 == 0
    assert batchA == batchB or batchA == 1 or batchB == 1
    cpmk.gemm_int8_scale_one(m, k, n, batchA, batchB, 1 if aT else 0, 1 if bT else 0, A, B, scale_row, scale_col,
                             1 if broad_cast_row else 0, 1 if broad_cast_col else 0, out, stream)


def gemm_quantize_cols_ld(batch: int, n: int, m: int, mat: DevicePointer,
                          row_scale: DevicePointer,   # (batch, n) fp16, (n) if broad_cast_row, or None
                          broad_cast_row: bool,
                          scale: DevicePointer,       # (batch, m)        fp16
                          out_t: DevicePointer,       # (batch, m, ld_t)  int8, or None
                          ld_t: int,
                          out_n: DevicePointer,       # (batch, n, ld_n)  int8, or None
                          ld_n: int,
                          stream: CUDAStream):
    """Per-column quantisation of mat (times row_scale: gemm_backward_scale_round) in the transposed and / or the matrix's
    own layout, rows filled up with zeros to ld_t / ld_n bytes."""
    cpmk.gemm_quantize_cols_ld(batch, n, m, mat, row_scale, 1 if broad_cast_row else 0, scale, out_t, ld_t, out_n, ld_n, stream)


def gemm_quantize_pair_ld(rows0: int, mat0: DevicePointer, scale0: DevicePointer, out0: DevicePointer,
                          rows1: int, mat1: DevicePointer, scale1: DevicePointer, out1: DevicePointer,
                          m: int, ld: int, stream: CUDAStream):
    """gemm_quantize_pair with int8 rows filled up with zeros to ld bytes; m <= 16384."""
    cpmk.gemm_quantize_pair_ld(rows0, mat0, scale0, out0, rows1, mat1, scale1, out1, m, ld, stream)


def gemm_quantize_cols_rows(batch: int, n: int, m: int, mat: DevicePointer, scale: DevicePointer,
                            out_t: DevicePointer, ld_t: int, out_n: DevicePointer, ld_n: int,      # as in gemm_quantize_cols_ld
                            rows: int,
                            row_mat: DevicePointer,     # (rows, n)     fp16
                            row_scale: DevicePointer,   # (rows)        fp16
                            row_out: DevicePointer,     # (rows, ld_t)  int8
                            stream: CUDAStream):
    """The two operands of a product, one quantised along its columns and the other along its rows, in one launch; n <= 16384."""
    cpmk.gemm_quantize_cols_rows(batch, n, m, mat, scale, out_t, ld_t, out_n, ld_n, rows, row_mat, row_scale, row_out, stream)


def gemm_backward_round_scale_ld(batch: int, n: int, m: int, mat: DevicePointer, scale_y: DevicePointer,
                                 out: DevicePointer,        # (batch, n, ld)  int8
                                 ld: int,
                                 scale_x: DevicePointer,    # (batch, n)      fp16
                                 broad_cast_y: bool, stream: CUDAStream):
    """gemm_backward_round_scale with rows filled up with zeros to ld bytes."""
    cpmk.gemm_backward_round_scale_ld(batch, n, m, mat, scale_y, out, ld, scale_x, 1 if broad_cast_y else 0, stream)


def gemm_backward_quantize_both(batch: int, n: int, m: int,
                                mat: DevicePointer,        # (batch, n, m)     fp16
                                row_scale: DevicePointer, broad_cast_row: bool,        # (batch, n) or (n)
                                scale: DevicePointer,      # (batch, m)        fp16
                                out_t: DevicePointer,      # (batch, m, ld_t)  int8
                                ld_t: int,
                                scale_y: DevicePointer, broad_cast_y: bool,            # (batch, m) or (m)
                                out: DevicePointer,        # (batch, n, ld)    int8
                                ld: int,
                                scale_x: DevicePointer,    # (batch, n)        fp16
                                stream: CUDAStream):
    """gemm_quantize_cols_ld of mat with row scales (transposed) and gemm_backward_round_scale_ld of it in one launch: a gradient on its way
    to both products of a backward pass."""
    cpmk.gemm_backward_quantize_both(batch, n, m, mat, row_scale, 1 if broad_cast_row else 0, scale, out_t, ld_t, scale_y, 1 if broad_cast_y else 0, out, ld,
                                     scale_x, stream)


def gemm_sum_groups(m: int, n: int, batch: int) -> int:
    """Partial sums that gemm_int8_scale_sum / gemm_fp16_sum form for (n, m) outputs over `batch` entries: as few as
    keep the device busy (a divisor of the batch)."""
    return cpmk.gemm_sum_groups(m, n, batch)


def gemm_sum_krows_groups(m: int, k: int, n: int, batch: int) -> int:
    """Groups (up to the batch) for gemm_fp16_parts with k_first, 0 where one product per entry and the sum of them is the quicker."""
    return cpmk.gemm_sum_krows_groups(m, k, n, batch)


def gemm_sum_groups_for(kind: int, m: int, k: int, n: int, batch: int) -> int:
    """The same for a depth of k an entry, or `batch` where one product per entry and the sum of them is the quicker.
    kind 0: gemm_int8_scale_sum, 1: gemm_fp16_sum, 2: gemm_fp16_parts with k_first."""
    return cpmk.gemm_sum_groups_for(kind, m, k, n, batch)


def gemm_sum_groups_timed(kind: int, m: int, k: int, n: int, batch: int) -> int:
    """The quickest number of groups, also where it leaves part of the device idle."""
    return cpmk.gemm_sum_groups_timed(kind, m, k, n, batch)


def gemm_int8_scale_sum(m: int, k: int, n: int, batch: int, groups: int,
                        A: DevicePointer,           # (batch, m, k)     int8
                        B: DevicePointer,           # (batch, n, k)     int8
                        scale_row: DevicePointer,   # (batch, n)        fp16
                        out: DevicePointer,         # (groups, n, m)    fp16
                        stream: CUDAStream):
    """out[g] = sum over the entries of group g of scale_row * (B x A^T): the reference's gemm_int8 + gemm_scale_x +
    sum over the batch (torch/gemm.py:115-186), each sum in fp32 and rounded once.  k is a multiple of 128."""
    assert m % 4 == 0 and n % 4 == 0 and k % 128 == 0
    cpmk.gemm_int8_scale_sum(m, k, n, batch, groups, A, B, scale_row, out, stream)


def gemm_fp16_sum(m: int, k: int, n: int, batch: int, groups: int,
                  A: DevicePointer,         # (batch, m, k)     fp16
                  B: DevicePointer,         # (batch, n, k)     fp16
                  out: DevicePointer,       # (groups, n, m)    fp16
                  stream: CUDAStream):
    """out[g] = sum over the entries of group g of B x A^T: gemm_fp16 + sum over the batch (torch/gemm.py:219-239)."""
    assert m % 4 == 0 and n % 4 == 0 and k % 2 == 0 and k > 32
    cpmk.gemm_fp16_sum(m, k, n, batch, groups, A, B, out, stream)


def gemm_int8_scale_parts(m: int, k: int, n: int, batch: int, groups: int,
                          A: DevicePointer, B: DevicePointer, scale_row: DevicePointer,    # as in gemm_int8_scale_sum
                          parts: DevicePointer,       # (groups, n, m)    fp32
                          stream: CUDAStream):
    """gemm_int8_scale_sum with the groups' sums as fp32, for gemm_add_parts."""
    assert m % 4 == 0 and n % 4 == 0 and k % 128 == 0
    cpmk.gemm_int8_scale_parts(m, k, n, batch, groups, A, B, scale_row, parts, stream)


def gemm_fp16_parts(m: int, k: int, n: int, batch: int, groups: int, k_first: int,
                    A: DevicePointer,         # (batch, m, k)     fp16   [(batch, k, m) if k_first]
                    B: DevicePointer,         # (batch, n, k)     fp16   [(batch, k, n) if k_first]
                    parts: DevicePointer,     # (groups, n, m)    fp32
                    stream: CUDAStream):
    """gemm_fp16_sum with the groups' sums as fp32, for gemm_add_parts.  k_first 2: any sizes and addresses."""
    assert m % 2 == 0 and n % 2 == 0 and k % 2 == 0
    cpmk.gemm_fp16_parts(m, k, n, batch, groups, int(k_first), A, B, parts, stream)


def gemm_add_parts(groups: int, n: int,
                   parts: DevicePointer,      # (groups, n)       fp32
                   out: DevicePointer,        # (n)               fp16
                   stream: CUDAStream):
    """out = sum of the parts, rounded once."""
    assert n % 4 == 0
    cpmk.gemm_add_parts(groups, n, parts, out, stream)


def gemm_depth_parts(f16: bool, m: int, k: int, n: int, batchA: int, batchB: int, aT: bool, bT: bool) -> int:
    """Parts that the depth of a product is worth dividing into (gemm_int8_scale_split, gemm_fp16_split), 1 if none."""
    return cpmk.gemm_depth_parts(1 if f16 else 0, m, k, n, batchA, batchB, 1 if aT else 0, 1 if bT else 0)


def gemm_fp16_copy_pays(m: int, k: int, n: int, batch: int, bT: bool) -> bool:
    """Whether gemm_fp16 of A (batch, k, m) beside one B for all of them is quicker with a copy of A as (batch, m, k)."""
    return cpmk.gemm_fp16_copy_pays(m, k, n, batch, 1 if bT else 0) != 0


def gemm_int8_scale_split(m: int, k: int, n: int, batchA: int, batchB: int, aT: bool, bT: bool,
                          A: DevicePointer, B: DevicePointer, scale_row: DevicePointer, scale_col: DevicePointer,
                          broad_cast_row: bool, broad_cast_col: bool,
                          out: DevicePointer,         # (batch, n, m)  fp16
                          parts: int,
                          workspace: DevicePointer,   # (parts, batch, n, m)  int32
                          stream: CUDAStream):
    """gemm_int8_scale_one with the depth divided into parts that are formed side by side."""
    cpmk.gemm_int8_scale_split(m, k, n, batchA, batchB, 1 if aT else 0, 1 if bT else 0, A, B, scale_row, scale_col,
                               1 if broad_cast_row else 0, 1 if broad_cast_col else 0, out, parts, workspace, stream)


def gemm_fp16_split(m: int, k: int, n: int, batchA: int, batchB: int, aT: bool, bT: bool,
                    A: DevicePointer, B: DevicePointer,
                    out: DevicePointer,         # (batch, n, m)         fp16
                    parts: int,
                    workspace: DevicePointer,   # (parts, batch, n, m)  fp32
                    stream: CUDAStream):
    """gemm_fp16 with the depth divided into parts that are formed side by side, their fp32 sums added and rounded once."""
    cpmk.gemm_fp16_split(m, k, n, batchA, batchB, 1 if aT else 0, 1 if bT else 0, A, B, out, parts, workspace, stream)


def gemm_fp16(m: int, k: int, n: int,
              batchA: int, batchB: int,
              aT: bool, bT: bool,
              A: DevicePointer,      # (bA, k, m) fp16   [(bA, m, k) if aT]
              B: DevicePointer,      # (bB, n, k) fp16   [(bB, k, n) if bT]
              out: DevicePointer,    # (max(bA, bB), n, m) fp16
              stream: CUDAStream):
    """reference: kernels/gemm.py:188-256 (cuBLASLt); same asserts (:200-201).  fp32 accumulation."""
    assert m % 2 == 0 and n % 2 == 0 and k % 2 == 0
    assert batchA == batchB or batchA == 1 or batchB == 1
    cpmk.gemm_fp16(m, k, n, batchA, batchB, int(bool(aT)), int(bool(bT)), A, B, out, stream)


def gemm_backward_round_scale(batch: int, n: int, m: int,
                              mat: DevicePointer,        # (batch, n, m) fp16
                              scale_y: DevicePointer,    # (batch, m)    fp16
                              out: DevicePointer,        # (batch, n, m) int8
                              scale_x: DevicePointer,    # (batch, n)    fp16
                              broad_cast_y: bool,
                              stream: CUDAStream):
    """Row scales and int8 rounding of mat * scale_y.  reference: kernels/gemm.py:261-283"""
    cpmk.gemm_backward_round_scale(batch, n, m, mat, scale_y, out, scale_x, int(bool(broad_cast_y)), stream)


def gemm_backward_scale_round(batch: int, n: int, m: int,
                              mat: DevicePointer,        # (batch, n, m) fp16
                              scale_x: DevicePointer,    # (batch, n)    fp16
                              out: DevicePointer,        # (batch, n, m) int8
                              scale_y: DevicePointer,    # (batch, m)    fp16
                              broad_cast_x: bool,
                              stream: CUDAStream):
    """Column scales and int8 rounding of mat * scale_x.  reference: kernels/gemm.py:285-307"""
    cpmk.gemm_backward_scale_round(batch, n, m, mat, scale_x, out, scale_y, int(bool(broad_cast_x)), stream)
