"""Token-embedding gathers with the signatures of cpm_kernels/kernels/embedding.py ."""
from ..library import cpmk
from .base import DevicePointer, CUDAStream


def embedding_forward(batch: int,
                      hidden_size: int,          # hidden size
                      seq_len: int,              # sequence length
                      ids: DevicePointer,        # (batch, seq_len) int32
                      weights: DevicePointer,    # (vocab_size, hidden_size) fp16
                      out: DevicePointer,        # (batch, hidden_size, seq_len) fp16
                      stream: CUDAStream):
    """reference: kernels/embedding.py:14-34"""
    cpmk.embedding_forward(batch, hidden_size, seq_len, ids, weights, out, stream)


def embedding_step(batch: int, embedding_size: int,
                   ids: DevicePointer,            # (batch,) int32
                   weights: DevicePointer,        # (vocab_size, embedding_size) fp16
                   out: DevicePointer,            # (batch, embedding_size) fp16
                   stream: CUDAStream):
    """reference: kernels/embedding.py:88-105"""
    cpmk.embedding_step(batch, embedding_size, ids, weights, out, stream)


def embedding_backward_stage1(batch: int, seq_len: int, hidden_size: int,
                              grad_out: DevicePointer,        # (batch * n, m)
                              argsort_ids: DevicePointer,     # (batch, n)
                              sorted_ids: DevicePointer,      # (batch, n)
                              grad: DevicePointer,            # (vocab_size, m)
                              aux_grad: DevicePointer,        # (batch, m)
                              aux_grad_idx: DevicePointer,    # (batch)
                              stream: CUDAStream):
    """Sums runs of equal sorted ids inside each batch entry.  reference: kernels/embedding.py:36-65"""
    cpmk.embedding_backward_stage1(batch, seq_len, hidden_size, grad_out, argsort_ids, sorted_ids, grad, aux_grad,
                                   aux_grad_idx, stream)


def embedding_backward_stage2(batch: int, hidden_size: int,
                              aux_grad: DevicePointer,        # (batch, m)
                              aux_grad_idx: DevicePointer,    # (batch)
                              grad: DevicePointer,            # (vocab_size, m)
                              stream: CUDAStream):
    """Adds the per-entry tail runs into grad.  reference: kernels/embedding.py:67-86"""
    cpmk.embedding_backward_stage2(batch, hidden_size, aux_grad, aux_grad_idx, grad, stream)


def embedding_order_ids(tokens: int,
                        ids: DevicePointer,             # (tokens) int32
                        order: DevicePointer,           # (tokens) int32
                        sorted_ids: DevicePointer,      # (tokens) int32
                        stream: CUDAStream):
    """The tokens in the order of their ids, equal ids in the order of the tokens (quadratic in the number of tokens)."""
    cpmk.embedding_order_ids(tokens, ids, order, sorted_ids, stream)


def embedding_backward_rows(tokens: int, hidden_size: int,
                            grad_rows: DevicePointer,   # (tokens, hidden_size) fp16
                            order: DevicePointer,       # (tokens) int32: tokens sorted by their ids
                            sorted_ids: DevicePointer,  # (tokens) int32
                            grad: DevicePointer,        # (vocab_size, hidden_size) fp16, rows of absent ids are left alone
                            partials: DevicePointer,    # 2 * ceil(tokens / 32) * hidden_size fp32
                            stream: CUDAStream):
    """What embedding_backward_stage1 and _stage2 compute together, summed in fp32 and rounded once."""
    cpmk.embedding_backward_rows(tokens, hidden_size, grad_rows, order, sorted_ids, grad, partials, stream)


def embedding_backward_prepare(batch: int, hidden_size: int, seq_len: int, vocab_size: int,
                               ids: DevicePointer,          # (batch * seq_len) int32, or None: order and sorted_ids are there already
                               order: DevicePointer, sorted_ids: DevicePointer,     # as in embedding_order_ids
                               grad_out: DevicePointer,     # (batch, hidden_size, seq_len) fp16
                               grad_rows: DevicePointer,    # (batch * seq_len, hidden_size) fp16
                               grad: DevicePointer,         # (vocab_size, hidden_size) fp16: cleared
                               stream: CUDAStream):
    """What embedding_backward_rows needs, in one launch: the order of the ids, grad_out as rows, zeros in the table."""
    cpmk.embedding_backward_prepare(batch, hidden_size, seq_len, vocab_size, ids, order, sorted_ids, grad_out, grad_rows, grad, stream)
