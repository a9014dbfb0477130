"""Token embedding with the interface of cpm_kernels/torch/embedding.py: ids (batch, seq) ->
(batch, embedding_size, seq); the gradient sums the rows of equal ids, as the two-stage sorted scatter-add of the
reference does."""
import torch
from ..kernels import embedding_forward, embedding_backward_prepare, embedding_backward_rows
from ._common import cur_stream, check_half

# More tokens than this are put in order by a radix sort: counting ranks is quadratic in their number (4096 tokens: 10 us
# against 35 us for the sort's launches, 16384: 26 against 35 us, 32768: 75 against 44 us).
MAX_RANKED = 16384


class OpEmbedding(torch.autograd.Function):
    """reference: torch/embedding.py:4-76"""

    @staticmethod
    def forward(ctx, ids: torch.Tensor, weight: torch.Tensor):
        assert ids.is_cuda and weight.is_cuda and ids.device == weight.device
        assert ids.ndim == 2 and ids.dtype == torch.int32
        check_half(weight, 2)
        if not ids.is_contiguous():
            ids = ids.contiguous()
        ctx.save_for_backward(ids, weight)
        out = torch.empty((ids.size(0), weight.size(1), ids.size(1)), device=ids.device, dtype=torch.half)
        embedding_forward(ids.size(0), weight.size(1), ids.size(1), ids.data_ptr(), weight.data_ptr(), out.data_ptr(),
                          cur_stream())
        return out

    @staticmethod
    def backward(ctx, grad_output: torch.Tensor):
        ids, weight = ctx.saved_tensors
        batch, n, m = grad_output.size()           # (batch, embedding_size, seq)
        assert grad_output.device == ids.device and grad_output.dtype == torch.half
        assert m == ids.size(1) and n == weight.size(1)
        if not grad_output.is_contiguous():
            grad_output = grad_output.contiguous()
        tokens, st = ids.numel(), cur_stream()
        # one workspace: the gradient rows, fp32 partial sums, and the order of the ids
        rows_bytes, partial_bytes = 2 * tokens * n, 8 * ((tokens + 31) // 32) * n
        rows_bytes += -rows_bytes % 16
        work = torch.empty((rows_bytes + partial_bytes + 8 * tokens,), device=grad_output.device, dtype=torch.uint8)
        rows = work.data_ptr()
        partials = rows + rows_bytes
        order = partials + partial_bytes
        sorted_ids = order + 4 * tokens
        unordered = ids.data_ptr()
        if tokens > MAX_RANKED:
            sort_result = ids.view(-1).sort()
            indices = sort_result.indices.to(torch.int32)
            order, sorted_ids, unordered = indices.data_ptr(), sort_result.values.data_ptr(), None
        ret = torch.empty((weight.size(0), n), device=grad_output.device, dtype=torch.half)
        embedding_backward_prepare(batch, n, m, weight.size(0), unordered, order, sorted_ids, grad_output.data_ptr(), rows, ret.data_ptr(), st)
        embedding_backward_rows(tokens, n, rows, order, sorted_ids, ret.data_ptr(), partials, st)
        return None, ret


class Embedding(torch.nn.Module):
    """reference: torch/embedding.py:78-84 (the weight is allocated uninitialised there too)."""

    def __init__(self, vocab_size: int, embedding_size: int):
        super().__init__()
        self.weight = torch.nn.Parameter(torch.empty((vocab_size, embedding_size), dtype=torch.half))

    def forward(self, ids: torch.Tensor):
        return OpEmbedding.apply(ids, self.weight)


class EmbeddingTH(torch.nn.Module):
    """reference: torch/embedding.py:86-99"""

    def __init__(self, vocab_size: int, embedding_size: int):
        super().__init__()
        self.weight = torch.nn.Parameter(torch.empty((vocab_size, embedding_size), dtype=torch.half))

    def forward(self, ids: torch.Tensor):
        assert ids.ndim == 2
        v = torch.embedding(self.weight, ids)
        assert v.ndim == 3
        return v.transpose(1, 2)
