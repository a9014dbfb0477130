import torch

_raw_stream, _device = getattr(torch._C, "_cuda_getCurrentRawStream", None), getattr(torch._C, "_cuda_getDevice", None)


def cur_stream() -> int:
    """Raw hipStream_t of torch's current stream (ROCm builds keep the ``cuda`` names).  Asked for by its number: the stream
    object in between costs 2.5 us, as much as a launch, and a training step of the ffn block asks nineteen times.  (A build of torch without these two calls is asked for the object.)"""
    if _raw_stream is None or _device is None or not torch.cuda.is_initialized():         # (nor in a forked child: torch's own call initialises or refuses)
        return torch.cuda.current_stream().cuda_stream
    return _raw_stream(_device())


def check_half(x: torch.Tensor, ndim=None):
    assert x.is_cuda and x.is_contiguous() and x.dtype == torch.float16
    if ndim is not None:
        assert x.ndim == ndim
