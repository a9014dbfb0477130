"""The stream that the torch-level operators launch on."""
import threading

import pytest
import torch

from cpm_kernels_amd.torch._common import cur_stream

pytestmark = pytest.mark.gpu


def test_current_stream_is_torchs():
    assert cur_stream() == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert cur_stream() == side.cuda_stream != 0
        seen = []
        t = threading.Thread(target=lambda: seen.append(cur_stream()))      # (a thread has a current stream of its own)
        t.start()
        t.join()
        assert seen == [torch.cuda.default_stream().cuda_stream]
    assert cur_stream() == torch.cuda.current_stream().cuda_stream
    with torch.cuda.device(0), torch.cuda.stream(torch.cuda.Stream(0)):
        assert cur_stream() == torch.cuda.current_stream().cuda_stream
