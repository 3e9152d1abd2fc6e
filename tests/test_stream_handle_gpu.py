"""The raw handle of a device's current stream, for every way a caller may name the device."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_every_name_of_a_device():
    from gbx_lm_amd import mixer_ops, ops
    side = torch.cuda.Stream()
    for stream in (torch.cuda.current_stream(), side):
        with torch.cuda.stream(stream):
            for name in ("cuda:0", "cuda", 0, torch.device("cuda"), torch.device("cuda:0"), torch.device("cuda", 0)):
                assert ops._stream_ptr(name) == mixer_ops._stream(name) == stream.cuda_stream
