"""The stream that calls go to is torch's current one, whichever it is."""
import pytest
import torch

from luisaml_amd import capi

pytestmark = pytest.mark.gpu


def test_current_stream(dev):
    assert capi._stream() == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert capi._stream() == side.cuda_stream == torch.cuda.current_stream().cuda_stream
        x = torch.full((1 << 22,), 3.0, device=dev)
        y = capi.activation(x, capi.ACT_NONE)
        z = y + 1.0  # on the same stream: ordered after the call
    side.synchronize()
    assert bool((z == 4.0).all())
    assert capi._stream() == torch.cuda.current_stream().cuda_stream
    assert capi._stream(side) == side.cuda_stream and capi._stream(123) == 123
