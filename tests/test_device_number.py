"""A python number as a device tensor, and the handle of the current stream."""
import math

import pytest
import torch

from rubix_amd import _lib, ops


@pytest.mark.parametrize("value", [0, 1, True, 2.5, 1 / 3, -1e-40, 3.4028234e38, 1e300, math.inf, math.nan])
@pytest.mark.parametrize("shape", [(), (3,), (2, 0)])
@pytest.mark.parametrize("dtype", [None, torch.float32, torch.float64])
def test_device_number_is_the_tensor_of_the_number(value, shape, dtype):
    want = torch.tensor(float(value), dtype=dtype).expand(shape)
    got = ops.device_number(value, shape, torch.device("cpu"), dtype)
    assert got.dtype == want.dtype and got.shape == want.shape and got.is_contiguous()
    assert torch.equal(got.nan_to_num(nan=7.0, posinf=8.0), want.nan_to_num(nan=7.0, posinf=8.0))


@pytest.mark.gpu
def test_stream_handle_is_the_current_stream():
    dev = torch.zeros(1, device="cuda").device
    side = torch.cuda.Stream()
    for d in (dev, "cuda", None, 0):
        assert (_lib.stream_handle(d).value or 0) == torch.cuda.current_stream().cuda_stream
        with torch.cuda.stream(side):
            assert _lib.stream_handle(d).value == side.cuda_stream
