"""GPU: convolutions over no lines."""
import pytest
import torch

from rubix_amd import _lib

pytestmark = pytest.mark.gpu


def test_dot_of_no_lines():
    """n_outer = 0 is a sum of nothing, not an error."""
    buf = torch.ones(64, device="cuda")
    taps = torch.ones(3, dtype=torch.float64, device="cuda")
    res = torch.full((), 7.0, dtype=torch.float64, device="cuda")
    ws = torch.empty(1 << 16, dtype=torch.uint8, device="cuda")
    _lib.call("rbx_conv_axis_dot", _lib.ptr(buf), _lib.ptr(buf), 0, 4, 16, _lib.ptr(taps), 3, 1,
              _lib.ptr(res), _lib.ptr(ws), ws.numel(), _lib.stream_handle(buf.device))
    assert float(res) == 0.0
