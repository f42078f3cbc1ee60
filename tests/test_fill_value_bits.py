"""The G-buffer collect's fill value holds what torch.tensor makes of the
default, bit for bit: signed zeros, and values past float32's range."""
import pytest
import torch

from diffrp_amd import deferred


@pytest.mark.parametrize('default', [
    [0.0, -0.0, 0.0], [-0.0, 0.0], [-0.0], [1e39, 0.0], [0.0, -1e39, 1e-50], [float('inf'), float('-inf'), 2.0],
    [float('nan'), 1.0], [1.0, float('nan')], [0.1, 0.1, 0.2], [2 ** 70, True], []])
def test_fill_value_bits(default):
    want = torch.tensor(default, dtype=torch.float32)
    got = deferred._fill_value(default, 'cpu')
    assert got.dtype == torch.float32 and got.shape == want.shape
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))
