"""The G-buffer's fill value on the CPU: what a caller may pass as ``default``
(lists, tuples, arrays, tensors, NaN, none at all) gives the values that
torch.tensor gives."""
import numpy as np
import pytest
import torch

from diffrp_amd.deferred import _fill_value

NAN = float('nan')


@pytest.mark.parametrize('default', [
    [0.0], [1.0, 0.0, 1.0], (0, 1), [], [NAN, 0.0], [0.0, NAN], [NAN, NAN], [float('inf'), -1e30],
    np.array([0.0, 0.5, 1.0]), np.zeros(4, np.float32), torch.tensor([0.1, 0.2]), torch.zeros(3),
], ids=str)
def test_fill_value_matches_tensor(default):
    want = torch.as_tensor(default, dtype=torch.float32)
    got = _fill_value(default, torch.device('cpu'))
    assert got.dtype == torch.float32 and got.shape == want.shape
    assert torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))
