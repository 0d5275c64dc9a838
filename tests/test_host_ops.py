"""Host side of packkv_amd/ops.py: checks that come before any launch, on tensors without a GPU."""
import pytest
import torch

from packkv_amd import ops


def test_rotary_tables_on_another_device_than_the_tokens_are_refused():
    """The kernels get bare addresses, so a host table must not pass: the tokens are on the meta device here."""
    like = torch.empty(2, 5, 7, 128, dtype=torch.float16, device="meta")
    here, there = torch.empty(2, 7, 128, dtype=torch.float16, device="meta"), torch.zeros(2, 7, 128, dtype=torch.float16)
    for cos, sin in ((there, there), (there, here), (here, there)):
        with pytest.raises(RuntimeError, match="one device"):
            ops._rotary_rows(cos, sin, like)
