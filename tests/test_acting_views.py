"""Which observation views the one-launch actor reads in place: row r, column c at r * pitch + c, as the kernel does."""

import itertools

import pytest
import torch

from robolearn_amd import kernels as K


@pytest.mark.parametrize("rows,columns", itertools.product((1, 2, 5), (1, 2, 6)))
def test_rows_are_read_in_place_or_after_a_copy(rows, columns):
    storage = torch.arange(400.0)
    for s0, s1, obs_dim in itertools.product((0, 1, 2, 5, 6, 9), (0, 1, 2, 5, 6), range(1, columns + 1)):
        view = storage.as_strided((rows, columns), (s0, s1), 3)
        expected = view[:, :obs_dim].clone()
        x = view if K.actor_rows_readable(view, obs_dim) else view[:, :obs_dim].contiguous()
        assert K.actor_rows_readable(x, obs_dim), (s0, s1, obs_dim)
        pitch = max(x.stride(0), obs_dim)
        read = x.as_strided((rows, obs_dim), (pitch, 1))
        assert torch.equal(read, expected), (s0, s1, obs_dim)
        # the last value read lies inside the tensor's storage
        assert x.storage_offset() + (rows - 1) * pitch + obs_dim <= x.untyped_storage().nbytes() // 4
