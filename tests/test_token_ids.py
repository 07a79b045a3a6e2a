"""Token ids on their way to the device: int32 or an error, never another token."""
import numpy as np
import pytest
import torch

from nl_hecate_amd.serving import host_ids


@pytest.mark.parametrize("make", [list, np.array, torch.tensor, tuple, lambda x: np.array(x, np.uint8), lambda x: np.array(x, np.uint32),
                                  lambda x: torch.tensor(x, dtype=torch.int32), lambda x: np.array(x, np.float64),
                                  lambda x: [np.int64(t) for t in x], lambda x: [torch.tensor(t) for t in x]])
def test_whole_numbers_of_any_type(make):
    got = host_ids(make([0, 5, 127]))
    assert got.dtype == np.int32 and got.tolist() == [0, 5, 127]


def test_range():
    assert host_ids([]).dtype == np.int32 and host_ids([]).size == 0
    assert host_ids([-1, -2 ** 31, 2 ** 31 - 1]).tolist() == [-1, -2 ** 31, 2 ** 31 - 1]   # targets outside the vocabulary are skipped
    assert host_ids([True, 2.9]).tolist() == [1, 2]


@pytest.mark.parametrize("bad", [[2 ** 32 + 5], [2 ** 31], [-2 ** 31 - 1], [2 ** 63], [2 ** 70], [2.0 ** 40], np.array([2 ** 31], np.uint32),
                                 torch.tensor([2 ** 40])])
def test_ids_that_do_not_fit_are_refused(bad):
    with pytest.raises((RuntimeError, OverflowError)):
        host_ids(bad)


@pytest.mark.parametrize("bad", [[float("nan")], [float("inf")]])
def test_ids_that_are_no_numbers_are_refused(bad):
    with pytest.raises((ValueError, OverflowError)):
        host_ids(bad)
