"""The comparison helper: what is not a number is never close."""
import pytest
import torch

from tests.util import assert_close


def test_nan_and_infinities():
    nan, inf = float("nan"), float("inf")
    t = torch.tensor
    assert_close(t([1., inf, -inf]), t([1. + 1e-7, inf, -inf]), 1e-5, 1e-5)
    for got, want in (([nan, 1.], [1., 1.]), ([1.], [nan]), ([inf], [1.]), ([inf], [-inf]), ([1.], [inf])):
        with pytest.raises(AssertionError):
            assert_close(t(got), t(want), 1e-2, 1e-2)
    with pytest.raises(AssertionError, match="shape"):
        assert_close(torch.zeros(2, 3), torch.zeros(1, 3), 1e-2, 1e-2)
