"""GPU kernels at the sizes where their launch shapes change, word for word against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import oracle as O  # noqa: E402
import stwo_hip as S  # noqa: E402


@pytest.mark.parametrize("log_n", [0, 1, 2, 3, 4, 9, 10, 11, 12, 13, 14, 17])
@pytest.mark.parametrize("start", [1, 3, 0x155])
def test_twiddle_tree_levels(log_n, start):
    """One block writes 2^12 values of level 0 and every level above them: sizes below, at and past
    one block, with starting points other than the canonic one."""
    c = S.Coset((start << (29 - log_n)) & 0x7FFFFFFF, (1 << (31 - log_n)) & 0x7FFFFFFF, log_n)
    tree = S.precompute_twiddles(c)
    tw, itw = O.precompute_twiddles(c.initial_index, c.step_size, c.log_size)
    assert (tree.twiddles.to_numpy() == tw).all()
    assert (tree.itwiddles.to_numpy() == itw).all()
