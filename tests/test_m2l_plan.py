"""Host side of the FP64 M2L (csrc/m2l_plan.hpp), without a GPU."""
import numpy as np
import pytest

import m2l_plan


def ranks():
    rng = np.random.default_rng(3)
    yield np.full(56, 1)
    yield np.full(56, 64)
    for lo, hi in ((4, 14), (8, 40), (1, 64)):
        yield rng.integers(lo, hi + 1, 56)


@pytest.mark.parametrize("rank", list(ranks()), ids=lambda r: f"sum{int(r.sum())}")
def test_masked_rows_lie_past_every_buffer(rank):
    """In every part of the rows, a row's place is within the part's C, and a
    masked lane's address (kNowhere plus that place) neither falls before kNowhere
    nor wraps: also for the rows that fill the last block."""
    tau, off, last, rboff = m2l_plan.rows(rank)
    nowhere = m2l_plan.lib().plan_nowhere()
    nrb = len(rboff) - 1
    assert rboff[nrb] < 1 << 20
    for rb0 in range(0, nrb, 2):
        at = off[16 * rb0:].astype(np.int64) - int(rboff[rb0])
        assert (at >= 0).all(), rb0
        assert (last[16 * rb0:].astype(np.int64) - int(rboff[rb0]) + nowhere < 1 << 32).all(), rb0
        filler = tau[16 * rb0:] == 56
        assert (last[16 * rb0:][~filler] < rboff[nrb]).all()
