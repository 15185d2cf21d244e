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


GB = 1 << 30
SIZES = [1 << 20, 100 << 20, GB, 4 * GB - 1, 4 * GB, 12 * GB, 32 * GB, 60 * GB]


@pytest.mark.parametrize("want", SIZES)
@pytest.mark.parametrize("free", [0, 50 << 20, GB, 6 * GB, 40 * GB, 280 * GB])
def test_workspace_leaves_three_quarters(want, free):
    """A context alone takes a quarter of the free memory at most, at every size;
    what it has it keeps."""
    room = m2l_plan.lib().plan_room
    assert room(want, 0, 0, free) == min(want, free // 4)
    for own in (GB, 8 * GB):
        got = room(want, own, own, free)
        assert min(want, own) <= got <= max(own, (free + own) // 4)


def test_workspaces_of_several_contexts():
    """Contexts one after the other, 2 GB of other buffers each: together at most a
    quarter of what the other buffers leave, but for a sixteenth of the wish each."""
    room = m2l_plan.lib().plan_room
    total, want, free, held = 288 * GB, 12 * GB, 288 * GB, 0
    for n in range(60):
        free -= 2 * GB
        got = room(want, 0, held, free)
        assert want // 16 <= got <= free // 4
        held, free = held + got, free - got
        assert held <= total // 4 + (n + 1) * (want // 16)
    assert free > 0


@pytest.mark.parametrize("rank", list(ranks()), ids=lambda r: f"sum{int(r.sum())}")
@pytest.mark.parametrize("step", [1, 2])
def test_parts_fit_the_room(rank, step):
    """The parts cover the rows in whole steps; C and the partial locals fit the room,
    or a part is one step; one part only where all of it fits."""
    rboff = m2l_plan.rows(rank)[3].astype(np.int64)
    nrb, ncell, max_part = len(rboff) - 1, 20011, 116
    whole, acc = int(rboff[-1]) * ncell, 4096 * ncell
    for room in (0, whole // 50, whole // 5, whole // 2, whole - 1, whole, 2 * whole):
        cut, size = m2l_plan.cut(rboff, step, max_part, ncell, acc, room)
        assert cut[0] == 0 and cut[-1] == nrb
        assert (np.diff(cut) > 0).all() and (np.diff(cut) <= max_part).all() and (cut[:-1] % step == 0).all()
        widths = (rboff[cut[1:]] - rboff[cut[:-1]]) * ncell
        assert size == widths.max()
        if len(cut) == 2:
            assert size <= room or nrb <= step
        else:
            assert whole > room or nrb > max_part
            assert (widths[np.diff(cut) > step] + acc <= room).all()
