"""How a step's long portions are cut into chunks and calls (kernels/recurrent.py): every token once and in order, no call
beyond its room, long portions not held up by short ones."""
import random

import numpy as np
import pytest

from herbert_rs_amd.kernels import recurrent


def covered(starts, least, room):
    """Walk through the calls and return how many there are; each portion's tokens must come once, in order."""
    at = {i: int(row) for i, row in enumerate(starts[:-1])}
    calls = recurrent.chunk_calls(np.array(starts, dtype=np.int32), least, room)
    for runs, chunks in calls:
        assert 0 < len(chunks) <= room
        assert [run[3] for run in runs] == sorted((run[3] for run in runs), reverse=True)
        places = []
        for seq, first, row, tokens in runs:
            assert row == at[seq] and starts[seq + 1] - starts[seq] >= least
            n = -(-tokens // recurrent.CHUNK)
            assert chunks[first:first + n] == [(row + 64 * i, min(64, tokens - 64 * i)) for i in range(n)]
            assert tokens % 64 == 0 or row + tokens == starts[seq + 1]         # (only a portion's end leaves a chunk short)
            at[seq] = row + tokens
            places += range(first, first + n)
        assert sorted(places) == list(range(len(chunks)))
    for i, row in at.items():
        n = starts[i + 1] - starts[i]
        assert row == (starts[i + 1] if n >= least else starts[i])
    return len(calls)


@pytest.mark.parametrize("seed", range(20))
def test_every_token_once_and_no_call_beyond_its_room(seed):
    rng = random.Random(seed)
    portions = [int(np.exp(rng.uniform(0, 7))) for _ in range(rng.randint(1, 60))] + [0, 64, 128, 129]
    starts = [0] + list(np.cumsum(portions))
    for room in (1, 2, 7, 64, 10000):
        covered(starts, rng.choice((1, 40, 96)), room)


def test_short_portions_leave_their_room_to_a_long_one():
    starts = [0, 2048] + [2048 + i for i in range(1, 65)]
    assert covered(starts, 40, 32) == 1                                   # one prompt beside 64 single tokens: its 32 chunks
    starts = [0, 2048] + [2048 + 40 * i for i in range(1, 65)]
    assert covered(starts, 40, 96) == 1                                   # beside 64 portions of one chunk each


def test_many_short_portions_keep_the_scratch_bounded():
    """256 portions of 64 tokens, 32 heads of 128 x 128: a chunk each would take 1.2 GB in one call."""
    size = recurrent.chunk_floats(128, 128, True)
    room = recurrent.CHUNK_SCRATCH // (32 * size)
    calls = recurrent.chunk_calls(np.arange(0, 257 * 64, 64), 40, room)
    assert max(len(chunks) for _, chunks in calls) * 32 * size <= recurrent.CHUNK_SCRATCH
    assert sum(len(chunks) for _, chunks in calls) == 256


def test_the_portions_that_take_chunks_decide():
    """The lines for many portions count those that are long enough, not the single tokens beside them."""
    ones = [1] * 47
    for few, many, form in ((112, 32, (True, False)), (96, 40, (True, True)), (48, 20, (False, True))):
        assert recurrent.chunks_from(np.array([few - 1] + ones), 16, *form) == few                # none
        assert recurrent.chunks_from(np.array([few] + ones), 16, *form) == few
        assert recurrent.chunks_from(np.array([many] * 8 + ones), 16, *form) == many
        assert recurrent.chunks_from(np.array([many - 1] * 80 + ones), 16, *form) == many         # none


@pytest.mark.parametrize("portions,least,launches", [([1, 1], 96, 1), ([0, 0], 96, 0), ([3, 0, 1], 96, 1), ([5] + [1] * 8, 96, 2),
                                                     ([9, 2, 30], 24, 1), ([2, 1, 1, 1, 1, 0], 2, 1), ([40, 1], 1, 0)])
def test_every_other_portion_is_in_one_walk(portions, least, launches):
    walks = recurrent.walks_of(np.array(portions), least, 16)
    assert len(walks) == launches and all(w == sorted(w) for w in walks)
    assert sorted(i for w in walks for i in w) == [i for i, n in enumerate(portions) if 0 < n < least]
