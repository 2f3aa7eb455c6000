"""How a step's tokens are cut into the plain attention's tiles (kernels/ops.py)."""
import pytest

from herbert_rs_amd.kernels.ops import token_tiles


@pytest.mark.parametrize("portions,held", [([512] + [1] * 15, [512] + [4096] * 15), ([2] * 9, [100, 3, 700, 64, 65, 2, 9, 10, 11]),
                                           ([1], [1]), ([70, 3, 100, 1], [70, 3, 129, 200])])
@pytest.mark.parametrize("most", [2, 5, 16])
def test_no_tile_holds_tokens_of_two_sequences(portions, held, most):
    """Every token is in one tile, a tile's tokens are neighbours of one sequence, and the tiles that see the most keys come first."""
    starts = [0]
    for n in portions:
        starts.append(starts[-1] + n)
    tiles = token_tiles(starts, held, most)
    assert sorted(t for first, n in tiles for t in range(first, first + n)) == list(range(starts[-1]))
    owner = [i for i, n in enumerate(portions) for _ in range(n)]
    position = [held[i] - n + j for i, n in enumerate(portions) for j in range(n)]
    for first, n in tiles:
        assert 0 < n <= most and len(set(owner[first:first + n])) == 1
    assert [position[first] for first, _ in tiles] == sorted((position[first] for first, _ in tiles), reverse=True)
    assert len(tiles) == sum(-(-n // most) for n in portions)
