"""The launch order of a batch of different circuits: every tile of every pass once, a circuit's
passes in one branch and in order, the longest passes of a launch first."""
from types import SimpleNamespace

import pytest

from qandle_amd._engine.uneven import BRANCHES, _Levels


@pytest.mark.parametrize("passes", [[1], [1, 1, 2], [3, 1, 7, 4, 5, 2, 1], [9, 8]])
def test_levels(passes):
    levels, tiles, k = _Levels(), {}, 0
    owner = {}
    for ci, npass in enumerate(passes):
        c = SimpleNamespace(plan=SimpleNamespace(passes=[None] * npass))
        for level in range(npass + 1):  # one step more than passes, as a backward has
            tiles[k], owner[k] = 1 + (3 * k) % 4, (ci, level, 10 + (7 * k) % 5)
            levels.add(level, k, tiles[k], c, owner[k][2])
            k += 1
    items, counts, branches = levels.build("cpu")
    assert [len(t) // 2 for t in items] == counts and sum(counts) == sum(tiles.values())
    assert len(branches) == len({min(p, BRANCHES) for p in passes})
    seen, where = [], {}
    for b, branch in enumerate(branches):
        assert [x[0] for x in branch] == sorted({x[0] for x in branch})
        for level, first, cnt in branch:
            its = items[level].view(-1, 2)[first:first + cnt].tolist()
            words = [owner[d][2] for d, _t in its]
            assert words == sorted(words, reverse=True)
            for d, t in its:
                assert owner[d][1] == level and where.setdefault(owner[d][0], b) == b
                seen.append((d, t))
    assert sorted(seen) == sorted((d, t) for d in tiles for t in range(tiles[d]))
