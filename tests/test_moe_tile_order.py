"""In which order workgroups of an expert product take its tiles
(csrc/moe.h): every tile once, row tiles of an expert together."""

import pytest


def _order(experts, n_blocks, split, tile_rows=256):
    try:
        from vllm_amd.ops import hip_ops
    except (ImportError, OSError) as e:
        pytest.skip(f"extension not built: {e}")
    flat = hip_ops._C.moe_tile_order(experts, n_blocks, split, tile_rows)
    return [tuple(flat[i:i + 3]) for i in range(0, len(flat), 3)]


# Experts of one tile, of a group, of one more, and of more than the 64 tiles
# that a wave looks at together; fewer tiles than parts.
@pytest.mark.parametrize("counts", [
    [1], [1, 1, 1], [8, 9, 1, 17], [3, 64, 65, 130, 2], [1] * 70 + [200]])
@pytest.mark.parametrize("n_blocks,split", [(1, 1), (6, 2), (28, 4), (112, 8)])
def test_every_tile_once_and_experts_together(counts, n_blocks, split):
    experts = [e for e, n in enumerate(counts) for _ in range(n)]
    order = _order(experts, n_blocks, split)
    assert sorted((m, n) for _, m, n in order) == [
        (m, n) for m in range(len(experts)) for n in range(n_blocks)]
    for xcd in range(8):
        mine = [(m, n) for x, m, n in order if x == xcd]
        tiles = sorted({m for m, _ in mine})
        if len(tiles) <= 8:
            # All together: the row tiles of a column block follow each other.
            assert mine == [(m, n) for n in sorted({n for _, n in mine})
                            for m in tiles]
            continue
        # An expert's tiles before the next one's, and as few groups as hold
        # eight tiles each: a group is done with a block before the next.
        assert [experts[m] for m, _ in mine] == sorted(
            experts[m] for m, _ in mine)
        for e in {experts[m] for m in tiles}:
            own = [m for m in tiles if experts[m] == e]
            first = [m for m, n in mine if experts[m] == e
                     and n == min(n for _, n in mine)]
            assert first == own
            runs = [(m, n) for m, n in mine if experts[m] == e]
            groups = 1 + sum(b[1] < a[1] for a, b in zip(runs, runs[1:]))
            blocks = len({n for _, n in runs})
            assert blocks == 1 or groups == -(-len(own) // 8)


# Tiles of 128 rows of which an XCD has all: up to 16 stay in groups of eight
# across experts, where one has two of them.
@pytest.mark.parametrize("counts,across", [
    ([1, 2, 1, 1, 2, 1, 1], True), ([2] * 8, True), ([1] * 7 + [9], True),
    ([1] * 15 + [2], False), ([1] * 12, False), ([2, 1, 1], None)])
@pytest.mark.parametrize("split,tile_rows", [(8, 128), (8, 256), (4, 128)])
def test_few_tiles_of_uneven_experts(counts, across, split, tile_rows):
    experts = [e for e, n in enumerate(counts) for _ in range(n)]
    tiles, n_blocks = len(experts), 28
    order = _order(experts, n_blocks, split, tile_rows)
    assert sorted((m, n) for _, m, n in order) == [
        (m, n) for m in range(tiles) for n in range(n_blocks)]
    for xcd in range(8):
        mine = [(m, n) for x, m, n in order if x == xcd]
        blocks = sorted({n for _, n in mine})
        here = sorted({m for m, _ in mine})
        if across and split == 8 and tile_rows == 128:
            groups = [here[:8], here[8:]]
        elif len(here) <= 8:
            groups = [here]
        else:
            groups = [[m for m in here if experts[m] == e]
                      for e in range(len(counts))]
            groups = [h for g in groups for h in (
                [g] if len(g) <= 8 else [g[:len(g) // 2], g[len(g) // 2:]])]
        assert mine == [(m, n) for g in groups for n in blocks for m in g]
