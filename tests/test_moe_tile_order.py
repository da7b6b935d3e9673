"""In which order workgroups of an expert product take its tiles
(csrc/moe.h): every tile once, row tiles of an expert together."""

import pytest


def _order(experts, n_blocks, split):
    try:
        from vllm_amd.ops import hip_ops
    except (ImportError, OSError) as e:
        pytest.skip(f"extension not built: {e}")
    flat = hip_ops._C.moe_tile_order(experts, n_blocks, split)
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
