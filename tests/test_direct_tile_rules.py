"""Which products the tiles of eight waves by direct loads take over from the tile that was named for them (here without a
GPU): the measured ones, and over sizes drawn at random only where all their blocks find a place at once."""
import random

import pytest

from test_dispatch_rules import core      # noqa: F401 (fixture)

SHAPES = {10: (128, 128), 11: (128, 192), 12: (192, 128)}


@pytest.mark.parametrize("kind,m,n,k,pieces,want", [
    # (us before / with it: csrc/gemm.hip)
    (1, 384, 9728, 896, 1, 10), (1, 256, 11008, 2048, 1, 10), (1, 2048, 896, 4864, 2, 10), (2, 457, 3584, 18944, 2, 10),
    (1, 512, 9728, 896, 1, 12), (1, 1024, 4864, 896, 1, 12), (5, 1900, 9728, 896, 1, 12), (5, 900, 17920, 1536, 1, 12),
    (1, 640, 9728, 896, 1, 11), (1, 256, 17920, 1536, 1, 11),
    (1, 656, 2048, 1536, 1, -1), (1, 762, 2560, 2048, 1, -1), (1, 1384, 896, 4864, 1, -1),      # 64 x 128 finds a unit for every block
    (1, 520, 2048, 11008, 1, 10), (1, 154, 4608, 3584, 1, 10), (2, 656, 2048, 1536, 1, 10),
    (1, 1024, 2048, 1536, 1, -1), (1, 1025, 2048, 1536, 1, 10), (1, 1024, 2048, 5856, 1, -1), (1, 1024, 2048, 5864, 1, 10),
    (5, 1024, 17920, 1536, 1, -1), (5, 384, 37888, 3584, 1, -1), (1, 64, 896, 4864, 2, -1), (0, 512, 896, 896, 1, -1),
    (4, 2048, 37888, 3584, 1, -1), (1, 384, 9728, 2 ** 22 + 8, 1, -1),
])
def test_measured(core, kind, m, n, k, pieces, want):      # noqa: F811
    assert core.llmlab_direct_tile(kind, m, n, k, pieces, 0, 256) == want


def test_units_are_the_callers(core):      # noqa: F811
    """228 blocks of 128 x 128 on chips of 228 units and of one less; 228 of 192 x 128 likewise."""
    assert core.llmlab_direct_tile(1, 384, 9728, 896, 1, 0, 228) == 10 and core.llmlab_direct_tile(1, 384, 9728, 896, 1, 0, 227) != 10
    assert core.llmlab_direct_tile(1, 512, 9728, 896, 1, 0, 228) == 12 and core.llmlab_direct_tile(1, 512, 9728, 896, 1, 0, 227) == 11


def test_only_where_their_blocks_find_a_place(core):      # noqa: F811
    rng, seen = random.Random(11), set()
    for _ in range(20000):
        kind, heads = rng.randint(0, 5), rng.randint(0, 1)
        m, n, k = rng.randint(1, 3000), rng.randint(1, 40000), 8 * rng.randint(1, 2500)
        pieces, units = rng.choice([1, 1, 2, 4, 8]), rng.choice([256, 256, 304, 228, 64])
        tile = core.llmlab_direct_tile(kind, m, n, k, pieces, heads, units)
        if tile < 0:
            continue
        seen.add((kind, tile))
        bm, bn = SHAPES[tile]
        blocks = -(-m // bm) * -(-n // bn) * pieces
        assert m > 64 and (not heads or tile == 10)
        assert blocks <= units or (kind == 5 and pieces == 1 and k <= 2048), (kind, m, n, k, pieces, tile)
    assert seen == {(1, 10), (2, 10), (1, 11), (1, 12), (5, 12)}


def test_a_forced_tile_holds_whole_heads(core):      # noqa: F811
    """Forced for a product written by heads: 128 x 128 where the named tile is no wider (a head of 256 fits one of 256 columns)."""
    for force, tile in ((138, 10), (139, 11), (140, 12)):
        core.llmlab_debug_gemm_tile(force)
        try:
            for kind in range(6):
                assert core.llmlab_direct_tile(kind, 200, 1024, 256, 1, 0, 256) == tile
                assert core.llmlab_direct_tile(kind, 200, 1024, 256, 1, 1, 256) == (10 if force == 138 and kind < 3 else -1)
        finally:
            core.llmlab_debug_gemm_tile(0)
