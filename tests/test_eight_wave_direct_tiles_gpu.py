"""The tiles of eight waves whose operands come by direct loads (138: 128 x 128, 139: 128 x 192, 140: 192 x 128): inner sizes
around their rings, rows and columns that fill no block, every epilogue (q, k and v by heads: 128 x 128, the one of them that
takes it); and to the bit what the tile gives that they stand in for, since every sum has the same order."""
import pytest
import torch

import test_direct_load_tiles_gpu as direct
import test_register_epilogue_gpu as epilogue
from test_kernels_gpu import DEV, check_qkv_rope_cache, emu, ops      # noqa: F401 (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile,m", [(138, 129), (138, 256), (139, 200), (140, 193), (140, 384)])
@pytest.mark.parametrize("k", [8, 32, 56, 64, 72, 96, 128, 160, 192, 200, 256, 392, 776])
def test_inner_sizes_around_the_rings(ops, tile, m, k):      # noqa: F811
    direct.test_inner_sizes_around_the_rings(ops, tile, m, k)


@pytest.mark.parametrize("tile", [138, 139, 140])
@pytest.mark.parametrize("m,n,k", [(129, 256, 64), (193, 288, 136), (70, 33, 72), (257, 520, 200)])
@pytest.mark.parametrize("pad,shift", [(0, 0), (8, 8), (4, 4), (3, 1)])
def test_every_epilogue_into_any_rows(ops, emu, tile, m, n, k, pad, shift):      # noqa: F811
    epilogue.test_every_tile_into_any_rows(ops, emu, tile, m, n, k, pad, shift)


@pytest.mark.parametrize("tile", [138, 139, 140])
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh", "clamped"])
@pytest.mark.parametrize("m,inter,k,pad", [(129, 128, 64, 0), (193, 152, 136, 0), (70, 20, 72, 0), (200, 256, 96, 5)])
def test_paired_products(ops, emu, tile, activation, m, inter, k, pad):      # noqa: F811
    epilogue.test_paired_products(ops, emu, tile, activation, m, inter, k, pad)


@pytest.mark.parametrize("m,n,k,old,tile", [(384, 9728, 896, 130, 10), (512, 9728, 896, 130, 12), (640, 9728, 896, 130, 11),
                                            (1900, 9728, 896, 133, 12)])
def test_same_results_as_the_tile_before(ops, m, n, k, old, tile):      # noqa: F811
    kind = {130: 1, 133: 5}[old]
    assert ops._core.llmlab_direct_tile(kind, m, n, k, 1, 0, ops.num_cus) == tile
    gen = torch.Generator(device=DEV).manual_seed(m)
    x = torch.randn(m, k, device=DEV, generator=gen).bfloat16()
    w = ops.prepare_weight(torch.randn(n, k, device=DEV, generator=gen).bfloat16())
    got, want = (torch.empty(m, n // 2, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    ops.linear_swiglu(x, w, got)
    with ops.debug.force(gemm_tile=old):
        ops.linear_swiglu(x, w, want)
    assert torch.equal(got, want)


QKV_STARTS = [([70, 1, 130], (3, 40, 0, 7)), ([300, 2, 2, 90], (3, 40, 0, 7)),
              # (values of four positions written together: starts and rows that line up, that do not, and short requests between)
              ([72, 4, 124], (0, 64, 8)), ([70, 6, 125], (2, 61, 9)), ([8, 4, 4, 180], (12, 0, 28, 100))]
MORE_ROWS = [([300, 2, 2, 90], (3, 40, 0, 7)), ([272, 4, 124], (0, 64, 8)), ([270, 6, 125], (2, 61, 9)), ([200, 4, 4, 190], (12, 0, 28, 100))]


@pytest.mark.parametrize("nq,nkv,d,page,hidden", [(4, 2, 16, 16, 64), (7, 1, 32, 16, 72), (14, 2, 64, 64, 896)])
@pytest.mark.parametrize("rows_per,starts", QKV_STARTS)
def test_queries_keys_and_values(ops, emu, nq, nkv, d, page, hidden, rows_per, starts):      # noqa: F811
    """Bias, rotation and the write into the cache; two to eight heads a tile of 128 columns, rows that end inside a tile."""
    with ops.debug.force(gemm_tile=138, few_rows_max=64, qkv_pieces_min_rows=1 << 30):
        assert ops.can_fuse_qkv_rope(sum(rows_per), torch.bfloat16, d, (nq + 2 * nkv) * d, hidden)
        check_qkv_rope_cache(ops, emu, nq, nkv, d, page, hidden, rows_per, starts)


def qkv_by(ops, tile, nq, nkv, d, page, hidden, rows_per, starts):      # noqa: F811
    """q, the keys and the values of a step by this tile (0: by the rule), what was there before included."""
    rows, n, reqs = sum(rows_per), (nq + 2 * nkv) * d, len(rows_per)
    ints, gen = dict(dtype=torch.int32, device=DEV), torch.Generator(device=DEV).manual_seed(rows)
    h, b = (torch.randn(*s, device=DEV, generator=gen).bfloat16() for s in ((rows, hidden), (n,)))
    w = ops.prepare_weight(torch.randn(n, hidden, device=DEV, generator=gen).bfloat16())
    need = [(s + r + page - 1) // page for s, r in zip(starts, rows_per)]
    table = torch.full((reqs, max(need)), -1, dtype=torch.int32)
    for i in range(reqs):
        table[i, :need[i]] = torch.arange(sum(need[:i]), sum(need[:i + 1])).int()
    positions = torch.cat([torch.arange(s, s + r) for s, r in zip(starts, rows_per)]).to(**ints)
    row_req = torch.cat([torch.full((r,), i) for i, r in enumerate(rows_per)]).to(**ints)
    kc, vc = (torch.randn(sum(need), nkv, *s, device=DEV, generator=gen).bfloat16() for s in ((page, d), (d, page)))
    q = torch.zeros(rows, nq * d, device=DEV, dtype=torch.bfloat16)
    inv_freq = (1e4 ** (-torch.arange(0, d, 2, device=DEV).double() / d)).float()
    with ops.debug.force(gemm_tile=tile, few_rows_max=64, qkv_pieces_min_rows=1 << 30):
        assert ops._core.llmlab_linear_heads_tile(rows, n, hidden, d, ops.num_cus) == 128
        ops.qkv_rope_cache(h, w, b, nq, nkv, d, inv_freq, positions, row_req, table.to(DEV), page, kc, vc, q)
    return q, kc, vc


@pytest.mark.parametrize("nq,nkv,page", [(22, 1, 16), (8, 8, 64)])
@pytest.mark.parametrize("rows_per,starts", MORE_ROWS)
def test_a_head_a_tile(ops, nq, nkv, page, rows_per, starts):      # noqa: F811
    """Heads of 128: to the bit what the tile of four waves gives, everywhere in the caches."""
    hidden = 1536
    got, want = (qkv_by(ops, tile, nq, nkv, 128, page, hidden, rows_per, starts) for tile in (138, 129))
    assert all(torch.equal(x, y) for x, y in zip(got, want))


@pytest.mark.parametrize("rows,nq,nkv,hidden", [(1093, 16, 2, 2048), (1242, 12, 2, 1536), (603, 32, 8, 4096)])
def test_queries_keys_and_values_by_the_rule(ops, rows, nq, nkv, hidden):      # noqa: F811
    """Sizes that the rule sends to 128 x 128: to the bit what the tile before gives."""
    assert ops._core.llmlab_direct_tile(1, rows, (nq + 2 * nkv) * 128, hidden, 1, 1, ops.num_cus) == 10
    got, want = (qkv_by(ops, tile, nq, nkv, 128, 64, hidden, [rows - 7, 7], (5, 90)) for tile in (0, 130))
    assert all(torch.equal(x, y) for x, y in zip(got, want))
