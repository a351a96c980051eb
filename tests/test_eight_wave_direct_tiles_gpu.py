"""The tiles of eight waves whose operands come by direct loads (138: 128 x 128, 139: 128 x 192, 140: 192 x 128): inner sizes
around their rings, rows and columns that fill no block, every epilogue; and to the bit what the tile gives that they
stand in for, since every sum has the same order."""
import pytest
import torch

import test_direct_load_tiles_gpu as direct
import test_register_epilogue_gpu as epilogue
from test_kernels_gpu import DEV, emu, ops      # noqa: F401 (fixtures)

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
