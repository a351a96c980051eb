"""The tiles whose operands come by direct loads into LDS (the two of two groups of waves, and 64 x 64): every length of
the inner size at which their rings begin, wrap or end (pieces of x of two steps, steps of W, the last of them cut
short), whole and in pieces."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BF = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from llm_inference_lab_amd.kernels.hip_ops import HipOps
    return HipOps(DEV)


@pytest.mark.parametrize("tile,m", [(132, 257), (132, 400), (133, 193), (133, 300), (64, 65), (64, 200)])
@pytest.mark.parametrize("k", [8, 32, 56, 64, 72, 96, 128, 160, 192, 200, 224, 256, 352, 384, 392, 448, 776])
def test_inner_sizes_around_the_rings(ops, tile, m, k):
    gen = torch.Generator(device=DEV).manual_seed(k)
    x = torch.randn(m, k, device=DEV, generator=gen).to(BF)
    w = torch.randn(530, k, device=DEV, generator=gen).to(BF)
    want = x.double() @ w.double().T
    unit = (k + 16) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T + 1)      # float32 sums in any order
    pw = ops.prepare_weight(w)
    with ops.debug.force(gemm_tile=tile, few_rows_max=64):
        out = torch.empty(m, 530, device=DEV)
        ops.linear_logits(x, pw, out)
        assert bool(((out.double() - want).abs() <= unit).all())
        for count in (2, 3):
            parts = torch.zeros(count, m, 530, device=DEV)
            ops.linear_partials(x, pw, parts, count)
            assert bool(((parts.double().sum(0) - want).abs() <= unit).all())


def test_an_inner_size_beyond_their_addresses(ops):
    """65 rows of 34,087,048 (4.4 GB; the 64 rows of a tile span more bytes than 32 bits address): rows that are zero but
    for a few numbers, whose product is that of those columns."""
    m, n, k = 65, 16, 34_087_048
    gen = torch.Generator(device=DEV).manual_seed(4)
    w = torch.randn(n, k, device=DEV, generator=gen).to(BF)
    at = torch.tensor([0, 33, k // 2 + 1, k - 9, k - 1], device=DEV)
    x = torch.zeros(m, k, device=DEV, dtype=BF)
    x[:, at] = torch.randn(m, 5, device=DEV, generator=gen).to(BF)
    want = x[:, at].double() @ w[:, at].double().T
    unit = 8 * 2.0 ** -24 * (x[:, at].double().abs() @ w[:, at].double().abs().T + 1)
    pw = ops.prepare_weight(w)
    out = torch.empty(m, n, device=DEV)
    ops.linear_logits(x, pw, out)
    assert bool(((out.double() - want).abs() <= unit).all())
    for tile in (0, 4):                    # (kinds named by the caller)
        parts = torch.zeros(2, m, n, device=DEV)
        ops._call(ops._core.llmlab_linear_partials, x.data_ptr(), pw.data_ptr(), 1, parts.data_ptr(), None, 0, m, n, k, n,
                  2, m * n, tile, ops._stream())
        assert bool(((parts.double().sum(0) - want).abs() <= unit).all()), tile
