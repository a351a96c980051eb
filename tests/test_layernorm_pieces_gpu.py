"""The layer norm of a result left in pieces, added into the stream: few rows and many (a block or a
wave a row), widths around what a thread keeps in registers, odd widths, pieces in groups and beyond."""
import pytest
import torch

from llm_inference_lab_amd.parts.base import PendingSums

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from llm_inference_lab_amd.kernels.hip_ops import HipOps
    return HipOps(DEV)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,width,splits", [(1, 64, 1), (16, 2048, 2), (3, 4100, 8), (2, 20000, 5), (130, 896, 3),
                                               (200, 77, 6), (513, 896, 2), (600, 2048, 4), (515, 2052, 2), (520, 4, 1)])
def test_layernorm_of_pieces(ops, dtype, rows, width, splits):
    g = torch.Generator().manual_seed(rows + width)
    parts = torch.randn(splits, rows, width, generator=g) * 3 + 1
    stream, weight = torch.randn(rows, width, generator=g), (1 + 0.1 * torch.randn(width, generator=g)).to(dtype)
    y = parts.double().sum(0)
    norm = torch.nn.functional.layer_norm(y, (width,), weight.double(), None, 1e-6)
    want = stream.double() + norm
    got, copy = stream.to(DEV), torch.empty(rows, width, dtype=dtype, device=DEV)
    ops.layernorm_add(PendingSums(parts.to(DEV), splits), weight.to(DEV), 1e-6, got, copy)
    # the pieces' sum and the mean are off by up to (splits + a tree's depth) roundings of numbers of size 3 splits,
    # relative to a deviation of 3 sqrt(splits)
    limit = (splits + 20) * 2.0 ** -24 * (4 + norm.abs().max()) * (1 + splits ** 0.5)
    assert float((got.cpu().double() - want).abs().max()) <= limit
    assert torch.equal(copy, got.to(dtype))
    out = torch.empty(rows, width, dtype=torch.float32, device=DEV)
    order = torch.arange(rows - 1, -1, -1, dtype=torch.int32)
    ops.layernorm(parts[0].to(DEV), weight.to(DEV), 1e-6, out, order.to(DEV))
    want = torch.nn.functional.layer_norm(parts[0].double(), (width,), weight.double(), None, 1e-6).flip(0)
    assert float((out.cpu().double() - want).abs().max()) <= 24 * 2.0 ** -24 * (4 + want.abs().max())
