"""The layer norm at the edges of its launches: one, two and three groups a thread and rows beyond, whole rows and rows
in pieces (fewer and more than are asked for at once), a block and a wave a row."""
import pytest
import torch

from test_layernorm_pieces_gpu import ops, test_layernorm_of_pieces as against_64_bits      # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,width,splits", [
    (1, 4, 1), (128, 4096, 1), (128, 4096, 6), (128, 4100, 1), (5, 8192, 4), (5, 8196, 1), (5, 8196, 3), (5, 12288, 2),
    (5, 12292, 1), (5, 12292, 8), (129, 1024, 1), (129, 1024, 5), (129, 1028, 2), (512, 2048, 1), (512, 2052, 3), (513, 1024, 1),
    (513, 1028, 1), (700, 2048, 3), (521, 12, 2)])
def test_edges(ops, dtype, rows, width, splits):      # noqa: F811
    against_64_bits(ops, dtype, rows, width, splits)
