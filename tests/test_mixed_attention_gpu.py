"""Mixed steps of many requests: a block of a launch for one kind of requests finds its request by counting
(64 requests a load), wherever the portions stand among the decoding requests."""
import pytest
import torch

from test_kernels_gpu import emu, ops, run_attention  # noqa: F401 (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("nq,nkv,d,page", [(14, 2, 64, 16), (4, 1, 128, 16)])
@pytest.mark.parametrize("requests,portions", [(2, [0]), (2, [1]), (64, [0, 63]), (65, [63, 64]), (130, [0, 64, 127, 129])])
def test_portions_anywhere(ops, emu, dtype, nq, nkv, d, page, requests, portions):  # noqa: F811
    spec = [((37 * i) % 70 + 1, 1) for i in range(requests)]
    for n, at in enumerate(portions):
        spec[at] = ((0, 50, 7, 33)[n], (40, 21, 70, 19)[n])
    if requests > 64:
        spec[5] = (0, 0)                     # a request without rows counts among the short ones
    run_attention(ops, emu, dtype, nq, nkv, d, page, None, spec, seed=95)


@pytest.mark.parametrize("path", [1, 2, 3, 4, 5, 6])
def test_every_launch(ops, emu, path):  # noqa: F811
    spec = [(60 + i, 1) for i in range(70)]
    spec[3], spec[66] = (30, 90), (0, 65)
    with ops.debug.force(attention_path=(64, path)):
        run_attention(ops, emu, torch.bfloat16, 14, 2, 64, 16, None, spec, seed=96)


@pytest.mark.parametrize("window", [None, 40])
@pytest.mark.parametrize("nq,nkv,d,page", [(14, 2, 64, 64), (7, 1, 16, 16), (12, 2, 128, 32), (4, 4, 112, 16)])
def test_tiles_of_16_rows(ops, emu, window, nq, nkv, d, page):  # noqa: F811
    """The step in one launch with small tiles: portions that fill no tile, begin in one, or see no key of some waves,
    behind histories whose keys are split over blocks and not."""
    for spec in ([(0, 3), (5, 1)], [(0, 17), (900, 1), (64, 1)], [(700, 1), (33, 50), (1500, 1), (0, 129)]):
        run_attention(ops, emu, torch.bfloat16, nq, nkv, d, page, window, spec, seed=97)
