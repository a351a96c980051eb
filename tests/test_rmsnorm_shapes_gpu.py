"""RMSNorm at every way its kernel is launched: a group a thread or several, one wave a row or more, rows longer than
what the threads hold, with and without pieces owed to the rows, gathered rows, rows that are not aligned."""
import pytest
import torch

from llm_inference_lab_amd.parts.base import PendingSums
from test_kernels_gpu import DEV, close, ops, rnd      # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [1, 128, 129, 1024, 1025])
@pytest.mark.parametrize("hidden", [4, 33, 896, 1024, 1028, 4100, 16400])
@pytest.mark.parametrize("splits", [0, 2, 3, 8])
def test_against_64_bits(ops, dtype, rows, hidden, splits):      # noqa: F811
    if rows * hidden > 5_000_000:
        rows = rows % 128 + 129
    x, w = rnd((rows, hidden), torch.float32, 1), (1 + 0.1 * rnd((hidden,), torch.float32, 2)).to(dtype)
    pieces = rnd((max(splits, 1), rows, hidden), torch.float32, 3)
    whole = x.double() + (pieces.double().sum(0) if splits else 0)
    want = whole * torch.rsqrt(whole.square().mean(-1, keepdim=True) + 1e-6) * w.double()
    got_x, got = x.to(DEV), torch.empty(rows, hidden, dtype=dtype, device=DEV)
    ops.rmsnorm(got_x, w.to(DEV), 1e-6, got, pending=PendingSums(pieces.to(DEV), splits) if splits else None)
    close(got, want, dtype, "norm", want.abs().max().item())
    close(got_x, whole, torch.float32, "rows made whole", whole.abs().max().item())
    if not splits:
        picked = torch.randint(0, rows, (min(rows, 40),), generator=torch.Generator().manual_seed(4)).int()
        got = torch.empty(len(picked), hidden, dtype=dtype, device=DEV)
        ops.rmsnorm(got_x, w.to(DEV), 1e-6, got, picked.to(DEV))
        close(got, want[picked.long()], dtype, "gathered", want.abs().max().item())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hidden", [4, 33, 64, 260, 512, 772, 896, 1024])
@pytest.mark.parametrize("splits", [0, 1, 2, 3, 8])
def test_a_row_is_the_same_among_any_number_of_rows(ops, dtype, hidden, splits):      # noqa: F811
    """Rows of up to 1,024 numbers: however a launch spreads them, a row's sum meets in one order."""
    x, w = rnd((2000, hidden), torch.float32, 1), (1 + 0.1 * rnd((hidden,), torch.float32, 2)).to(dtype).to(DEV)
    pieces = rnd((max(splits, 1), 2000, hidden), torch.float32, 3)
    got = {}
    for rows in (1, 100, 129, 1024, 1025, 2000):
        out = torch.empty(rows, hidden, dtype=dtype, device=DEV)
        ops.rmsnorm(x[:rows].to(DEV), w, 1e-6, out,
                    pending=PendingSums(pieces[:, :rows].contiguous().to(DEV), splits) if splits else None)
        got[rows] = out
    for rows, out in got.items():
        assert torch.equal(out, got[2000][:rows]), f"{rows} rows"
