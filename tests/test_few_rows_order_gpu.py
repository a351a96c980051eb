"""The few-row kernels and decode attention where their loads are ordered by hand: what the epilogue
needs is asked for at the start of a kernel, pieces in fours and eights, block-table rows as a whole."""
import pytest
import torch

from llm_inference_lab_amd.parts.base import PendingSums
from test_kernels_gpu import DEV, close, emu, ops, rnd, run_attention      # noqa: F401 (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("pages", [1, 63, 64, 65, 127, 128, 129, 200])
def test_decode_reads_tables_of_any_length(ops, emu, dtype, pages):      # noqa: F811
    """Rows of up to 128 pages are read ahead as a whole, longer ones page by page."""
    last = pages * 16 - 1
    run_attention(ops, emu, dtype, 7, 1, 64, 16, None, [(last, 1), (last // 2, 1), (0, 1)])
    run_attention(ops, emu, dtype, 4, 2, 128, 16, 40, [(last, 1), (3, 1)])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m", [1, 5, 16, 40])
@pytest.mark.parametrize("splits", [1, 3, 4, 5, 8])
def test_owed_pieces_of_any_number(ops, emu, dtype, m, splits):      # noqa: F811
    """Pieces owed to rows that a fused norm reads and that a product adds into, with a bias in either type."""
    n, k = 272, 1216
    x, w = rnd((m, k), dtype, 1), rnd((n, k), dtype, 2, 0.1)
    pieces, resid = rnd((ops.MAX_SPLITS, m, n), torch.float32, 9), rnd((m, n), torch.float32, 3)
    pending, want_pending = PendingSums(pieces.to(DEV), splits), PendingSums(pieces, splits)
    whole = resid + pieces[:splits].sum(0)
    x2, w2 = rnd((m, 96), dtype, 4), rnd((n, 96), dtype, 5, 0.1)
    got = resid.clone().to(DEV)
    ops.linear_residual(x2.to(DEV), ops.prepare_weight(w2.to(DEV)), got, pending=pending)
    want = whole + x2.float() @ w2.float().t()
    close(got, want, torch.float32, "pieces folded with a product", want.abs().max().item())
    for wdtype in (torch.float32, torch.bfloat16):
        norm_w, head = (1 + 0.1 * rnd((n,), torch.float32, 6)).to(wdtype), rnd((48, n), dtype, 7, 0.1)
        logits = torch.zeros(m, 48, device=DEV)
        ops.fused_norm_logits(resid.to(DEV), None, norm_w.to(DEV), 1e-6, ops.prepare_weight(head.to(DEV)), logits,
                              pending=pending)
        rows = whole.double()
        want_l = (rows * torch.rsqrt(rows.square().mean(-1, keepdim=True) + 1e-6) * norm_w.double()) @ head.double().t()
        # (bfloat16: a row times the norm's weight is rounded once, to 2^-9 of its size, in each of 272 terms)
        close(logits, want_l, dtype, "pieces under a norm", want_l.abs().max().item())
    for bdtype in (torch.float32, torch.bfloat16):
        bias = rnd((n,), torch.float32, 8).to(bdtype)
        out, want_o = torch.empty(m, n, dtype=dtype, device=DEV), torch.empty(m, n, dtype=dtype)
        ops.linear(x.to(DEV), ops.prepare_weight(w.to(DEV)), out, bias.to(DEV))
        emu.linear(x, w, want_o, bias)
        close(out, want_o, dtype, "bias", want_o.float().abs().max().item())


@pytest.mark.parametrize("splits,waves,steps,large", [(3, 3, 20, 1), (6, 8, 97, 1), (2, 4, 17, 1), (2, 2, 13, 2)])
def test_a_shorter_last_group_is_shared_out_evenly(ops, splits, waves, steps, large):      # noqa: F811
    """The inner size in groups of steps, the last one shorter: its steps, too, go to the waves in equal portions.  One
    number a step: a large one, one half a unit of its last place, and the large one's negative; the second is lost
    where it meets the first in one wave and kept where it meets the third there."""
    group = -(-steps // splits)
    rest = steps - (splits - 1) * group
    portion = -(-rest // waves)
    assert 0 < rest < group and portion < -(-group // waves) and portion == large + 1
    k, n = 32 * steps, 32
    w, x = torch.zeros(n, k, dtype=torch.bfloat16), torch.ones(3, k, dtype=torch.bfloat16)
    first = (splits - 1) * group
    w[:, 32 * (first + large)], w[:, 32 * (first + large + 1)], w[:, 32 * (first + large + 2)] = 2.0 ** 24, 1.0, -2.0 ** 24
    parts = torch.full((splits, 3, n), float("nan"), device=DEV)
    with ops.debug.force(skinny_shape=(1, waves, 0, 1)):
        ops.linear_partials(x.to(DEV), ops.prepare_weight(w.to(DEV)), parts, splits)
    assert bool((parts[:-1] == 0).all()) and bool((parts[-1] == 1.0).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [96, 896, 2048, 3584])
def test_a_norm_of_weights_in_either_type(ops, dtype, n):      # noqa: F811
    """Weights of one value in bfloat16 and in float32 are read by instances of their own: a row's squares meet in one
    order, to the bit."""
    weight, head = (1 + 0.1 * rnd((n,), torch.float32, 6)).bfloat16().to(DEV), ops.prepare_weight(rnd((48, n), dtype, 7, 0.1).to(DEV))
    for m in range(1, 65):
        if not ops.can_fuse(m, dtype, n):
            continue
        x = rnd((m, n), torch.float32, m).to(DEV)
        narrow, wide = torch.empty(m, 48, device=DEV), torch.empty(m, 48, device=DEV)
        ops.fused_norm_logits(x, None, weight, 1e-6, head, narrow)
        ops.fused_norm_logits(x, None, weight.float(), 1e-6, head, wide)
        assert torch.equal(narrow, wide), f"{m} rows"
