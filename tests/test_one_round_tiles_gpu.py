"""The tiles whose widths are 3, 5 and 7 times 32 columns (few rows of wide matrices): every epilogue at
ragged edges in all three dimensions, and the rule that picks them."""
import pytest
import torch

from llm_inference_lab_amd.parts.feed_forward import interleave_gate_up

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BF = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from llm_inference_lab_amd.kernels.hip_ops import HipOps
    return HipOps(DEV)


def rnd(shape, seed, scale=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale).to(BF)


@pytest.mark.parametrize("tile", [134, 135, 136, 137])
@pytest.mark.parametrize("m,n,k", [(65, 130, 72), (127, 449, 136), (129, 64, 1160), (70, 300, 24), (200, 1000, 64)])
def test_epilogues(ops, tile, m, n, k):
    x, w = rnd((m, k), 1), rnd((n, k), 2, 0.1)
    bias, old = torch.randn(n, generator=torch.Generator().manual_seed(3)), torch.randn(m, n)
    want = x.double() @ w.double().T
    unit = (k + 16) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T + 4)      # float32 sums in any order
    dx, dw = x.to(DEV), ops.prepare_weight(w.to(DEV))
    with ops.debug.force(gemm_tile=tile, few_rows_max=64):
        out = torch.empty(m, n, device=DEV)
        ops.linear_logits(dx, dw, out)
        assert bool(((out.cpu().double() - want).abs() <= unit).all())
        got = old.to(DEV)
        ops.linear_residual(dx, dw, got)
        assert bool(((got.cpu().double() - want - old.double()).abs() <= unit).all())
        low = torch.empty(m, n, dtype=BF, device=DEV)
        ops.linear(dx, dw, low, bias.to(DEV))
        full = want + bias.double()
        assert bool(((low.cpu().double() - full).abs() <= unit + full.abs() / 256).all())
        inter = n // 2 + 3
        gate, up = rnd((inter, k), 4, 0.1), rnd((inter, k), 5, 0.1)
        act = torch.empty(m, inter, dtype=BF, device=DEV)
        ops.linear_swiglu(dx, ops.prepare_weight(interleave_gate_up(gate, up).to(DEV)), act)
        g, u = x.double() @ gate.double().T, x.double() @ up.double().T
        full = g * torch.sigmoid(g) * u
        sums = lambda a: (k + 16) * 2.0 ** -24 * (x.double().abs() @ a.double().abs().T)  # noqa: E731
        assert bool(((act.cpu().double() - full).abs()
                     <= 1.1 * sums(gate) * u.abs() + sums(up) * g.abs() + full.abs() / 128 + 1e-6).all())


@pytest.mark.parametrize("m,n,k,columns", [(17, 24448, 1024, 96), (64, 37888, 1024, 160), (40, 49000, 3072, 224),
                                           (65, 37888, 1024, 160), (128, 17920, 1024, 160), (64, 152064, 1024, 128)])
def test_one_round_of_blocks(ops, m, n, k, columns):
    """The chosen width, and one product by it against the same product by another tile."""
    if ops.num_cus == 256:
        assert ops._core.llmlab_plain_tile(m, n, k, 256) == columns
    x, w = rnd((m, k), 6).to(DEV), (torch.randn(n, k, device=DEV) * 0.05).to(BF)
    pw = ops.prepare_weight(w)
    out, other = torch.empty(m, n, device=DEV), torch.empty(m, n, device=DEV)
    with ops.debug.force(few_rows_max=64):
        ops.linear_logits(x, pw, out)
    with ops.debug.force(gemm_tile=130):
        ops.linear_logits(x, pw, other)
    assert float((out - other).abs().max()) <= 2 * (k + 16) * 2.0 ** -24 * float((x.float().abs() @ w.float().abs().T).max())
