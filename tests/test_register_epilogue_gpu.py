"""The epilogue of the bfloat16 tiles that writes sums from where the matrix instructions leave them: every tile, rows
and columns that fill no block of 16, outputs whose rows are not aligned for whole stores, every activation."""
import pytest
import torch

from test_kernels_gpu import DEV, close, emu, ops, rnd      # noqa: F401 (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [64, 130, 129, 131, 132, 133])
@pytest.mark.parametrize("m,n,k", [(129, 256, 64), (193, 288, 136), (70, 33, 72), (257, 520, 200)])
@pytest.mark.parametrize("pad,shift", [(0, 0), (8, 8), (4, 4), (3, 1)])
def test_every_tile_into_any_rows(ops, emu, tile, m, n, k, pad, shift):      # noqa: F811
    bf = torch.bfloat16
    x, w, b = rnd((m, k), bf, 1), rnd((n, k), bf, 2, 0.1), rnd((n,), torch.float32, 3)
    dx, dw = x.to(DEV), ops.prepare_weight(w.to(DEV))

    def place(dtype, *pieces):
        """Rows of a wider and longer matrix (a tile's rows longer) that begin at an odd place of it; what lies around
        them stays as it is."""
        whole = torch.full((*pieces, m + 256, n + pad + shift), 7.0, dtype=dtype, device=DEV)
        return whole, whole[..., :m, shift:shift + n]

    def alone(whole, out):
        out.fill_(7.0)
        return bool((whole == 7.0).all())

    y = x.float() @ w.float().t()
    scale = y.abs().max().item()
    with ops.debug.force(gemm_tile=tile):
        whole, out = place(bf)
        ops.linear(dx, dw, out, b.to(DEV))
        close(out, (y + b).to(bf), bf, "store", (y + b).abs().max().item())
        assert alone(whole, out), "written beside the output"
        whole_f, out_f = place(torch.float32)
        ops.linear_logits(dx, dw, out_f)
        close(out_f, y, torch.float32, "float32", scale)
        assert alone(whole_f, out_f), "written beside the output"
        before = rnd((m, n), torch.float32, 4)
        out_f.copy_(before)
        ops.linear_residual(dx, dw, out_f)
        close(out_f, before + y, torch.float32, "into the residual", scale)
        assert alone(whole_f, out_f), "written beside the output"
        whole_p, parts = place(torch.float32, 3)
        ops.linear_partials(dx, dw, parts, 3)
        close(parts.sum(0), y, torch.float32, "pieces", scale)
        assert alone(whole_p, parts), "written beside the pieces"


@pytest.mark.parametrize("tile", [64, 130, 129, 131, 132, 133])
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh", "clamped"])
@pytest.mark.parametrize("m,inter,k,pad", [(129, 128, 64, 0), (193, 152, 136, 0), (70, 20, 72, 0), (200, 256, 96, 5)])
def test_paired_products(ops, emu, tile, activation, m, inter, k, pad):      # noqa: F811
    bf = torch.bfloat16
    rows = 2 * ((inter + 15) // 16 * 16)
    x, w = rnd((m, k), bf, 5), rnd((rows, k), bf, 6, 0.1)
    constants = (1.5, 1.7, 1.0) if activation == "clamped" else None
    want = torch.empty(m, inter, dtype=bf)
    emu.linear_swiglu(x, w, want, activation, constants)
    got = torch.full((m + 256, inter + pad), 7.0, dtype=bf, device=DEV)
    with ops.debug.force(gemm_tile=tile):
        ops.linear_swiglu(x.to(DEV), ops.prepare_weight(w.to(DEV)), got[:m, :inter], activation, constants)
    close(got[:m, :inter], want, bf, "paired", want.float().abs().max().item())
    assert bool((got[:, inter:] == 7.0).all()) and bool((got[m:] == 7.0).all())


@pytest.mark.parametrize("tile", [64, 132])
def test_gates_of_any_size(ops, tile):      # noqa: F811
    """Gates whose exponential overflows or vanishes give 0 and the gate itself, infinite ones what a division gives."""
    x = torch.zeros(96, 64, dtype=torch.bfloat16)
    sizes = [0.0, 1e-30, -1e-30, 5.0, -5.0, 80.0, -80.0, 95.0, -95.0, 3e38, -3e38, 3e38, -3e38]
    x[:len(sizes), 0] = torch.tensor(sizes).bfloat16()
    x[11, 2], x[12, 2] = 3e38, -3e38     # (sums beyond the largest number)
    w = torch.zeros(32, 64, dtype=torch.bfloat16)
    w[:16, 0] = w[:16, 2] = 1.0          # gates
    x[:, 1], w[16:, 1] = 1.0, 1.0        # up values: one
    z = (x[:, 0].float() + x[:, 2].float()).double()
    want = (z / (1 + torch.exp(-z)))[:, None].expand(96, 16)
    got = torch.empty(96, 16, dtype=torch.bfloat16, device=DEV)
    with ops.debug.force(gemm_tile=tile):
        ops.linear_swiglu(x.to(DEV), ops.prepare_weight(w.to(DEV)), got)
    got = got.cpu().double()
    assert torch.equal(got.isnan(), want.isnan())
    fine = want.isfinite()
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    # (one rounding to bfloat16; numbers below 2^-126 may be zero)
    assert bool(((got - want).abs()[fine] <= 2.0 ** -8 * want.abs()[fine] + 2.0 ** -126).all())


@pytest.mark.parametrize("tile", [64, 130, 129, 131, 132, 133])
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh", "clamped"])
def test_gates_as_in_the_few_row_kernel(ops, tile, activation):      # noqa: F811
    """The same function of the same sums, to the bit: gates and up values of one term each."""
    bf, m = torch.bfloat16, 520
    gen = torch.Generator().manual_seed(8)
    x = torch.zeros(m, 64, dtype=bf)
    x[:, 0] = torch.linspace(-100.0, 100.0, m).to(bf)
    x[:, 1] = torch.randn(m, generator=gen).to(bf)
    w = torch.zeros(32, 64, dtype=bf)
    w[:16, 0] = (0.05 + 0.95 * torch.rand(16, generator=gen)).to(bf)
    w[0, 0] = 0.879                      # (gates of the size at which one over the denominator is no normal number)
    w[16:, 1] = torch.randn(16, generator=gen).to(bf)
    constants = (7.0, 1.7, 1.0) if activation == "clamped" else None
    dx, dw = x.to(DEV), ops.prepare_weight(w.to(DEV))
    got, want = torch.empty(m, 16, dtype=bf, device=DEV), torch.empty(m, 16, dtype=bf, device=DEV)
    with ops.debug.force(gemm_tile=tile):
        ops.linear_swiglu(dx, dw, got, activation, constants)
    for r in range(0, m, 8):      # (so few rows take the other kernel)
        ops.linear_swiglu(dx[r:r + 8], dw, want[r:r + 8], activation, constants)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
