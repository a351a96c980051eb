"""The few-row product kernel in float32 (``skinny_block_kernel<float, ...>``): every epilogue, alone
and under the fused norm, at the edges of its tiles of 16 rows and 16 columns, against 64 bits."""
import pytest
import torch

from llm_inference_lab_amd.parts.base import PendingSums
from llm_inference_lab_amd.parts.feed_forward import interleave_gate_up

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from llm_inference_lab_amd.kernels.hip_ops import HipOps
    return HipOps(DEV)


def rnd(shape, seed, scale=1.0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale


def check(got, want, x, w, what, extra=0.0):
    """32-bit sums of ``k`` products in any order: ``k`` roundings of half a unit of the sum of the absolute
    products, a handful more for what the epilogue does; ``extra`` the size of what is added to the sums."""
    limit = (x.shape[1] + 16) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T + extra)
    assert bool(((got.cpu().double() - want).abs() <= limit).all()), what


@pytest.mark.parametrize("m,n,k", [(3, 16, 16), (5, 17, 896), (16, 100, 48), (17, 130, 160), (33, 64, 272), (64, 31, 1600)])
def test_products(ops, m, n, k):
    assert ops.few_rows_take_float32(m, k)
    x, w, bias, old = rnd((m, k), 1), rnd((n, k), 2), rnd((n,), 3), rnd((m, n), 4)
    dx, dw = x.to(DEV), w.to(DEV)
    plain = x.double() @ w.double().T
    out = torch.empty(m, n, device=DEV)
    ops.linear(dx, dw, out, bias.to(DEV))
    check(out, plain + bias.double(), x, w, "store", 4.0)
    ops.linear_relu2(dx, dw, out)
    got, want = out.cpu().double(), plain.clamp(min=0) ** 2
    assert bool(((got - want).abs() <= 2 * (k + 16) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) * (want.sqrt() + 1)).all())
    parts = torch.full((2, m, n), float("nan"), device=DEV)
    pending = ops.linear_partials(dx, dw, parts, 2)
    check(parts.cpu().double().sum(0), plain, x, w, "pieces")
    got = old.to(DEV)
    ops.linear_residual(dx, dw, got, pending=pending)
    check(got, old.double() + 2 * plain, x, w, "into the stream", 4.0 + plain.abs().max().item())


@pytest.mark.parametrize("m,k,inter", [(1, 64, 20), (4, 896, 33), (16, 256, 16), (21, 160, 48), (64, 48, 40)])
def test_fused_norm(ops, m, k, inter):
    assert ops.can_fuse(m, torch.float32, k, 2 * inter)
    x, nw, pieces = rnd((m, k), 5, 3.0), 1 + rnd((k,), 6, 0.1), rnd((3, m, k), 7)
    whole = (x.double() + pieces.double().sum(0))
    normed = whole * torch.rsqrt(whole.square().mean(1, keepdim=True) + 1e-6) * nw.double()
    gate, up, w = rnd((inter, k), 8, 0.2), rnd((inter, k), 9, 0.2), rnd((37, k), 10)
    pend = PendingSums(pieces.to(DEV), 3)
    out = torch.empty(m, 37, device=DEV)
    ops.fused_norm_logits(x.to(DEV), None, nw.to(DEV), 1e-6, w.to(DEV), out, pending=pend)
    check(out, normed @ w.double().T, normed, w, "logits")
    act = torch.empty(m, inter, device=DEV)
    ops.fused_norm_swiglu(x.to(DEV), nw.to(DEV), 1e-6, interleave_gate_up(gate, up).to(DEV), act, pending=pend)
    g, u = normed @ gate.double().T, normed @ up.double().T
    want = g * torch.sigmoid(g) * u
    unit = (k + 24) * 2.0 ** -24       # of the gate's and the up value's sums, each scaled by the other factor (|silu'| <= 1.1)
    sums = lambda w: normed.abs() @ w.double().abs().T  # noqa: E731
    assert bool(((act.cpu().double() - want).abs()
                 <= unit * (1.1 * sums(gate) * u.abs() + sums(up) * g.abs() + want.abs()) + 1e-12).all())


@pytest.mark.parametrize("m,d,nq,nkv", [(1, 64, 2, 1), (8, 64, 14, 2), (19, 32, 4, 2), (5, 48, 3, 3), (2, 256, 2, 1)])
def test_fused_norm_qkv(ops, m, d, nq, nkv):
    from llm_inference_lab_amd.cache import layout
    k, page = 96, 16
    n = (nq + 2 * nkv) * d
    x, nw, w, bias = rnd((m, k), 11, 2.0), 1 + rnd((k,), 12, 0.1), rnd((n, k), 13, 0.2), rnd((n,), 14)
    positions = torch.arange(m, dtype=torch.int32) * 7 % 40
    requests = torch.arange(m, dtype=torch.int32)
    table = torch.arange(m * 3, dtype=torch.int32).view(m, 3)
    freq = 1e4 ** (-2.0 * torch.arange(d // 2).double() / d)
    kc, vc = torch.zeros(m * 3, nkv, page, d, device=DEV), torch.zeros(m * 3, nkv, d, page, device=DEV)
    q = torch.empty(m, nq * d, device=DEV)
    ops.fused_norm_qkv(x.to(DEV), nw.to(DEV), 1e-6, w.to(DEV), bias.to(DEV), nq, nkv, d, freq.float().to(DEV), positions.to(DEV),
                       requests.to(DEV), table.to(DEV), page, kc, vc, q)
    xd = x.double()
    normed = xd * torch.rsqrt(xd.square().mean(1, keepdim=True) + 1e-6) * nw.double()
    y = (normed @ w.double().T + bias.double()).view(m, nq + 2 * nkv, d)
    size = (normed.abs() @ w.double().abs().T + bias.double().abs()).max().item()
    angle = positions.double()[:, None] * freq.float().double()[None]
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    lo, hi = y[..., :d // 2], y[..., d // 2:]
    turned = torch.cat([lo * c - hi * s, hi * c + lo * s], -1)
    limit = ((k + 16) * 2.0 ** -24 + 40 * 2.0 ** -24) * 2 * size       # (the angle is rounded to 24 bits: up to 40 radians)
    assert float((q.cpu().double().view(m, nq, d) - turned[:, :nq]).abs().max()) <= limit
    keys = layout.keys_from_cache_order(kc.cpu())
    values = layout.values_from_cache_order(vc.cpu())
    for r in range(m):
        p, off = int(table[r, int(positions[r]) // page]), int(positions[r]) % page
        assert float((keys[p, :, off].double() - turned[r, nq:nq + nkv]).abs().max()) <= limit
        assert float((values[p, :, :, off].double() - y[r, nq + nkv:]).abs().max()) <= limit


@pytest.mark.parametrize("m,n,k", [(3, 16, 16), (5, 17, 896), (16, 100, 48), (17, 130, 160), (64, 31, 1600)])
def test_infinities(ops, m, n, k):
    """An infinity among the inputs gives an infinity, NaN gives NaN, in their rows alone: in every epilogue, whole
    and in pieces, wherever in the row it lies (the last steps of a wave's share are filled up with zeros)."""
    x, w = rnd((m, k), 15), rnd((n, k), 16)
    x[0, k - 1], x[1, 0], x[2, k // 2] = float("inf"), -float("inf"), float("nan")
    want = x.double() @ w.double().T
    limit = (k + 16) * 2.0 ** -24 * (x[3:].double().abs() @ w.double().abs().T)
    dx, dw = x.to(DEV), w.to(DEV)
    for what in ("store", "logits", "stream", "pieces"):
        out = torch.zeros(m, n, device=DEV)
        if what == "store":
            ops.linear(dx, dw, out)
        elif what == "logits":
            ops.linear_logits(dx, dw, out)
        elif what == "stream":
            ops.linear_residual(dx, dw, out)
        else:
            parts = torch.full((2, m, n), float("nan"), device=DEV)
            ops.linear_partials(dx, dw, parts, 2)
            out = parts.sum(0)
        got = out.cpu().double()
        assert torch.equal(got[:2], want[:2]) and bool(got[2].isnan().all()), what
        assert bool(((got[3:] - want[3:]).abs() <= limit).all()), what


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh", "clamped"])
@pytest.mark.parametrize("m,k,inter", [(3, 64, 20), (16, 96, 16), (21, 160, 48)])
def test_pairs(ops, activation, m, k, inter):
    """The three pairs of gate and up value, from far below zero to far above."""
    x, gate, up = rnd((m, k), 17, 3.0), rnd((inter, k), 18, 0.5), rnd((inter, k), 19, 0.5)
    out = torch.empty(m, inter, device=DEV)
    constants = (7.0, 1.702, 1.0) if activation == "clamped" else None
    assert ops.few_rows_take_float32(m, k)
    ops.linear_swiglu(x.to(DEV), interleave_gate_up(gate, up).to(DEV), out, activation, constants)
    g, u = x.double() @ gate.double().T, x.double() @ up.double().T
    # the sums are off by e_g and e_u; |slope| of each activation is at most 1.2 (silu 1.1, tanh gelu 1.13, the clamped
    # 1.1), its own evaluation a few units of the result, and the tanh form's 1 + tanh one unit of the gate's number where it cancels
    unit = (k + 16) * 2.0 ** -24
    e_g, e_u = (unit * (x.double().abs() @ t.double().abs().T) for t in (gate, up))
    if activation == "clamped":
        limit, slope, shift = constants
        g = g.clamp(max=limit)
        v = g * torch.sigmoid(slope * g)
        u = u.clamp(-limit, limit) + shift
    elif activation == "silu":
        v = g * torch.sigmoid(g)
    else:
        v = 0.5 * g * (1 + torch.tanh(0.7978845608028654 * (g + 0.044715 * g ** 3)))
    bound = 1.2 * e_g * u.abs() + e_u * v.abs() + 2.0 ** -20 * (v * u).abs() + 2.0 ** -23 * (g * u).abs() + 1e-12
    assert bool(((out.cpu().double() - v * u).abs() <= bound).all())
