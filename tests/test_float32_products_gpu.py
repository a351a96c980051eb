"""The float32 products of many rows that split every number into three bfloat16 parts
(``gemm_f32_split_kernel``): all tiles, whole and in pieces, against 64 bits at the edges of the
tiles, with numbers of very different sizes, and with numbers that have no such parts."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from llm_inference_lab_amd.kernels.hip_ops import HipOps
    return HipOps(DEV)


def rnd(shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed))


def bound(x, w):
    """What 32-bit sums of ``k`` products in any order may be off by: ``k`` roundings (and, of the split, the
    three left-out terms, below two more) of half a unit of the sum of the absolute products."""
    return (x.shape[1] + 4) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)


@pytest.mark.parametrize("tile", [64, 128, 131, None])
@pytest.mark.parametrize("m,n,k", [(65, 64, 32), (66, 65, 33), (127, 63, 31), (128, 128, 64), (129, 130, 100),
                                   (192, 257, 1), (193, 36, 1153)])
def test_against_64_bits(ops, tile, m, n, k):
    # (sizes spread over 2^-30 .. 2^30: all three parts of a number matter)
    x = rnd((m, k), 1) * torch.exp2(torch.randint(-30, 31, (m, k), generator=torch.Generator().manual_seed(2)).float())
    w = rnd((n, k), 3)
    want, limit = x.double() @ w.double().T, bound(x, w)
    dx, dw = x.to(DEV), ops.prepare_weight(w.to(DEV))
    with ops.debug.force(gemm_tile=tile):
        out = torch.empty(m, n, device=DEV)
        ops.linear_logits(dx, dw, out)
        assert bool(((out.cpu().double() - want).abs() <= limit).all())
        for pieces in (2, 3):
            parts = torch.full((pieces, m, n), float("nan"), device=DEV)
            ops.linear_partials(dx, dw, parts, pieces)
            got = parts.cpu().double().sum(0)
            assert bool(((got - want).abs() <= limit).all()), f"{pieces} pieces"


@pytest.mark.parametrize("tile", [64, 128, 131])
@pytest.mark.parametrize("one_part", [False, True])
def test_numbers_without_parts(ops, tile, one_part):
    """Infinities, numbers that bfloat16 rounds to infinity and NaN: as plain 32-bit FMAs give them.  ``one_part``: W's
    numbers are bfloat16 ones, infinite and NaN among them and one below the smallest normal number."""
    m, n, k = 70, 66, 40
    x, w = rnd((m, k), 5), rnd((n, k), 6)
    x[3, 7], x[10, 0], x[20, 39], x[65, 1] = float("inf"), 3.4e38, float("nan"), -float("inf")
    w[:, 0] = 1e-38 * w[:, 0]
    if one_part:
        w[5, 2], w[9, 35], w[40, 39], w[64, 3] = float("inf"), -float("inf"), float("nan"), 2.0 ** -130
        w = w.bfloat16().float()
    want = x.double() @ w.double().T
    out = torch.empty(m, n, device=DEV)
    with ops.debug.force(gemm_tile=tile):
        ops.linear_logits(x.to(DEV), w.to(DEV), out)
    got = out.cpu().double()
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isinf(), want.isinf()) and torch.equal(got[want.isinf()], want[want.isinf()])
    fine = want.isfinite()
    limit = torch.where(fine, bound(x, w), torch.zeros(()).double())
    assert bool(((got - want).abs()[fine] <= limit[fine]).all())


@pytest.mark.parametrize("tile", [64, 128, 131])
@pytest.mark.parametrize("m,n,k", [(70, 66, 40), (129, 130, 100), (65, 64, 33)])
@pytest.mark.parametrize("size", [-100, -104, -107, -110, -111, -112, -116, -120, -124, -126, -140])
@pytest.mark.parametrize("one_part", [False, True])
def test_small_numbers(ops, tile, m, n, k, size, one_part):
    """Numbers whose last bits lie under bfloat16's smallest (or that are below float32's smallest normal number), in
    one row among ordinary ones, in a few places among zeros, and on the other side of the product; beside
    numbers of three parts and of one."""
    x, w = rnd((m, k), 7), rnd((n, k), 8) * 2.0 ** 90
    if one_part:
        w = w.bfloat16().float()
    x[3] *= 2.0 ** size
    alone = torch.arange(m - 9, m)
    x[alone] = 0
    x[alone, alone % k] = rnd((9,), 11) * 2.0 ** size
    for a, b in ((x, w), (w, x)):
        want, limit = a.double() @ b.double().T, bound(a, b)
        # (a product below float32's smallest normal number is a whole number of its steps, 2^-149)
        limit = limit + a.shape[1] * 2.0 ** -149
        one = (a != 0).sum(1, keepdim=True) * (b != 0).sum(1) < 2 * a.shape[1]      # (a product alone: no sum to round)
        limit = torch.where(one, 4 * 2.0 ** -24 * want.abs() + 2.0 ** -149, limit)
        out = torch.empty(a.shape[0], b.shape[0], device=DEV)
        with ops.debug.force(gemm_tile=tile):
            ops.linear_logits(a.to(DEV), b.to(DEV), out)
            parts = torch.full((2, a.shape[0], b.shape[0]), float("nan"), device=DEV)
            ops.linear_partials(a.to(DEV), b.to(DEV), parts, 2)
        assert bool(((out.cpu().double() - want).abs() <= limit).all())
        assert bool(((parts.cpu().double().sum(0) - want).abs() <= limit).all())


@pytest.mark.parametrize("tile", [64, 128, 131])
@pytest.mark.parametrize("one_part", [False, True])
def test_sums_that_overflow(ops, tile, one_part):
    """Numbers that have parts and a product past the largest float32: infinite, not NaN; a product just below it,
    whose leading parts' product is past it: finite.  ``one_part``: W's numbers are bfloat16 ones."""
    m, n, k = 70, 66, 40
    x, w = rnd((m, k), 9), rnd((n, k), 10)
    x[0], x[1], x[2] = 0, 0, 0
    x[0, 5], w[:33, 5] = 1e38, 1003000.0
    x[1, 6], w[7, 6] = 1e30, 1.0037e12
    root = 2.0 ** 64 * (1 - 2.0 ** -10)          # (its leading part is 2^64)
    x[2, 9], w[11, 9] = root, root
    if one_part:
        w[11, 9] = 2.0 ** 64
        w = w.bfloat16().float()
    want = (x.double() @ w.double().T)
    limit = bound(x, w)
    want = torch.where(want.abs() >= 2.0 ** 128 * (1 - 2.0 ** -25), want.sign() * float("inf"), want)
    assert bool(want[0, :33].isinf().all()) and bool(want[1, 7].isinf()) and bool(want[2, 11].isfinite())
    out = torch.empty(m, n, device=DEV)
    with ops.debug.force(gemm_tile=tile):
        ops.linear_logits(x.to(DEV), w.to(DEV), out)
    got = out.cpu().double()
    fine = want.isfinite()
    assert torch.equal(got[~fine], want[~fine])
    assert bool(((got - want).abs()[fine] <= limit[fine]).all())


@pytest.mark.parametrize("tile", [64, 128, 131])
@pytest.mark.parametrize("m,n,k", [(65, 64, 32), (128, 256, 64), (129, 257, 96), (127, 255, 36), (130, 300, 100), (70, 66, 33),
                                   (200, 520, 1152)])
@pytest.mark.parametrize("odd", [None, 0, -1])
def test_weights_of_one_part(ops, tile, m, n, k, odd):
    """Matrices whose numbers are bfloat16 numbers take half of the part products; one other number, in the first
    step of the inner size or in the last, makes its blocks take all.  Whole, in pieces and paired."""
    x, w = rnd((m, k), 21), rnd((n, k), 22).bfloat16().float()
    if odd is not None:
        w[n // 2, odd] = 1.0 + 2.0 ** -20
    want, limit = x.double() @ w.double().T, bound(x, w)
    dx, dw = x.to(DEV), ops.prepare_weight(w.to(DEV))
    with ops.debug.force(gemm_tile=tile):
        out = torch.empty(m, n, device=DEV)
        ops.linear_logits(dx, dw, out)
        assert bool(((out.cpu().double() - want).abs() <= limit).all())
        parts = torch.full((3, m, n), float("nan"), device=DEV)
        ops.linear_partials(dx, dw, parts, 3)
        assert bool(((parts.cpu().double().sum(0) - want).abs() <= limit).all())
        if n % 32 == 0:
            paired = torch.empty(m, n // 2, device=DEV)
            ops.linear_swiglu(dx, dw, paired)
            both = out.cpu().reshape(m, n // 32, 2, 16).double()
            want_p = (both[:, :, 0] * torch.sigmoid(both[:, :, 0]) * both[:, :, 1]).reshape(m, n // 2)
            # (the same sums; the activation and two products in 32 bits: a few roundings of 2^-24, the exponential 2 ulp)
            assert bool(((paired.cpu().double() - want_p).abs() <= 2.0 ** -20 * want_p.abs() + 1e-30).all())


def test_products_of_many_steps_of_one_part_and_three_agree(ops):
    """The part products left out are zeros: the sums are the same to the bit."""
    m, n, k = 150, 512, 640
    x, w = rnd((m, k), 23).to(DEV), rnd((n, k), 24).bfloat16().float().to(DEV)
    # (a row of other numbers behind every 31: all blocks of this matrix take three parts)
    mixed = torch.full((n + n // 31 + 1, k), 1.0 + 2.0 ** -20, device=DEV)
    places = torch.tensor([i for i in range(mixed.shape[0]) if i % 32 != 31][:n], device=DEV)
    mixed[places] = w
    for tile in (64, 128, 131):
        with ops.debug.force(gemm_tile=tile):
            one, three = torch.empty(m, n, device=DEV), torch.empty(m, mixed.shape[0], device=DEV)
            ops.linear_logits(x, ops.prepare_weight(w), one)
            ops.linear_logits(x, ops.prepare_weight(mixed), three)
            assert torch.equal(one, three[:, places]), f"tile {tile}"


@pytest.mark.parametrize("tile", [64, 128, 131])
@pytest.mark.parametrize("k", [32, 160, 330, 352])
def test_a_number_of_three_parts_in_any_step(ops, tile, k):
    """From the step on that holds the first such number a block takes all parts; its sums are those of a block that
    takes all parts from the start, to the bit."""
    m, n = 140, 300
    x, w = rnd((m, k), 25).to(DEV), rnd((n, k), 26).bfloat16().float()
    rows = [5, 150, 290]      # (one a block of every tile at least)
    rest = torch.tensor([r for r in range(n) if r not in [b + 1 for b in range(0, n, 64)]], device=DEV)
    general = w.clone()
    general[[b + 1 for b in range(0, n, 64)], 0] = 1.0 + 2.0 ** -20      # (a row of every block, left out below)
    with ops.debug.force(gemm_tile=tile):
        for at in range(0, k, 32):
            for row in rows:
                late, first = w.clone(), general.clone()
                late[row, min(at + 7, k - 1)] = first[row, min(at + 7, k - 1)] = 1.0 + 2.0 ** -19
                got, want = torch.empty(m, n, device=DEV), torch.empty(m, n, device=DEV)
                ops.linear_logits(x, ops.prepare_weight(late.to(DEV)), got)
                ops.linear_logits(x, ops.prepare_weight(first.to(DEV)), want)
                assert torch.equal(got[:, rest], want[:, rest]), f"step {at // 32}, row {row}"


@pytest.mark.parametrize("tile", [64, 128, 131])
def test_a_late_number_of_three_parts_costs_no_second_walk(ops, tile):
    """A matrix with one such number a block, in the last step, takes little longer than one of such numbers (which
    takes about as long as a walk by itself; two walks would take 1.6 times as long)."""
    m, n, k = 1536, 4096, 896
    x, w = rnd((m, k), 27).to(DEV), rnd((n, k), 28)
    late = w.bfloat16().float()
    late[::64, -1] = 1.0 + 2.0 ** -20
    out = torch.empty(m, n, device=DEV)

    def time(weight):
        weight, best = ops.prepare_weight(weight.to(DEV)), float("inf")
        for _ in range(12):
            marks = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            marks[0].record()
            for _ in range(10):
                ops.linear_logits(x, weight, out)
            marks[1].record()
            torch.cuda.synchronize()
            best = min(best, marks[0].elapsed_time(marks[1]))
        return best

    with ops.debug.force(gemm_tile=tile):
        assert time(late) < 1.25 * time(w)
