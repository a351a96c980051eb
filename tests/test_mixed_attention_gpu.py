"""Mixed steps of many requests: a block of a launch for one kind of requests finds its request by counting
(64 requests a load), wherever the portions stand among the decoding requests."""
import pytest
import torch

from llm_inference_lab_amd.cache import layout as cache_layout
from llm_inference_lab_amd.parts.base import ShortRequests
from test_kernels_gpu import DEV, emu, make_cache, ops, rnd, run_attention  # noqa: F401 (fixtures)

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
    behind histories short and long (the switch takes it to that launch whatever the rule says)."""
    for spec in ([(0, 3), (5, 1)], [(0, 17), (900, 1), (64, 1)], [(700, 1), (33, 50), (1500, 1), (0, 129)]):
        with ops.debug.force(attention_small_tiles=d):
            run_attention(ops, emu, torch.bfloat16, nq, nkv, d, page, window, spec, seed=97)


@pytest.mark.parametrize("splits", [1, 2, 3, 7])
@pytest.mark.parametrize("nq,nkv,d,portion", [(14, 2, 64, 464), (8, 2, 32, 300), (12, 2, 128, 100)])
def test_tiles_of_16_rows_beside_split_keys(ops, nq, nkv, d, portion, splits):  # noqa: F811
    """Steps that the rule itself takes there, with the decoding requests' keys split over blocks and merged by the
    last block to arrive and by a kernel: the same as in a launch for each kind."""
    decoding = 60 if d < 128 else 40
    spec = [(1400 - 23 * i, 1) for i in range(decoding)] + [(150, portion), (0, 33)]
    run, counted = step(ops, torch.bfloat16, nq, nkv, d, 64, spec, 99)
    how = ops._attention_lib(d).llmlab_attention_mixed_launches(nq, nkv, len(spec), decoding, portion, 1401, 1401, 0, ops.num_cus)
    assert how == 3, how
    with ops.debug.force(attention_two_launches=d):
        want = run(counted)
    bound = 2e-2 * max(1.0, want.abs().max().item())
    assert (run(counted) - want).abs().max().item() <= bound
    for merged in ("attention_merge_kernel", "attention_merge_in_place"):
        with ops.debug.force(attention_small_tiles=d, attention_splits=(d, splits), **{merged: d}):
            for described in (counted, tuple(counted)):
                assert (run(described) - want).abs().max().item() <= bound, (merged, len(described))
    assert int(ops.arrived.abs().sum()) == 0


def step(ops, dtype, nq, nkv, d, page, spec, seed):  # noqa: F811
    """A step over requests ``(start, tokens)``; a function that takes its description and returns its rows, and
    the description as it is counted."""
    per = max(-(-(s + n) // page) for s, n in spec)
    starts = [0]
    for _, n in spec:
        starts.append(starts[-1] + n)
    q = rnd((starts[-1], (nq + 2 * nkv) * d), dtype, seed).to(DEV)
    kc, vc = make_cache(per * len(spec) + 1, nkv, page, d, dtype, seed + 1)
    kc, vc = cache_layout.keys_to_cache_order(kc).to(DEV), cache_layout.values_to_cache_order(vc).to(DEV)
    table = torch.arange(per * len(spec), dtype=torch.int32, device=DEV).view(len(spec), per)
    row_req = torch.cat([torch.full((n,), b) for b, (_, n) in enumerate(spec)]).int().to(DEV)
    q_start, start_pos = (torch.tensor(v, dtype=torch.int32, device=DEV) for v in (starts, [s for s, _ in spec]))
    longest, most = max(n for _, n in spec), max(s + n for s, n in spec)
    counted = ShortRequests.count(row_req, ops.attention_short_limit(nq, nkv, dtype, longest), starts, [s for s, _ in spec],
                                  len(spec))

    def run(short):
        out = torch.full((starts[-1], nq * d), 777.0, dtype=dtype, device=DEV)
        ops.paged_attention(q, nq, nkv, d, kc, vc, table, page, q_start, start_pos, len(spec), longest, most, None,
                            d ** -0.5, out, short)
        return out.float()
    return run, counted


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("nq,nkv,d", [(14, 2, 64), (8, 2, 128)])
@pytest.mark.parametrize("portion", [21, 300])
def test_a_count_that_the_caller_only_claims(ops, dtype, nq, nkv, d, portion):  # noqa: F811
    """A count of short requests that is not that of the step (one too many, one too few, nearly all) leaves no row
    unwritten: only a counted description bounds the blocks of a launch."""
    spec = [(60 + 7 * i, 1) for i in range(9)] + [(500, portion), (0, 40), (33, portion)]
    run, counted = step(ops, dtype, nq, nkv, d, 64, spec, 98)
    assert counted[2:] == (9, 117)
    want = run(None)
    bound = (2e-5 if dtype == torch.float32 else 2e-2) * max(1.0, want.abs().max().item())
    assert (run(counted) - want).abs().max().item() <= bound
    for claimed in (1, 8, 9, 10, 11):
        got = run((counted[0], counted[1], claimed, 117))
        assert (got - want).abs().max().item() <= bound, claimed
