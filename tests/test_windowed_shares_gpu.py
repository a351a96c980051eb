"""The shares that a decoding row's keys are cut into follow from the row and the number of rows of the launch, not
from the longest history announced: a step that is told of longer ones (as one replayed from a graph is) gives the
same bits."""
import pytest
import torch

from test_vivevik_mechanisms import Paged, close, ops_of, randn

pytestmark = pytest.mark.gpu


# (one tile, two, an odd number, many; a window whose first tile is cut; one kernel's share against several)
@pytest.mark.parametrize("lengths", [[7, 33], [36, 70, 1], [64, 97, 300], [1500, 129]])
@pytest.mark.parametrize("window,keep_first", [(None, 0), (100, 8)])
def test_longer_histories_announced_change_nothing(lengths, window, keep_first):
    heads, kv_heads, dim, values, dtype = 6, 2, 64, 96, torch.bfloat16
    ops = ops_of("hip")
    cache = Paged(ops, dtype, lengths, kv_heads, dim, values, seed=3)
    for b, n in enumerate(lengths):
        proj = torch.cat([torch.zeros(n, heads * dim), randn(n, kv_heads * dim, seed=4 + b),
                          randn(n, kv_heads * values, seed=20 + b)], 1)
        cache.write(proj, heads, list(range(n)), [b] * n)
    rows = len(lengths)
    q = randn(rows, heads * dim, seed=40).to(dtype).to(ops.device)
    ints = dict(dtype=torch.int32, device=ops.device)
    positions = torch.tensor([n - 1 for n in lengths], **ints)
    sink = torch.linspace(-1, 1, heads).to(ops.device)
    reach = max(lengths) * 99 if window is None else window + keep_first      # (no more is ever announced)
    outs = []
    for keys in (max(lengths), max(128, 2 * max(lengths)), 4096):
        out = torch.full((rows, heads * values), float("nan"), dtype=dtype, device=ops.device)
        ops.sink_window_attention(q, heads, kv_heads, dim, values, cache.k_cache, cache.v_cache, cache.table, cache.page,
                                  positions, torch.arange(rows, **ints), window, keep_first, sink, 0.3, out,
                                  torch.arange(rows + 1, **ints), 4, 1, min(keys, reach))
        outs.append(out)
    assert bool(torch.isfinite(outs[0].float()).all())
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("values,shares", [(e, z) for e in (16, 64, 96, 128) for z in (2, 15, 16, 17, 33)] +
                         [(e, z) for e in (192, 256) for z in (2, 7, 8, 9, 17)])
@pytest.mark.parametrize("sink_on", [True, False])
def test_any_number_of_shares_is_merged(values, shares, sink_on):
    """Shares around the chunks that a merge asks for at once (16, or 8 of wide values), against the plain reference: a row
    that fills them all, one that fills a few and leaves the others empty, one of a single key.  Nothing is read
    from scratch that was not written."""
    heads, kv_heads, dim, dtype = 6, 2, 64, torch.bfloat16
    announced = 32 * (2 * shares - 1)
    lengths = [announced, min(300, announced), 1]
    sink = torch.linspace(-1, 1, heads)
    outs = {}
    for backend in ("emu", "hip"):
        ops = ops_of(backend)
        cache = Paged(ops, dtype, lengths, kv_heads, dim, values, seed=3)
        for b, n in enumerate(lengths):
            proj = torch.cat([torch.zeros(n, heads * dim), randn(n, kv_heads * dim, seed=4 + b),
                              randn(n, kv_heads * values, seed=20 + b)], 1)
            cache.write(proj, heads, list(range(n)), [b] * n)
        rows = len(lengths)
        q = randn(rows, heads * dim, seed=40).to(dtype).to(ops.device)
        ints = dict(dtype=torch.int32, device=ops.device)
        if backend == "hip":
            ops.workspace.fill_(float("nan"))
        outs[backend] = torch.full((rows, heads * values), float("nan"), dtype=dtype, device=ops.device)
        ops.sink_window_attention(q, heads, kv_heads, dim, values, cache.k_cache, cache.v_cache, cache.table, cache.page,
                                  torch.tensor([n - 1 for n in lengths], **ints), torch.arange(rows, **ints), None, 0,
                                  sink.to(ops.device) if sink_on else None, 0.3, outs[backend],
                                  torch.arange(rows + 1, **ints), 4, 1, announced)
    close(outs["hip"], outs["emu"], dtype, f"{shares} shares of {values}")
