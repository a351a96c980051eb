"""Prompts of the windowed attention with two groups of waves a block, each with every second tile of keys: rows whose second
group has no tile, an odd number of them, a window and a prefix, a sink, sigmoid weights, several requests in a tile; and the
decays of a gated recurrence, one to four rows a block, at the edges of their blocks."""
import pytest
import torch

from test_vivevik_mechanisms import Paged, close, ops_of, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups", [1, 2])
@pytest.mark.parametrize("lengths", [[20], [40], [70, 33], [5, 6, 7, 200], [333]])
@pytest.mark.parametrize("window,keep_first,chunk", [(None, 0, None), (50, 8, None), (None, 0, 64)])
@pytest.mark.parametrize("dim,values,sink_on,weights", [(64, 64, True, "softmax"), (32, 16, False, "softmax"),
                                                        (128, 96, True, "sigmoid"), (64, 128, False, "sigmoid")])
def test_prompts(groups, lengths, window, keep_first, chunk, dim, values, sink_on, weights):
    heads, kv_heads, dtype = 10, 2, torch.bfloat16
    sink, outs = torch.linspace(-1, 1, heads), {}
    for backend in ("emu", "hip"):
        ops = ops_of(backend)
        cache = Paged(ops, dtype, lengths, kv_heads, dim, values, seed=3)
        for b, n in enumerate(lengths):
            proj = torch.cat([torch.zeros(n, heads * dim), randn(n, kv_heads * dim, seed=4 + b),
                              randn(n, kv_heads * values, seed=20 + b)], 1)
            cache.write(proj, heads, list(range(n)), [b] * n)
        rows, starts = sum(lengths), [sum(lengths[:i]) for i in range(len(lengths) + 1)]
        q = randn(rows, heads * dim, seed=40).to(dtype).to(ops.device)
        ints = dict(dtype=torch.int32, device=ops.device)
        outs[backend] = torch.full((rows, heads * values), float("nan"), dtype=dtype, device=ops.device)
        if backend == "hip":
            ops._mixer_lib("windowed_attention").llmlab_debug_windowed_attention_groups(groups)
        try:
            ops.sink_window_attention(q, heads, kv_heads, dim, values, cache.k_cache, cache.v_cache, cache.table, cache.page,
                                      torch.tensor([i for n in lengths for i in range(n)], **ints),
                                      torch.tensor([b for b, n in enumerate(lengths) for _ in range(n)], **ints), window,
                                      keep_first, sink.to(ops.device) if sink_on else None, 0.3, outs[backend],
                                      torch.tensor(starts, **ints), 1, 2, 0, weights, chunk)
        finally:
            if backend == "hip":
                ops._mixer_lib("windowed_attention").llmlab_debug_windowed_attention_groups(0)
    close(outs["hip"], outs["emu"], dtype, f"{groups} groups")


@pytest.mark.parametrize("kind", ["sigmoid", "double_exp"])
@pytest.mark.parametrize("rows,channels,rank", [(1, 448, 32), (257, 448, 32), (512, 300, 30), (701, 448, 7), (1401, 256, 32),
                                                (2049, 100, 1028)])
def test_decays(rows, channels, rank, kind):
    """Against 64 bits, and to the bit what a row by itself gets (its sum has one order however many share its block)."""
    ops = ops_of("hip")
    low, w2, bias = (randn(*s, seed=i).to(ops.device) for i, s in ((50, (rows, rank)), (51, (channels, rank)), (52, (channels,))))
    w2 *= rank ** -0.5
    out, alone = torch.empty(rows, channels, device=ops.device), torch.empty(1, channels, device=ops.device)

    def run(low, out):
        ops._call(ops._mixer_lib("linear_attention").llmlab_gla_decay, low.data_ptr(), low.stride(0), low.shape[0], rank, w2.data_ptr(),
                  bias.data_ptr(), 0 if kind == "sigmoid" else 1, 8.0, out.data_ptr(), channels, 0, ops._stream(),
                  lib=ops._mixer_lib("linear_attention"))
    run(low, out)
    z = bias.double() + (low.double() if kind == "sigmoid" else low.double().tanh()) @ w2.double().T
    want = z.sigmoid() ** (1 / 8) if kind == "sigmoid" else (-z.exp()).exp()
    # (a sum of `rank` terms in 32 bits, through functions of slope 1 at most, and their own few units)
    bound = (rank + 16) * 2.0 ** -24 * (1 + low.double().abs().max() * w2.double().abs().sum(1).max())
    assert (out.double() - want).abs().max() <= bound
    for r in {0, rows // 2, rows - 1}:
        run(low[r:r + 1], alone)
        assert torch.equal(alone[0], out[r])
