"""float32 attention of many rows whose waves split the keys of a tile (heads up to 64: blocks of four waves, or of eight where
tiles are few and histories long): the edges of tiles of rows and of the waves' shares of the keys, against the emulation."""
import pytest
import torch

from test_kernels_gpu import DEV, emu, ops, rnd, run_attention  # noqa: F401 (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("window", [None, 40])
@pytest.mark.parametrize("nq,nkv,d,page", [(14, 2, 64, 16), (6, 1, 32, 64), (4, 4, 48, 32)])
def test_edges(ops, emu, window, nq, nkv, d, page):  # noqa: F811
    """One row more and less than a tile; keys one more and less than the four waves' steps; waves without keys; requests of
    different lengths in one launch; a score that stands out late and early."""
    g = nq // nkv
    with ops.debug.force(attention_path=(d, 1)):
        for rows in (16, 32):
            n = max(rows // g, 16 // g + 1)
            run_attention(ops, emu, torch.float32, nq, nkv, d, page, window, [(0, n), (63 - n, n + 1), (64, n)], seed=111,
                          amplify=(0, 1, 30.0))
        run_attention(ops, emu, torch.float32, nq, nkv, d, page, window, [(0, 257), (255, 33), (31, 32)], seed=112,
                      amplify=(0, 200, 30.0))


@pytest.mark.parametrize("nq,nkv,d,page", [(14, 2, 64, 16), (6, 1, 32, 64)])
@pytest.mark.parametrize("spec", [[(767, 1 + 16), (750, 40)], [(740, 20)], [(4090, 60)]])
def test_few_tiles_behind_histories(ops, emu, nq, nkv, d, page, spec):  # noqa: F811
    """On both sides of the length from which eight waves share a tile; more steps than page numbers are read at once."""
    run_attention(ops, emu, torch.float32, nq, nkv, d, page, None, spec, seed=113, amplify=(0, 300, 30.0))


@pytest.mark.parametrize("start", [50, 140 * 64 - 50])
def test_missing_pages_stay_out(ops, start):  # noqa: F811
    """Pages without a number, in the launch by four waves, by eight, and by a wave per tile (bound: the sums' orders)."""
    nq, nkv, page, d, n = 4, 1, 64, 64, 50
    pages = (start + n + page - 1) // page
    q = rnd((n, (nq + 2 * nkv) * d), torch.float32, 114).to(DEV)
    kc, vc = (rnd((pages, nkv, *s), torch.float32, i).to(DEV) for i, s in ((115, (page, d)), (116, (d, page))))
    vc[0] = float("nan")          # (what a missing page reads)
    table = torch.arange(pages, dtype=torch.int32, device=DEV).view(1, -1).clone()
    table[0, 0] = -1
    table[0, pages // 2] = -1 if pages > 2 else pages // 2
    q_start, start_pos = (torch.tensor(v, dtype=torch.int32, device=DEV) for v in ([0, n], [start]))
    got = []
    for path in (1, 2):
        out = torch.full((n, nq * d), 777.0, device=DEV)
        with ops.debug.force(attention_path=(d, path)):
            ops.paged_attention(q, nq, nkv, d, kc, vc, table, page, q_start, start_pos, 1, n, start + n, None, d ** -0.5, out)
        got.append(out)
    assert got[0].isfinite().all()
    assert (got[0] - got[1]).abs().max().item() <= 2e-5 * max(1.0, got[1].abs().max().item())


@pytest.mark.parametrize("window", [None, 768])
@pytest.mark.parametrize("nq,nkv,d", [(8, 8, 64), (8, 8, 48), (8, 4, 32), (8, 8, 16)])
def test_wide_tiles_behind_histories(ops, emu, window, nq, nkv, d):  # noqa: F811
    """Tiles of 32 rows by eight waves, which the rule takes behind histories: rows that end inside a tile and in its first half,
    one row, histories of other lengths in one launch."""
    spec = [(768, 129), (700, 33), (3, 17), (760, 128), (0, 1 + 16 * nkv // nq)]
    assert ops._attention_lib(d).llmlab_attention_f32_blocks(nq, nkv, len(spec), 129, 768 + 129, window or 0, ops.num_cus) == 3
    run_attention(ops, emu, torch.float32, nq, nkv, d, 64, window, spec, seed=117, amplify=(0, 300, 30.0))


@pytest.mark.parametrize("nq,nkv,d,reqs,longest,how", [(8, 8, 64, 16, 257, 1), (8, 8, 64, 8, 257, 17), (16, 16, 32, 8, 300, 1)])
def test_order_of_blocks(ops, emu, nq, nkv, d, reqs, longest, how):  # noqa: F811
    """More tiles than the chip holds, request by request, and the same kernel by tiles: ragged portions, the longest last."""
    assert ops._attention_lib(d).llmlab_attention_f32_blocks(nq, nkv, reqs, longest, longest, 0, ops.num_cus) == how
    with ops.debug.force(attention_path=(d, 1)):
        run_attention(ops, emu, torch.float32, nq, nkv, d, 64, None, [(0, 1 + 31 * i % 97) for i in range(reqs - 1)] + [(0, longest)], seed=118)


@pytest.mark.parametrize("nq,nkv,d,reqs", [(8, 8, 64, 33), (16, 8, 64, 49), (16, 16, 32, 33), (14, 2, 32, 300)])
@pytest.mark.parametrize("window", [None, 20])
def test_dense_decode(ops, emu, nq, nkv, d, reqs, window):  # noqa: F811
    """Decode steps of more blocks than units hold by the plain kernel: histories of one key and of all waves' shares and one more."""
    assert ops._attention_lib(d).llmlab_attention_f32_dense(reqs * nkv, window or 130, ops.num_cus) == 1
    run_attention(ops, emu, torch.float32, nq, nkv, d, 16, window, [((0, 1, 15, 16, 127, 128, 129)[i % 7], 1) for i in range(reqs)], seed=119)
