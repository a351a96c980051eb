"""Attention of many rows by keys staged in LDS (heads of 64 and 128): every block shape it is launched with, at the edges
of its tiles of rows and stages of keys, against the emulation; fixed from outside, whatever the rule would take."""
import pytest
import torch

from test_kernels_gpu import DEV, emu, ops, rnd, run_attention  # noqa: F401 (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("window", [None, 40])
@pytest.mark.parametrize("path", [2, 3, 4, 6])
@pytest.mark.parametrize("nq,nkv,d,page", [(14, 2, 64, 16), (4, 4, 64, 128), (7, 1, 128, 64)])
def test_edges(ops, emu, window, path, nq, nkv, d, page):  # noqa: F811
    """One row more and less than a tile of 32, 64 and 128; keys one more and less than a stage; waves without rows."""
    g = nq // nkv
    with ops.debug.force(attention_path=(d, path)):
        for rows in (32, 64, 128):
            n = max(rows // g, 17 // g + 1)
            run_attention(ops, emu, torch.bfloat16, nq, nkv, d, page, window, [(0, n), (127 - n, n + 1), (128, n)],
                          seed=101, amplify=(0, 1, 30.0))
        run_attention(ops, emu, torch.bfloat16, nq, nkv, d, page, window, [(0, 257), (255, 33), (31, 32)], seed=102,
                      amplify=(0, 200, 30.0))


@pytest.mark.parametrize("path", [2, 3, 6])
@pytest.mark.parametrize("nq,nkv,d,page", [(14, 2, 64, 16), (6, 1, 128, 64)])
def test_more_tiles_than_are_located_at_once(ops, emu, path, nq, nkv, d, page):  # noqa: F811
    with ops.debug.force(attention_path=(d, path)):
        run_attention(ops, emu, torch.bfloat16, nq, nkv, d, page, None, [(8180, 40), (4090, 40)], seed=103)


@pytest.mark.parametrize("path", [2, 3, 4, 6])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("lost", [[3], [0], [130], [2, 70, 139]])
def test_missing_pages_stay_out(ops, path, d, lost):  # noqa: F811
    """Pages without a number: as in the launch whose waves split the keys of a tile (bound: the results' rounding)."""
    nq, nkv, page, start, n = 4, 1, 64, 140 * 64 - 50, 50
    pages = 140
    q = rnd((n, (nq + 2 * nkv) * d), torch.bfloat16, 104).to(DEV)
    kc, vc = (rnd((pages, nkv, *s), torch.bfloat16, i).to(DEV) for i, s in ((105, (page, d)), (106, (d, page))))
    vc[0] = float("nan")          # (what a missing page reads)
    table = torch.arange(pages, dtype=torch.int32, device=DEV).view(1, -1).clone()
    table[0, lost] = -1
    table[0, 0] = -1
    q_start, start_pos = (torch.tensor(v, dtype=torch.int32, device=DEV) for v in ([0, n], [start]))
    got = {}
    for p in (1, path):
        out = torch.full((n, nq * d), 777.0, dtype=torch.bfloat16, device=DEV)
        with ops.debug.force(attention_path=(d, p)):
            ops.paged_attention(q, nq, nkv, d, kc, vc, table, page, q_start, start_pos, 1, n, start + n, None, d ** -0.5, out)
        got[p] = out.float()
    assert got[path].isfinite().all()
    assert (got[path] - got[1]).abs().max().item() <= 2e-2 * max(1.0, got[1].abs().max().item())
