"""Attention of many rows at heads of 64 and 128: a value that is not finite belongs to its position alone. Rows whose tile ends
before it, or whose windows begin behind it, give what they give without it, to the bit."""
import pytest
import torch

from llm_inference_lab_amd.cache import layout
from test_kernels_gpu import DEV, ops, rnd  # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu
TILE = 32          # rows (a token and a head of a group each) that share their products


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("window", [None, 40])
@pytest.mark.parametrize("path", [0, 2, 3, 4, 6])
@pytest.mark.parametrize("nq,nkv,d", [(2, 2, 64), (7, 1, 64), (2, 2, 128), (4, 1, 128)])
@pytest.mark.parametrize("start", [0, 70])
def test_rows_before_and_behind(ops, start, nq, nkv, d, path, window, value):  # noqa: F811
    page, n, group = 64, 200, nq // nkv
    pages = (start + n + page - 1) // page
    q = rnd((n, (nq + 2 * nkv) * d), torch.bfloat16, 121).to(DEV)
    keys = layout.keys_to_cache_order(rnd((pages, nkv, page, d), torch.bfloat16, 122)).to(DEV)
    plain = rnd((pages, nkv, d, page), torch.bfloat16, 123)
    table = torch.arange(pages, dtype=torch.int32, device=DEV).view(1, -1)
    q_start, start_pos = (torch.tensor(v, dtype=torch.int32, device=DEV) for v in ([0, n], [start]))

    def run(values):
        values = layout.values_to_cache_order(values).to(DEV)
        out = torch.full((n, nq * d), 777.0, dtype=torch.bfloat16, device=DEV)
        with ops.debug.force(attention_path=(d, path)):
            ops.paged_attention(q, nq, nkv, d, keys, values, table, page, q_start, start_pos, 1, n, start + n, window, d ** -0.5, out)
        return out
    clean = run(plain)
    for token in (0, 31, 32, 101, 130):
        at = start + token
        marked = plain.clone()
        marked[at // page, :, :, at % page] = value
        got = run(marked)
        before = token * group // TILE * TILE // group      # tokens of the tiles that end before the marked one's
        assert torch.equal(got[:before], clean[:before]), (token, "before")
        if window is not None:
            # ... and of the first tile on whose first window begins behind the 32 positions with the marked one
            tile = next(t for t in range(n * group) if start + t * TILE // group - window + 1 >= at // 32 * 32 + 32)
            behind = -(-tile * TILE // group)
            assert torch.equal(got[behind:], clean[behind:]), (token, "behind")
    # (the marked token's own row has it in its sum)
    assert not got[130].isfinite().any()
