"""The last pass of a gated recurrence in chunks, by two waves a sub-block of rows (decays, heads of 64 key channels and more):
chunks that end inside a sub-block, halves of unequal width, value sizes that fill no tile, decays that forget everything."""
import pytest
import torch

from test_mazanex_mechanisms import Recurrence, close, ints, ops_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("harsh", [False, True])
@pytest.mark.parametrize("heads,D,E", [(2, 64, 16), (1, 64, 32), (3, 72, 40), (2, 63, 136), (2, 64, 128), (1, 80, 130), (2, 128, 256),
                                       (1, 49, 64), (1, 48, 64)])
def test_edges(heads, D, E, harsh):
    ops = ops_of("hip")
    lengths = [1, 15, 16, 17, 63, 64, 65, 130]
    r = Recurrence("decay", heads, D, E, lengths, seed=7, harsh=harsh)
    state = torch.zeros(len(lengths), heads, D, E, device=ops.device)
    out = r.step(ops, [(0, n) for n in lengths], ints(list(range(len(lengths))), ops.device), state, None, "chunks", torch.float32)
    close(out, torch.cat(r.want), torch.float32, "outputs", f32=1e-4)
    for b, last in enumerate(r.last):
        close(state[b], last, torch.float32, f"state of request {b}", f32=3e-5)
