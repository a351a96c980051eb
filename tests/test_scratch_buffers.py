"""Scratch buffers asked for in the middle of a run: a new one moves none of the others, so the calls that a block
has written down stay and later blocks' are written down; one that grows moves, and drops them."""
import pytest
import torch

import helpers as H
import vivevik_cases as V
from emu_ops import EmuOps


def vivevik(**kw):
    return V.make_engine("P", 1, "bf16", ops=EmuOps(), device="cpu", **kw)


def test_first_decode_step_writes_all_blocks_down():
    """A prompt of many rows cuts no product; the first decode step does and asks for the pieces' buffers: its
    blocks' calls are written down all the same, and the second step makes them from the list."""
    engine = vivevik()
    engine.ops.rules.min_steps_per_split = 1
    ids = V.random_ids(V.config_of("P"), 72, 3)
    request = engine.open("r")
    engine.step([H.lab.StepEntry(request, ids[:70], [])])
    made = engine.step_fn.ctx.scratch_allocations
    prompt = engine.model.launches_recorded
    keeping = sum(engine.model.blocks[v.block].keeps_launches for v in engine.model.entries)
    engine.step([H.lab.StepEntry(request, [ids[70]], [0])])
    assert engine.step_fn.ctx.scratch_allocations > made
    assert engine.model.launches_recorded - prompt == keeping > 0
    replayed = engine.model.launches_replayed
    engine.step([H.lab.StepEntry(request, [ids[71]], [0])])
    assert engine.model.launches_replayed - replayed == keeping
    engine.close(request)


def test_a_buffer_that_grows_moves(monkeypatch):
    ctx = vivevik().step_fn.ctx
    small = ctx.scratch("a", (4, 4), torch.float32)
    assert ctx.scratch("a", (2, 4), torch.float32).data_ptr() == small.data_ptr()
    before = ctx.scratch_version
    ctx.scratch("b", (4, 4), torch.float32)
    assert ctx.scratch_version == before
    ctx.scratch("a", (8, 4), torch.float32)
    assert ctx.scratch_version == before + 1

    def full(*args, **kw):
        raise RuntimeError("no memory")
    with monkeypatch.context() as m:
        m.setattr(torch, "empty", lambda *a, **kw: full() if a and a[0] == 64 else torch.zeros(*a, **kw))
        with pytest.raises(RuntimeError):
            ctx.scratch("a", (16, 4), torch.float32)
    assert ctx.scratch_version == before + 2          # (the old one has been given back: nothing may still point at it)
    assert ctx.scratch("a", (8, 4), torch.float32).shape == (8, 4)


@pytest.mark.parametrize("backend", ["emu", pytest.param("hip", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("design,name", [("vivevik", "P"), ("qwen2", "B")])
def test_no_memory_left_for_pieces(backend, dtype, design, name):
    """A step that fits while its products are taken whole still runs when the rules would cut them and nothing
    is left for the pieces: the same bits as whole."""
    cases = V if design == "vivevik" else H
    kw = dict(ops=EmuOps(), device="cpu") if backend == "emu" else {}
    engine = cases.make_engine(name, 1, dtype, **kw)
    ids = cases.random_ids(cases.config_of(name), 21, 3)
    outs = []
    for least in (10 ** 6, 1):
        engine.ops.rules.min_steps_per_split = least
        request = engine.open(least)
        outs.append([engine.step([H.lab.StepEntry(request, ids[:20], [19])]).clone(),
                     engine.step([H.lab.StepEntry(request, ids[20:], [0])]).clone()])
        engine.close(request)
        engine.step_fn.ctx._memory_available = lambda enough: 0
    made = engine.step_fn.ctx.scratch_allocations
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    assert engine.step_fn.ctx.scratch_allocations == made


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_no_memory_left_for_pieces_under_capture(dtype):
    """Memory that turns up while a graph is captured makes no buffer inside it: the graph does what the eager
    step before it did, at every replay."""
    runs = []
    for graph in (False, True):
        engine = V.make_engine("P", 1, dtype, graph=graph)
        ids = V.random_ids(V.config_of("P"), 40, 5)
        engine.ops.rules.min_steps_per_split = 10 ** 6
        requests = [engine.open(i) for i in range(3)]
        engine.step([H.lab.StepEntry(r, ids[:20 + i], [19]) for i, r in enumerate(requests)])
        engine.step([H.lab.StepEntry(r, [ids[29]], [0]) for r in requests])
        ctx = engine.step_fn.ctx
        if graph:
            engine.ops.rules.min_steps_per_split = 1
            ctx._memory_available = lambda enough: (1 << 40) if torch.cuda.is_current_stream_capturing() else 0
        outs = []
        for i in range(6):
            outs.append(engine.step([H.lab.StepEntry(r, [ids[30 + i]], [0]) for r in requests]).clone())
            torch.cuda.synchronize()
        if graph:
            assert engine.step_fn.graph_captures > 0 and engine.step_fn.graph_replays > 0
            assert not any(name.endswith(".pieces") for name, _ in ctx._scratch)
        runs.append(outs)
    assert all(torch.equal(a, b) for a, b in zip(*runs))
