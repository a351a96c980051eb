"""What the norm behind a sublayer is handed: a whole result, one left in pieces, or a pair of normed results
(``SublayerNormBlock``), with layer norms and RMS norms."""
import types

import pytest
import torch

import helpers as H          # noqa: F401  (puts the repository on the path)
from emu_ops import EmuOps
from llm_inference_lab_amd.config.spec import PartSpec
from llm_inference_lab_amd.parts.base import Mixer
from llm_inference_lab_amd.parts.blocks import SublayerNormBlock
from llm_inference_lab_amd.parts.registry import register_part
from llm_inference_lab_amd.weights.loader import MATRIX, TensorSpec

BACKENDS = ["emu", pytest.param("hip", marks=pytest.mark.gpu)]


def ops_of(backend):
    if backend == "emu":
        return EmuOps()
    from llm_inference_lab_amd.kernels.hip_ops import HipOps
    return HipOps("cuda:0")


class OneProduct(Mixer):
    """A mixer that is one product of its input, whole or left in pieces."""

    writes_output = True

    def __init__(self, size, tensors):
        super().__init__(tensors)
        self.size = size

    def tensor_specs(self):
        return {self.tensor_names["w"]: TensorSpec((self.size, self.size), MATRIX)}

    def bind(self, tensors, ops, dtype):
        super().bind(tensors, ops, dtype)
        self.w = ops.prepare_weight(tensors[self.tensor_names["w"]])

    def forward_into(self, h, out, ctx, entry):
        self.ops.linear_logits(h, self.w, out)

    def forward_split(self, h, out, ctx, entry):
        return self._product_split(h, self.w, out, ctx)

    def weight_bytes(self):
        return self.w.numel() * self.w.element_size()


register_part("mixer", "one_product_of_the_tests", OneProduct)


class Step:
    """The least a block needs of a step."""

    def __init__(self, device, rows):
        self.device, self.n_rows, self.n_reqs, self.pending, self.memo = device, rows, 1, None, {}

    def scratch(self, name, shape, dtype):
        return torch.full(shape, float("nan"), dtype=dtype, device=self.device)


def normed(y, kind, weight, eps):
    if kind == "layernorm":
        y = y - y.mean(1, keepdim=True)
    return y * torch.rsqrt(y.square().mean(1, keepdim=True) + eps) * weight


@pytest.mark.parametrize("backend", BACKENDS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", ["layernorm", "rmsnorm"])
@pytest.mark.parametrize("mixer", ["pair", "sum", "pieces", "whole"])
@pytest.mark.parametrize("feed_forward", [True, False])
def test_what_a_norm_is_handed(backend, dtype, kind, mixer, feed_forward):
    """``pair``: two mixers with norms of their results; ``sum``: the same without; ``pieces``: a product that is
    cut along its inner size; ``whole``: the same product not cut; each with and without a feed-forward."""
    rows, size, inter, eps = 5, 96, 128, 1e-5
    ops = ops_of(backend)
    if mixer == "pieces":
        ops.rules.min_steps_per_split = 1
    gen = torch.Generator().manual_seed(1)
    rnd = lambda *shape: torch.randn(shape, generator=gen)
    one = lambda name: PartSpec("one_product_of_the_tests", dict(size=size), dict(w=name))
    if mixer in ("pair", "sum"):
        normed_too = dict(norm_eps=1e-3, hidden_size=size) if mixer == "pair" else {}
        spec = PartSpec("parallel", dict(left=one("left"), right=one("right"), left_scale=0.7, right_scale=1.2, **normed_too),
                        dict(left_norm="ln", right_norm="rn") if mixer == "pair" else {})
    else:
        spec = one("left")
    norm = lambda name: PartSpec(kind, dict(size=size, eps=eps), dict(weight=name))
    ff = PartSpec("dense", dict(hidden_size=size, intermediate_size=inter, activation="relu2"),
                  dict(up_weight="up", down_weight="down")) if feed_forward else None
    block = SublayerNormBlock(size, spec, norm("n1"), ff, norm("n2") if feed_forward else None)
    t = {name: (rnd(*shape) * scale + offset).to(dtype) for name, shape, scale, offset in (
        ("left", (size, size), 0.1, 0), ("right", (size, size), 0.1, 0), ("up", (inter, size), 0.1, 0),
        ("down", (size, inter), 0.1, 0), ("ln", (size,), 0.1, 1), ("rn", (size,), 0.1, 1), ("n1", (size,), 0.1, 1),
        ("n2", (size,), 0.1, 1))}
    block.bind({name: w.to(ops.device) for name, w in t.items()}, ops, dtype)
    x = rnd(rows, size)
    calls = []
    partials = ops.linear_partials
    ops.linear_partials = lambda *a, **kw: calls.append(1) or partials(*a, **kw)
    stream = x.clone().to(ops.device)
    block.forward(stream, Step(ops.device, rows), types.SimpleNamespace(index=0))
    assert bool(calls) == (mixer == "pieces" and (backend == "hip" or dtype == torch.bfloat16))

    d = {name: w.double() for name, w in t.items()}
    h = x.to(dtype).double()
    y = h @ d["left"].T
    if mixer == "pair":
        y = 0.7 * normed(y, "rmsnorm", d["ln"], 1e-3) + 1.2 * normed(h @ d["right"].T, "rmsnorm", d["rn"], 1e-3)
    elif mixer == "sum":
        y = 0.7 * y + 1.2 * (h @ d["right"].T)
    want = x.double() + normed(y, kind, d["n1"], eps)
    if feed_forward:
        act = ((want.float().to(dtype).double() @ d["up"].T).clamp(min=0) ** 2).to(dtype).double()
        want = want + normed(act @ d["down"].T, kind, d["n2"], eps)
    # float32: sums of up to 128 products, twice, under norms of numbers of order one.  bfloat16: the mixer's input is
    # rounded in both; a unit in the last place of the stream's copy and of the activation may fall the other way,
    # 2^-8 of a number, spread by a product over rows of 96 and 128 of them
    limit = 2e-5 if dtype == torch.float32 else 2e-2
    assert float((stream.cpu().double() - want).abs().max()) <= limit


@pytest.mark.parametrize("backend", BACKENDS)
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("design,name", [("vivevik", "P"), ("vivevik", "Q"), ("mazanex", "R")])
def test_models_whose_products_are_cut(backend, dtype, design, name):
    """Recurrent, windowed and feed-forward sublayers whose last products are left in pieces for the norms: the
    logits of the plain implementation, as without pieces."""
    import mazanex_cases
    import test_mazanex_engine
    import test_vivevik_engine
    import vivevik_cases
    cases, bounds = ((vivevik_cases, test_vivevik_engine) if design == "vivevik" else (mazanex_cases, test_mazanex_engine))
    cfg = cases.config_of(name)
    seqs = {f"r{i}": cases.random_ids(cfg, n, 10 + i) for i, n in enumerate((9, 30, 41))}
    want = {rid: cases.plain_logits(name, 1, ids) for rid, ids in seqs.items()}
    made = {}
    for least in (1, 10 ** 6):
        kw = dict(ops=EmuOps(), device="cpu") if backend == "emu" else {}
        engine = cases.make_engine(name, 1, dtype, **kw)
        engine.ops.rules.min_steps_per_split = least
        calls = []
        partials = engine.ops.linear_partials
        engine.ops.linear_partials = lambda *a, **kw: calls.append(1) or partials(*a, **kw)
        got = H.run_trace(engine, seqs, H.steps_mixed(seqs, max_live=3))
        made[least] = len(calls)
        if dtype == "f32":
            assert H.first_wrong(got, want, bounds.TOL["f32"]) is None
        else:
            err = torch.cat([(got[rid].double() - want[rid].double()).flatten() for rid in seqs])
            assert float(err.square().mean().sqrt()) <= bounds.TOL_BF16[0] and float(err.abs().max()) <= bounds.TOL_BF16[1]
    assert made[10 ** 6] == 0 and (made[1] > 0) == (backend == "hip" or dtype == "bf16")


@pytest.mark.parametrize("shape,splits", [((2, 3, 8), 3), ((1, 3, 8), 2), ((2, 3, 8), 0), ((3, 8), 1)])
def test_pieces_that_are_not_there(shape, splits):
    """A layer norm of more pieces than the buffer holds is refused before any launch."""
    from llm_inference_lab_amd.kernels.hip_ops import HipOps
    from llm_inference_lab_amd.parts.base import PendingSums
    ops = HipOps.__new__(HipOps)          # (its checks alone: no library, no GPU)
    ops.device = torch.device("cpu")

    class Library:
        llmlab_layernorm_add = None
    ops._core = Library()
    launched = []
    ops._call = lambda *a: launched.append(a)
    ops._stream = lambda: None
    with pytest.raises(ValueError):
        ops.layernorm_add(PendingSums(torch.zeros(shape), splits), torch.ones(8), 1e-6, torch.zeros(3, 8))
    assert not launched
    ops.layernorm_add(PendingSums(torch.zeros(2, 3, 8), 2), torch.ones(8), 1e-6, torch.zeros(3, 8))
    assert len(launched) == 1
