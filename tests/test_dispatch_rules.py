"""The host-side choices of the matrix products (which tile, how many pieces along the inner
size, which block shape for few rows) are plain functions of the sizes: they run here without
a GPU, over sizes drawn at random, against what every choice must satisfy, and a few
measured decisions are pinned so that a change of a constant shows."""
import ctypes
import math
import random
import shutil

import pytest

from llm_inference_lab_amd.kernels import build

CUS = 256
KINDS = {0: (64, 64), 1: (64, 128), 2: (128, 128), 3: (128, 256), 4: (256, 256), 5: (192, 256)}


@pytest.fixture(scope="module")
def core():
    if shutil.which("hipcc") is None and not build.hipcc_path():
        pytest.skip("no hipcc to build the library with")
    try:
        lib = ctypes.CDLL(build.core_library())
    except (OSError, RuntimeError) as err:
        pytest.skip(f"the core library does not load here: {err}")
    lib.llmlab_linear_tile.restype = ctypes.c_int
    lib.llmlab_linear_plan.restype = None
    lib.llmlab_skinny_shape.restype = None
    return lib


def plan(core, m, n, k, max_pieces=16, min_tiles=8):
    out = (ctypes.c_int * 2)()
    core.llmlab_linear_plan(m, n, k, CUS, max_pieces, min_tiles, out)
    return out[0], out[1]


def test_tile_and_pieces_of_products_of_many_rows(core):
    rng = random.Random(5)
    for _ in range(3000):
        m = rng.choice([rng.randint(1, 64), rng.randint(65, 600), rng.randint(601, 9000)])
        n = rng.randint(1, 60000)
        k = 8 * rng.randint(1, 4000)
        width = core.llmlab_linear_tile(m, n, k, CUS)
        assert width in (64, 128, 256), (m, n, k, width)
        # the tiles of 256 columns are for steps of many rows (of a wide matrix: from 129 on),
        # and inner sizes they were measured at
        if width == 256:
            one_tile = 64 < m <= 128 and 32768 <= n <= 65536 and k >= 1024      # (the 128 x 256 tile of eight waves)
            assert ((m >= 512 or (m > 128 and n >= 16384)) and k >= 896) or one_tile, (m, n, k)
        pieces, kind = plan(core, m, n, k)
        assert 1 <= pieces <= 16 and kind in KINDS, (m, n, k, pieces, kind)
        if pieces > 1:
            tiles = (k + 63) // 64
            assert (tiles + pieces - 1) // pieces >= 8, (m, n, k, pieces)      # whole K tiles, enough of them
            assert kind != 3, "the 128 x 256 tile of eight waves makes no pieces"
        if kind in (4, 5):
            assert (m >= 512 or (m > 128 and n >= 16384 and pieces == 1)) and k >= 896, (m, n, k, kind)


DIRECT = {10: (128, 128), 11: (128, 192), 12: (192, 128)}      # (by direct loads: put in the place of a tile of KINDS)


def launched_width(core, m, n, k, cus=CUS):
    """Of a whole product whose tile the estimates name."""
    out = (ctypes.c_int * 2)()
    core.llmlab_linear_plan(m, n, k, cus, 1, 8, out)
    direct = core.llmlab_direct_tile(out[1], m, n, k, 1, 0, cus)
    return (KINDS[out[1]] if direct < 0 else DIRECT[direct])[1]


def test_a_plan_in_one_piece_names_the_tile_of_the_whole_product(core):
    """That the estimates name, and with the direct tiles in their place that which is launched."""
    rng = random.Random(9)
    whole = direct = 0
    for _ in range(20000):
        m, n, k = rng.randint(17, 2560), 16 * rng.randint(4, 700), 8 * rng.randint(8, 900)
        pieces, kind = plan(core, m, n, k)
        if pieces == 1:
            whole += 1
            assert KINDS[kind][1] == core.llmlab_linear_tile(m, n, k, CUS), (m, n, k, kind)
            if m > 128 or k < 1024:      # (else one_round_tile is asked first)
                assert core.llmlab_plain_tile(m, n, k, CUS) == launched_width(core, m, n, k), (m, n, k, kind)
                direct += launched_width(core, m, n, k) != KINDS[kind][1]
    assert whole > 5000 and direct > 100


@pytest.mark.parametrize("m,n,k,pieces,want", [
    (384, 5120, 3072, 2, 1),          # 33.8 us in two pieces against 40.5 with the tile of the whole product
    (256, 4608, 3584, 3, 1), (128, 3584, 18944, 4, 2), (192, 2560, 2048, 2, 0),
])
def test_tile_of_a_number_of_pieces_that_is_not_the_plans(core, m, n, k, pieces, want):
    assert core.llmlab_pieces_tile(m, n, k, CUS, pieces) == want


def test_limits_of_the_plan_are_kept(core):
    for max_pieces, min_tiles in ((1, 8), (3, 8), (16, 100), (16, 1)):
        for (m, n, k) in ((40, 3584, 18944), (576, 3584, 18944), (2048, 5120, 27648), (100, 896, 4864)):
            pieces, _ = plan(core, m, n, k, max_pieces, min_tiles)
            assert pieces <= max_pieces
            assert pieces == 1 or ((k + 63) // 64 + pieces - 1) // pieces >= min_tiles


@pytest.mark.parametrize("m,n,k,want", [
    # (measured: see the comments in csrc/gemm.hip)
    (2048, 37888, 3584, (1, 4)),      # gate/up of a 2,048-token step, 7B shape: 256 x 256, two groups of waves
    (2048, 55296, 5120, (1, 4)),
    (576, 3584, 18944, (6, 5)),       # down product of a mixed step: six pieces with the 192 x 256 tile
    (2048, 3584, 18944, (2, 4)),
    (576, 37888, 3584, (1, 5)),       # three tiles of 192 rows
    (2048, 4608, 3584, (1, 5)),
    (576, 1152, 896, (1, 0)),         # a small product: 64 x 64
    (2048, 9728, 896, (1, 5)),        # gate/up of the 0.5B shape
    (2048, 9728, 512, (1, 2)),        # an inner size shorter than any measured: no tile of two groups of waves
    (192, 55296, 5120, (1, 5)),       # one or two tiles of rows of a wide matrix already fill the chip:
    (256, 55296, 5120, (1, 4)),       # the tiles of two groups of waves (153 / 171 us against 187 / 199)
    (384, 27648, 5120, (1, 5)),
    (192, 27648, 5120, (1, 1)),       # ... not where half the units would stay idle
    (192, 4608, 3584, (1, 0)),        # 216 blocks of 64 x 64 are one round (26 us against 29 with 64 x 128),
    (1536, 896, 896, (1, 0)),         # ... and so are 336 by direct loads, three to a unit (with the norm 16.5 against 18.7)
    (2048, 1152, 896, (1, 0)),
    (1400, 2304, 768, (1, 1)),        # 792 are a round and a bit
    (384, 5120, 27648, (4, 2)),       # three tiles of 128 rows in four pieces (150 us against 183 in two of 64 x 128)
    (256, 8192, 8192, (4, 2)),
    (192, 5120, 27648, (4, 1)),       # ... from 256 rows on (a step of 192 requests of the 32B shape loses 5 % with them)
    (272, 5120, 27648, (2, 1)),       # ... and only well-filled tiles
])
def test_measured_decisions(core, m, n, k, want):
    assert plan(core, m, n, k) == want


@pytest.mark.parametrize("m,n,k,columns", [
    # (us with this tile and with the best of the others; blocks of 64 x 64 that find no place any more with three
    # to a unit cost a round, and a block of 128 x 128 more than units as well)
    (700, 5632, 1024, 128),      # 64 x 128: 18.2 us against 23.7 (128 x 128) and 22.6
    (576, 6144, 768, 128),       # 14.1 against 16.6
    (640, 5632, 1024, 128),      # 17.8 against 20.6
    (640, 5216, 1000, 128),      # 17.9 against 21.1
    (384, 9216, 1152, 128),      # 20.4 against 24.1
    (300, 10240, 1280, 128),     # 22.9 against 26.0
    (1400, 2304, 768, 128),      # 15.2 against 19.4
    (1536, 2304, 1792, 128),     # 25.1 against 31.3
    (2048, 1792, 1280, 128),     # 21.1 against 26.0
    (1801, 2048, 1024, 128),     # 18.5 against 22.6
    (2300, 1536, 1536, 128),     # 32.2 against 36.4
    (1400, 3584, 3584, 128),     # 70.4 against 76.3 with the 192 x 256 tile
    (768, 6144, 4096, 128),      # 64.0 against 69.9
    (512, 896, 896, 64), (2048, 896, 896, 64), (2048, 1152, 896, 64), (700, 2048, 2048, 64),
])
def test_tiles_of_few_blocks(core, m, n, k, columns):
    assert core.llmlab_linear_tile(m, n, k, CUS) == columns


@pytest.mark.parametrize("m,n,k,want", [
    (576, 1536, 8960, (4, 1)),       # with the norm 40.9 us against 46.1 (64 x 64 in two pieces)
    (1024, 1792, 7168, (4, 5)),      # 46.4 against 65.9 (64 x 64 whole)
    (300, 3584, 3584, (3, 1)),       # 30.6 against 33.3 (64 x 64 in three)
    (512, 2560, 2560, (3, 1)),       # 26.0 against 30.1 (64 x 64 whole)
    (512, 896, 4864, (4, 0)),        # 17.8 against 24.7 (64 x 128 in six)
    (1100, 4096, 4096, (2, 5)),      # 59.3 against 72.3 (64 x 128 whole)
    (900, 3584, 3584, (3, 5)),       # 44.9 against 53.4 (64 x 128 whole)
    (1400, 4096, 4096, (2, 5)),      # 66.1 against 85.0 (192 x 256 whole)
    (2048, 896, 4864, (2, 1)),
])
def test_pieces_of_few_blocks(core, m, n, k, want):
    assert plan(core, m, n, k) == want
    assert plan(core, m, n, k, 8) == want


def test_one_tile_of_rows_of_a_wide_matrix(core):
    """Up to 128 rows: the tile that the estimates pick, measured inside decode steps of 96 and 128 requests.  (A
    product that is neither cut nor written by heads follows it only where no width makes one round of blocks:
    ``test_one_round_of_blocks``.)"""
    assert core.llmlab_linear_tile(128, 37888, 3584, CUS) == 256      # 128 x 256: 77 us against 84
    assert core.llmlab_linear_tile(96, 55296, 5120, CUS) == 256
    assert core.llmlab_linear_tile(128, 152064, 3584, CUS) == 128     # a vocabulary gains nothing from it
    assert core.llmlab_linear_tile(128, 27648, 5120, CUS) == 128
    assert core.llmlab_linear_tile(64, 37888, 3584, CUS) == 128       # (64 x 128)


@pytest.mark.parametrize("m,n,k,columns", [
    # (measured: see the comment at the rule in csrc/gemm.hip)
    (64, 37888, 3584, 160), (17, 37888, 3584, 160), (64, 22016, 2048, 96), (64, 17920, 1536, 96),
    (64, 27648, 5120, 128), (64, 55296, 5120, 224), (128, 37888, 3584, 160), (128, 17920, 1536, 160),
    # 128 columns from an inner size of 1,152 on, 224 from 3,072 on (below, the estimates' picks are faster)
    (17, 28672, 1152, 128), (17, 28672, 1024, 64), (32, 49152, 3072, 224), (32, 49152, 2048, 128), (17, 24448, 1024, 96),
    # no width makes a round: what the estimates pick
    (128, 55296, 5120, 256), (128, 152064, 3584, 128), (64, 152064, 3584, 128), (64, 4608, 3584, 64),
])
def test_one_round_of_blocks(core, m, n, k, columns):
    """The tile of gate and up, of logits and of other whole products of up to 128 rows."""
    assert core.llmlab_plain_tile(m, n, k, CUS) == columns


def test_one_round_of_blocks_is_one_round(core):
    """Over sizes drawn at random: where the tile is not the one that the estimates pick (or the direct one in its place), its blocks
    find a compute unit each and leave few without one; beyond 128 rows and at short inner sizes it is the estimates' always."""
    rng = random.Random(7)
    differs = 0
    for _ in range(5000):
        m = rng.choice([rng.randint(17, 64), rng.randint(65, 128), rng.randint(129, 3000)])
        n, k = rng.randint(64, 70000), 8 * rng.randint(16, 1500)
        cus = rng.choice([CUS, 304, 64])
        columns, estimates = core.llmlab_plain_tile(m, n, k, cus), launched_width(core, m, n, k, cus)
        if m > 128 or k < 1024:
            assert columns == estimates, (m, n, k)
        if columns == estimates:
            continue
        differs += 1
        assert columns in ((96, 128, 160, 224) if m <= 64 else (160,)), (m, n, k)
        rounds = [(n + columns - 1) // columns * tiles / cus for tiles in ((1,) if m <= 64 else (1, 2))]
        assert any((0.7 if columns == 96 else 0.8) <= r <= 1.0 for r in rounds), (m, n, k, columns)
    assert differs > 300


@pytest.mark.parametrize("m", [1, 65, 200, 600, 2048])
@pytest.mark.parametrize("k", [2 ** 22 + 8, 34_087_048, 40_000_000])
def test_inner_sizes_beyond_the_addresses_of_direct_loads(core, m, k):
    """The 64 x 64 tile and the two of two groups of waves address a tile's rows by 32 bits of bytes (63 rows of
    34,087,042 numbers wrap): beyond their limit nothing is given to them, whether estimated, cut or named."""
    direct = (0, 4, 5)
    for n in (7, 16, 896):
        assert core.llmlab_linear_tile(m, n, k, CUS) in (128,) and core.llmlab_plain_tile(m, n, k, CUS) in (128,)
        assert core.llmlab_linear_heads_tile(m, n, k, 64, CUS) == 128
        assert plan(core, m, n, k)[1] not in direct and plan(core, m, n, k, 1)[1] not in direct
        for tile in (64, 132, 133):
            core.llmlab_debug_gemm_tile(tile)
            try:
                assert core.llmlab_linear_tile(m, n, k, CUS) == 128 and plan(core, m, n, k)[1] not in direct
                assert core.llmlab_linear_tile(m, n, 2 ** 22, CUS) == (64 if tile == 64 else 256)
            finally:
                core.llmlab_debug_gemm_tile(0)


def test_block_shapes_of_products_of_few_rows(core):
    rng = random.Random(6)
    out = (ctypes.c_int * 5)()
    for _ in range(2000):
        epilogue = rng.choice([0, 1, 2, 3, 5])
        m = rng.randint(1, 64)
        n = 16 * rng.randint(1, 9500)
        if epilogue == 3:
            n = 32 * rng.randint(1, 3000)
        k = 8 * rng.randint(1, 3500)
        ksplit = rng.randint(2, 8) if epilogue == 5 else 1
        core.llmlab_skinny_shape(epilogue, int(epilogue in (2, 3) and rng.random() < 0.5), m, n, k, 0, CUS, ksplit, out)
        nsb, kw, stage, qsplit, mb = list(out)
        if nsb == 0:
            continue                                        # no shape fits: the caller takes another kernel
        assert nsb in (1, 2, 4, 8, 16) and kw >= 1 and nsb * kw <= 16, (epilogue, m, n, k, list(out))
        assert mb in (1, 2, 4) and 16 * mb <= max(16, 2 * m), (m, mb)
        assert stage in (0, 1) and qsplit == 1


@pytest.mark.parametrize("m,n,k,want", [
    (16, 17920, 1536, (8, 1, 1, 1, 1)),      # 16.6 us; 2 strips x 2 slices 21.7
    (5, 37888, 3584, (2, 4, 1, 1, 1)),       # 52; 2 x 2 57
    (10, 37888, 3584, (16, 1, 1, 1, 1)),     # 55; 4 x 2 59
])
def test_measured_block_shapes_of_gate_and_up(core, m, n, k, want):
    """Behind a norm, weights from memory."""
    out = (ctypes.c_int * 5)()
    core.llmlab_skinny_shape(3, 1, m, n, k, 0, CUS, 1, out)
    assert tuple(out) == want


def test_when_a_decode_graph_pays():
    """``graph="auto"``: the rule on measured cases.  At the 0.5B shape (151 calls a step, 1 GB
    of weights) the host cannot keep up and the graph is taken, also with 3.2 GB of cache
    behind 64 requests; at the 7B and 32B shapes the step streams for longer than the host
    needs and is launched call by call; a small model behind a very long context is no
    longer misjudged by its weights alone."""
    from llm_inference_lab_amd.kernels.debug import DispatchRules
    rules = DispatchRules()
    assert rules.graph_pays(151, 0.988e9, 0.4e9)
    assert rules.graph_pays(151, 0.988e9, 3.2e9)
    assert not rules.graph_pays(171, 14.1e9, 1.9e9)
    assert not rules.graph_pays(387, 64.0e9, 17e9)
    assert rules.graph_pays(151, 0.988e9, 0.0) and not rules.graph_pays(151, 0.988e9, 12e9)


def test_the_engine_counts_a_decode_step_and_decides_step_by_step():
    """Over the kernel references on the CPU: the first decode step of ``graph="auto"`` runs
    eagerly and its calls are counted; what the rules are asked is the number of calls, the
    weights of one step and the cache that the step's requests hold at that moment, at
    every decode step anew.  (The rules here always say no: a CPU has no graphs.)"""
    import helpers as H
    import llm_inference_lab_amd as lab
    from emu_ops import EmuOps
    from llm_inference_lab_amd.kernels.debug import DispatchRules

    class Asked(DispatchRules):
        def __init__(self):
            super().__init__()
            self.questions = []

        def graph_pays(self, calls, weight_bytes, cache_bytes):
            self.questions.append((calls, weight_bytes, cache_bytes))
            return False

    ops = EmuOps()
    ops.rules = Asked()
    engine = H.make_engine("B", 1, "f32", ops=ops, device="cpu", graph="auto", num_pages=24)
    cfg = H.config_of("B")
    a, b = engine.open("a"), engine.open("b")
    engine.step([lab.StepEntry(a, H.random_ids(cfg, 30, 1), [29]), lab.StepEntry(b, H.random_ids(cfg, 7, 2), [6])])
    assert engine.step_fn.decode_calls is None and ops.rules.questions == []      # a prefill step decides nothing
    before = ops.calls_made
    engine.step([lab.StepEntry(a, [1], [0]), lab.StepEntry(b, [2], [0])])
    calls = ops.calls_made - before
    assert engine.step_fn.decode_calls == calls > 0 and engine.step_fn.use_graph is False
    engine.step([lab.StepEntry(a, [3], [0]), lab.StepEntry(b, [4], [0])])
    engine.step([lab.StepEntry(a, [5], [0])])
    assert [q[0] for q in ops.rules.questions] == [calls] * 3
    assert all(q[1] == engine.model.weight_bytes_per_step() for q in ops.rules.questions)
    # config B: one layer sees everything, two see the last 24 positions; 1 kv head of 32, float32
    per_token = 2 * 32 * 4
    seen = lambda n: per_token * (n + 2 * min(n, 24))
    assert [q[2] for q in ops.rules.questions] == [seen(31) + seen(8), seen(32) + seen(9), seen(33)]


# ----------------------------------------------------------------- attention
def attention_library(head_dim):
    if shutil.which("hipcc") is None and not build.hipcc_path():
        pytest.skip("no hipcc to build the library with")
    try:
        lib = ctypes.CDLL(build.attention_library(head_dim))
    except (OSError, RuntimeError) as err:
        pytest.skip(f"the attention library does not load here: {err}")
    lib.llmlab_attention_launch.restype = ctypes.c_int
    return lib


BF16, F32 = 1, 0        # (the dtype codes of the libraries)


@pytest.mark.parametrize("head_dim,nq,nkv", [(64, 14, 2), (96, 28, 4), (128, 28, 4), (256, 8, 8)])
def test_attention_launch_is_one_the_head_size_has(head_dim, nq, nkv):
    """Over steps drawn at random: a decode step is told apart, the launches with two groups of
    waves and with 32 rows a wave only where the head size has them, pairs of tiles only at the
    start of prompts without a window, keys staged in LDS at heads of 64 and 128 only."""
    lib = attention_library(head_dim)
    rng = random.Random(head_dim)
    group = nq // nkv
    for _ in range(3000):
        reqs = rng.choice([1, 2, 4, 8, 16, 64])
        q = rng.choice([1, 2, 3, rng.randint(4, 64), rng.randint(65, 4096)])
        ctx = q + rng.choice([0, rng.randint(0, 300), rng.randint(0, 9000)])
        window = rng.choice([0, 0, 0, 128, 4096])
        for dtype in (BF16, F32):
            path = lib.llmlab_attention_launch(dtype, nq, nkv, reqs, q, ctx, window, CUS)
            if q * group <= 16:
                assert path == 0, (q, path)
                continue
            if dtype == F32:
                assert path in (1, 2), (reqs, q, ctx, path)
                continue
            assert path in {64: (1, 7, 8, 9, 10), 96: (1, 2, 3, 4, 6), 256: (1, 3, 4)}.get(head_dim, (1, 8, 10, 11)), (reqs, q, ctx, path)
            if path == 3:
                assert window == 0 and 16 * (ctx - q) <= q
            if path == 1:
                assert -(-q * group // 64) * nkv * reqs <= CUS // 2       # few tiles of rows only


@pytest.mark.parametrize("head_dim,nq,nkv,dtype,reqs,q,behind,want", [
    # (measured: see the comments in csrc/attention.hip; 1 = a block's waves split the keys of a tile of
    # rows, 2 = 32 rows a wave, 4 = 16 rows a wave, 6 = 4 with two groups of waves a block; keys staged in LDS: 7, 8, 9, 10, 11 =
    # tiles of 32 rows by groups of waves 1 x 4, 2 x 4, 4 x 2, 4 x 1, 2 x 2)
    (64, 14, 2, BF16, 1, 48, 1500, 1),       # few rows behind a history: 14.5 us and 14.8
    (64, 14, 2, BF16, 1, 48, 4000, 1),       # 24.0 against 27.4
    (64, 14, 2, BF16, 1, 48, 500, 7),        # 9.7 against 10.4
    (64, 14, 2, BF16, 1, 48, 1024, 1), (64, 14, 2, BF16, 1, 48, 1023, 7),
    (64, 14, 2, BF16, 1, 1024, 0, 7),        # a prompt from its start, 224 tiles of 64 rows: 12.9 us against 13.3 and 18.1
    (64, 14, 2, BF16, 1, 1025, 0, 8),
    (64, 14, 2, BF16, 1, 1536, 0, 8),        # 18.3 against 19.6 and 23.7
    (64, 14, 2, BF16, 64, 24, 0, 10),        # many short prompts: 7.0 against 12.9 and 10.5
    (64, 8, 4, BF16, 64, 93, 0, 10),         # 7.9 against 13.6 with 2 x 4
    (64, 16, 4, BF16, 8, 318, 0, 10),        # 10.3 against 14.4
    (64, 1, 1, BF16, 64, 229, 0, 8),         # a block a unit: 7.4 against 9.6 with 4 x 1
    (64, 28, 4, BF16, 1, 1210, 36, 8),       # 17.8 against 23.6 with 4 x 1
    (64, 16, 2, BF16, 32, 512, 0, 10),       # 31 against 42 with 4 x 2
    (64, 1, 1, BF16, 224, 64, 1, 7), (64, 1, 1, BF16, 225, 64, 1, 8), (64, 1, 1, BF16, 64, 64, 0, 10),
    (64, 1, 1, BF16, 257, 64, 128, 10), (64, 1, 1, BF16, 257, 64, 129, 8), (64, 1, 1, BF16, 256, 64, 128, 8),
    (64, 1, 1, BF16, 513, 64, 480, 10), (64, 1, 1, BF16, 513, 64, 481, 8), (64, 1, 1, BF16, 512, 64, 480, 8),
    (64, 1, 1, BF16, 768, 64, 481, 8), (64, 1, 1, BF16, 769, 64, 481, 9), (64, 1, 1, BF16, 1024, 64, 481, 9),
    (64, 1, 1, BF16, 1025, 64, 481, 10), (64, 1, 1, BF16, 1025, 64, 1504, 10), (64, 1, 1, BF16, 1025, 64, 1505, 9),
    (64, 1, 1, BF16, 2048, 64, 1505, 9), (64, 1, 1, BF16, 2049, 64, 1505, 10),
    (64, 14, 2, BF16, 1, 8192, 0, 9),        # a long prompt: 148 us against 153 with 4 x 1 and 160 with 2 x 4
    (128, 28, 4, BF16, 1, 4, 1500, 8),       # 21 us against 27 with the key split
    (128, 28, 4, BF16, 1, 96, 4000, 8),      # 43 against 47
    (128, 28, 4, BF16, 1, 128, 2560, 8),
    (128, 28, 4, BF16, 1, 464, 3000, 8),     # 42.5 against 51 and 81
    (128, 28, 4, BF16, 1, 768, 0, 11),       # 20 against 24 and 25
    (128, 28, 4, BF16, 1, 3072, 0, 10),      # 90 against 126 and 98
    (128, 8, 1, BF16, 32, 7, 5500, 1),       # keys of many requests from memory: 64 us against 78 with 2 x 4
    (128, 1, 1, BF16, 16, 35, 7284, 1),      # 80 against 98
    (128, 4, 4, BF16, 8, 49, 1891, 1),       # 28.0 against 32.9
    (128, 4, 1, BF16, 16, 116, 5873, 8),     # 70.0 against 71.4: more tiles than half the units
    (128, 1, 1, BF16, 32, 32, 1568, 1), (128, 1, 1, BF16, 32, 32, 1567, 8), (128, 1, 1, BF16, 128, 32, 1568, 1),
    (128, 1, 1, BF16, 129, 32, 1568, 8),
    (128, 4, 2, BF16, 64, 186, 0, 10),       # 13.6 against 18.6 with 2 x 2
    (128, 1, 1, BF16, 512, 64, 192, 10), (128, 1, 1, BF16, 512, 64, 193, 11), (128, 1, 1, BF16, 511, 64, 192, 11),
    (128, 1, 1, BF16, 256, 64, 353, 8), (128, 1, 1, BF16, 256, 64, 352, 11), (128, 1, 1, BF16, 257, 64, 353, 11),
    (128, 1, 1, BF16, 1024, 64, 193, 11), (128, 1, 1, BF16, 1025, 64, 193, 10),
    (128, 1, 1, BF16, 8, 32, 0, 10), (128, 1, 1, BF16, 8, 32, 1, 11),
    (128, 28, 4, BF16, 64, 24, 0, 10),       # 12 against 29 and 18
    (96, 28, 4, BF16, 1, 128, 1024, 6),      # (heads beside them: as those were measured without staged keys)
    (96, 28, 4, BF16, 1, 128, 2560, 1), (96, 28, 4, BF16, 8, 128, 0, 2), (96, 28, 4, BF16, 1, 64, 0, 4),
    (48, 14, 2, BF16, 1, 512, 1536, 1), (48, 14, 2, BF16, 1, 2048, 0, 6), (48, 14, 2, BF16, 1, 8192, 0, 2), (48, 14, 2, BF16, 16, 64, 0, 4),
    (64, 14, 2, F32, 1, 512, 1024, 1),       # 31 us against 120
    (64, 14, 2, F32, 1, 1531, 0, 1),         # 49 against 122
    (64, 14, 2, F32, 16, 512, 0, 2),         # (3,584 blocks of 32 rows)
    (64, 8, 4, F32, 64, 121, 0, 2),          # 26.4 against 33.6 with the key split
    (64, 16, 4, F32, 64, 629, 0, 2),         # 594 against 613
    (64, 56, 8, F32, 8, 505, 0, 2), (64, 56, 8, F32, 8, 513, 0, 1),
    (64, 8, 4, F32, 64, 134, 0, 1),          # 35.5 against 41.9: a last block of 12 rows
    (32, 32, 8, F32, 16, 123, 0, 2),         # 16.6 against 22.6
    (32, 64, 8, F32, 64, 464, 65, 2),        # 754 against 1,002
    (32, 4, 2, F32, 64, 749, 0, 1),          # 127 against 152
    (32, 14, 2, F32, 64, 571, 0, 1),         # 263 against 355
    # (borders, tiles of 32 rows by fours)
    (64, 4, 1, F32, 112, 32, 16, 2), (64, 4, 1, F32, 111, 32, 16, 1), (64, 4, 1, F32, 112, 32, 17, 1),
    (64, 4, 1, F32, 224, 32, 96, 2), (64, 4, 1, F32, 223, 32, 96, 1), (64, 4, 1, F32, 224, 32, 97, 1),
    (64, 4, 1, F32, 448, 32, 160, 2), (64, 4, 1, F32, 447, 32, 160, 1), (64, 4, 1, F32, 448, 32, 161, 1),
    (64, 4, 1, F32, 896, 32, 480, 2), (64, 4, 1, F32, 895, 32, 480, 1), (64, 4, 1, F32, 896, 32, 481, 1),
    (64, 4, 1, F32, 3584, 32, 992, 2), (64, 4, 1, F32, 3583, 32, 992, 1), (64, 4, 1, F32, 3584, 32, 993, 1),
    (64, 3, 1, F32, 600, 32, 160, 2), (64, 3, 1, F32, 600, 31, 161, 1), (64, 3, 1, F32, 600, 31, 97, 2),
    (32, 4, 1, F32, 112, 32, 32, 2), (32, 4, 1, F32, 112, 32, 33, 1), (32, 4, 1, F32, 224, 32, 160, 2), (32, 4, 1, F32, 224, 32, 161, 1),
    (32, 4, 1, F32, 448, 32, 224, 2), (32, 4, 1, F32, 448, 32, 225, 1), (32, 4, 1, F32, 6400, 32, 992, 2), (32, 4, 1, F32, 6400, 32, 993, 1),
    (32, 4, 1, F32, 6399, 32, 481, 1),
    (128, 28, 4, F32, 4, 256, 0, 2),         # 58 against 81
    (128, 28, 4, F32, 1, 256, 1024, 1),      # 77 against 226
    (128, 28, 4, F32, 1, 1024, 0, 1),        # a long portion's tiles are uneven: 148 against 184
    (128, 28, 4, F32, 2, 1024, 1024, 1),     # 620 against 656
    (128, 28, 4, F32, 4, 1024, 0, 2),        # 501 against 562
])
def test_measured_attention_launches(head_dim, nq, nkv, dtype, reqs, q, behind, want):
    lib = attention_library(head_dim)
    assert lib.llmlab_attention_launch(dtype, nq, nkv, reqs, q, behind + q, 0, CUS) == want


@pytest.mark.parametrize("head_dim,nq,nkv,reqs,q,behind,window,want", [
    # (a window bounds what a tile walks, and what all requests read)
    (64, 14, 2, 2, 1521, 0, 33, 10),         # 9.1 us against 14.0 with 2 x 4
    (64, 8, 8, 25, 45, 5578, 0, 8), (64, 8, 8, 20, 45, 5578, 0, 7),       # 200 and 160 tiles of 64 rows: 78 us by 1 x 4 for the first, 62.5 (beside 5 decoding)
    (64, 8, 8, 25, 45, 447, 0, 8), (64, 8, 8, 25, 45, 446, 0, 7), (64, 8, 8, 25, 45, 600, 447, 8), (64, 8, 8, 25, 45, 600, 446, 7),      # 24 MB
    (64, 16, 8, 8, 298, 0, 32, 10),          # 7.9 against 11.9
    (64, 1, 1, 513, 64, 4000, 512, 10), (64, 1, 1, 513, 64, 4000, 513, 8),
    (128, 8, 2, 1, 80, 6665, 50, 11),        # 7.7 against 9.5
    (128, 1, 1, 16, 35, 7284, 1000, 8),
    (128, 16, 4, 2, 1827, 0, 49, 10),        # 15.7 against 21.2 with 2 x 2
])
def test_launches_in_a_window(head_dim, nq, nkv, reqs, q, behind, window, want):
    lib = attention_library(head_dim)
    assert lib.llmlab_attention_launch(BF16, nq, nkv, reqs, q, behind + q, window, CUS) == want


@pytest.mark.parametrize("head_dim,nq,nkv,reqs,q,behind,window,want", [
    # (us by 16 rows in the order of the tiles / by 16 rows request by request / by 32 rows request by request; 1 and 2 are 16 rows by
    # four and eight waves, 3 the tile of 32, 16 more the order of the tiles)
    (64, 14, 2, 1, 1531, 0, 0, 17),
    (64, 16, 8, 1, 867, 0, 0, 17),              # 28.5 / 38.4 / --
    (64, 14, 2, 8, 1786, 4794, 0, 3),           # 1,733 / 850 / 887 (portions of up to so many)
    (64, 14, 2, 21, 444, 4141, 0, 3),           # 2,446 / 1,308 / 1,365
    (64, 16, 8, 22, 61, 5007, 0, 3),            # 531 with 16 rows, 380 with 32: 457 MB of keys and values
    (16, 8, 2, 5, 160, 5847, 0, 3),             # 60 / 59 / 43: 200 tiles of 32 rows
    (64, 8, 8, 1, 100, 3000, 0, 18), (64, 8, 8, 1, 100, 667, 0, 17), (64, 8, 8, 1, 100, 668, 0, 18),     # 768 keys in all
    (64, 8, 8, 4, 129, 767, 0, 17), (64, 8, 8, 4, 129, 768, 0, 3),      # 768 keys of history
    (64, 8, 8, 4, 128, 5000, 0, 18),                                    # (half a tile of 32 rows a unit)
    (64, 8, 8, 1, 1056, 768, 0, 3), (64, 8, 8, 1, 1088, 768, 0, 17),    # 264 and 272 tiles: a round of the units and a bit
    (64, 8, 8, 1, 1536, 768, 0, 17), (64, 8, 8, 1, 1537, 768, 0, 3),    # 384 and 392: one and a half
    (64, 8, 8, 1, 1537, 768, 767, 17), (64, 8, 8, 1, 1537, 768, 768, 3),
    (64, 8, 8, 16, 256, 0, 0, 17), (64, 8, 8, 16, 257, 0, 0, 1),        # 2,048 and 2,176 tiles of 16 rows
    (32, 8, 2, 32, 513, 0, 0, 1), (32, 8, 2, 32, 500, 0, 0, 17),        # 8 MB of keys and values
    (16, 8, 2, 16, 1025, 0, 0, 1), (16, 8, 2, 16, 1024, 0, 0, 17),      # 512 keys that a tile walks
    (64, 8, 8, 32, 1023, 0, 0, 1), (64, 8, 8, 32, 1024, 0, 0, 3),       # 128 MB
    (128, 28, 4, 1, 1500, 0, 0, 3), (256, 8, 8, 4, 100, 0, 0, 3),
])
def test_blocks_of_float32(head_dim, nq, nkv, reqs, q, behind, window, want):
    lib = attention_library(head_dim)
    assert lib.llmlab_attention_f32_blocks(nq, nkv, reqs, q, behind + q, window, CUS) == want


@pytest.mark.parametrize("head_dim,blocks,keys,want", [
    (64, 256, 71, 0), (64, 257, 71, 1),              # 34 requests of 8 heads over 8 at 95 9.5 us alone, 8.9 dense
    (64, 257, 256, 1), (64, 257, 257, 0), (64, 384, 257, 0), (64, 385, 257, 1),
    (64, 2040, 1024, 1), (64, 2040, 1025, 0),
    (32, 512, 65, 0), (32, 513, 65, 1), (32, 513, 1025, 0),
    (16, 4096, 65, 0), (48, 4096, 65, 0), (128, 4096, 65, 0),
])
def test_dense_decode_blocks_of_float32(head_dim, blocks, keys, want):
    assert attention_library(head_dim).llmlab_attention_f32_dense(blocks, keys, CUS) == want


@pytest.mark.parametrize("head_dim,nq,nkv,portion,behind,decoding,their_keys,want", [
    # (us in two launches / in one with the portion by tiles of 32 rows / in one by tiles of 16; the rules are in
    # csrc/attention.hip.  2: two launches, 1: one by tiles of 32 rows, 3: one by tiles of 16)
    (64, 14, 2, 128, 2048, 63, 2048, 1),     # 30.9 / 19.1 / 15.3
    (64, 14, 2, 256, 1024, 31, 1024, 1),     # 20.0 / 12.7 / 13.2
    (64, 14, 2, 512, 1536, 31, 1024, 3),     # 23.4 / 16.5 / 18.6
    (64, 14, 2, 512, 1536, 127, 1024, 3),    # 31.6 / 27.3 / 25.7
    (64, 14, 2, 512, 1536, 63, 512, 3),      # 21.0 / 19.3 / 19.4
    (64, 14, 2, 464, 1100, 48, 1400, 3),     # 24.9 / 21.0 / 16.4
    (64, 14, 2, 64, 0, 48, 300, 3),          # 11.6 / -- / 6.8
    (64, 14, 2, 1024, 1100, 48, 1400, 3),    # 28.6 / -- / 30.4: 896 blocks, three and a half a unit (from its start 17.2 / 17.7)
    (64, 14, 2, 1025, 1100, 48, 1400, 2),    # 29.1 / -- / 30.1
    (64, 14, 2, 512, 2560, 48, 1400, 3),     # 30.7 / 27.7 / 25.7: 3,072 keys
    (64, 14, 2, 512, 2600, 48, 1400, 1),     # 31.6 / 27.8 / 28.3
    (128, 28, 4, 128, 2048, 63, 2048, 1),    # 72.0 / 51.7 / 45.2
    (128, 40, 8, 128, 2048, 127, 1024, 3),   # 130 / 119 / 116
    (128, 28, 4, 512, 512, 63, 2048, 2),     # 62.2 / -- / 69.3
    (128, 28, 4, 146, 0, 48, 1400, 3),       # 36.0 / -- / 25.5: 256 blocks, one a unit
    (128, 28, 4, 147, 0, 48, 1400, 2),       # 35.7 / -- / 25.4
    (128, 28, 4, 900, 1100, 48, 1400, 2),    # 59 / -- / 85
    (256, 8, 8, 64, 0, 8, 300, 2),           # (no small tiles at such heads)
])
def test_measured_launches_of_a_mixed_step(head_dim, nq, nkv, portion, behind, decoding, their_keys, want):
    lib = attention_library(head_dim)
    lib.llmlab_attention_mixed_launches.restype = ctypes.c_int
    got = lib.llmlab_attention_mixed_launches(nq, nkv, decoding + 1, decoding, portion, behind + portion,
                                              their_keys, 0, CUS)
    assert got == want
    lib.llmlab_debug_attention_two_launches(-2)                  # (as the switch forces it; heads up to 128)
    try:
        assert lib.llmlab_attention_mixed_launches(nq, nkv, decoding + 1, decoding, portion, behind + portion,
                                                   their_keys, 0, CUS) == (3 if head_dim <= 128 else want)
    finally:
        lib.llmlab_debug_attention_two_launches(0)
    # not a mixed step: nobody decodes, or everybody
    assert lib.llmlab_attention_mixed_launches(nq, nkv, 4, 0, portion, behind + portion, 0, 0, CUS) == 0
    assert lib.llmlab_attention_mixed_launches(nq, nkv, 4, 4, portion, behind + portion, their_keys, 0, CUS) == 0


@pytest.mark.parametrize("head_dim,nkv,reqs,beside,keys,want", [
    # (a block reads keys times 4 times the head size bytes; us unsplit / split in csrc/attention.hip)
    (64, 2, 20, 0, 1400, 6),                 # 12.0 / 9.7
    (64, 2, 20, 0, 1280, 6), (64, 2, 20, 0, 1279, 1),         # 320 KB where three splits and more are to be had
    (64, 2, 42, 0, 1280, 3), (64, 2, 42, 0, 1279, 1),
    (64, 2, 43, 0, 1536, 2), (64, 2, 43, 0, 1535, 1),         # 384 KB with two, at heads up to 64
    (64, 2, 64, 0, 1700, 2),                 # 17.1 / 16.2
    (64, 2, 65, 0, 4096, 1),                 # (more blocks than half the units)
    (128, 2, 40, 0, 1400, 3),                # 22.5 / 18.2
    (128, 2, 43, 0, 1200, 2), (128, 2, 43, 0, 1199, 1),       # 600 KB with two at heads above, up to three eighths of the units
    (128, 2, 48, 0, 1200, 2), (128, 2, 49, 0, 1535, 1), (128, 2, 49, 0, 1536, 2),      # 768 KB beyond
    (128, 2, 56, 0, 1400, 1),                # 24.1 / 27
    (256, 2, 40, 0, 320, 3), (256, 2, 40, 0, 319, 1), (32, 2, 20, 0, 2560, 6), (32, 2, 20, 0, 2559, 1),
    # beside portions: 384 KB from five splits on, 768 below
    (64, 2, 20, 1, 1536, 6), (64, 2, 20, 1, 1535, 1), (64, 2, 48, 1, 1500, 1), (64, 2, 32, 1, 2000, 1),
    (64, 2, 32, 1, 3071, 1), (64, 2, 32, 1, 3072, 4), (128, 2, 43, 1, 1535, 1), (128, 2, 43, 1, 1536, 2),
])
def test_key_splits_of_decoding_requests(head_dim, nkv, reqs, beside, keys, want):
    lib = attention_library(head_dim)
    assert lib.llmlab_attention_decode_splits(7 * nkv, nkv, reqs + beside, reqs, keys, 0, CUS) == want


def first_float32_sum(m, n, k, max_pieces, min_steps):
    """Steps of a sum by the estimate of the kernels that add all part products in one sum (64 x 64 and 128 x 128)."""
    steps, best = -(-k // 32), None
    for tile in (64, 128):
        for pieces in range(1, max_pieces + 1):
            s = -(-steps // pieces)
            if pieces > 1 and s < min_steps:
                break
            share = -(-m // tile) * -(-n // tile) * pieces / CUS
            whole = math.ceil(share - 1e-9)
            if tile == 128:
                t = whole * (5.4 + s * (1.31 + 0.12 * min(share, 1.0)))
            else:
                t, shared = 2.0 + 0.863 * s, (whole if share <= 3 else share) * (1.0 + 0.58 * s)
                t = shared if shared > t and whole > 1 else t
            t += pieces * (m * n * 2.2e-6 + 0.3) if pieces > 1 else 0.0
            if best is None or t < best[0]:
                best = (t, s)
    return best[1]


def test_float32_sums_are_no_longer_than_their_tile_allows(core):
    """A product that may be cut: the 128 x 256 tile, which adds everything in one sum, adds no more steps than the first
    kernels did (nor than 64, where more pieces are to be had), the others three times as many at most."""
    core.llmlab_linear_plan_f32.restype = None
    out, rng, kinds = (ctypes.c_int * 2)(), random.Random(9), set()
    shapes = [(896, 4864), (896, 896), (1536, 1536), (2048, 2048), (1536, 8960), (1024, 4096)]
    for i in range(6000):
        n, k = rng.choice(shapes) if i % 2 else (16 * rng.randint(20, 400), 16 * rng.randint(8, 800))
        m = rng.choice([rng.randint(65, 1024), rng.randint(1025, 9000)])
        max_pieces, min_steps = rng.choice([(8, 8), (8, 8), (1, 1), (8, 40), (3, 8)])
        core.llmlab_linear_plan_f32(m, n, k, CUS, max_pieces, min_steps, out)
        pieces, kind = out
        steps = -(-k // 32)
        s = -(-steps // pieces)
        assert 1 <= pieces <= max_pieces and kind in (0, 2, 3) and (pieces == 1 or s >= min_steps), (m, n, k, pieces, kind)
        first = first_float32_sum(m, n, k, max_pieces, min_steps)
        assert s <= (first if kind == 3 else 3 * first), (m, n, k, max_pieces, min_steps, pieces, kind, first)
        if kind == 3 and pieces < max_pieces and -(-steps // (pieces + 1)) >= min_steps:
            assert s <= 64, (m, n, k, pieces)
        kinds.add((kind, pieces > 1))
    assert len(kinds) == 6


@pytest.mark.parametrize("tile,kind", [(64, 0), (128, 2), (131, 3)])
def test_a_forced_float32_tile_is_planned_at_any_size(core, tile, kind):
    core.llmlab_linear_plan_f32.restype = None
    out, rng = (ctypes.c_int * 2)(), random.Random(10)
    core.llmlab_debug_gemm_tile(tile)
    try:
        for _ in range(2000):
            m, n, k = rng.randint(65, 9000), rng.randint(1, 6000), rng.randint(1, 20000)
            core.llmlab_linear_plan_f32(m, n, k, CUS, rng.randint(1, 8), rng.choice([1, 8, 40, 500]), out)
            assert out[1] == kind and 1 <= out[0] <= 8, (m, n, k, out[0], out[1])
    finally:
        core.llmlab_debug_gemm_tile(0)


@pytest.mark.parametrize("dim,values,rows,heads,kv_heads,keys,want", [
    # (us with one group of waves a block / with two: csrc/windowed_attention.hip)
    (64, 64, 20, 14, 2, 20, 0),              # 5.15 / 5.61
    (64, 64, 384, 14, 2, 24, 0),             # 6.92 / 7.41
    (64, 64, 512, 14, 2, 512, 1),            # 18.8 / 14.5
    (64, 64, 1900, 14, 2, 1032, 1),          # 41.6 / 35.0
    (64, 64, 4096, 14, 2, 4096, 0),          # 58.7 / 64.6
    (64, 64, 4144, 8, 1, 72, 0),             # 10.85 / 12.89
    (64, 64, 1024, 14, 2, 32, 0), (64, 64, 1024, 14, 2, 33, 1), (64, 64, 1025, 14, 2, 128, 0), (64, 64, 1025, 14, 2, 129, 1),
    (64, 64, 2560, 14, 2, 2560, 1), (64, 64, 2561, 14, 2, 2561, 0), (64, 64, 20, 14, 2, 0, 1),
    (128, 64, 120, 8, 2, 30, 0),             # 6.96 / 7.90
    (128, 128, 1000, 16, 2, 1000, 1),        # 40.5 / 30.1
    (128, 128, 1900, 16, 2, 1032, 0),        # 51.2 / 60.1
    (96, 96, 164, 28, 4, 72, 1),              # 9.51 / 8.66
    (128, 128, 96, 16, 2, 72, 1), (128, 128, 96, 16, 2, 71, 0), (128, 128, 95, 16, 2, 72, 0),
])
def test_groups_of_waves_of_windowed_attention(dim, values, rows, heads, kv_heads, keys, want):
    try:
        lib = ctypes.CDLL(build.mixer_library("windowed_attention"))
    except (OSError, RuntimeError) as err:
        pytest.skip(f"the library does not load here: {err}")
    assert lib.llmlab_windowed_two_groups(dim, values, rows, heads, kv_heads, keys, CUS) == want
