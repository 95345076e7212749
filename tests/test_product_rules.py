"""Which kernel serves a product of many rows: the rule of csrc/gemm_tile.hip on both sides of its lines, without a GPU."""

from types import SimpleNamespace

import pytest

from clockwork_amd import ops

CUS = 256


def _choice(mode, M, N, K):
    code = ops._load("gemm_tile").cw_gemm_bf16_mid_choice(mode, M, N, K, K, CUS)
    return (code & 1023, code >> 10 & 1023, code >> 20) if code else None


# (mode, rows, N, K) where the library's product was measured to be the faster one
@pytest.mark.parametrize("mode,M,N,K", [
    # narrow outputs with a long K: a few workgroups walk the whole of it
    (0, 128, 64, 16384), (0, 144, 16, 1536), (0, 1000, 64, 1536), (0, 256, 128, 4096), (0, 144, 512, 896), (0, 700, 256, 1536),
    # tiles enough for the library
    (0, 700, 4096, 896), (0, 1500, 2048, 896), (0, 1500, 4096, 512), (0, 1000, 4096, 256), (0, 144, 2048, 1536),
    # sums for a norm: large outputs, small tiles beyond 1024 rows, whole sums of a long K, rounds that stay empty
    (3, 2048, 5120, 27648), (3, 640, 8192, 29568), (3, 2048, 8192, 29568), (3, 1434, 2048, 11008), (3, 1356, 2048, 11008), (3, 1600, 3584, 18944),
    (3, 152, 7376, 2304),
    # gated products of a narrow output
    (2, 165, 896, 4864), (2, 250, 368, 9600), (2, 92, 1280, 3072), (2, 670, 9728, 896)])
def test_products_that_stay_with_the_library(mode, M, N, K):
    assert _choice(mode, M, N, K) is None


@pytest.mark.parametrize("mode,M,N,K,wide", [
    (0, 144, 1152, 896, False), (0, 400, 2048, 1536, False), (0, 256, 64, 512, False), (0, 1000, 1152, 512, False),
    (3, 160, 1536, 8960, False), (3, 2048, 1536, 8960, True), (3, 1024, 1536, 8960, True), (3, 2048, 3584, 18944, True), (3, 256, 8192, 29568, False),
    (3, 1536, 5120, 27648, True), (3, 160, 1536, 1536, False), (3, 1000, 896, 896, False), (3, 700, 2048, 11008, True), (3, 1600, 2048, 11008, True), (3, 1000, 2048, 6144, False), (3, 2048, 256, 1024, False),
    (2, 160, 17920, 1536, False), (2, 400, 9728, 896, False), (2, 257, 8192, 2048, False)])
def test_products_on_the_tiles_between(mode, M, N, K, wide):
    bm, bn, planes = _choice(mode, M, N, K)
    assert (bm == 256) == wide and (planes == 1 or mode == 3)


def _wide_choice(mode, M, N, K, ldx=None):
    code = ops._load("gemm_tile").cw_gemm_bf16_wide_choice(mode, M, N, K, ldx or K, CUS)
    return (code & 1023, code >> 10 & 1023, code >> 20) if code else None


@pytest.mark.parametrize("mode,M,N,K,there", [
    # few columns of a long K, few outputs; both sides of each line
    (0, 144, 512, 896, False), (0, 144, 896, 896, True), (0, 300, 2048, 1536, True), (0, 200, 2048, 1536, False), (0, 1000, 1152, 1536, False),
    (0, 500, 3584, 3584, True), (0, 400, 3584, 3584, False), (0, 1000, 512, 2048, False), (0, 1000, 4096, 4160, False), (0, 700, 8200, 512, False),
    # gated: up to 136 M elements, no narrow output of a long K
    (2, 72, 37888, 3584, True), (2, 512, 27648, 5120, False), (2, 165, 896, 4864, False), (2, 2048, 2048, 1024, True),
    # sums for a norm
    (3, 2048, 1536, 8960, True), (3, 1500, 5120, 13824, True), (3, 1600, 5120, 27648, False), (3, 250, 8192, 29568, True), (3, 640, 8192, 29568, False),
    (3, 780, 1536, 1536, True), (3, 790, 1536, 1536, False), (3, 500, 2048, 2048, True), (3, 520, 2048, 2048, False), (3, 152, 7376, 2304, False),
    # rows that are no multiples of 16 bytes, rows of x that are none, too few rows and too many
    (0, 256, 1028, 512, False), (2, 256, 8200, 512, False), (3, 256, 514, 2048, False), (0, 64, 1152, 896, False), (0, 2049, 1152, 896, False)])
def test_products_on_the_wide_kernels_tiles(mode, M, N, K, there):
    choice = _wide_choice(mode, M, N, K)
    assert (choice is not None) == there
    if there:
        bm, bn, planes = choice
        assert planes == 1 or (mode == 3 and K // planes >= 256)
        assert _wide_choice(mode, M, N, K, K + 4) is None   # rows of x at no 16 bytes


@pytest.mark.parametrize("M,N,K,hd,there", [(2048, 1152, 896, 64, True), (2049, 1152, 896, 64, False), (1024, 2048, 1536, 128, True),
                                           (1152, 2048, 1536, 128, True), (1153, 2048, 1536, 128, False), (72, 2048, 1536, 128, True), (72, 2560, 2048, 128, False),
                                           (128, 2560, 2048, 128, True), (336, 4608, 3584, 128, False), (64, 1152, 896, 64, False), (160, 1152, 896, 48, False),
                                           (160, 1150, 896, 64, False), (160, 1152, 900, 64, False)])
def test_queries_keys_and_values_rotated_by_their_product(M, N, K, hd, there):
    assert bool(ops._load("gemm_tile").cw_gemm_bf16_pairs_ok(M, N, K, K, hd)) == there


def test_tiles_follow_the_rounds_that_they_need():
    """Gate/up of the 1.5B shape: the tile whose rounds over the compute units are fullest for what they cost."""
    tiles = {M: _wide_choice(2, M, 17920, 1536)[:2] for M in (100, 160, 336, 512, 1000, 2048)}
    assert tiles[1000] == tiles[2048] == (256, 288)      # 252 and 504 tiles
    assert tiles[336] == (192, 160)                      # 224
    assert tiles[100] == tiles[160] == (160, 96)         # 187, the fewest columns that one round of a row tile takes
    assert all(_wide_choice(3, M, 1536, 8960)[2] <= _wide_choice(3, 160, 1536, 8960)[2] for M in (336, 1000, 2048))


def test_no_choice_outside_what_the_kernels_take():
    for mode in (0, 2, 3):
        for M, N, K in ((64, 1152, 896), (2049, 1152, 896), (144, 1152, 900), (144, 1152, 192), (144, 0, 896)):
            assert _choice(mode, M, N, K) is None
    assert _choice(2, 160, 9729, 896) is None and _choice(1, 160, 1152, 896) is None


def test_planes_of_many_rows_only_for_a_norm_that_adds_them(monkeypatch):
    """A product of a portion, and any in float32, may come as planes of partial sums where its block hands it to a norm
    that adds them in its kernel; any other reader would add a dozen planes with a dozen launches."""
    from clockwork_amd.parts.block import PreNormBlock, TwoNormParallelBlock
    from clockwork_amd.parts.mlp import SwiGLU
    from clockwork_amd.parts.norm import LayerNorm, RMSNorm

    assert RMSNorm.adds_partial_sums and not getattr(LayerNorm, "adds_partial_sums", False)
    asked = []
    monkeypatch.setattr(ops, "linear_swiglu", lambda x, *a, **k: x)
    monkeypatch.setattr(ops, "linear", lambda *a, **k: asked.append(k["portions_partial_ok"]))
    monkeypatch.setattr(ops, "gated_residual_add", lambda *a: None)
    feed_forward = SwiGLU(None)
    feed_forward.gate_up = feed_forward.down = None

    class Mixer:
        def forward(self, x, ctx, cache):
            asked.append(("mixer", ctx.reader_adds_sums))

    def norm(adds):
        return SimpleNamespace(forward=lambda resid, delta: resid, adds_partial_sums=adds)

    resid = SimpleNamespace(shape=(300, 8), dtype=None)
    for inner in (False, True):
        for after in (False, True):
            ctx = SimpleNamespace(next_norm_adds_sums=after, next_norm_accepts_pending=False, products=None)
            PreNormBlock(Mixer(), norm(False), feed_forward, norm(inner)).forward(resid, None, ctx, None)
            assert asked == [("mixer", inner), after]
            asked.clear()
            PreNormBlock(Mixer(), norm(False)).forward(resid, None, ctx, None)
            assert asked == [("mixer", after)]
            asked.clear()
            ctx.next_norm_accepts_pending = inner
            TwoNormParallelBlock(Mixer(), norm(True), feed_forward, norm(True)).forward(resid, None, ctx, None)
            assert asked == [("mixer", False), inner and after]
            asked.clear()
    # a part that no block has told anything
    feed_forward.forward(resid, SimpleNamespace(products=None))
    assert asked == [False]


def test_the_model_says_whether_the_next_norm_adds_planes():
    from clockwork_amd.config.spec import LayerSpec, ModelSpec, RunEntry
    from clockwork_amd.parts.model import DecoderModel
    from clockwork_amd.parts.specs import AttentionSpec, RMSNormSpec, SwiGLUSpec

    norm = RMSNormSpec(16, 1e-6)
    layer = LayerSpec("prenorm", AttentionSpec(16, 1, 1, 16, False, False, 0.25), SwiGLUSpec(16, 32), norm, norm)
    model = DecoderModel(ModelSpec("toy", 10, 16, [layer], [RunEntry(0)] * 4, norm))
    said = []

    class Block:
        def __init__(self, adds):
            self.first_norm = lambda: SimpleNamespace(adds_partial_sums=adds)

        def forward(self, resid, delta, ctx, cache):
            said.append((ctx.next_norm_adds_sums, ctx.reader_adds_sums))
            ctx.reader_adds_sums = True   # does not reach the next block
            return delta

    model.layers = [Block(True), Block(True), Block(False), Block(True)]
    model.spec.run = [RunEntry(0), RunEntry(1), RunEntry(2), RunEntry(3)]
    model.embedding = type("E", (), {"forward": lambda self, ctx: None})()
    assert model.forward(SimpleNamespace(num_logit_rows=0, sequence_positions=None), [None] * 4) is None
    assert said == [(True, False), (False, False), (True, False), (True, False)]


@pytest.mark.parametrize("N,K,parts", [(4096, 14336, 8), (8192, 29568, 8), (3584, 18944, 8), (1536, 8960, 7), (5120, 27648, 11), (896, 4864, 4)])
def test_parts_over_k_do_not_come_to_more_workgroups_than_units(N, K, parts):
    """Products of up to 16 rows: a workgroup takes ceil(tiles * parts / 256) tiles of a part."""
    tiles = -(-N // 16)
    assert -(-tiles // -(-tiles * parts // CUS)) * parts <= CUS
    assert all(ops._load("gemm").cw_gemm_bf16_skinny_ksplits(M, N, K) == parts for M in (1, 8, 16))


def test_several_products_of_few_rows():
    """Which are taken together, and that operands of other kinds are not."""
    import torch

    from clockwork_amd import ops

    ok = ops._load("gemm").cw_gemm_bf16_group_ok
    for M in (1, 16):
        assert ok(2, 0, M, 2, 8) and ok(4, 1, M, 5000, 1536)
    # beyond 16 rows: one x, and tiles and a K that the streaming kernel takes
    assert ok(3, 1, 64, 610, 1536) and not ok(3, 0, 64, 610, 1536) and not ok(3, 1, 64, 200, 1536) and not ok(3, 1, 17, 610, 512)
    # one product, five, no rows, more rows, columns that are not whole 16 bytes
    assert not (ok(1, 1, 8, 96, 1536) or ok(5, 1, 8, 480, 1536) or ok(2, 1, 0, 96, 1536) or ok(2, 1, 65, 610, 1536) or ok(2, 1, 8, 96, 1532))
    x, w = torch.zeros(4, 64, dtype=torch.bfloat16), torch.zeros(32, 64, dtype=torch.bfloat16)
    for xs, ws in (([x, x], [w, w.float()]), ([x.float(), x.float()], [w, w]), ([x, x[:2]], [w, w]), ([x, x], [w, w[:, :32]]),
                   ([x, x], [w, w.t().contiguous().t()]), ([x[:, :32], x[:, :32]], [w[:, :32].contiguous()] * 2), ([x], [w])):
        assert ops.linear_several(xs, ws) is None


def test_float32_queries_keys_and_values_of_few_rows():
    from clockwork_amd import ops

    ok = ops._load("gemm").cw_gemm_f32_pairs_ok
    assert ok(1, 896, 14, 2, 64) and ok(16, 1920, 2, 2, 32)
    # rows, blocks of K, whole blocks, whole tiles of a head, heads
    assert not (ok(0, 896, 14, 2, 64) or ok(17, 896, 14, 2, 64) or ok(1, 1936, 14, 2, 64) or ok(1, 888, 14, 2, 64) or ok(1, 896, 14, 2, 24)
                or ok(1, 896, 0, 2, 64) or ok(1, 896, 2, 0, 64) or ok(1, 896, 1000, 20, 64))


@pytest.mark.parametrize("N,K,planes", [(896, 896, 2), (1536, 1536, 2), (1536, 8960, 5), (3584, 3584, 2), (4096, 14336, 8), (8192, 28672, 16), (768, 512, 2)])
def test_planes_of_17_to_64_rows(N, K, planes):
    """A workgroup takes ceil(tiles * planes / 256) tiles of a part; no more workgroups than units."""
    lib = ops._load("gemm")
    assert lib.cw_gemm_bf16_skinny_planes(33, N, K) == planes
    for M in (17, 32, 33, 64):
        s = lib.cw_gemm_bf16_skinny_planes(M, N, K)
        tiles = -(-N // 16)
        assert 2 <= s <= 16 and K // s >= 256 and -(-tiles // -(-tiles * s // CUS)) * s <= CUS
    # rows, an output of more than 512 tiles, K too short to cut, an output that leaves the units idle however K is cut
    assert all(lib.cw_gemm_bf16_skinny_planes(*shape) == 1 for shape in ((16, N, K), (65, N, K), (33, 8193, K), (33, N, 511), (33, 64, 512)))


def test_a_table_of_angles_is_kept_for_a_pass_over_the_model_only(monkeypatch):
    """Layers of one pass share a table; a layer that is called by itself, with a context whose positions have been
    written again since, makes its own, also after a pass."""
    import types

    import torch

    from clockwork_amd.engine.batch import StepContext
    from clockwork_amd.parts import rope
    from clockwork_amd.parts.model import DecoderModel
    from clockwork_amd.parts.specs import RopeNeoxSpec

    made = []
    monkeypatch.setattr(rope.ops, "qkv_rope_rows_ok", lambda *a: True)
    monkeypatch.setattr(rope.ops, "rope_angles", lambda positions, inv_freq: made.append(positions.clone()) or made[-1])
    monkeypatch.setattr(rope.ops, "qkv_rope_rows", lambda x, w, b, angles, *a: angles)
    part = rope.RopeNeox(RopeNeoxSpec(rotary_dim=64, theta=1e6))
    part.bind({}, "cpu", torch.bfloat16)
    ctx = StepContext()
    ctx.positions = torch.arange(100, dtype=torch.int32)

    def layer():
        return part.project_rotate_store_rows(None, None, None, ctx, torch.zeros(100), 2, 1, 64, None, None)

    assert torch.equal(layer(), ctx.positions)
    ctx.positions += 100
    assert torch.equal(layer(), ctx.positions) and len(made) == 2
    # a model of two layers: one table, and nothing left of it
    block = types.SimpleNamespace(forward=lambda *a: layer())
    entries = [types.SimpleNamespace(layer=i, add_input=False, reenter=None) for i in range(2)]
    model = types.SimpleNamespace(embedding=types.SimpleNamespace(forward=lambda ctx: None), own_caches=lambda: [], layers=[block, block],
                                  spec=types.SimpleNamespace(run=entries), final_norm=None)
    model._pass = types.MethodType(DecoderModel._pass, model)
    DecoderModel.forward(model, ctx, [None, None])
    assert len(made) == 3
    ctx.positions += 100
    assert torch.equal(layer(), ctx.positions) and len(made) == 4


@pytest.mark.parametrize("mode,M,N,K,there", [
    # whole rows: many columns and few outputs of a middling K are the narrow tiles' by lines of their own
    (0, 72, 8704, 512, True), (0, 400, 8704, 512, True), (0, 512, 8704, 512, False), (0, 160, 9728, 896, True), (0, 320, 9728, 896, False),
    (0, 322, 1536, 1536, True), (0, 319, 1536, 1536, False), (0, 2048, 2048, 1536, True),
    # rows that end inside 16 bytes
    (0, 300, 4097, 896, True), (2, 160, 8008, 640, True), (3, 144, 1538, 8960, True), (0, 300, 9729, 1536, False)])
def test_one_rule_names_the_tiles_of_a_product(monkeypatch, mode, M, N, K, there):
    """What the engine asks: for whole rows ``cw_gemm_bf16_wide_choice`` alone, for others ``cw_gemm_bf16_mid_choice`` alone."""
    import torch

    monkeypatch.setattr(ops, "_compute_units", lambda device: CUS)
    code = ops._tile_rule(mode, torch.empty(M, K, dtype=torch.bfloat16), torch.empty(N, K, dtype=torch.bfloat16))
    whole = N % {0: 8, 2: 16, 3: 4}[mode] == 0
    assert ((code & 1023, code >> 10 & 1023, code >> 20) if code else None) == (_wide_choice if whole else _choice)(mode, M, N, K)
    assert (code != 0) == there
    if whole and there and not (N <= 8192 and M * N >= 500000):
        assert code == 64 | 64 << 10 | 1 << 20


def test_long_sums_of_many_rows_are_whole_on_large_tiles_only():
    """Smaller ones ask L2 for more than it gives (7B shape's down product, 1280 rows 199 us by 160 x 128, 173 in runs)."""
    for M in range(641, 2049, 7):
        for N, K in ((3584, 18944), (2048, 11008), (4096, 14336), (5120, 27648)):
            choice = _wide_choice(3, M, N, K)
            assert choice is None or choice[2] > 1 or choice[0] + choice[1] >= 352
    assert _wide_choice(3, 1280, 3584, 18944) == (192, 160, 3) and _wide_choice(3, 2048, 3584, 18944) == (192, 160, 1)


@pytest.mark.parametrize("M,N,K,want", [(208, 896, 4864, (64, 64, 4)), (320, 1024, 4096, (64, 64, 3)), (160, 2048, 2048, (64, 64, 2)), (640, 1536, 1536, (64, 64, 1))])
def test_few_small_tiles_rather_than_many_runs(M, N, K, want):
    """Sums that tiles of 64 x 128 in more runs were named for, 6 to 13 % slower (11.8 / 13.3, 13.1 / 14.5, 11.0 / 12.0, 14.2 / 15.2 us with the norm)."""
    assert _wide_choice(3, M, N, K) == want


@pytest.mark.parametrize("M,N,K,there", [(1500, 6144, 3072, True), (1600, 6144, 3072, False), (2048, 6144, 3072, False), (2048, 5120, 2048, True), (2048, 4608, 3584, True)])
def test_large_outputs_of_a_long_k_are_the_librarys(M, N, K, there):
    assert (_wide_choice(0, M, N, K) is not None) == there


# cards of 304 compute units down to 64, and a part of one
@pytest.mark.parametrize("units", [304, 256, 128, 64, 32])
def test_a_joining_product_has_room_for_its_outputs(units):
    """A workgroup owns no more outputs than its kernel has room for (eight waves: 8), and the workgroups all of them."""
    rule, taken = ops._load("gemm").cw_gemm_bf16_join_rule, 0
    for N in (64, 72, 512, 896, 1000, 1024, 1536, 2048, 2056, 3584, 4096):
        for K in (256, 896, 1536, 2048, 2056, 4864, 8960):
            code = rule(1, N, K, units)
            rows, slots, waves = code & 255, code >> 8 & 255, code >> 16
            assert rows <= slots and (not code or (waves, slots) in ((8, 8), (16, 4), (16, 8), (16, 16)))
            assert not code or -(-N // rows) <= min(units, 256)
            taken += code != 0
    assert taken
    if units == 256:   # as its kernels were timed
        assert [rule(8, N, K, units) for N, K in ((896, 896), (896, 4864), (1536, 1536), (1536, 8960), (3584, 3584))] == [
            8 | 8 << 8 | 8 << 16, 4 | 4 << 8 | 16 << 16, 8 | 8 << 8 | 8 << 16, 6 | 8 << 8 | 16 << 16, 14 | 16 << 8 | 16 << 16]


@pytest.mark.parametrize("n", [1, 32, 33, 64, 512, 65535])
@pytest.mark.parametrize("V", [1, 2048, 151936, (1 << 21) + 1, (1 << 24) + 5, (1 << 26) - 3, 1 << 27])
def test_chunks_of_a_row_of_logits_have_few_enough_tokens_for_float64_sums(n, V):
    """4 tokens of every 1024 a thread, each a weight of up to 2^40: at most 2^53 in all (2^27 logits are 64 chunks of 2^21)."""
    need = ops._load("sampling").cw_sample_workspace_bytes
    one = need(1, 1) - 64 - 32   # what a row of one chunk needs beside the chunk's
    chunks = ((need(n, V) - 64) // n - one) // 32
    per = -(-(-(-V // chunks)) // 4) * 4
    assert 1 <= chunks <= 64 and 4 * -(-per // 1024) * 2 ** 40 <= 2 ** 53


@pytest.mark.parametrize("N,K,rows,not_rows", [(896, 4864, (1, 8, 13), (14, 16)), (1536, 8960, (1, 4, 7), (8, 16)), (2048, 11008, (1, 4, 5), (6, 8)), (3584, 18944, (), (1, 2, 3)),
                                               (2560, 9728, (1,), (2, 4, 8)), (4096, 14336, (1,), (2, 4)), (1536, 1536, (1, 8, 16), ()), (3584, 3584, (1, 8, 16), ()), (4096, 4096, (16,), ())])
def test_outputs_join_the_stream_where_that_is_the_faster_way(N, K, rows, not_rows):
    """The parts ask what pays; the kernel takes more than that (few rows of a long K, timed both ways in whole steps)."""
    import torch

    from clockwork_amd.parts.mlp import SwiGLU

    ffn, norm = SwiGLU.__new__(SwiGLU), SimpleNamespace(weight=torch.ones(N))
    ffn.down = torch.zeros(1, dtype=torch.bfloat16).expand(N, K)
    assert not ffn.joins_stream(1, norm)   # rows with gaps
    ffn.down = torch.empty(N, K, dtype=torch.bfloat16)
    assert all(ffn.joins_stream(M, norm) for M in rows) and not any(ffn.joins_stream(M, norm) for M in not_rows)
    assert all(ops.linear_join_ok(M, ffn.down, norm.weight) == (M <= 16 and M * K <= 72 * 1024) for M in (*rows, *not_rows, 17))


def test_few_rows_join_the_stream_between_blocks_only():
    """The mixer's output begins the second norm and the feed-forward's the next block's first one, where the parts take such
    rows and another block follows; the last block leaves its outputs to the final norm."""
    import torch

    from clockwork_amd.parts.block import PreNormBlock

    calls = []

    class Piece:
        def __init__(self, name, most):
            self.name, self.most = name, most

        def takes_begun_norm(self, n, *cache):
            return n <= self.most

        def joins_stream(self, n, norm):
            return n <= self.most

        def forward(self, x, *rest):
            calls.append((self.name, type(x).__name__))
            return torch.zeros(1)

        def forward_joined(self, x, *rest):
            calls.append((self.name + " joins", type(x).__name__, rest[-1].name))
            return ops.BegunNorm(torch.zeros(1), torch.zeros(1), 1e-6)

    def norm(name, begun=True):
        return SimpleNamespace(name=name, can_be_begun=begun, forward=lambda resid, delta: calls.append(name) or torch.zeros(1))

    def run(rows, follows, nxt, delta=None, begun=True):
        calls.clear()
        block = PreNormBlock(Piece("mixer", 16), norm("n1", begun), Piece("ffn", 16), norm("n2", begun))
        ctx = SimpleNamespace(block_follows=follows, norm_to_begin=nxt)
        out = block.forward(SimpleNamespace(shape=(rows, 8)), delta, ctx, None)
        return list(calls), isinstance(out, ops.BegunNorm), block.norm_to_begin(rows, None)

    nxt, begun = norm("next"), ops.BegunNorm(torch.zeros(1), torch.zeros(1), 1e-6)
    got, joined, first = run(4, True, nxt)
    assert got == ["n1", ("mixer joins", "Tensor", "n2"), ("ffn joins", "BegunNorm", "next")] and joined and first.name == "n1"
    got, joined, _ = run(4, True, nxt, begun)
    assert got == [("mixer joins", "BegunNorm", "n2"), ("ffn joins", "BegunNorm", "next")] and joined
    assert run(4, True, None)[:2] == (["n1", ("mixer joins", "Tensor", "n2"), ("ffn", "BegunNorm")], False)
    assert run(4, False, None, begun)[:2] == ([("mixer", "BegunNorm"), "n2", ("ffn", "Tensor")], False)
    assert run(17, True, None) == (["n1", ("mixer", "Tensor"), "n2", ("ffn", "Tensor")], False, None)
    assert run(4, True, None, begun=False) == (["n1", ("mixer", "Tensor"), "n2", ("ffn", "Tensor")], False, None)


def _mixer_kinds():
    import importlib
    import inspect

    from clockwork_amd import registry

    kinds = []
    for module, name in registry._BUILTIN_PARTS.values():
        cls = getattr(importlib.import_module(module), name)
        if list(inspect.signature(getattr(cls, "forward", lambda: None)).parameters)[:4] == ["self", "x", "ctx", "cache"]:
            kinds.append(cls)
    return kinds


@pytest.mark.parametrize("cls", _mixer_kinds(), ids=lambda cls: cls.__name__)
def test_every_mixer_in_a_block_whose_parts_join_the_stream(cls, monkeypatch):
    """Few rows of bfloat16 in a block whose feed-forward and norms take part: a mixer that does not is run by ``forward``."""
    import torch

    from clockwork_amd.parts.block import PreNormBlock

    mixer, out = cls.__new__(cls), torch.zeros(4, 8)
    mixer.out_bias = torch.zeros(8)   # (plain attention with a bias behind its last product leaves the add to the norm)
    monkeypatch.setattr(cls, "forward", lambda self, x, ctx, cache: out)
    ffn = SimpleNamespace(takes_begun_norm=lambda n: True, joins_stream=lambda n, norm: False, forward=lambda x, ctx: x)
    norm = SimpleNamespace(can_be_begun=True, forward=lambda resid, delta: torch.zeros(4, 8) if delta is None else delta)
    got = PreNormBlock(mixer, norm, ffn, norm).forward(SimpleNamespace(shape=(4, 8)), None, SimpleNamespace(block_follows=True), None)
    assert got is out


def test_a_scaled_pair_refuses_mixers_without_a_place_between_products():
    from clockwork_amd.parts.pair import PairMixer
    from clockwork_amd.parts.specs import AttentionSpec, PairMixerSpec

    side = AttentionSpec(hidden_size=64, num_heads=2, num_kv_heads=1, head_dim=32, qkv_bias=False, out_bias=False, scale=1.0)
    with pytest.raises(NotImplementedError):
        PairMixer(PairMixerSpec(hidden_size=64, left=side, right=side, scales=(0.5, 0.5)))


@pytest.mark.parametrize("joint", [False, True])
def test_blocks_take_chosen_rows_of_mixers_that_make_them(joint):
    """A scaled pair whose mixers share one output product makes all rows, in either block; two mixers with outputs of their own make
    the chosen ones; a mixer that does not know of it makes all."""
    from clockwork_amd.parts.attention import PagedAttention
    from clockwork_amd.parts.block import ParallelBlock, PreNormBlock
    from clockwork_amd.parts.pair import PairMixer

    pair = PairMixer.__new__(PairMixer)
    pair.joint = joint
    pair.left = pair.right = SimpleNamespace(before_output=None)
    ffn, norm = SimpleNamespace(by_rows=True), SimpleNamespace()
    for mixer, takes in ((pair, not joint), (PagedAttention.__new__(PagedAttention), True), (SimpleNamespace(), False)):
        pre, par = PreNormBlock(mixer, norm, ffn, norm), ParallelBlock(mixer, norm, ffn)
        assert pre.takes_rows(100, 1) == par.takes_rows(100, 1) == takes
        assert not PreNormBlock(mixer, norm, SimpleNamespace(), norm).takes_rows(100, 1)
        # as few rows as are not worth it, none, more than half
        for rows, chosen in ((16, 1), (100, 0), (100, 51)):
            assert not pre.takes_rows(rows, chosen) and not par.takes_rows(rows, chosen)
        assert not pre.takes_rows(32, 1) and pre.takes_rows(33, 16) == pre.takes_rows(64, 17) == takes
        assert par.takes_rows(17, 1) == par.takes_rows(64, 16) == par.takes_rows(65, 17) == takes and not par.takes_rows(64, 17)


def test_parts_with_a_forward_of_their_own_are_not_passed_by():
    """A part derived from a built-in one, or an object given a method, is run by that method: the hooks that go past it say no."""
    import torch

    from clockwork_amd.parts import attention, block, mlp, norm, pair, rope
    from clockwork_amd.parts.base import EntryCache
    from clockwork_amd.parts.specs import AttentionSpec, GatedMLPSpec, LayerNormSpec, RMSNormSpec, RopeNeoxSpec, SwiGLUSpec

    cpu, H, I, hd = "cpu", 512, 1024, 64
    begun = norm.RMSNorm(RMSNormSpec(H, 1e-6))
    begun.weight = torch.ones(H)

    def attn(cls, position=rope.RopeNeox):
        part = cls(AttentionSpec(H, 8, 2, hd, False, False, 0.1, position=RopeNeoxSpec(hd, 1e4)))
        part.position = position(part.spec.position)
        part.bind({"qkv_weight": torch.zeros(12 * hd, H, dtype=torch.bfloat16), "out_weight": torch.zeros(H, H, dtype=torch.bfloat16)}, cpu, torch.bfloat16)
        return part

    def ffn(cls, spec=SwiGLUSpec(H, I)):
        part = cls(spec)
        part.bind({"gate_up_weight": torch.zeros(2 * I, H, dtype=torch.bfloat16), "down_weight": torch.zeros(H, I, dtype=torch.bfloat16)}, cpu, torch.bfloat16)
        return part

    def two(cls):
        part = cls.__new__(cls)
        part.joint, part.left, part.right = False, SimpleNamespace(before_output=None), SimpleNamespace(before_output=None)
        return part

    def pre(cls):
        return cls(attn(attention.PagedAttention), begun, ffn(mlp.SwiGLU), begun)

    def par(cls):
        return cls(two(pair.PairMixer), begun, ffn(mlp.SwiGLU))

    cache = EntryCache()
    kinds = [(attention.PagedAttention, attn, "forward", [lambda p: p.takes_begun_norm(4, cache), lambda p: p.joins_stream(4, begun), lambda p: p.takes_rows()]),
             (rope.RopeNeox, lambda cls: attn(attention.PagedAttention, cls), "project_rotate_store", [lambda p: p.takes_begun_norm(4, cache)]),
             (mlp.SwiGLU, ffn, "forward", [lambda p: p.takes_begun_norm(4), lambda p: p.joins_stream(4, begun), lambda p: p.by_rows]),
             (mlp.GatedMLP, lambda cls: ffn(cls, GatedMLPSpec(H, I)), "forward", [lambda p: p.by_rows]),
             (norm.RMSNorm, lambda cls: cls(RMSNormSpec(H, 1e-6)), "forward", [lambda p: p.can_be_begun, lambda p: p.takes_all_rows]),
             (norm.LayerNorm, lambda cls: cls(LayerNormSpec(H, 1e-6)), "forward", [lambda p: p.takes_all_rows]),
             (pair.PairMixer, two, "forward", [lambda p: p.takes_rows()]),
             (block.PreNormBlock, pre, "forward", [lambda p: p.takes_rows(100, 1), lambda p: p.norm_to_begin(4, cache) is begun]),
             (block.ParallelBlock, par, "forward", [lambda p: p.takes_rows(100, 1)])]
    for cls, build, method, hooks in kinds:
        same = type("Same", (cls,), {})
        own = type("Own", (cls,), {method: lambda self, *args: None})
        for hook in hooks:
            assert hook(build(cls)) and hook(build(same)), cls
            assert not hook(build(own)), cls
        if cls is not rope.RopeNeox:
            given = build(cls)
            setattr(given, method, lambda *args: None)
            assert not any(hook(given) for hook in hooks), cls


@pytest.mark.parametrize("taken", [False, True])
def test_chosen_rows_keep_the_first_products_of_a_pair_in_one_launch(taken, monkeypatch):
    """The last block of a portion of few rows makes its mixers' first products as every other block does."""
    import torch

    from clockwork_amd.parts.block import ParallelBlock

    weights, asked, got = [torch.zeros(2, 8), torch.ones(3, 8)], [], {}

    def several(xs, ws):
        asked.append((len(xs), [w is v for w, v in zip(ws, weights)]))
        return ["left", "right"] if taken else None

    def forward_rows(x, ctx, cache, rows, *others, made=None):
        got["made"] = made
        return x[rows], [o[rows] for o in others]

    monkeypatch.setattr(ops, "linear_several", several)
    x = torch.randn(40, 8)
    mixer = SimpleNamespace(input_weights=lambda: list(weights), forward_rows=forward_rows)
    block = ParallelBlock(mixer, SimpleNamespace(forward=lambda resid, delta: x))
    resid, pending = block.forward_rows(torch.zeros(40, 8), None, SimpleNamespace(next_norm_accepts_gated=True), None, torch.tensor([39]))
    assert asked == [(2, [True, True])] and got["made"] == (["left", "right"] if taken else None)
    assert resid.shape == (1, 8) and torch.equal(pending.a, x[39:])


@pytest.mark.parametrize("counts", [[2048, 1, 2, 64], [300, 8], [48, 24]])
def test_choices_for_few_rows_are_timed_on_the_step_of_few_rows(counts, monkeypatch):
    """A tuning start-up runs it ahead of the long portions, whose last block multiplies one row."""
    import contextlib

    import torch

    from clockwork_amd.engine.model_runner import ModelRunner

    ran = []
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    monkeypatch.setattr(ops, "library_tuning", lambda policy: contextlib.nullcontext())
    runner = SimpleNamespace(dtype=torch.bfloat16, cfg=SimpleNamespace(model=SimpleNamespace(max_model_len=4096)), _table_width=256, products=None,
                             manager=SimpleNamespace(block_size=16, can_admit=lambda *a: True), FEW_ROWS_SAMPLE=ModelRunner.FEW_ROWS_SAMPLE,
                             reserve=lambda *a, **k: None, release=lambda s: None, step=lambda entries: ran.append(len(entries[0].tokens)))
    few = min(counts) <= ops.SKINNY_MAX_ROWS
    large = sorted((c for c in counts if c > ops.SKINNY_MAX_ROWS), reverse=True)
    assert ModelRunner.tune_products(runner, counts) == large + [8] * few
    assert ran == [8] * few + large
