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
