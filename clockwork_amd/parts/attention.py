"""Grouped-query softmax attention over the paged cache (clockwork/engine/model.py:66-128).

Steps: one fused q/k/v product; bias, rotation and the cache write in one kernel (keys
and values of every token of the step are in the cache before any query reads it,
model.py:100); attention straight from the pages through the block table, prompt
portions and single tokens in the same step; output product.
"""

from __future__ import annotations

import math
from dataclasses import dataclass
from functools import lru_cache
from types import SimpleNamespace
from typing import Optional

import numpy as np
import torch

from clockwork_amd import ops
from clockwork_amd.config.spec import KVPagesSpec, ParamSpec
from clockwork_amd.parts.base import EntryCache, Part, own_method
from clockwork_amd.parts.rope import NoPosition
from clockwork_amd.parts.specs import AttentionSpec
from clockwork_amd.registry import build_part


@dataclass
class AttentionPlan:
    """Work items of the attention kernels for one head geometry (see csrc/attention.hip).

    Requests with one token go to the 16-row kernel, cut over their keys into
    ``single_splits`` parts; longer portions are cut into tiles of the 64-row kernel."""

    wide_items: Optional[torch.Tensor] = None
    n_wide: int = 0
    gh_wide: int = 1
    wide_splits: int = 1       # parts every wide item's key range is cut into (few items with many keys)
    mfma_items: Optional[torch.Tensor] = None   # the same portions cut for the bfloat16 matrix-core kernel
    n_mfma: int = 0
    mfma_row_blocks: int = 4   # row blocks of that kernel's workgroups: 2 when 4 would leave compute units idle
    mfma_parts: int = 1        # the most parts an item's key range is shared among (1: no item is cut)
    single_items: Optional[torch.Tensor] = None
    n_single: int = 0
    gh_single: int = 1
    chunks_single: int = 1
    single_splits: int = 1
    decode_splits: int = 1   # splits of the bfloat16 decode kernel (finer: it walks 16-key tiles)
    decode_split_keys: int = 0    # keys of each of those splits, at fixed places (a multiple of 32)
    decode_max_ctx: int = 0       # the longest context the fixed places were planned for
    single_identity: bool = False  # a batch of single tokens only: item i is request i, token row i
    together: bool = False        # the matrix-core kernels' portions and single tokens go as one launch


# a portion's key ranges count as long when its tokens see this many keys or more on average
LONG_RANGE_KEYS = 3072


def portions_have_short_ranges(q_lens, ctx_lens) -> bool:
    """The rule by which a step's portions (entries of more than one token) choose the shape of
    the matrix-core kernel's workgroups: True while their tokens see fewer than 3072 keys on
    average. Behind a long cached prefix every workgroup's key range is long and about the same,
    and sharing the keys among more rows wins (2048 tokens of 12 heads of 128 on 2, us, two row blocks / four: no
    prefix 31.8 / 36.9, behind 1024 tokens 49.4 / 50.5, 2048 68.0 / 64.0, 6144 142.7 / 118.1; 1000 tokens, whose
    workgroups of four are 96, behind 2500 41.5 / 56.5, the keys not cut into parts)."""
    tokens = sum(q for q in q_lens if q > 1)
    keys = sum(q * (c - q / 2.0) for q, c in zip(q_lens, ctx_lens) if q > 1)
    return tokens > 0 and keys / tokens < LONG_RANGE_KEYS


# a part of an item's key range is at least this many keys (two stages of the kernel), and an item
# is cut into at most this many parts
MIN_PART_KEYS = 256
MAX_PARTS = 64
# Parts of a single token's keys for the float32 kernel: a workgroup of eight waves takes 128 keys in one turn of some
# 1.5 us, and the kernel that merges the parts takes 4 us however many there are. Up to 384 keys stay whole (one
# request of the 0.5B shape, one part / parts of 128 keys: 300 keys 10.3 / 10.5 us, 510 keys 12.9 / 10.9): a rule for steps
# that are not captured. Captured ones are planned for a multiple of 512 keys and always have four parts or more.
F32_PART_KEYS = 128
F32_WHOLE_KEYS = 384


def _share_long_key_ranges(items: np.ndarray, ctx, workgroups_per_item: int):
    """A compute unit holds one workgroup of the kernel for portions at a time (its tiles fill the
    unit's LDS), so a launch with fewer workgroups than half the compute units (a short portion behind a long cached
    prefix: the end of a long prompt, a new turn of a long conversation) leaves most of the card
    idle while a few units walk through thousands of keys. Such a launch's items stand in the
    list once for each of several parts, one after the other, as ``part | parts << 8`` in the
    fourth field; the kernel gives each part a run of the item's keys and a second kernel puts
    them together. Launches that fill the card are left alone: there the parts cost more than
    they bring (measured). Returns the flat item list and the most parts of an item (1: nothing
    was cut)."""
    workgroups = len(items) * workgroups_per_item
    spare = ctx.num_compute_units // max(workgroups, 1)
    if len(items) == 0 or spare < 2:
        return items.reshape(-1), 1
    ctx_lens = np.asarray(ctx.h_ctx_lens, dtype=np.int64)
    q_lens = np.asarray(ctx.h_q_lens, dtype=np.int64)
    req = items[:, 0]
    keys = ctx_lens[req] - q_lens[req] + items[:, 1] + items[:, 2]  # keys that the item's last token sees
    parts = np.minimum(spare, keys // MIN_PART_KEYS).clip(1, MAX_PARTS).astype(np.int64)
    most = int(parts.max())
    if most == 1:
        return items.reshape(-1), 1
    out = np.repeat(items, parts, axis=0)
    first = np.cumsum(parts) - parts  # where each item's parts begin
    part = np.arange(len(out)) - np.repeat(first, parts)
    out[:, 3] = part | (np.repeat(parts, parts) << 8)
    return out.astype(np.int32).reshape(-1), most


def typical_start(start: int) -> int:
    """Where the portions that one captured step serves are taken to begin when it is planned: nowhere behind cached
    keys, or behind the nearest power of two of them, from 512 on. (How many parts a portion's keys are cut into follows
    their number, and a captured step for each number would be one for each request: with a power of two the parts are
    at most 1.4 times too long or too short, and they stop growing where they fill the card.)"""
    near = 1 << round(math.log2(start)) if start > 0 else 0
    return near if near >= 512 else 0


def _typical_lens(q_lens, ctx_lens) -> tuple:
    """The contexts that a captured step is planned for: every portion where the portions of its kind begin."""
    return tuple(c if q == 1 else q + typical_start(c - q) for q, c in zip(q_lens, ctx_lens))


@lru_cache(maxsize=4096)
def captured_choices(q_lens: tuple, ctx_lens: tuple, *how) -> tuple:
    """What the plan of a captured step decides by its portions' cached keys: steps of the same tokens and the same choices
    have the same plan. ``how``: (heads, kv heads, compute units, whether the portions run on the bfloat16 matrix-core kernel,
    and ``attention_plan``'s ``narrow_ok``, ``whole_keys`` and ``together_ok``). (A portion's start is hardly ever one that was
    there before, what it counts as nearly always is.)"""
    return _choices_of(q_lens, _typical_lens(q_lens, ctx_lens), *how)


@lru_cache(maxsize=1024)
def _choices_of(q_lens: tuple, ctx_lens: tuple, nh: int, nkv: int, units: int, mfma: bool, narrow_ok: bool, whole_keys: int,
                together_ok: bool) -> tuple:
    step = SimpleNamespace(h_q_lens=q_lens, h_ctx_lens=ctx_lens, num_compute_units=units, upload=lambda arrays: arrays)
    plan = _make_plan(step, nh, nkv, narrow_ok and any(q > 1 for q in q_lens), whole_keys, together_ok)
    if not mfma:
        return ("parts", plan.wide_splits)
    parts = np.maximum(np.asarray(plan.mfma_items).reshape(-1, 4)[:, 3] >> 8, 1)
    edges = np.flatnonzero(np.diff(parts, prepend=0))  # runs of items of the same number of parts
    return (plan.mfma_row_blocks, plan.together, plan.decode_splits, tuple(zip(edges.tolist(), parts[edges].tolist())))


def attention_plan(ctx, nh: int, nkv: int, narrow_ok: bool = False, whole_keys: int = 0, together_ok: bool = False,
                   together_split_keys: int = 0, captured: bool = False) -> AttentionPlan:
    """The step's work items for heads of this geometry, made once a step and kept in
    ``ctx.plans``. ``narrow_ok``: the matrix-core kernel for portions also comes with two row
    blocks a workgroup (see ``ops.prefill_row_blocks_ok``). ``whole_keys``: up to this many keys of a single
    token stay with one workgroup (see ``whole_single_keys``). ``together_ok``: the caller can run portions and single
    tokens as one launch (see ``_share_the_card``), whose splits take ``together_split_keys`` keys at most (0: any).
    ``captured``: the plan is for all steps of the same ``captured_choices``, not for this one's portions alone."""
    # a batch of single tokens has no portions: one plan, whatever the kernel for portions offers
    narrow_ok = bool(narrow_ok) and any(q > 1 for q in ctx.h_q_lens)
    key = ("attention", nh, nkv, narrow_ok, whole_keys, together_ok, together_split_keys, captured)
    plan = ctx.plans.get(key)
    if plan is None:
        step = ctx
        if captured:
            step = SimpleNamespace(h_q_lens=ctx.h_q_lens, h_ctx_lens=_typical_lens(ctx.h_q_lens, ctx.h_ctx_lens),
                                   num_compute_units=ctx.num_compute_units, upload=ctx.upload)
        plan = ctx.plans[key] = _make_plan(step, nh, nkv, narrow_ok, whole_keys, together_ok, together_split_keys)
    return plan


def _split_keys(longest: int, splits: int) -> int:
    """Keys of each of ``splits`` fixed places that cover ``longest`` keys: a multiple of 32."""
    return 32 * -(-(-(-longest // splits)) // 32)


def _share_the_card(plan: AttentionPlan, room: int, base: int, longest: int, most_keys: int) -> None:
    """One launch for a step's portions and single tokens, where all workgroups of both are at work at once: ``room``
    compute units are left beside the portions' workgroups, a split of every single token takes ``base`` of them. The splits
    are then as many as fit, but not fewer than half of those that the single tokens alone would be cut into. Measured
    on both sides of that line, us a layer's attention as two launches / as one with the splits that fit (12 heads of 128 on
    2): 16 requests of 1500 keys (8 splits) beside 64 tokens 20.0 / 12.8 with 7, 320 tokens 22.6 / 16.0 with 6, 448 23.9 / 17.1
    with 5; below it 760 tokens 27.1 / 19.2 with 3, 900 28.8 / 20.6 with 2; 32 of 1500 (4) beside 320 26.7 / 18.1 with 3, 760
    30.8 / 17.0 with 1; 64 of 2000 (2) beside 320 42.7 / 33.6 with 1. So one launch is the faster one below the line as well:
    the line is cautious, not where the two meet. (A step of 15 requests of 1500 beside 300 tokens, 1.5B shape: 3.30 ms with
    8 splits behind the portions, 3.04 with 6 beside them.) A split of more than ``most_keys`` keys
    (of the ``longest`` context) has more pages than the launch takes: two launches then, whose splits are shorter."""
    splits = min(room // base, plan.decode_splits)
    if splits >= 1 and 2 * splits >= plan.decode_splits and not 0 < most_keys < _split_keys(longest, splits):
        plan.together, plan.decode_splits = True, splits


def whole_single_keys(head_dim: int) -> int:
    """Heads of up to 128 elements come with eight waves a workgroup, which take 512 keys in two turns: as
    long as the kernel that merges the parts of a request would take alone (us for one request, one part
    against two for 300 keys and three for 500: heads of 64 4.8 / 6.7 and 5.6 / 6.8; of 128, 7.0 / 7.9 and
    8.7 / 8.0)."""
    return 512 if head_dim <= 128 else 0


def _make_plan(ctx, nh: int, nkv: int, narrow_ok: bool, whole_keys: int = 0, together_ok: bool = False,
               together_split_keys: int = 0) -> AttentionPlan:
    group = nh // nkv
    gh_wide = min(group, 64)
    tokens_per_tile = 64 // gh_wide
    gh_single = min(group, 16)
    wide: list = []   # one array of items per portion
    mfma: list = []
    # Workgroups of four row blocks share each key among the most rows, but the one with the longest key range
    # decides the launch's time. Unless the key ranges are long, two row blocks are the faster way where their workgroups
    # are at most one for every compute unit (us, two row blocks / four: 1024 tokens of 16 heads of 64 on 8, 256
    # workgroups of two, 12.8 / 17.0); beyond, a second round of them costs their chain of first loads again, which pays
    # for key ranges of ten stages and more (1800 tokens of 12 heads of 128 on 2, 360 of two, 26.5 / 33.1; 2500 tokens, 500,
    # 40.4 / 43.4; 1000 tokens of 28 on 4, 448, 28.7 / 24.2; 640 of 32 on 8, 320, 22.1 / 18.3), while four would leave a
    # twentieth of the units idle. Groups of more than 32 heads, whose last chunk leaves rows idle: up to 1.5
    # workgroups of four a unit (6 % either way).
    tokens_of_four = 4 * 32 // min(group, 32)
    workgroups = sum(-(-q // tokens_of_four) for q in ctx.h_q_lens if q > 1) * nkv * -(-group // 32)
    short_ranges = portions_have_short_ranges(ctx.h_q_lens, ctx.h_ctx_lens)
    longest = max((c for q, c in zip(ctx.h_q_lens, ctx.h_ctx_lens) if q > 1), default=0)
    units = ctx.num_compute_units
    two = 2 * workgroups <= units or (workgroups < 1.5 * units if group > 32 else longest >= 1280 and workgroups < 0.95 * units)
    row_blocks = 2 if narrow_ok and short_ranges and two else 4
    tokens_per_mfma_item = row_blocks * 32 // min(group, 32)
    single: list[int] = []
    longest_single = 0

    def items_of(r: int, q_len: int, step: int, longest_first: bool) -> np.ndarray:
        """(request, first token, tokens, 0) for runs of ``step`` tokens of one portion."""
        tok0 = np.arange(0, q_len, step, dtype=np.int32)
        if longest_first:
            tok0 = tok0[::-1]
        out = np.zeros((tok0.size, 4), dtype=np.int32)
        out[:, 0] = r
        out[:, 1] = tok0
        out[:, 2] = np.minimum(step, q_len - tok0)
        return out.reshape(-1)

    for r, q_len in enumerate(ctx.h_q_lens):
        if q_len == 1:
            single += [r, 0, 1, 0]
            longest_single = max(longest_single, ctx.h_ctx_lens[r])
        else:
            wide.append(items_of(r, q_len, tokens_per_tile, False))
            # longest key ranges first: the last tokens of a portion have the most work
            mfma.append(items_of(r, q_len, tokens_per_mfma_item, True))
    wide = np.concatenate(wide) if wide else np.zeros(0, dtype=np.int32)
    mfma = np.concatenate(mfma) if mfma else np.zeros(0, dtype=np.int32)
    plan = AttentionPlan(gh_wide=gh_wide, gh_single=gh_single, mfma_row_blocks=row_blocks)
    mfma, plan.mfma_parts = _share_long_key_ranges(mfma.reshape(-1, 4), ctx, nkv * -(-group // 32))
    plan.n_wide, plan.n_single, plan.n_mfma = len(wide) // 4, len(single) // 4, len(mfma) // 4
    if plan.n_wide:
        # the 64-row kernel cuts every item's keys the same number of ways: as many as there are idle
        # compute units for, while the longest portion's keys give each part MIN_PART_KEYS
        spare = ctx.num_compute_units // (plan.n_wide * nkv * -(-group // gh_wide))
        most_keys = max(c for q, c in zip(ctx.h_q_lens, ctx.h_ctx_lens) if q > 1)
        plan.wide_splits = int(max(1, min(spare, most_keys // MIN_PART_KEYS, MAX_PARTS)))
    plan.chunks_single = -(-group // gh_single)
    if plan.n_single:
        # as many parts as still give every workgroup a compute unit of its own (64 requests of 1500 keys, heads of
        # 128 on 2 kv heads: 42 us with 2 parts, 47 with 4, 62 with 8)
        by_occupancy = ctx.num_compute_units // (plan.n_single * nkv * plan.chunks_single)
        plan.single_splits = 1 if longest_single <= min(F32_WHOLE_KEYS, whole_keys) else max(
            1, min(by_occupancy, longest_single // F32_PART_KEYS, 64))
        # decode kernel: a workgroup per (request, kv head, split); a split is at least 128 keys
        # (one 32-key tile for each of its four waves). As many splits as still give every
        # workgroup a compute unit of its own: one more and some units run a second round (24
        # requests of 2100 keys on 2 kv heads, kernel and merge: 19.2 us with 4 splits, 22.4 with 6;
        # 96 requests: 42.5 us with 1, 50.6 with 3). More than 64 splits never paid: one request
        # with 30000 keys takes 16 us with 64 to 128 splits and 19 us with 235.
        base = plan.n_single * nkv * -(-group // min(group, 16))
        plan.decode_splits = 1 if longest_single <= whole_keys else max(
            1, min(ctx.num_compute_units // base, longest_single // 128, 64))
        if together_ok and plan.n_mfma and plan.mfma_parts == 1:
            _share_the_card(plan, ctx.num_compute_units - plan.n_mfma * nkv * -(-group // 32), base, longest_single, together_split_keys)
        # fixed places for the splits: a workgroup then knows its pages before it knows the
        # request's length, which saves it a trip to memory
        plan.decode_split_keys = _split_keys(longest_single, plan.decode_splits)
        plan.decode_max_ctx = longest_single
        plan.single_identity = plan.n_single == len(ctx.h_q_lens)
    plan.wide_items, plan.single_items, plan.mfma_items = ctx.upload([wide, single, mfma])
    return plan


class PagedAttention(Part):
    compute_units = 256  # of the card that the part is bound to
    _choices = None      # what ``captured_choices`` takes beside the step, the same for every step

    @property
    def graph_safe(self) -> bool:
        """A fixed sequence of launches if the position encoding is one too."""
        return bool(getattr(self.position, "graph_safe", False))

    def __init__(self, spec: AttentionSpec) -> None:
        self.spec = spec
        self.position = build_part(spec.position) if spec.position is not None else NoPosition()
        self.q_width = spec.num_heads * spec.head_dim
        self.kv_width = spec.num_kv_heads * spec.head_dim

    def param_specs(self):
        s = self.spec
        width = self.q_width + 2 * self.kv_width
        specs = {
            "qkv_weight": ParamSpec((width, s.hidden_size)),
            "out_weight": ParamSpec((s.hidden_size, self.q_width)),
        }
        if s.qkv_bias:
            specs["qkv_bias"] = ParamSpec((width,), precision="stored", init=("normal", 0.02))
        if s.out_bias:
            specs["out_bias"] = ParamSpec((s.hidden_size,), precision="compute", init=("normal", 0.02))
        return specs

    def cache_need(self):
        return KVPagesSpec(self.spec.num_kv_heads, self.spec.head_dim, self.spec.window)

    def kernel_libraries(self) -> list:
        return [("attention", int(self.spec.head_dim))]

    def _plan(self, ctx, dtype) -> AttentionPlan:
        hd = self.spec.head_dim
        narrow_ok = ops.prefill_attention_supported(hd, dtype) and ops.prefill_row_blocks_ok(hd, 2)
        together_keys = ops.together_attention_split_keys(hd, dtype, ctx.block_size)
        return attention_plan(ctx, self.spec.num_heads, self.spec.num_kv_heads, narrow_ok=narrow_ok, whole_keys=whole_single_keys(hd),
                              together_ok=together_keys > 0, together_split_keys=together_keys, captured=ctx.captured)

    def prepare(self, ctx) -> None:
        """The step's work items, before ``forward`` (a captured step must not make them)."""
        self._plan(ctx, self.dtype)

    def shape_class(self, q_lens, ctx_lens):
        """Portions behind few and many cached keys run other workgroups, cut their keys into other numbers of parts and
        leave the single tokens another share of the card: what of that the plan of a captured step decides."""
        if not any(q > 1 for q in q_lens):
            return "single tokens"
        if self._choices is None:
            nh, nkv, hd = self.spec.num_heads, self.spec.num_kv_heads, self.spec.head_dim
            mfma = ops.prefill_attention_supported(hd, self.dtype)
            self._choices = (nh, nkv, self.compute_units, mfma, mfma and ops.prefill_row_blocks_ok(hd, 2), whole_single_keys(hd),
                             ops.together_attention_supported(hd, self.dtype))
        return captured_choices(tuple(q_lens), tuple(ctx_lens), *self._choices)

    def bind(self, params, device, dtype) -> None:
        self.qkv_weight = params["qkv_weight"]
        self.qkv_bias = params.get("qkv_bias")
        self.out_weight = params["out_weight"]
        self.out_bias = params.get("out_bias")
        self.dtype = dtype
        self._choices = None
        if torch.device(device).type == "cuda":
            self.compute_units = ops._compute_units(device)
        self.position.bind({}, device, dtype)

    def takes_begun_norm(self, n_tokens: int, cache: EntryCache) -> bool:
        """May ``forward``'s input be an ``ops.BegunNorm`` of that many rows?"""
        takes = getattr(self.position, "takes_begun_norm", None)
        return takes is not None and own_method(self, PagedAttention) and cache.writes and takes(n_tokens, self.qkv_weight, self.spec.head_dim)

    def joins_stream(self, n_tokens: int, norm) -> bool:
        """Does ``forward_joined`` add that many rows to the stream and begin ``norm``?"""
        return own_method(self, PagedAttention) and self.out_bias is None and ops.linear_join_pays(n_tokens, self.out_weight, norm.weight)

    def forward_joined(self, x, ctx, cache: EntryCache, resid, norm) -> "ops.BegunNorm":
        """``forward``, its output added to ``resid`` and ``norm`` of that begun."""
        return ops.linear_join(self._before_output(x, ctx, cache), self.out_weight, resid, norm.weight, norm.spec.eps)

    def forward(self, x: torch.Tensor, ctx, cache: EntryCache) -> torch.Tensor:
        return self.output(self._before_output(x, ctx, cache), ctx)

    def takes_rows(self) -> bool:
        """Can ``forward_rows`` make chosen rows of the output alone?"""
        return own_method(self, PagedAttention)

    def forward_rows(self, x, ctx, cache: EntryCache, rows, *others) -> tuple:
        """``forward``'s ``rows``, the cache being left as by all of them, and the same rows of ``others``."""
        out, *others = ops.take_rows(rows, self._before_output(x, ctx, cache), *others)
        return self.output(out, ctx), others

    def output(self, out: torch.Tensor, ctx):
        return ops.linear(out, self.out_weight, self.out_bias, partial_ok=True, policy=getattr(ctx, "products", None),
                          portions_partial_ok=getattr(ctx, "reader_adds_sums", False))

    def _before_output(self, x, ctx, cache: EntryCache) -> torch.Tensor:
        """All but the product with ``out_weight``, [T, heads * head_dim]."""
        s = self.spec
        nh, nkv, hd = s.num_heads, s.num_kv_heads, s.head_dim
        policy = getattr(ctx, "products", None)
        fused = getattr(self.position, "project_rotate_store", None) if cache.writes else None
        qkv = None
        if fused is not None:
            qkv = fused(x, self.qkv_weight, self.qkv_bias, ctx.positions, ctx.slots[cache.group], nh, nkv, hd, cache.k, cache.v)
        rows = getattr(self.position, "project_rotate_store_rows", None) if cache.writes and qkv is None else None
        if rows is not None:
            qkv = rows(x, self.qkv_weight, self.qkv_bias, ctx, ctx.slots[cache.group], nh, nkv, hd, cache.k, cache.v)
        if qkv is not None:
            pass  # q only, [T, nh * hd]: keys and values are in the cache already
        elif cache.writes:
            qkv = ops.linear(x, self.qkv_weight, policy=policy)
            self.position.rotate_and_store(
                qkv, self.qkv_bias, ctx.positions, ctx.slots[cache.group], nh, nkv, hd, cache.k, cache.v
            )
        else:
            # the keys and values of another entry are read: only queries are made here
            qkv = ops.linear(x, self.qkv_weight[: self.q_width], policy=policy)
            bias = self.qkv_bias[: self.q_width] if self.qkv_bias is not None else None
            self.position.rotate_and_store(qkv, bias, ctx.positions, None, nh, 0, hd, None, None)
        return self.attend(qkv, ctx, cache)

    def attend(self, q: torch.Tensor, ctx, cache: EntryCache) -> torch.Tensor:
        """Attention of the step's rotated queries (the first ``num_heads * head_dim`` columns of
        ``q``, one row a token) over the keys and values that ``cache`` holds, [T, heads * head_dim]:
        the kernels and work items that the step's plan names, and nothing else of the layer."""
        s = self.spec
        nh, nkv, hd = s.num_heads, s.num_kv_heads, s.head_dim
        T = q.shape[0]
        out = torch.empty((T, self.q_width), dtype=q.dtype, device=q.device)
        mfma = ops.prefill_attention_supported(hd, q.dtype)
        plan = self._plan(ctx, q.dtype)
        common = dict(
            q=q, q_stride=q.shape[1], out=out, k_cache=cache.k, v_cache=cache.v,
            block_tables=ctx.block_tables[cache.group], ctx_lens=ctx.ctx_lens, cu_q=ctx.cu_q,
            nh=nh, nkv=nkv, hd=hd, block_size=cache.block_size, window=s.window or 0,
            scale=s.scale, n_tokens=T, n_requests=ctx.num_requests,
        )
        if plan.together:
            workspace = None
            if plan.decode_splits > 1:
                need = ops.decode_attention_workspace_floats(hd, plan.n_single, nh, nkv, plan.decode_splits)
                workspace = torch.empty(need, dtype=torch.float32, device=q.device)
            ops.attention_together(portions=plan.mfma_items, n_portions=plan.n_mfma, row_blocks=plan.mfma_row_blocks,
                                   singles=plan.single_items, n_singles=plan.n_single, n_splits=plan.decode_splits,
                                   split_keys=plan.decode_split_keys, max_ctx=plan.decode_max_ctx, workspace=workspace, **common)
            return out
        if plan.n_wide and mfma:
            workspace = None
            if plan.mfma_parts > 1:
                need = ops.prefill_attention_workspace_floats(hd, plan.n_mfma, nh, nkv, plan.mfma_row_blocks)
                workspace = torch.empty(need, dtype=torch.float32, device=q.device)
            ops.attention_prefill(items=plan.mfma_items, n_items=plan.n_mfma, row_blocks=plan.mfma_row_blocks,
                                  workspace=workspace, **common)
        elif plan.n_wide:
            workspace = None
            if plan.wide_splits > 1:
                need = ops.attention_workspace_floats(hd, 64, plan.n_wide, nkv, -(-(nh // nkv) // plan.gh_wide), plan.wide_splits)
                workspace = torch.empty(need, dtype=torch.float32, device=q.device)
            ops.attention(items=plan.wide_items, n_items=plan.n_wide, rows=64, gh=plan.gh_wide,
                          n_splits=plan.wide_splits, workspace=workspace, **common)
        if plan.n_single and ops.decode_attention_supported(hd, q.dtype):
            workspace = None
            if plan.decode_splits > 1:
                need = ops.decode_attention_workspace_floats(hd, plan.n_single, nh, nkv, plan.decode_splits)
                workspace = torch.empty(need, dtype=torch.float32, device=q.device)
            ops.attention_decode(items=plan.single_items, n_items=plan.n_single, n_splits=plan.decode_splits,
                                 workspace=workspace, identity=plan.single_identity,
                                 split_keys=plan.decode_split_keys, max_ctx=plan.decode_max_ctx, **common)
        elif plan.n_single:
            workspace = None
            if plan.single_splits > 1:
                need = ops.attention_workspace_floats(hd, 16, plan.n_single, nkv, plan.chunks_single, plan.single_splits)
                workspace = torch.empty(need, dtype=torch.float32, device=q.device)
            ops.attention(items=plan.single_items, n_items=plan.n_single, rows=16, gh=plan.gh_single,
                          n_splits=plan.single_splits, workspace=workspace, **common)
        return out
