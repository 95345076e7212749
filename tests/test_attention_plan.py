"""The attention part's planning of work items, on the CPU (no kernel runs)."""

import numpy as np
import pytest
import torch

from clockwork_amd import ops
from clockwork_amd.parts.attention import MAX_PARTS, MIN_PART_KEYS, PagedAttention, _share_long_key_ranges, attention_plan, portions_have_short_ranges, typical_start
from clockwork_amd.parts.specs import AttentionSpec


class _Step:
    def __init__(self, q_lens, ctx_lens, num_compute_units=256):
        self.h_q_lens, self.h_ctx_lens, self.num_compute_units = list(q_lens), list(ctx_lens), num_compute_units
        self.block_size, self.captured, self.plans, self.upload = 16, False, {}, lambda arrays: [np.asarray(a, dtype=np.int32) for a in arrays]


def _items(q_lens, tokens_per_item):
    rows = []
    for r, q in enumerate(q_lens):
        for tok0 in range(0, q, tokens_per_item):
            rows.append((r, tok0, min(tokens_per_item, q - tok0), 0))
    return np.asarray(rows, dtype=np.int32).reshape(-1, 4)


def _unpack(flat):
    items = flat.reshape(-1, 4)
    return items, items[:, 3] & 255, (items[:, 3] >> 8) & 255


def test_a_launch_that_fills_the_card_is_left_alone():
    step = _Step([2048], [2048])
    items = _items(step.h_q_lens, 10)  # 205 items on 2 key/value heads: 410 workgroups
    flat, most = _share_long_key_ranges(items, step, workgroups_per_item=2)
    assert most == 1 and (flat.reshape(-1, 4) == items).all()


def test_a_short_portion_behind_a_long_prefix_is_cut_into_parts():
    step = _Step([200], [8392])
    items = _items(step.h_q_lens, 20)  # 10 items on 2 heads: 20 workgroups for 256 compute units
    flat, most = _share_long_key_ranges(items, step, workgroups_per_item=2)
    out, part, parts = _unpack(flat)
    assert most == 12 and len(out) == 120 and (parts == 12).all()
    for i in range(10):  # the parts of an item follow one another and keep its first three fields
        block = out[12 * i : 12 * i + 12]
        assert (block[:, :3] == items[i, :3]).all() and list(part[12 * i : 12 * i + 12]) == list(range(12))


def test_parts_are_bounded_by_the_keys_and_by_the_list_format():
    step = _Step([16], [30016])
    flat, most = _share_long_key_ranges(_items([16], 10), step, workgroups_per_item=2)
    assert most == MAX_PARTS and MAX_PARTS <= 255  # eight bits in the item's fourth field
    step = _Step([16], [600])  # 600 keys: two parts of at least MIN_PART_KEYS
    flat, most = _share_long_key_ranges(_items([16], 10), step, workgroups_per_item=2)
    assert most == 600 // MIN_PART_KEYS == 2
    step = _Step([100, 1, 1], [100, 500, 700])  # few workgroups, but of few keys: nothing to share
    flat, most = _share_long_key_ranges(_items([100], 10), step, workgroups_per_item=2)
    assert most == 1
    flat, most = _share_long_key_ranges(np.zeros((0, 4), dtype=np.int32), step, workgroups_per_item=2)
    assert most == 1 and flat.size == 0


def test_items_of_different_lengths_get_parts_of_their_own():
    step = _Step([10, 10], [300, 5000])  # two portions: one behind 290 keys, one behind 4990
    flat, most = _share_long_key_ranges(_items(step.h_q_lens, 10), step, workgroups_per_item=1)
    out, part, parts = _unpack(flat)
    assert list(parts[out[:, 0] == 0]) == [1] and most == 5000 // MIN_PART_KEYS
    assert (parts[out[:, 0] == 1] == most).all() and (out[:, 0] == 1).sum() == most


def test_short_and_long_key_ranges():
    assert portions_have_short_ranges([2048], [2048])
    assert not portions_have_short_ranges([2048], [8192])
    assert not portions_have_short_ranges([1, 1], [500, 600])  # no portion at all


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("block_size", [1, 3, 16])
@pytest.mark.parametrize("requests,keys", [(60, 50000), (60, 32736), (60, 32737), (16, 300000), (15, 1500)])
def test_one_launch_is_planned_only_where_it_takes_a_splits_pages(hd, block_size, requests, keys):
    """60 requests of 50,000 keys in pages of one key beside a portion of 64 tokens: a split of the one launch would have more
    pages than it takes, while two launches take the step (with splits of their own length)."""
    most = ops.together_attention_split_keys(hd, torch.bfloat16, block_size)
    assert most % 32 == 0 and most // block_size >= 32000
    how = dict(narrow_ok=True, whole_keys=512)
    plan = attention_plan(_Step([1] * requests + [64], [keys] * requests + [64]), 12, 2, together_ok=True, together_split_keys=most, **how)
    apart = attention_plan(_Step([1] * requests + [64], [keys] * requests + [64]), 12, 2, **how)
    free = attention_plan(_Step([1] * requests + [64], [keys] * requests + [64]), 12, 2, together_ok=True, **how)
    if plan.together:
        assert plan.decode_split_keys <= most and plan.decode_splits == free.decode_splits
    else:
        assert (plan.decode_splits, plan.decode_split_keys) == (apart.decode_splits, apart.decode_split_keys) and free.decode_split_keys > most
    assert plan.together == (free.decode_split_keys <= most) and plan.decode_split_keys * plan.decode_splits >= keys


def test_heads_without_the_one_launch_have_no_keys_for_it():
    assert ops.together_attention_split_keys(256, torch.bfloat16, 16) == 0 == ops.together_attention_split_keys(48, torch.bfloat16, 16)
    assert ops.together_attention_split_keys(128, torch.float32, 16) == 0 == ops.together_attention_split_keys(128, torch.bfloat16, 0)


def _captured_plan(part, q_lens, ctx_lens):
    step = _Step(q_lens, ctx_lens)
    step.captured = True
    plan = part._plan(step, part.dtype)
    if ops.prefill_attention_supported(part.spec.head_dim, part.dtype):  # the fields that this type's kernels read
        return (plan.n_mfma, plan.mfma_row_blocks, plan.mfma_parts, plan.mfma_items.tobytes(), plan.n_single, plan.single_items.tobytes(),
                plan.decode_splits, plan.decode_split_keys, plan.decode_max_ctx, plan.single_identity, plan.together)
    return (plan.n_wide, plan.wide_splits, plan.wide_items.tobytes(), plan.n_single, plan.single_items.tobytes(), plan.single_splits)


@pytest.mark.parametrize("nh,nkv,hd,dtype", [(12, 2, 128, torch.bfloat16), (14, 2, 64, torch.bfloat16), (28, 4, 128, torch.bfloat16),
                                             (40, 1, 64, torch.bfloat16), (16, 4, 256, torch.bfloat16), (14, 2, 64, torch.float32)])
def test_captured_steps_of_one_class_have_one_plan(nh, nkv, hd, dtype):
    """A captured step is kept under its token counts, the decoding requests' context and its class, and serves whatever
    portion comes under the same: where the first one began must not decide how the others run. Portions behind 0 to 12,000
    cached keys, alone and beside single tokens: one plan for each class, and few classes."""
    part = PagedAttention(AttentionSpec(hidden_size=nh * hd, num_heads=nh, num_kv_heads=nkv, head_dim=hd, qkv_bias=False, out_bias=False,
                                        scale=hd ** -0.5))
    part.dtype = dtype
    starts = [*range(0, 1200, 40), *range(1200, 4000, 190), *range(4000, 12000, 900)]
    for decoders, capacity in ((0, 0), (1, 512), (16, 2048), (64, 1024)):
        for size in (12, 60, 160, 320, 512, 1000, 2048):
            plans = {}
            for start in starts:
                q_lens, ctx_lens = [1] * decoders + [size], [capacity] * decoders + [start + size]
                plans.setdefault(part.shape_class(q_lens, ctx_lens), set()).add(_captured_plan(part, q_lens, ctx_lens))
            assert all(len(of) == 1 for of in plans.values()), (decoders, size, {k: len(v) for k, v in plans.items()})
            assert len(plans) <= 6, (decoders, size, len(plans))


def test_portions_of_a_captured_step_begin_near_those_that_it_serves():
    assert [typical_start(s) for s in (0, 1, 300, 362, 363, 512, 724, 725, 7000, 10000)] == [0, 0, 0, 0, 512, 512, 512, 1024, 8192, 8192]
    assert all(s / 1.42 < typical_start(s) < 1.42 * s for s in range(363, 40000, 77))
