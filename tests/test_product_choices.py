"""What a tuning start-up measured for the package's own kernels is kept in a file and read again."""

import json

import pytest
import torch

from clockwork_amd import ops


def test_choices_written_and_read_back(tmp_path):
    path = str(tmp_path / "choices.json")
    first = ops.ProductPolicy()
    first.k_split_choices[(1536, 8960)] = 6
    first.wide_partial_choices[(1536, 8960)] = 4
    first.swiglu_choices[(17920, 1536)] = False
    first.product_choices[(3584, 1024, True)] = True
    first.write_choices(path)

    later = ops.ProductPolicy()
    later.k_split_choices[(1536, 8960)] = 3          # what this process measured itself stays
    assert later.read_choices(path) == 4
    # remembered, not in use: another model's shapes never show among this engine's choices
    assert later.k_split_choices == {(1536, 8960): 3} and not later.wide_partial_choices and not later.swiglu_choices
    assert later.recall("k_split_choices", (1536, 8960)) is None          # its own choice stands
    assert later.recall("wide_partial_choices", (1536, 8960)) == 4
    assert later.recall("wide_partial_choices", (1536, 8960)) is None     # in use now: nothing left to recall
    assert later.recall("swiglu_choices", (17920, 1536)) is False
    assert later.recall("swiglu_choices", (9, 9)) is None
    assert later.wide_partial_choices == {(1536, 8960): 4} and later.swiglu_choices == {(17920, 1536): False}
    assert not later.product_choices and not ops.DEFAULT_POLICY.k_split_choices
    # what it leaves behind: everything remembered, its own choices on top
    again = str(tmp_path / "again.json")
    later.write_choices(again)
    third = ops.ProductPolicy()
    assert third.read_choices(again) == 4
    assert third.recall("k_split_choices", (1536, 8960)) == 3
    assert third.recall("product_choices", (3584, 1024, True)) is True


def test_choices_of_another_build_or_a_broken_file_are_passed_over(tmp_path):
    path = tmp_path / "choices.json"
    policy = ops.ProductPolicy()
    assert policy.read_choices(str(path)) == 0                      # no file
    path.write_text("{ not json")
    assert policy.read_choices(str(path)) == 0
    record = {"made_for": ["another card", 1, 2, "0.0", "gemm-0.so", "gemm_tile-0.so", "core-0.so"],
              "k_split_choices": [[[1536, 8960], 6]]}
    path.write_text(json.dumps(record))
    assert policy.read_choices(str(path)) == 0 and policy.recall("k_split_choices", (1536, 8960)) is None
    record["made_for"] = ops._choices_made_for()
    path.write_text(json.dumps(record))
    assert policy.read_choices(str(path)) == 1 and policy.recall("k_split_choices", (1536, 8960)) == 6
    assert policy.k_split_choices == {(1536, 8960): 6}
    # a folder that cannot be written: nothing is kept, nothing is raised
    policy.write_choices(str(tmp_path / "missing" / "choices.json"))


def test_choices_file_follows_the_environment(monkeypatch, tmp_path):
    monkeypatch.setenv("CLOCKWORK_AMD_CHOICES_FILE", str(tmp_path / "c.json"))
    assert ops.choices_file() == str(tmp_path / "c.json")
    monkeypatch.delenv("CLOCKWORK_AMD_CHOICES_FILE")
    assert "clockwork_amd_choices_" in ops.choices_file()


def test_the_card_is_known_by_more_than_its_name(monkeypatch):
    """Under a profiler the card's marketing name comes back empty: what identifies it to the
    choices file is its architecture, its compute units and its memory, and another card has
    another file."""
    import types

    def card(arch, units):
        return types.SimpleNamespace(name="", gcnArchName=arch, multi_processor_count=units, total_memory=1 << 38)

    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda d: card("gfx950:sramecc+:xnack-", 256))
    made_for, path = ops._choices_made_for(), ops.choices_file()
    assert made_for[:3] == ["gfx950:sramecc+:xnack-", 256, 1 << 38]
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda d: card("gfx950:sramecc+:xnack-", 128))
    assert ops._choices_made_for() != made_for and ops.choices_file() != path


@pytest.mark.parametrize("limit", [0.0, 7.0, ops.RELU_GATE, ops.GELU_GATE])
def test_a_gated_product_is_timed_and_kept_with_its_own_activation(monkeypatch, tmp_path, limit):
    ran = []
    monkeypatch.setattr(ops, "_timed_us", lambda fn: fn() or 1.0)
    monkeypatch.setattr(ops, "_library_product", lambda *a: ran.append("product"))
    monkeypatch.setattr(ops, "silu_mul", lambda gate_up, out, limit=0.0: ran.append(("gate", limit)))
    monkeypatch.setattr(ops, "gelu_tanh_mul", lambda gate_up, out: ran.append(("gate", ops.GELU_GATE)))
    monkeypatch.setattr(ops, "linear_tiled", lambda *a, limit=0.0, **k: ran.append(("own", limit)))
    assert ops._measure_swiglu(None, None, None, limit)
    assert ran == ["product", ("gate", limit), ("own", limit)]
    # another activation's choice for the same sizes is not taken, also behind a file
    policy, path = ops.ProductPolicy(), str(tmp_path / "choices.json")
    policy.swiglu_choices[ops._swiglu_key(17920, 1536, limit)] = False
    policy.write_choices(path)
    later = ops.ProductPolicy()
    assert later.read_choices(path) == 1
    for other in (0.0, 7.0, ops.RELU_GATE, ops.GELU_GATE):
        assert (later.recall("swiglu_choices", ops._swiglu_key(17920, 1536, other)) is False) == (other == limit)


def test_the_tiles_between_leave_a_product_that_was_timed_to_the_library(monkeypatch, tmp_path):
    """A tuning start-up times the rule's kernel against the library's tuned product, for the rows that it runs with;
    the faster one stays, also behind a file, and other numbers of rows follow the rule."""
    timed = []
    monkeypatch.setattr(ops, "_compute_units", lambda device: 256)
    monkeypatch.setattr(ops, "_measure_mid", lambda mode, choice, x, weight, bias, limit: timed.append((mode, x.shape[0], limit)) or False)
    rows = {m: torch.zeros(m, 896, dtype=torch.bfloat16) for m in (128, 160)}
    weight, path = torch.zeros(1152, 896, dtype=torch.bfloat16), str(tmp_path / "choices.json")
    policy = ops.ProductPolicy()
    by_rule = ops._mid_choice(0, rows[128], weight, policy)
    assert by_rule and not timed
    policy.tuning = True
    for _ in range(2):
        assert ops._mid_choice(0, rows[128], weight, policy) == 0
    assert ops._mid_choice(2, rows[128], weight, policy, limit=ops.GELU_GATE) == 0
    assert timed == [(0, 128, 0.0), (2, 128, ops.GELU_GATE)]
    policy.tuning = False
    assert ops._mid_choice(0, rows[128], weight, policy) == 0 and ops._mid_choice(0, rows[160], weight, policy) == by_rule
    assert ops._mid_choice(2, rows[128], weight, policy) != 0     # another activation: not timed
    policy.write_choices(path)
    later = ops.ProductPolicy()
    assert later.read_choices(path) == 2 and ops._mid_choice(0, rows[128], weight, later) == by_rule   # (not in use before it asks)
    later.tuning = True
    assert ops._mid_choice(0, rows[128], weight, later) == 0 and len(timed) == 2


def test_runs_of_k_that_a_start_up_timed_come_before_the_rules_tiles(monkeypatch):
    """A long portion's product with a timed (N, K): the timed runs, or what the rule names where they were not the fastest;
    and they are timed against that as well as against the library."""
    M, N, K = 1024, 1536, 8960
    x, w = torch.zeros(M, K, dtype=torch.bfloat16), torch.zeros(N, K, dtype=torch.bfloat16)
    costs = {"library": 50.0, "tiles": 40.0}
    monkeypatch.setattr(ops, "_gpu", lambda *a: None)
    monkeypatch.setattr(ops, "_compute_units", lambda device: 256)
    monkeypatch.setattr(ops, "_library_product", lambda *a: "library")
    monkeypatch.setattr(ops, "linear_mid", lambda *a, **k: "tiles")
    monkeypatch.setattr(ops, "linear_wide_partial", lambda x, w, runs: runs)
    monkeypatch.setattr(ops, "add_rmsnorm", lambda resid, y, *a, **k: y)
    monkeypatch.setattr(ops, "_timed_us", lambda fn: costs.get(fn(), 45.0))
    run = lambda policy: ops.linear(x, w, partial_ok=True, portions_partial_ok=True, policy=policy)  # noqa: E731
    policy = ops.ProductPolicy()
    assert run(policy) == "tiles"
    policy.wide_partial_choices[(N, K)] = 3
    assert run(policy) == 3
    policy.wide_partial_choices[(N, K)] = 0
    assert run(policy) == "tiles"
    for four, want in ((45.0, "tiles"), (39.5, "tiles"), (30.0, 4)):
        costs[4] = four
        policy = ops.ProductPolicy()
        policy.tuning = True
        assert run(policy) == want
        policy.tuning = False
        assert run(policy) == want and policy.wide_partial_choices[(N, K)] == (4 if want == 4 else 0)
