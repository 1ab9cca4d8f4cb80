"""Compacted loops run on the common paths of their checked functions and
turn to the full ones where a lane needs them: bit for bit the plain loop."""

import numpy as np
import pytest

from checked_cases import checked_call, checked_data


@pytest.mark.parametrize("kind, mode, want", [
    ("div", "reproducible", True), ("explog", "reproducible", True), ("pow", "safe", True),
    ("div", "safe", False),  # the compiler's division: no branch
    ("branch", "reproducible", False),  # branches of its own
    ("div", "fast", False),
])
def test_which_loops_turn(kind, mode, want):
    src = checked_call(4096, kind, mode).bound(*checked_data(4096)).hip_source
    assert ("bool _odd" in src) is want


@pytest.mark.gpu
@pytest.mark.parametrize("kind, mode", [("div", "reproducible"), ("explog", "reproducible"), ("pow", "reproducible"),
                                        ("pow", "safe"), ("branch", "reproducible")])
@pytest.mark.parametrize("n, regular", [(1000, False), (1000, True), (70_001, False)])
def test_odd_operands_match_the_plain_loop(monkeypatch, kind, mode, n, regular):
    print(f"[checked] {kind} {mode} n={n} regular={regular}", flush=True)
    args = checked_data(n, regular)
    got = checked_call(n, kind, mode)(*args)
    monkeypatch.setenv("PALLADIUM_WHILE_COMPACTION", "0")
    plain = checked_call(n, kind, mode)
    assert "bool _odd" not in plain.bound(*args).hip_source
    for g, w in zip(got, plain(*args)):
        np.testing.assert_array_equal(np.asarray(g).view(np.int32), np.asarray(w).view(np.int32))
