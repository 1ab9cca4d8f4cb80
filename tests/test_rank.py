"""Which loops lane compaction ranks by progress (tests/test_gpu_rank.py runs them)."""

import numpy as np
import pytest

from palladium_amd.workloads import bs3_vdp_call
from rank_cases import ranked_call


def _ranked(call, n, args=1):
    return "ph_rank_cut" in call.bound(*[np.ones(n, np.float32)] * args).hip_source


@pytest.mark.parametrize("kwargs, want", [
    ({}, True), ({"test": "le"}, True), ({"test": "gt"}, True), ({"start": -1.0}, True),
    ({"test": "int"}, False),  # no float carry with a bound
    ({"start": None}, False),  # starts at data
    ({"ops": 20}, False),  # a short body
    ({"mode": "fast"}, False),
])
def test_ranked_loops(kwargs, want):
    assert _ranked(ranked_call(65_537, **kwargs), 65_537) is want


@pytest.mark.parametrize("n, mode, want", [(4096, "safe", True), (65_536, "safe", False), (65_537, "safe", True), (131_073, "reproducible", True),
                                           (262_144, "fast", False)])
def test_ranked_bs3(n, mode, want):
    assert _ranked(bs3_vdp_call(n, math_mode=mode), n, 3) is want
