"""Lane compaction ranked by progress: bit-identical to the uncompacted loop,
whatever the estimates say."""

import numpy as np
import pytest

from palladium_amd.workloads import bs3_inputs, bs3_vdp_call
from rank_cases import ranked_call, steps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["spread", "alike", "stuck"])
@pytest.mark.parametrize("n", [1000, 4096, 65_537, 131_072, 140_001])
def test_ranked_equals_the_plain_loop(monkeypatch, n, kind):
    print(f"[rank] n={n} {kind}", flush=True)
    r = steps(kind, n)
    call = ranked_call(n)
    assert "ph_rank_cut" in call.bound(r).hip_source
    got = call(r)
    monkeypatch.setenv("PALLADIUM_WHILE_COMPACTION", "0")
    plain = ranked_call(n)
    assert "ph_rank_cut" not in plain.bound(r).hip_source
    for g, w in zip(got, plain(r)):
        np.testing.assert_array_equal(np.asarray(g).view(np.int32), np.asarray(w).view(np.int32))


@pytest.mark.parametrize("mode", ["reproducible", "safe"])
def test_ranked_bs3_equals_the_plain_loop(monkeypatch, mode):
    n = 131_200
    args = bs3_inputs(n)
    got = bs3_vdp_call(n, math_mode=mode)(*args)
    monkeypatch.setenv("PALLADIUM_WHILE_COMPACTION", "0")
    for g, w in zip(got, bs3_vdp_call(n, math_mode=mode)(*args)):
        np.testing.assert_array_equal(g, w)
