"""The strip height a Gray-Scott register pass takes for a grid: every row is
stored once whatever the height, explicit heights are kept, and the fields
equal the oracle's bit for bit at sizes that take short strips."""

import numpy as np
import pytest

import oracle
from palladium_amd import stencil
from palladium_amd.workloads import GS_CFG, gray_scott_initial
from test_stencil import _register_pass


@pytest.mark.parametrize("n", [76, 100, 333, 700, 1024, 2048, 4096, 8192])
@pytest.mark.parametrize("k", [1, 4, 6])
def test_height_is_in_range_and_costs_no_more_than_the_tallest(n, k):
    r = stencil.strip_height(n, k)
    assert 2 <= r <= stencil.DEFAULT_ROWS and r + 2 * k <= n

    def cost(h):
        waves = stencil.register_geometry(n, k, h)[1] * 4
        return -(-(h + 2 * k) // 4) * 4 * (-(-waves // stencil.SIMDS) + 1.3)

    assert cost(r) <= cost(stencil.DEFAULT_ROWS)


def test_default_adapts_and_explicit_heights_stay():
    assert stencil.RegisterGrayScott(200)._rows == {6: 2, 1: 2}
    assert stencil.RegisterGrayScott(4096)._rows == {6: 64, 1: 64}
    assert stencil.RegisterGrayScott(512, rows=40)._rows == {6: 40, 1: 40}
    assert stencil.RegisterGrayScott(512, rows=64)._rows == {6: 64, 1: 64}
    assert stencil.RegisterGrayScott(512, cols=2)._rows == {6: 64, 1: 64}
    with pytest.raises(ValueError, match="too small"):
        stencil.RegisterGrayScott(75)


@pytest.mark.parametrize("n,rows", [(78, 2), (81, 6)])
def test_short_strips_restated_match_oracle(n, rows):
    u0, v0 = gray_scott_initial(n)
    u, v = _register_pass(u0, v0, 6, rows, 4, GS_CFG)
    wu, wv = oracle.gray_scott(u0, v0, GS_CFG, 6)
    np.testing.assert_array_equal(u, wu)
    np.testing.assert_array_equal(v, wv)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [76, 200, 515, 700, 1030])
def test_short_strips_bit_exact_on_the_gpu(n):
    print(f"[stencil] adaptive strips n={n}", flush=True)
    u0, v0 = gray_scott_initial(n)
    f = stencil.RegisterGrayScott(n, math_mode="safe")
    u, v, _ = stencil.gray_scott_fused_run(f, u0, v0, 20)
    wu, wv = oracle.gray_scott(u0, v0, GS_CFG, 20)
    np.testing.assert_array_equal(u, wu)
    np.testing.assert_array_equal(v, wv)
