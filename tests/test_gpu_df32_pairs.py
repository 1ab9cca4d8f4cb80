"""df32 RK4 LV with two lanes per trajectory (small ensembles) and one: both
sides of the line between them, the smallest ensembles and the edges of a
workgroup, bit for bit the oracle's words."""

import numpy as np
import pytest

import oracle
from palladium_amd import df32
from palladium_amd.workloads import lv_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 31, 127, 128, 129, 255, 257, 5000, df32.PAIR_MAX, df32.PAIR_MAX + 1])
def test_bit_exact_vs_oracle(n):
    print(f"[df32] n={n}", flush=True)
    args = lv_inputs(n, n)
    steps = 120 if n < 10_000 else 20
    for g, w in zip(df32.lv_rk4_df32(*args, 0.01, steps), oracle.lv_rk4_df32(*args, 0.01, steps)):
        np.testing.assert_array_equal(g, w)


def test_zeros_and_no_steps():
    """A state at zero keeps its zero words; no steps returns the inputs."""
    x0, y0, a, b, c, d = (v.copy() for v in lv_inputs(300, 3))
    x0[::3] = 0.0
    y0[::5] = 0.0
    for steps in (0, 50):
        got = df32.lv_rk4_df32(x0, y0, a, b, c, d, 0.01, steps)
        for g, w in zip(got, oracle.lv_rk4_df32(x0, y0, a, b, c, d, 0.01, steps)):
            np.testing.assert_array_equal(g, w)
