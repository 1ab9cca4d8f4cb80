"""Compacted loops whose bodies divide, take logs, exponentials and powers, on
operands that leave those functions' common paths now and then."""

import numpy as np

import palladium_amd as pa
from palladium_amd.frontend import jnp, lax, pl


def checked_call(n, kind, mode):
    def step(x, k):
        if kind == "div":  # a zero, subnormal, huge or NaN divisor on some trips
            return 1.0 / x + 1.0 / (x - 3.0)
        if kind == "explog":  # exp overflows, log meets zero and negative numbers
            return jnp.exp(x * 0.25) - jnp.log(x)
        if kind == "pow":
            return jnp.power(x, 0.7) + jnp.power(jnp.abs(x), -0.3)
        return lax.cond(k > 3, lambda v: 1.0 / v, lambda v: 2.0 / v, x) + 1.0 / (x + 1.0)  # "branch"

    def kernel(x_ref, trips_ref, o_ref, c_ref):
        x0, trips = x_ref[0], trips_ref[0]

        def body(s):
            x, acc, k = s
            return jnp.where(k == 5, x * 0.0, x - 0.5), acc * 0.5 + step(x, k), k + 1

        x, acc, k = lax.while_loop(lambda s: s[2] < trips, body, (x0, x0, jnp.int32(0)))
        o_ref[0], c_ref[0] = acc, k

    one = pl.BlockSpec((1,), lambda i: (i,))
    return pa.hip_call(kernel, grid=(n,), in_specs=[one, one], out_specs=[one, one], math_mode=mode, out_shape=[
        pl.ShapeDtypeStruct((n,), np.float32), pl.ShapeDtypeStruct((n,), np.int32)])


def checked_data(n, regular=False):
    rng = np.random.default_rng(n)
    x = rng.uniform(100.0, 200.0, n).astype(np.float32)
    if not regular:
        x[::3] = rng.uniform(-4.0, 40.0, len(x[::3])).astype(np.float32)
        x[::7] = 3.0  # whole numbers and halves: divisors that are exactly zero
        for k, v in enumerate((0.0, -0.0, 1e-42, 3e38, np.inf, -np.inf, np.nan, 1.0)):
            x[5 + k :: 301] = v
    return x, rng.integers(0, 150, n).astype(np.int32)
