"""A loop long enough to be ranked by progress: t advances by the instance's
own step until a bound, or until `cap` trips."""

import numpy as np

import palladium_amd as pa
from palladium_amd.frontend import jnp, lax, pl


def ranked_call(n, test="lt", start=0.0, ops=40, cap=700, mode="safe"):
    def kernel(r_ref, o_ref, c_ref):
        r = r_ref[0]

        def cond(s):
            more = {"lt": lambda: s[0] < 20.0, "le": lambda: s[0] <= 20.0, "gt": lambda: 20.0 > s[0],
                    "int": lambda: s[2] < 20}[test]()
            return jnp.logical_and(more, s[2] < cap)

        def body(s):
            t, y, c = s
            for _ in range(ops):
                y = y * 0.999 + r
            return t + r, y, c + 1

        t, y, c = lax.while_loop(cond, body, (r if start is None else jnp.float32(start), r, jnp.int32(0)))
        o_ref[0], c_ref[0] = t + y, c

    one = pl.BlockSpec((1,), lambda i: (i,))
    return pa.hip_call(kernel, grid=(n,), in_specs=[one], out_specs=[one, one], math_mode=mode, out_shape=[
        pl.ShapeDtypeStruct((n,), np.float32), pl.ShapeDtypeStruct((n,), np.int32)])


def steps(kind, n, seed=0):
    """Steps whose trip counts are spread, alike, or never end by themselves."""
    rng = np.random.default_rng(seed)
    trips = np.exp(rng.uniform(np.log(20), np.log(500), n))
    if kind == "alike":
        trips = rng.uniform(200, 205, n)
    r = (20.0 / trips).astype(np.float32)
    if kind == "stuck":  # no progress, backwards, too small to show, NaN, one step
        for k, v in enumerate((0.0, -0.5, 1e-30, np.nan, np.inf)):
            r[k::11] = v
    return r
