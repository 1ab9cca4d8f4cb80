"""Integer maxima and minima over an instance's lanes, against the interpreter:
every lane sends its value, also those that keep their own."""

import numpy as np
import pytest

import palladium_amd as pa
from palladium_amd.frontend import jnp, lax, pl


def _call(lanes, dt):
    def kernel(x_ref, o_ref, lo_ref, hi_ref):
        x = lax.fori_loop(0, 3, lambda k, v: v * 3 + 1, x_ref[...])
        lo, hi = jnp.min(x), jnp.max(x)
        o_ref[...] = x + lo + hi
        lo_ref[0], hi_ref[0] = lo, hi

    blk, one = pl.BlockSpec((lanes,), lambda i: (i,)), pl.BlockSpec((1,), lambda i: (i,))
    return pa.hip_call(kernel, grid=(9,), in_specs=[blk], out_specs=(blk, one, one), math_mode="safe",
                       out_shape=(pl.ShapeDtypeStruct((9 * lanes,), dt), *[pl.ShapeDtypeStruct((9,), dt)] * 2))


def _data(lanes, dt):
    lo = -40_000_000 if dt == np.int32 else 0
    return np.random.default_rng(lanes).integers(lo, 40_000_000, 9 * lanes).astype(dt)


@pytest.mark.parametrize("dt", [np.int32, np.uint32])
def test_no_exchange_inside_a_choice(dt):
    src = _call(256, dt).bound(_data(256, dt)).hip_source
    lines = [line for line in src[src.index('extern "C"'):].splitlines() if "__shfl_xor" in line]
    assert lines and not any("?" in line for line in lines)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [np.int32, np.uint32])
@pytest.mark.parametrize("lanes", [64, 256])
def test_integer_extremes_match_the_interpreter(lanes, dt):
    print(f"[extremes] lanes={lanes} {dt.__name__}", flush=True)
    call, x = _call(lanes, dt), _data(lanes, dt)
    for g, w in zip(call(x), call.interpret(x)):
        np.testing.assert_array_equal(g, w)
