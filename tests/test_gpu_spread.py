"""Blocks spread over teams of lanes on the GPU: SAFE and REPRODUCIBLE bit
for bit against the interpreter (float sums in the traced order), FAST
against float64."""

import numpy as np
import pytest

from palladium_amd import dtypes
from spread_cases import CASES, CROSSED, LANE_ROWS, MOMENTS, OVERWRITTEN

pytestmark = pytest.mark.gpu


def _run(name, mode):
    call, args = {**CASES, **MOMENTS}[name](np.random.default_rng(7), math_mode=mode)
    print(f"[spread] {name} {mode}", flush=True)
    got, want = call(*args), call.interpret(*args)
    return [got] if isinstance(got, np.ndarray) else got, [want] if isinstance(want, np.ndarray) else want


@pytest.mark.parametrize("mode", ["safe", "reproducible"])
@pytest.mark.parametrize("name", sorted({**CASES, **MOMENTS}))
def test_bit_exact_against_the_interpreter(name, mode):
    for g, w in zip(*_run(name, mode)):
        if dtypes.is_bf16(g.dtype):
            g, w = g.view(np.uint16), w.view(np.uint16)
        np.testing.assert_array_equal(g, w)


@pytest.mark.parametrize("name", sorted(n for n in CASES if not n.startswith("loops")))
def test_fast_close_to_the_interpreter(name):
    """FAST reassociates: a sum of n terms in another order moves by at most
    n eps times the sum of magnitudes (n <= 5,001, standard normal data),
    plus a few roundings of the element-wise part; narrow types round each
    operation to their own eps."""
    for g, w in zip(*_run(name, "fast")):
        if dtypes.is_bf16(g.dtype):
            g, w, eps = dtypes.to_float(g), dtypes.to_float(w), 2.0**-8
        elif g.dtype.kind != "f":
            np.testing.assert_array_equal(g, w)
            continue
        else:
            eps = float(np.finfo(g.dtype).eps)
        g, w = g.astype(np.float64), w.astype(np.float64)
        # the interpreter's own ordered sum carries the larger part: n eps/2
        # of a partial sum of about sqrt(n) in the narrow type
        n = max(1, int(name.split("x")[1].split("_")[0])) if name.startswith(("rows", "dense_1", "dense_2")) else 64
        scale = np.abs(w).max() + np.sqrt(n)
        assert np.abs(g - w).max() <= 8 * eps * scale * np.sqrt(n)


@pytest.mark.parametrize("mode", ["fast", "relaxed"])
@pytest.mark.parametrize("name", ["flat_250_bf16", "flat_1250_bf16", "flat_wide_bf16", "dense_33x1x40_bf16"])
def test_bfloat16_operations_round_one_by_one(name, mode):
    """Sums and products rounded each: the interpreter's bits. (No operation
    here leaves the exactly rounded ones, and no value is subnormal.)"""
    for g, w in zip(*_run(name, mode)):
        np.testing.assert_array_equal(g.view(np.uint16), w.view(np.uint16))


@pytest.mark.parametrize("mode", ["safe", "fast"])
@pytest.mark.parametrize("name", sorted({**OVERWRITTEN, **CROSSED}))
def test_later_stores_win(name, mode):
    """Exact in both modes: one rounding an element."""
    call, args = {**OVERWRITTEN, **CROSSED}[name](np.random.default_rng(7), math_mode=mode)
    print(f"[spread] {name} {mode}", flush=True)
    got, want = call(*args), call.interpret(*args)
    if name in CROSSED:
        m, w = (int(v) for v in name.split("_")[1].split("x"))
        got, want = (v.reshape(5, m, w) for v in (got, want))
        for at in ((slice(None), m - 1), (slice(None), slice(None), w - 1), (slice(None), 0, 0)):
            np.testing.assert_array_equal(got[at], want[at])
        return
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("mode", ["safe", "fast"])
@pytest.mark.parametrize("name", sorted(LANE_ROWS))
def test_lanes_of_an_instance_keep_its_order(name, mode):
    """Exact in both modes: one rounding an operation, sums in their order."""
    call, args = LANE_ROWS[name](np.random.default_rng(7), math_mode=mode)
    print(f"[lanes] {name} {mode}", flush=True)
    got, want = call(*args), call.interpret(*args)
    for g, w in zip(*((v,) if isinstance(v, np.ndarray) else v for v in (got, want))):
        np.testing.assert_array_equal(g, w)


@pytest.mark.parametrize("block", [64, 512, 1024])
@pytest.mark.parametrize("name", ["rows_4x17_f32", "rows_8x128_f32", "rows_64x40_f32", "dense_64x21x17_f32"])
def test_results_do_not_depend_on_the_workgroup(name, block):
    for mode in ("safe", "fast"):
        call, args = CASES[name](np.random.default_rng(7), math_mode=mode, threadgroup=block)
        default, _ = CASES[name](np.random.default_rng(7), math_mode=mode)
        print(f"[spread] {name} {block} {mode}", flush=True)
        for g, w in zip(*((v,) if isinstance(v, np.ndarray) else v for v in (call(*args), default(*args)))):
            np.testing.assert_array_equal(g, w)
