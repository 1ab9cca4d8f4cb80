"""Host copies around a call: large readbacks through the pinned ring (its
slots' edges, several at once from threads) and inputs packed into one
upload (at and past the limit, mixed types, an empty one, launches in flight)."""

import threading

import numpy as np
import pytest

import palladium_amd as pa
from palladium_amd import runtime as rt
from palladium_amd.dispatch import PACK_LIMIT
from palladium_amd.frontend import jnp, pl

pytestmark = pytest.mark.gpu
MIB = 1 << 20


@pytest.mark.parametrize("nbytes", [8 * MIB - 4, 8 * MIB, 8 * MIB + 4, 20 * MIB, 22 * MIB + 12, 61 * MIB + 20])
def test_large_readback_is_exact(nbytes):
    x = np.random.default_rng(nbytes).integers(0, 2**32, nbytes // 4, dtype=np.uint32)
    buf = rt.Buffer.from_numpy(x)
    stream = rt.Stream()
    for _ in range(2):
        np.testing.assert_array_equal(buf.to_numpy(stream), x)


def test_readbacks_from_several_threads():
    data = [np.random.default_rng(k).integers(0, 2**32, 3 * MIB + k, dtype=np.uint32) for k in range(4)]
    bufs = [rt.Buffer.from_numpy(d) for d in data]
    got = [None] * 4

    def read(k):
        stream = rt.Stream()
        for _ in range(3):
            got[k] = bufs[k].to_numpy(stream)

    threads = [threading.Thread(target=read, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g, d in zip(got, data):
        np.testing.assert_array_equal(g, d)


@pytest.mark.parametrize("n", [1, 200, PACK_LIMIT // 12 - 100, PACK_LIMIT // 12 + 100])
def test_packed_inputs_of_mixed_types(n):
    def kernel(a_ref, b_ref, c_ref, o_ref):
        o_ref[...] = a_ref[...] + b_ref[...].astype(jnp.float32) * jnp.where(c_ref[...], 2.0, 1.0)

    s = pl.BlockSpec((1,), lambda i: (i,))
    f = pa.hip_call(kernel, grid=(n,), in_specs=[s] * 3, out_specs=s, out_shape=pl.ShapeDtypeStruct((n,), np.float32),
                    math_mode="safe")
    rng = np.random.default_rng(n)
    calls = [(rng.standard_normal(n).astype(np.float32), rng.integers(-9, 9, n).astype(np.int32),
              rng.integers(0, 2, n).astype(np.bool_)) for _ in range(9)]
    pending = [f.launch(*c) for c in calls]  # more than the sets in flight
    for p, (a, b, c) in zip(pending, calls):
        np.testing.assert_array_equal(p.wait(), a + b.astype(np.float32) * np.where(c, np.float32(2), np.float32(1)))


@pytest.mark.parametrize("shapes", [((5,), (0,), (5,)), ((0,), (5,), (5,)), ((5,), (5,), (0,))])
def test_packed_inputs_with_an_empty_one(shapes):
    """An input without elements takes no place among the packed ones."""
    full = [k for k, s in enumerate(shapes) if s != (0,)]

    def kernel(*refs):
        refs[-1][...] = refs[full[0]][...] - refs[full[1]][...]

    specs = [pl.BlockSpec((1,), lambda i: (i,)) if s != (0,) else pl.BlockSpec((0,), lambda i: (0,)) for s in shapes]
    f = pa.hip_call(kernel, grid=(5,), in_specs=specs, out_specs=pl.BlockSpec((1,), lambda i: (i,)),
                    out_shape=pl.ShapeDtypeStruct((5,), np.float32), math_mode="safe")
    args = [np.random.default_rng(k).standard_normal(s).astype(np.float32) for k, s in enumerate(shapes)]
    np.testing.assert_array_equal(f(*args), args[full[0]] - args[full[1]])


def test_nothing_but_empty_inputs():
    def kernel(e_ref, o_ref):
        o_ref[...] = jnp.full((3,), 2.0, jnp.float32)

    f = pa.hip_call(kernel, out_shape=pl.ShapeDtypeStruct((3,), np.float32), math_mode="safe")
    np.testing.assert_array_equal(f(np.zeros(0, np.float32)), np.full(3, 2, np.float32))
