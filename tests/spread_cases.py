"""Kernels whose blocks are spread over teams of lanes (emit/spread.py),
shared by the CPU and GPU tests: name -> (call factory, inputs). Sizes sit
at the edges of the layout: one lane's chunk, a wavefront's, a ragged last
chunk, the widest team, more than one run of slots."""

import numpy as np

import palladium_amd as pa
from palladium_amd import dtypes
from palladium_amd.frontend import jnp, lax, pl

F = np.float32
_DT = {"f32": np.dtype(np.float32), "f16": np.dtype(np.float16), "bf16": np.dtype(dtypes.bfloat16),
       "i32": np.dtype(np.int32), "u32": np.dtype(np.uint32), "bool": np.dtype(np.bool_)}


def _data(rng, shape, dt):
    if dt in ("f32", "f16"):
        return rng.standard_normal(shape).astype(_DT[dt])
    if dt == "bf16":
        return dtypes.from_float(rng.standard_normal(shape).astype(F))
    if dt == "bool":
        return rng.integers(0, 2, shape).astype(np.bool_)
    return rng.integers(0, 100, shape).astype(_DT[dt])


def flat(b, dt="f32", grid=5):
    """Element by element over blocks of b."""
    def kernel(x_ref, y_ref, o_ref):
        x, y = x_ref[...], y_ref[...]
        if dt == "bool":
            o_ref[...] = jnp.logical_xor(x, y)
        elif dt in ("i32", "u32"):
            o_ref[...] = x * y + 3
        else:
            z = x * y + 0.25 * x
            o_ref[...] = jnp.where(z > 0, z * 3.0, jnp.abs(y) - 0.5)

    def make(rng, **kw):
        s = pl.BlockSpec((b,), lambda i: (i,))
        call = pa.hip_call(kernel, grid=(grid,), in_specs=[s, s], out_specs=s,
                           out_shape=pl.ShapeDtypeStruct((grid * b,), _DT[dt]), **kw)
        return call, (_data(rng, grid * b, dt), _data(rng, grid * b, dt))

    return make


def flat2d(m, w, grid=3):
    """A whole block of rows, element by element, through two refs of other ranks."""
    def kernel(x_ref, o_ref):
        o_ref[...] = x_ref[...] * 2.0 + 1.0

    def make(rng, **kw):
        s = pl.BlockSpec((m, w), lambda i: (i, 0))
        call = pa.hip_call(kernel, grid=(grid,), in_specs=[s], out_specs=s,
                           out_shape=pl.ShapeDtypeStruct((grid * m, w), F), **kw)
        return call, (_data(rng, (grid * m, w), "f32"),)

    return make


def rows(m, w, dt="f32", grid=3):
    """Row maximum and sum, a row of biases, a value per row, both indices."""
    fl = dt in ("f32", "f16", "bf16")

    def kernel(x_ref, bias_ref, scale_ref, o_ref, top_ref, n_ref):
        x = x_ref[...]
        z = x + bias_ref[...]
        top = jnp.max(z, axis=-1, keepdims=True)
        low = jnp.min(z, axis=-1, keepdims=True)
        i = lax.broadcasted_iota(jnp.int32, (m, w), 0)
        j = lax.broadcasted_iota(jnp.int32, (m, w), 1)
        total = jnp.sum(z, axis=-1, keepdims=True)
        if fl:
            o_ref[...] = (z - top) * 0.5 + total * 0.125 + scale_ref[...]
        else:
            o_ref[...] = (z - top) * 3 + total + scale_ref[...]
        top_ref[...] = top - low
        n_ref[...] = jnp.sum(jnp.where(z > low, i * w + j, -1), axis=-1)

    def make(rng, **kw):
        s = pl.BlockSpec((m, w), lambda i: (i, 0))
        col = pl.BlockSpec((m, 1), lambda i: (i, 0))
        call = pa.hip_call(kernel, grid=(grid,),
                           in_specs=[s, pl.BlockSpec((w,), lambda i: (0,)), col],
                           out_specs=(s, col, pl.BlockSpec((m,), lambda i: (i,))),
                           out_shape=(pl.ShapeDtypeStruct((grid * m, w), _DT[dt]),
                                      pl.ShapeDtypeStruct((grid * m, 1), _DT[dt]),
                                      pl.ShapeDtypeStruct((grid * m,), np.int32)), **kw)
        return call, (_data(rng, (grid * m, w), dt), _data(rng, (w,), dt), _data(rng, (grid * m, 1), dt))

    return make


def loops(b, grid=4):
    """A loop whose carry starts the same everywhere, a loop until every
    element is done, a switch on a reduction, any and all."""
    def kernel(x_ref, o_ref, k_ref, f_ref):
        x = x_ref[...]
        y = lax.fori_loop(0, 7, lambda i, c: c * 0.5 + x * (i + 1), jnp.zeros((b,), jnp.float32))

        def body(c):
            v, n = c
            return jnp.where(v > 1.0, v * 0.5, v), n + 1

        v, n = lax.while_loop(lambda c: jnp.any(c[0] > 1.0), body, (jnp.abs(y) * 8.0, jnp.int32(0)))
        t = jnp.max(x)
        v = lax.cond(t > 2.0, lambda a: a - t, lambda a: a + 1.0, v)
        o_ref[...] = v
        k_ref[0] = n
        f_ref[0] = jnp.all(v < 2.0)

    def make(rng, **kw):
        s = pl.BlockSpec((b,), lambda i: (i,))
        one = pl.BlockSpec((1,), lambda i: (i,))
        call = pa.hip_call(kernel, grid=(grid,), in_specs=[s], out_specs=(s, one, one),
                           out_shape=(pl.ShapeDtypeStruct((grid * b,), F), pl.ShapeDtypeStruct((grid,), np.int32),
                                      pl.ShapeDtypeStruct((grid,), np.bool_)), **kw)
        return call, (_data(rng, grid * b, "f32"),)

    return make


def indexed(m, w, grid=3):
    """Rows and columns of a block one by one: a column per row's first
    lane, a row for all rows, single elements of a parameter array."""
    def kernel(x_ref, p_ref, o_ref, c_ref, r_ref):
        x = x_ref[...]
        a, b = p_ref[0], p_ref[2]
        o_ref[...] = x * a + b
        c_ref[:, 1] = x_ref[:, 0] * 2.0
        c_ref[:, 0] = jnp.sum(x, axis=1)
        r_ref[0, :] = x_ref[1, :] + b

    def make(rng, **kw):
        s = pl.BlockSpec((m, w), lambda i: (i, 0))
        call = pa.hip_call(kernel, grid=(grid,), in_specs=[s, pl.BlockSpec((3,), lambda i: (0,))],
                           out_specs=(s, pl.BlockSpec((m, 2), lambda i: (i, 0)), pl.BlockSpec((1, w), lambda i: (i, 0))),
                           out_shape=(pl.ShapeDtypeStruct((grid * m, w), F), pl.ShapeDtypeStruct((grid * m, 2), F),
                                      pl.ShapeDtypeStruct((grid, w), F)), **kw)
        return call, (_data(rng, (grid * m, w), "f32"), _data(rng, (3,), "f32"))

    return make


def dense(m, k, n, dt="f32", grid=3, transposed=False):
    """Rows times a matrix plus a bias and a value per row."""
    def kernel(a_ref, w_ref, b_ref, s_ref, o_ref):
        w = w_ref[...]
        y = lax.dot_general(a_ref[...], w, (((1,), (1,)), ((), ()))) if transposed else jnp.dot(a_ref[...], w)
        o_ref[...] = jnp.maximum(y + b_ref[...], 0.0) + s_ref[...]

    def make(rng, **kw):
        call = pa.hip_call(kernel, grid=(grid,),
                           in_specs=[pl.BlockSpec((m, k), lambda i: (i, 0)),
                                     pl.BlockSpec((n, k) if transposed else (k, n), lambda i: (0, 0)),
                                     pl.BlockSpec((n,), lambda i: (0,)), pl.BlockSpec((m, 1), lambda i: (i, 0))],
                           out_specs=pl.BlockSpec((m, n), lambda i: (i, 0)),
                           out_shape=pl.ShapeDtypeStruct((grid * m, n), _DT[dt]), **kw)
        return call, (_data(rng, (grid * m, k), dt), _data(rng, (n, k) if transposed else (k, n), dt), _data(rng, (n,), dt),
                      _data(rng, (grid * m, 1), dt))

    return make


def two_dots(m, k, n, grid=3):
    """Two products into one block, one of them with a matrix per instance, indices of both axes."""
    def kernel(a_ref, w_ref, v_ref, o_ref):
        y = jnp.dot(a_ref[...], w_ref[...]) - jnp.dot(a_ref[...], v_ref[...])
        i = lax.broadcasted_iota(jnp.int32, (m, n), 0)
        j = lax.broadcasted_iota(jnp.int32, (m, n), 1)
        o_ref[...] = jnp.where(i > j, y, y * 0.5)

    def make(rng, **kw):
        call = pa.hip_call(kernel, grid=(grid,),
                           in_specs=[pl.BlockSpec((m, k), lambda i: (i, 0)), pl.BlockSpec((k, n), lambda i: (0, 0)),
                                     pl.BlockSpec((k, n), lambda i: (i, 0))],
                           out_specs=pl.BlockSpec((m, n), lambda i: (i, 0)),
                           out_shape=pl.ShapeDtypeStruct((grid * m, n), F), **kw)
        return call, (_data(rng, (grid * m, k), "f32"), _data(rng, (k, n), "f32"), _data(rng, (grid * k, n), "f32"))

    return make


def single(n):
    """One instance, looping over a whole array."""
    def kernel(y_ref, r_ref, o_ref):
        r = r_ref[...]
        o_ref[...] = lax.fori_loop(0, 20, lambda _, y: y + 0.01 * r * y * (1.0 - y), y_ref[...])

    def make(rng, **kw):
        call = pa.hip_call(kernel, out_shape=pl.ShapeDtypeStruct((n,), F), **kw)
        return call, (_data(rng, n, "f32"), _data(rng, n, "f32"))

    return make


CASES = {
    **{f"flat_{b}_{dt}": flat(b, dt) for b, dt in
       ((32, "f32"), (33, "f32"), (100, "f16"), (250, "bf16"), (1000, "u32"), (1025, "f32"), (1250, "bf16"),
        (4096, "i32"), (5001, "f32"), (300, "bool"), (2048, "f16"))},
    "flat_16_f32": flat(16, "f32"),
    **{f"flat_one_{b}_f32": flat(b, "f32", grid=1) for b in (17, 1000, 4099)},
    "flat_wide_1024_f16": flat(1024, "f16", grid=2000),
    "flat_wide_f32": flat(1000, "f32", grid=1200),
    "flat_wide_bf16": flat(1000, "bf16", grid=2400),
    **{f"flat2d_{m}x{w}": flat2d(m, w) for m, w in ((3, 40), (8, 128), (7, 333), (1, 50))},
    **{f"rows_{m}x{w}_{dt}": rows(m, w, dt) for m, w, dt in
       ((1, 37, "f32"), (1, 64, "i32"), (1, 1000, "f32"), (1, 1025, "bf16"), (1, 3000, "f32"), (4, 17, "f32"),
        (5, 33, "f16"), (8, 128, "f32"), (8, 100, "bf16"), (64, 40, "f32"), (64, 8, "f32"), (12, 4, "f32"), (300, 8, "f32"), (3, 700, "u32"), (33, 34, "f32"))},
    **{f"loops_{b}": loops(b) for b in (48, 100, 777, 1500)},
    **{f"indexed_{m}x{w}": indexed(m, w) for m, w in ((4, 24), (6, 130))},
    **{f"dense_{m}x{k}x{n}_{dt}": dense(m, k, n, dt) for m, k, n, dt in
       ((128, 64, 32, "f32"), (64, 21, 17, "f32"), (100, 33, 3, "f32"), (16, 16, 16, "f32"), (1024, 16, 48, "f32"),
        (250, 40, 64, "bf16"), (64, 32, 30, "bf16"), (128, 96, 16, "f16"), (33, 7, 33, "f16"), (256, 128, 64, "f32"),
        (64, 15, 40, "f16"), (64, 3, 18, "bf16"), (64, 1, 20, "f16"), (64, 2, 24, "f32"), (128, 50, 20, "f32"),
        (64, 84, 24, "f16"), (64, 8, 17, "bf16"), (33, 1, 40, "bf16"))},
    "dense_64x24x20_transposed_f32": dense(64, 24, 20, "f32", transposed=True),
    "dense_64x40x20_transposed_bf16": dense(64, 40, 20, "bf16", transposed=True),
    "dense_wide_f32": dense(128, 24, 32, "f32", grid=600),
    "two_dots_64x24x16": two_dots(64, 24, 16),
    **{f"single_{n}": single(n) for n in (65, 200, 1024, 3000)},
}


def overwritten(b, order):
    """A block stored whole and in part, whose lanes would not be the same ones."""
    one_d = not isinstance(b, tuple)

    def kernel(x_ref, o_ref):
        x = x_ref[...]

        def whole():
            o_ref[...] = x * 2.0

        if order == "last":  # a boundary value after the block
            whole()
            if one_d:
                o_ref[b - 1] = 5.0
            else:
                o_ref[b[0] - 1, b[1] - 1] = 5.0
        elif order == "first":  # and before it
            if one_d:
                o_ref[b - 1] = 5.0
            else:
                o_ref[b[0] - 1, :] = x_ref[0, :]
            whole()
        elif order == "row":
            whole()
            o_ref[b[0] - 1, :] = x_ref[0, :]
        elif order == "column":
            whole()
            o_ref[:, b[1] - 1] = x_ref[:, 0] + 1.0
        elif order == "cross":  # a row and a column, without the block
            o_ref[b[0] - 1, :] = x_ref[0, :]
            o_ref[:, b[1] - 1] = x_ref[:, 0] + 1.0
            o_ref[0, 0] = 3.0
            o_ref[b[0] - 1, 0] = 7.0
        elif order == "loop":
            o_ref[...] = jnp.zeros((b,), jnp.float32)

            def body(i, c):
                o_ref[i * (b // 10)] = x_ref[i] + c
                return c + 1.0

            lax.fori_loop(0, 10, body, jnp.float32(0.0))
        elif order == "branch":
            whole()

            def put(v):
                o_ref[b - 2] = v
                return v

            lax.cond(x_ref[0] > 0.0, put, lambda v: v, jnp.float32(9.0))

    def make(rng, grid=5, **kw):
        shape = (b,) if one_d else b
        s = pl.BlockSpec(shape, lambda i: (i, *(0,) * (len(shape) - 1)))
        full = (grid * shape[0], *shape[1:])
        call = pa.hip_call(kernel, grid=(grid,), in_specs=[s], out_specs=s, out_shape=pl.ShapeDtypeStruct(full, F), **kw)
        return call, (_data(rng, full, "f32"),)

    return make


def _overwritten(*cases):
    return {f"{order}_{b if isinstance(b, int) else '%dx%d' % b}": overwritten(b, order) for order, b in cases}


# (In one lane a block lies in scratch, which every hardware queue keeps for
# all waves of the chip: the blocks that run are small.)
OVERWRITTEN = _overwritten(("last", 100), ("last", 300), ("first", 300), ("loop", 300), ("branch", 300), ("last", (3, 100)),
                           ("first", (3, 100)), ("row", (3, 100)), ("row", (70, 4)), ("column", (3, 100)), ("column", (20, 16)))
OVERWRITTEN_WIDE = _overwritten(("last", 1000), ("first", 1000), ("loop", 1000), ("branch", 3000), ("row", (8, 100)),
                                ("row", (300, 20)), ("column", (3, 700)))
# The rest of the block is not written: compared where it is.
CROSSED = {f"cross_{m}x{w}": overwritten((m, w), "cross") for m, w in ((3, 100), (16, 20))}


def read_by_all(b):
    """An output's element read by every lane after lane 0 stored it, its
    rows summed one by one after each lane stored its own."""
    def kernel(x_ref, o_ref, s_ref):
        s_ref[0] = jnp.max(x_ref[...])
        o_ref[...] = x_ref[...] - s_ref[0]
        s_ref[1] = o_ref[b - 1] * 2.0

        def body(i, c):
            s_ref[1] = s_ref[1] + o_ref[i * (b // 8)]
            return c

        lax.fori_loop(0, 8, body, jnp.float32(0.0))

    def make(rng, grid=5, **kw):
        s = pl.BlockSpec((b,), lambda i: (i,))
        call = pa.hip_call(kernel, grid=(grid,), in_specs=[s], out_specs=(s, pl.BlockSpec((2,), lambda i: (i,))),
                           out_shape=(pl.ShapeDtypeStruct((grid * b,), F), pl.ShapeDtypeStruct((grid * 2,), F)), **kw)
        return call, (_data(rng, grid * b, "f32"),)

    return make


# The same where a block's rows have a lane each.
LANE_ROWS = {**_overwritten(("last", 64), ("last", 256), ("first", 1024), ("loop", 256), ("branch", 128), ("last", (128, 4)),
                            ("first", (128, 4)), ("row", (256, 3)), ("row", (64, 3))),
             **{f"read_by_all_{b}": read_by_all(b) for b in (64, 256, 1024)}}


def moments(m, w, n, dt="f32"):
    """n sums along each row, one after another, in two accumulation types."""
    def kernel(x_ref, o_ref, n_ref):
        x = x_ref[...]
        z = x
        for _ in range(n):
            z = x - jnp.sum(z, axis=1, keepdims=True) * (0.5 / w)
        o_ref[...] = z
        n_ref[...] = jnp.sum(jnp.where(z > x, 0.5, 0.25), axis=1)

    def make(rng, grid=3, **kw):
        s = pl.BlockSpec((m, w), lambda i: (i, 0))
        call = pa.hip_call(kernel, grid=(grid,), in_specs=[s], out_specs=(s, pl.BlockSpec((m,), lambda i: (i,))),
                           out_shape=(pl.ShapeDtypeStruct((grid * m, w), _DT[dt]),
                                      pl.ShapeDtypeStruct((grid * m,), F)), **kw)
        return call, (_data(rng, (grid * m, w), dt),)

    return make


# Together past a workgroup's LDS, were each staged by itself.
MOMENTS = {f"moments_{m}x{w}_{n}_{dt}": moments(m, w, n, dt) for m, w, n, dt in
           ((64, 900, 3, "f32"), (64, 512, 5, "f32"), (128, 400, 4, "f32"), (256, 200, 4, "f32"), (4, 1000, 12, "f16"),
            (1, 4096, 4, "f32"), (1, 15000, 3, "f32"))}
