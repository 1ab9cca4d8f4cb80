"""The work this framework is timed on: its hot-path kernels and the ordinary
Pallas kernels its users write, through the public entry points.

Sizes are the configurations of `palladium_amd.workloads` (config 0 to 4b),
those of the tests and the benchmark, and generic ones between and around
them. A case is a dict of plain values; `kind` picks the program:

- `lv`        RK4 Lotka-Volterra ensemble, one trajectory per instance or
              blocks of trajectories (`lv_rk4_call`)
- `bs3`       adaptive BS3(2)+PI Van der Pol ensemble (`bs3_vdp_call`)
- `gbm`       GBM Monte Carlo, one path per instance (`gbm_call`)
- `gbm_fold`  the same with per-path, per-draw derived keys
              (`gbm_fold_in_call`)
- `df32`      RK4 Lotka-Volterra in compensated pairs (`lv_rk4_df32_device`)
- `gs_steps`  Gray-Scott, one launch per step, host arrays in and out
              (`gray_scott_run`)
- `gs_passes` Gray-Scott, several steps per launch, host arrays in and out
              (`gray_scott_fused_run`)
- `logistic`  a kernel without a grid over a whole array, called with host
              arrays as a first program does (`hip_call`)
- `softmax`   row-wise softmax in blocks of rows (`hip_call`)
- `pointwise` element-wise arithmetic in blocks of any size (`hip_call`)
- `dense`     rows times a small matrix plus a bias, tanh, in blocks of rows
              (`hip_call`)

Kernels called with device arrays run on the caller's current stream.
"""

import math

import numpy as np
import torch

import palladium_amd as pa
from palladium_amd import df32, dtypes, stencil, workloads
from palladium_amd.frontend import jnp, lax, pl, random as prandom

F32 = np.float32
DEV = "cuda"

_NP = {"float32": np.dtype(np.float32), "float16": np.dtype(np.float16), "bfloat16": np.dtype(dtypes.bfloat16)}
_TORCH = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
_BYTES = {"float32": 4, "float16": 2, "bfloat16": 2}


def listed():
    return [
        # The first program of a new user: a whole small array, no grid, NumPy
        # in and out (the tests' Euler steps of the logistic equation).
        {"name": "logistic_200", "kind": "logistic", "n": 200, "steps": 100},
        # Config 0: a small ensemble in blocks of 256, the last one ragged.
        {"name": "lv_100k_blocks", "kind": "lv", "n": 100_000, "steps": 1000, "dt": 0.01, "block": 256, "mode": "fast"},
        # Config 1: a large ensemble, the headline workload.
        {"name": "lv_1m", "kind": "lv", "n": 1_000_000, "steps": 4000, "dt": 0.005, "block": 1, "mode": "fast"},
        # Config 2: adaptive, divergent, step counts that a host can repeat.
        {"name": "bs3_262k", "kind": "bs3", "n": 262_144, "mode": "reproducible"},
        # Config 3: Monte Carlo pricing, counter-based random numbers.
        {"name": "gbm_4m", "kind": "gbm", "n": 4_194_304, "steps": 252, "mode": "fast"},
        # A price to a few digits with derived keys per path and draw.
        {"name": "gbm_fold_65k", "kind": "gbm_fold", "n": 65_536, "steps": 252, "mode": "fast"},
        # A small simulation driven step by step; the size fits no tile.
        {"name": "gs_500_steps", "kind": "gs_steps", "size": 500, "steps": 200, "mode": "fast"},
        # Config 4 whole: fields in from the host, 2,000 steps, fields out.
        {"name": "gs_4096_passes", "kind": "gs_passes", "size": 4096, "steps": 2000, "mode": "fast"},
        # Config 4b at config 0's size: compensated arithmetic, exact.
        {"name": "df32_100k", "kind": "df32", "n": 100_000, "steps": 1000, "dt": 0.01},
        # Rows normalised, one row per instance, a width that is no power of two.
        {"name": "softmax_8192x1000", "kind": "softmax", "rows": 8192, "width": 1000, "block": 1, "dtype": "float32", "mode": "fast"},
        # A long array in half precision, blocks larger than a workgroup.
        {"name": "pointwise_4m_bf16", "kind": "pointwise", "n": 4_000_000, "block": 1250, "dtype": "bfloat16", "mode": "fast"},
        # One layer of a small network over an ensemble's states.
        {"name": "dense_262k_64x32", "kind": "dense", "rows": 262_144, "k": 64, "cols": 32, "block": 128, "dtype": "float32", "mode": "fast"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["logistic", "lv", "lv", "bs3", "gbm", "gbm_fold", "gs_steps", "gs_passes", "df32",
                       "softmax", "softmax", "pointwise", "pointwise", "dense", "dense"])
    mode = rng.choice(["fast", "fast", "safe"])
    if kind == "logistic":
        return {"kind": kind, "n": _log(rng, 16, 240), "steps": _log(rng, 10, 200)}
    if kind == "lv":
        return {"kind": kind, "n": _log(rng, 1000, 1_000_000), "steps": _log(rng, 100, 2000), "dt": 0.005,
                "block": rng.choice([1, 1, 64, 256]), "mode": rng.choice(["fast", "fast", "safe", "reproducible"])}
    if kind == "bs3":
        return {"kind": kind, "n": _log(rng, 1000, 262_144), "mode": rng.choice(["reproducible", "safe"])}
    if kind == "gbm":
        return {"kind": kind, "n": _log(rng, 10_000, 4_194_304), "steps": rng.choice([12, 52, 252]), "mode": "fast"}
    if kind == "gbm_fold":
        return {"kind": kind, "n": _log(rng, 10_000, 500_000), "steps": rng.choice([12, 52, 252]), "mode": "fast"}
    if kind == "gs_steps":
        return {"kind": kind, "size": _log(rng, 64, 1500), "steps": _log(rng, 20, 400), "mode": mode}
    if kind == "gs_passes":
        return {"kind": kind, "size": _log(rng, 200, 4096), "steps": _log(rng, 60, 1500), "mode": mode}
    if kind == "df32":
        return {"kind": kind, "n": _log(rng, 1000, 400_000), "steps": _log(rng, 100, 1000), "dt": 0.005}
    dtype = rng.choice(["float32", "float32", "bfloat16", "float16"])
    if kind == "softmax":
        # one instance holds its whole block: 1,000 or so values at most
        block = rng.choice([1, 1, 4, 8, 64])
        width = _log(rng, 16, 1200 // block if block < 64 else 128)
        rows = max(1, min(_log(rng, 64, 32768), 16_000_000 // width) // block) * block
        return {"kind": kind, "rows": rows, "width": width, "block": block, "dtype": dtype,
                "mode": mode if dtype == "float32" else "fast"}
    if kind == "pointwise":
        block = rng.choice([1, 32, 64, 100, 256, 500, 1000, 1024, *([1250] if dtype != "float32" else [])])
        return {"kind": kind, "n": max(1, _log(rng, 1000, 16_000_000) // block) * block, "block": block, "dtype": dtype,
                "mode": mode}
    block = rng.choice([64, 128, 256])
    return {"kind": "dense", "rows": _log(rng, 1, 4096) * block, "k": _log(rng, 4, 128), "cols": _log(rng, 2, 64),
            "block": block, "dtype": dtype, "mode": mode}


# ---------------------------------------------------------------------------
# kernels that are not in palladium_amd.workloads


def _logistic_call(n, steps):
    dt = 0.01

    def logistic(y0_ref, r_ref, o_ref):
        r = r_ref[...]
        o_ref[...] = lax.fori_loop(0, steps, lambda _, y: y + dt * r * y * (1.0 - y), y0_ref[...])

    return pa.hip_call(logistic, out_shape=pl.ShapeDtypeStruct((n,), F32))


def _softmax_call(c):
    rows, width, block, dt = c["rows"], c["width"], c["block"], _NP[c["dtype"]]

    def softmax(x_ref, o_ref):
        v = x_ref[...]
        z = v - jnp.max(v, axis=-1, keepdims=True)
        e = jnp.exp(z)
        o_ref[...] = e / jnp.sum(e, axis=-1, keepdims=True)

    spec = pl.BlockSpec((block, width), lambda i: (i, 0))
    return pa.hip_call(softmax, grid=(rows // block,), in_specs=[spec], out_specs=spec,
                       out_shape=pl.ShapeDtypeStruct((rows, width), dt), math_mode=c["mode"])


def _pointwise_call(c):
    n, block, dt = c["n"], c["block"], _NP[c["dtype"]]

    def pointwise(x_ref, y_ref, o_ref):
        x, y = x_ref[...], y_ref[...]
        z = x * y + 0.1 * x - y / (x * x + 1.0)
        o_ref[...] = jnp.where(z > 0, z * 3.0, jnp.abs(z) - 0.5)

    spec = pl.BlockSpec((block,), lambda i: (i,))
    return pa.hip_call(pointwise, grid=(n // block,), in_specs=[spec, spec], out_specs=spec,
                       out_shape=pl.ShapeDtypeStruct((n,), dt), math_mode=c["mode"])


def _dense_call(c):
    rows, k, cols, block, dt = c["rows"], c["k"], c["cols"], c["block"], _NP[c["dtype"]]

    def dense(a_ref, w_ref, b_ref, o_ref):
        o_ref[...] = jnp.tanh(jnp.dot(a_ref[...], w_ref[...]) + b_ref[...])

    return pa.hip_call(
        dense, grid=(rows // block,),
        in_specs=[pl.BlockSpec((block, k), lambda i: (i, 0)), pl.BlockSpec((k, cols), lambda i: (0, 0)),
                  pl.BlockSpec((cols,), lambda i: (0,))],
        out_specs=pl.BlockSpec((block, cols), lambda i: (i, 0)),
        out_shape=pl.ShapeDtypeStruct((rows, cols), dt), math_mode=c["mode"])


# ---------------------------------------------------------------------------
# inputs


def _gs_cfg():
    return workloads.GS_CFG


def _host_inputs(c, seed):
    """The case's inputs as float32 (or uint32) NumPy arrays."""
    kind = c["kind"]
    rng = np.random.default_rng([seed, 77])
    if kind in ("lv", "df32"):
        return workloads.lv_inputs(c["n"], seed)
    if kind == "bs3":
        return workloads.bs3_inputs(c["n"], seed)
    if kind in ("gbm", "gbm_fold"):
        return (prandom.key(seed & 0x7FFFFFFF),)
    if kind in ("gs_steps", "gs_passes"):
        return workloads.gray_scott_initial(c["size"], seed)
    if kind == "logistic":
        return rng.uniform(0.1, 0.9, c["n"]).astype(F32), rng.uniform(0.5, 1.5, c["n"]).astype(F32)
    return ()


def _device_inputs(c, seed):
    """Inputs of the kernels that take device arrays, as torch tensors."""
    kind = c["kind"]
    if kind in ("softmax", "pointwise", "dense"):
        g = torch.Generator(device=DEV)
        g.manual_seed(seed)
        dt = _TORCH[c["dtype"]]

        def normal(*shape, scale=1.0):
            return (torch.randn(*shape, generator=g, device=DEV) * scale).to(dt)

        if kind == "softmax":
            return (normal(c["rows"], c["width"], scale=3.0),)
        if kind == "pointwise":
            return normal(c["n"], scale=2.0), normal(c["n"], scale=2.0)
        return (normal(c["rows"], c["k"]), normal(c["k"], c["cols"], scale=c["k"] ** -0.5),
                normal(c["cols"], scale=0.1))
    return tuple(torch.from_numpy(np.ascontiguousarray(a)).to(DEV) for a in _host_inputs(c, seed))


def _call_of(c):
    kind = c["kind"]
    if kind == "lv":
        return workloads.lv_rk4_call(c["n"], c["dt"], c["steps"], block=c["block"], math_mode=c["mode"])
    if kind == "bs3":
        return workloads.bs3_vdp_call(c["n"], math_mode=c["mode"])
    if kind == "gbm":
        return workloads.gbm_call(workloads.GBMConfig(n_steps=c["steps"]), n_paths=c["n"], math_mode=c["mode"])
    if kind == "gbm_fold":
        return workloads.gbm_fold_in_call(workloads.GBMConfig(n_steps=c["steps"]), n_paths=c["n"], math_mode=c["mode"])
    return {"softmax": _softmax_call, "pointwise": _pointwise_call, "dense": _dense_call}[kind](c)


def _shape_structs(c, tensors):
    names = {torch.float32: np.dtype(F32), torch.uint32: np.dtype(np.uint32), torch.float16: np.dtype(np.float16),
             torch.bfloat16: np.dtype(dtypes.bfloat16)}
    return [pl.ShapeDtypeStruct(tuple(t.shape), names[t.dtype]) for t in tensors]


def _output_like(info):
    if dtypes.is_bf16(info.dtype):
        dt = torch.bfloat16
    else:
        dt = {"float32": torch.float32, "float16": torch.float16, "int32": torch.int32}[np.dtype(info.dtype).name]
    return torch.empty(info.array_shape, dtype=dt, device=DEV)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "logistic":
        call = _logistic_call(c["n"], c["steps"])
        arrays = _host_inputs(c, seed)
        call.bound(*arrays)
        return {"case": c, "call": call, "arrays": arrays}
    if kind == "gs_steps":
        call = workloads.gray_scott_call(size=c["size"], math_mode=c["mode"])
        u, v = _host_inputs(c, seed)
        call.bound(u, v)
        return {"case": c, "call": call, "arrays": (u, v)}
    if kind == "gs_passes":
        passes = stencil.RegisterGrayScott(c["size"], math_mode=c["mode"])
        return {"case": c, "call": passes, "arrays": _host_inputs(c, seed)}
    ins = _device_inputs(c, seed)
    if kind == "df32":
        df32.lv_kernel().load()
        return {"case": c, "ins": ins, "outs": tuple(torch.empty(c["n"], device=DEV) for _ in range(4))}
    bound = _call_of(c).bound(*_shape_structs(c, ins))
    return {"case": c, "bound": bound, "ins": ins, "outs": tuple(_output_like(i) for i in bound.spec.outputs)}


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "logistic":
        return state["call"](*state["arrays"])
    if kind == "gs_steps":
        return workloads.gray_scott_run(state["call"], *state["arrays"], c["steps"])[:2]
    if kind == "gs_passes":
        return stencil.gray_scott_fused_run(state["call"], *state["arrays"], c["steps"])[:2]
    stream = torch.cuda.current_stream()
    if kind == "df32":
        df32.lv_rk4_df32_device(state["ins"], state["outs"], c["dt"], c["steps"], c["n"], stream)
    else:
        state["bound"].launch_device(*state["ins"], *state["outs"], stream=stream)
    return state["outs"]


# ---------------------------------------------------------------------------
# what a pass cannot do without

# Attempts per trajectory of the Van der Pol ensemble (262.6 million over
# config 2's 262,144 trajectories) and operations per attempt.
_BS3_ATTEMPTS, _BS3_OPS = 1002, 99
_GBM_OPS = 97  # per path-step: 72 of Threefry, 25 of Box-Muller and the update
_GBM_FOLD_OPS = 319  # per path-step: four Threefry blocks instead of one
_GS_OPS = 29  # per cell-step


def work(case):
    c, kind = case, case["kind"]
    if kind == "lv":
        return {"bytes": c["n"] * 32, "flops": c["n"] * c["steps"] * workloads.LV_FLOP_PER_STEP}
    if kind == "df32":
        return {"bytes": c["n"] * 40, "flops": c["n"] * c["steps"] * df32.LV_DF32_FLOPS_PER_STEP}
    if kind == "bs3":
        return {"bytes": c["n"] * 32, "flops": c["n"] * _BS3_ATTEMPTS * _BS3_OPS}
    if kind == "gbm":
        return {"bytes": c["n"] * 4 + 8, "flops": c["n"] * c["steps"] * _GBM_OPS}
    if kind == "gbm_fold":
        return {"bytes": c["n"] * 4 + 8, "flops": c["n"] * c["steps"] * _GBM_FOLD_OPS}
    if kind in ("gs_steps", "gs_passes"):
        return {"bytes": c["size"] ** 2 * 16, "flops": c["size"] ** 2 * c["steps"] * _GS_OPS}
    if kind == "logistic":
        return {"bytes": c["n"] * 12, "flops": c["n"] * c["steps"] * 5}
    size = _BYTES[c["dtype"]]
    if kind == "softmax":
        return {"bytes": c["rows"] * c["width"] * 2 * size, "flops": c["rows"] * c["width"] * 5}
    if kind == "pointwise":
        return {"bytes": c["n"] * 3 * size, "flops": c["n"] * 11}
    return {"bytes": (c["rows"] * (c["k"] + c["cols"]) + (c["k"] + 1) * c["cols"]) * size,
            "flops": c["rows"] * c["cols"] * (2 * c["k"] + 2)}


def tolerance(case):
    kind, mode = case["kind"], case.get("mode")
    if kind in ("bs3", "df32"):
        return "exact"  # deterministic modes: states and step counts are bits
    if kind in ("lv", "gs_steps", "gs_passes") and mode in ("safe", "reproducible"):
        return "exact"  # every operation's order is fixed
    # About four times the error against 64 bits that was measured.
    if kind in ("gs_steps", "gs_passes"):
        return {"rel": 6e-5, "max": 1.2e-3}
    if kind == "lv":
        return {"rel": 2e-5, "max": 4e-4}
    if kind in ("gbm", "gbm_fold"):
        return {"rel": 1.4e-5, "max": 1e-4}
    if kind == "logistic":
        return {"rel": 1e-6, "max": 3e-6}
    if case["dtype"] == "float32":
        return {"rel": 2.5e-6, "max": 1.5e-5} if kind == "softmax" else {"rel": 5e-7, "max": 7e-6}
    if case["dtype"] == "bfloat16":
        return {"rel": 1.4e-2, "max": 0.25}
    # float16 sums are rounded to float16 term by term: a softmax's row sum
    # carries that error, and other orders of adding another one
    return {"rel": 2.5e-2, "max": 0.1} if kind == "softmax" else {"rel": 2e-3, "max": 1e-2}


# ---------------------------------------------------------------------------
# the same in 64 bits, plain torch

_ROT = ((13, 15, 26, 6), (17, 29, 16, 24))


def _rotl(x, r):
    return (x << r) | ((x >> (32 - r)) & ((1 << r) - 1))


def _threefry(k0, k1, x0, x1):
    """Threefry-2x32-20 on int32 tensors (arithmetic wraps)."""
    ks = (k0, k1, k0 ^ k1 ^ 0x1BD11BDA)
    x0, x1 = x0 + ks[0], x1 + ks[1]
    for g in range(5):
        for r in _ROT[g % 2]:
            x0 = x0 + x1
            x1 = _rotl(x1, r) ^ x0
        x0 = x0 + ks[(g + 1) % 3]
        x1 = x1 + ks[(g + 2) % 3] + (g + 1)
    return x0, x1


def _uniform(bits):
    return ((bits >> 9) & 0x7FFFFF).double() * 2.0**-23


def _gbm64(c, seed):
    cfg = workloads.GBMConfig(n_steps=c["steps"])
    f = lambda v: float(F32(v))  # noqa: E731  the program's constants are float32
    drift, vol, twopi = f(cfg.drift_dt), f(cfg.vol_sqdt), f(2.0 * math.pi)
    key = torch.from_numpy(np.asarray(prandom.key(seed & 0x7FFFFFFF)).view(np.int32).copy()).to(DEV)
    k0, k1 = key[0], key[1]
    path = torch.arange(c["n"], dtype=torch.int32, device=DEV)
    zero = torch.zeros_like(path)
    s = torch.full((c["n"],), cfg.s0, dtype=torch.float64, device=DEV)
    if c["kind"] == "gbm_fold":
        k0, k1 = _threefry(k0, k1, zero, path)
    for i in range(c["steps"]):
        if c["kind"] == "gbm":
            b0, b1 = _threefry(k0, k1, path, zero + i)
        else:
            bits = []
            for d in (2 * i, 2 * i + 1):
                a, b = _threefry(*_threefry(k0, k1, zero, zero + d), zero, zero)
                bits.append(a ^ b)
            b0, b1 = bits
        u1, u2 = torch.clamp(_uniform(b0), min=f(1e-7)), _uniform(b1)
        z = torch.sqrt(-2.0 * torch.log(u1)) * torch.cos(twopi * u2)
        s = s * torch.exp(drift + vol * z)
    return torch.clamp(s - cfg.strike, min=0.0)


def _lv64(c, seed):
    x, y, a, b, cc, d = (t.double() for t in _device_inputs(c, seed))
    dt = c["dt"]

    def rhs(x, y):
        xy = x * y
        return a * x - b * xy, cc * xy - d * y

    for _ in range(c["steps"]):
        k1x, k1y = rhs(x, y)
        k2x, k2y = rhs(x + 0.5 * dt * k1x, y + 0.5 * dt * k1y)
        k3x, k3y = rhs(x + 0.5 * dt * k2x, y + 0.5 * dt * k2y)
        k4x, k4y = rhs(x + dt * k3x, y + dt * k3y)
        x = x + dt / 6.0 * (k1x + 2.0 * k2x + 2.0 * k3x + k4x)
        y = y + dt / 6.0 * (k1y + 2.0 * k2y + 2.0 * k3y + k4y)
    return x, y


def _gs64(c, seed):
    g = _gs_cfg()
    u, v = (torch.from_numpy(a).to(DEV).double() for a in _host_inputs(c, seed))
    f = lambda q: float(F32(q))  # noqa: E731
    du, dv, ff, fk, dt = f(g.du), f(g.dv), f(g.f), f(g.f + g.k), f(g.dt)
    for _ in range(c["steps"]):
        lu = torch.roll(u, 1, 0) + torch.roll(u, -1, 0) + torch.roll(u, 1, 1) + torch.roll(u, -1, 1) - 4.0 * u
        lv = torch.roll(v, 1, 0) + torch.roll(v, -1, 0) + torch.roll(v, 1, 1) + torch.roll(v, -1, 1) - 4.0 * v
        uvv = u * v * v
        u, v = u + dt * (du * lu - uvv + ff * (1.0 - u)), v + dt * (dv * lv + uvv - fk * v)
    return u.cpu().numpy(), v.cpu().numpy()


def _bs364(c, seed):
    """The adaptive solver in 64 bits: its states at the end (its step
    counts are its own, so they have no 64-bit value)."""
    cfg = workloads.BS3_CFG
    x, v, mu = (t.double() for t in _device_inputs(c, seed))
    t, dt, prev = torch.zeros_like(x), torch.full_like(x, cfg.dt0), torch.ones_like(x)
    c1, c2 = (cfg.icoeff + cfg.pcoeff) / 3, -cfg.pcoeff / 3

    def rhs(x, v):
        return v, mu * (1.0 - x * x) * v - x

    k1x, k1v = rhs(x, v)
    for it in range(8000):
        if it % 64 == 0 and bool((t >= cfg.t1).all()):
            break
        dt = torch.minimum(dt, cfg.t1 - t)
        k2x, k2v = rhs(x + 0.5 * dt * k1x, v + 0.5 * dt * k1v)
        k3x, k3v = rhs(x + 0.75 * dt * k2x, v + 0.75 * dt * k2v)
        yx = x + dt * (2 / 9 * k1x + 1 / 3 * k2x + 4 / 9 * k3x)
        yv = v + dt * (2 / 9 * k1v + 1 / 3 * k2v + 4 / 9 * k3v)
        k4x, k4v = rhs(yx, yv)
        ex = yx - (x + dt * (7 / 24 * k1x + 1 / 4 * k2x + 1 / 3 * k3x + 1 / 8 * k4x))
        ev = yv - (v + dt * (7 / 24 * k1v + 1 / 4 * k2v + 1 / 3 * k3v + 1 / 8 * k4v))
        err = torch.maximum(ex.abs() / (cfg.atol + cfg.rtol * yx.abs()), ev.abs() / (cfg.atol + cfg.rtol * yv.abs()))
        ok = err <= 1.0
        t, x, v = torch.where(ok, t + dt, t), torch.where(ok, yx, x), torch.where(ok, yv, v)
        k1x, k1v = torch.where(ok, k4x, k1x), torch.where(ok, k4v, k1v)
        inv = 1.0 / err.clamp(min=1e-9)
        dt = dt * torch.clamp(0.9 * inv**c1 * prev**c2, 0.2, 10.0)
        prev = torch.where(ok, inv, prev)
    return t, x, v, None, None


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("gbm", "gbm_fold"):
        return (_gbm64(c, seed),)
    if kind == "lv":
        return _lv64(c, seed)
    if kind == "df32":
        x, y = _lv64(c, seed)
        return x, None, y, None  # the low words hold what the high ones round away
    if kind == "bs3":
        return _bs364(c, seed)
    if kind in ("gs_steps", "gs_passes"):
        return _gs64(c, seed)
    if kind == "logistic":
        y, r = (a.astype(np.float64) for a in _host_inputs(c, seed))
        for _ in range(c["steps"]):
            y = y + float(F32(0.01)) * r * y * (1.0 - y)
        return y
    ins = [t.double() for t in _device_inputs(c, seed)]
    if kind == "softmax":
        return (torch.softmax(ins[0], dim=-1),)
    if kind == "pointwise":
        x, y = ins
        z = x * y + 0.1 * x - y / (x * x + 1.0)
        return (torch.where(z > 0, z * 3.0, z.abs() - 0.5),)
    a, w, b = ins
    return (torch.tanh(a @ w + b),)
