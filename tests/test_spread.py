"""Blocks spread over teams of lanes, on the CPU: which kernels take the
form, that its lanes cover every element once, and the forms it leaves to
the other lowerings. (The results are compared on the GPU.)"""

import re

import numpy as np
import pytest

import palladium_amd as pa
from palladium_amd.emit import RULES, emit_hip, launch_geometry
from palladium_amd.emit.core import plan_of
from palladium_amd.emit.lanes import LanePlan
from palladium_amd.emit.spread import MAX_LANES, MAX_SLOTS, ORDERED_LDS, SpreadPlan
from palladium_amd.frontend import jnp, lax, pl
from palladium_amd.frontend.core import current_builder
from palladium_amd.ir import ShapedArray
from palladium_amd.trace import trace
from spread_cases import CASES, CROSSED, LANE_ROWS, MOMENTS, OVERWRITTEN, OVERWRITTEN_WIDE

F = np.float32


def _spec(name):
    call, args = CASES[name](np.random.default_rng(1))
    return trace(call._staged, *args)


@pytest.mark.parametrize("name", sorted(CASES))
def test_every_element_has_one_lane(name):
    spec = _spec(name)
    plan = plan_of(spec)
    assert isinstance(plan, SpreadPlan)
    assert 1 < plan.lanes <= MAX_LANES and plan.slots <= MAX_SLOTS and plan.slots % plan.vec == 0
    if plan.tile:
        down, across = plan.tile
        seen = [(lane // 64 * 16 * down + 16 * a + 4 * (lane % 64 // 16) + i, 16 * b + lane % 16)
                for lane in range(plan.lanes) for a in range(down) for b in range(across) for i in range(4)]
        assert len(seen) == plan.lanes * plan.slots
        kept = [(r, c) for r, c in seen if r < plan.rows and c < plan.width]
        assert sorted(kept) == [(r, c) for r in range(plan.rows) for c in range(plan.width)]
        return
    seen = sorted(e for q in range(plan.chunks) for t in range(plan.team) for v in range(plan.vec)
                  if (w := (q * plan.team + t) * plan.vec) < plan.width for e in [w + v])
    assert seen == list(range(plan.width))
    m, w = plan.block
    assert plan.rows * plan.width == m * w
    geo = launch_geometry(spec)
    assert geo.lanes == plan.lanes and geo.block % 64 == 0
    assert geo.blocks * geo.block >= spec.num_programs * plan.lanes
    if plan.reduces:  # a team inside a wavefront, or a workgroup of its own
        assert plan.team & (plan.team - 1) == 0
        assert geo.block % plan.team == 0 and (plan.team <= 64 or geo.block == plan.team)


@pytest.mark.parametrize("name", ["flat_1250_bf16", "rows_8x128_f32", "rows_1x3000_f32", "loops_777", "indexed_6x130",
                                  "dense_128x64x32_f32", "dense_250x40x64_bf16", "two_dots_64x24x16"])
@pytest.mark.parametrize("mode", ["safe", "relaxed", "fast", "reproducible"])
def test_compiles_without_scratch(name, mode):
    call, args = CASES[name](np.random.default_rng(1), math_mode=mode)
    assert call.explain(*args).resources.scratch_bytes == 0


@pytest.mark.parametrize("name", sorted(MOMENTS))
def test_sums_of_a_kernel_share_their_staging(name):
    """At most one row array of ORDERED_LDS, and the exchanges of wide teams."""
    for mode in ("safe", "reproducible"):
        call, args = MOMENTS[name](np.random.default_rng(1), math_mode=mode)
        assert isinstance(plan_of(trace(call._staged, *args)), SpreadPlan)
        assert call.explain(*args).resources.lds_bytes <= ORDERED_LDS + 1024


def _huge(kind, grid, m, w, k=8):
    """A kernel over shapes alone."""
    def loop(x_ref, o_ref):
        o_ref[...] = lax.fori_loop(0, 5, lambda _, y: y * 0.5 + 1.0, x_ref[...])

    def softmax(x_ref, o_ref):
        e = jnp.exp(x_ref[...] - jnp.max(x_ref[...], axis=-1, keepdims=True))
        o_ref[...] = e / jnp.sum(e, axis=-1, keepdims=True)

    def dense(x_ref, w_ref, o_ref):
        o_ref[...] = jnp.dot(x_ref[...], w_ref[...])

    def block(m, w):
        return pl.BlockSpec((m, w), lambda i: (i, 0))

    specs, shapes = [block(m, w)], [(grid * m, w)]
    if kind == "dense":
        specs, shapes = [block(m, k), pl.BlockSpec((k, w), lambda i: (0, 0))], [(grid * m, k), (k, w)]
    kernel = {"loop": loop, "softmax": softmax, "dense": dense}[kind]
    call = pa.hip_call(kernel, grid=(grid,), in_specs=specs, out_specs=block(m, w),
                       out_shape=pl.ShapeDtypeStruct((grid * m, w), F))
    return trace(call._staged, *[pl.ShapeDtypeStruct(s, F) for s in shapes])


@pytest.mark.parametrize("kind, m, w", [("loop", 1, 100), ("loop", 1, 1000), ("loop", 4, 25), ("softmax", 1, 33),
                                        ("softmax", 1, 1000), ("softmax", 4, 100), ("dense", 32, 20), ("dense", 48, 64)])
def test_large_grids_stay_below_the_lane_limit(kind, m, w):
    """A launch has fewer than 2**31 lanes: with more instances each takes
    fewer, or one."""
    free = plan_of(_huge(kind, 1000, m, w))
    assert isinstance(free, SpreadPlan)
    edge = (2**31 - 1) // plan_of(_huge(kind, 200_000, m, w)).lanes
    for grid in (edge, edge + 1, 2 * edge, 2**31 // 3):
        spec = _huge(kind, grid, m, w)
        geo, plan = launch_geometry(spec), plan_of(spec)
        assert geo.lanes * grid < 2**31 and (plan is None) == (geo.lanes == 1)
        if grid == edge:
            assert isinstance(plan, SpreadPlan)
        emit_hip(spec, math_mode="fast")


@pytest.mark.parametrize("name", sorted(n for n in {**CASES, **MOMENTS} if n.startswith(("rows", "moments"))))
def test_a_team_stages_every_sum_in_its_own_bytes(name):
    """A wavefront may be a sum ahead of the others, in another type."""
    call, args = {**CASES, **MOMENTS}[name](np.random.default_rng(1))
    text = emit_hip(trace(call._staged, *args), math_mode="safe")
    rows = re.findall(r"\((\w+)\*\)_rows \+ \(threadIdx.x / (\d+)u\) \* (\d+)u;", text)
    alone = re.findall(r"\(\w+\*\)_rows \+ 0;", text)
    total = re.search(r"_rows\[(\d+)\];", text)
    if not rows and not alone:
        assert total is None
        return
    assert not (rows and alone)
    places = {(int(team), int(pitch) * (2 if t == "_Float16" else 4)) for t, team, pitch in rows}
    assert len(places) <= 1
    for team, pitch in places:
        plan = plan_of(trace(call._staged, *args))
        assert pitch >= 4 * plan.width and pitch * (launch_geometry(trace(call._staged, *args)).block // team) <= int(total[1])


@pytest.mark.parametrize("name, rounds", [("flat_250_bf16", True), ("flat_1250_bf16", True), ("flat_wide_bf16", True),
                                          ("flat_100_f16", False), ("flat_5001_f32", False), ("rows_64x8_f32", False),
                                          ("rows_8x100_bf16", True), ("dense_250x40x64_bf16", True),
                                          ("dense_33x1x40_bf16", True), ("dense_64x32x30_bf16", False)])
def test_bfloat16_operations_are_not_regrouped(name, rounds):
    """Where one lane kept a block of bfloat16 values in memory, FAST and
    RELAXED round every operation, as the interpreter does."""
    for mode in ("fast", "relaxed"):
        text = emit_hip(_spec(name), math_mode=mode)
        assert all((f"= ph_bf16_{op}(" in text) == rounds for op in (("add",) if "dense" in name else ("add", "mul", "sub")))
    assert "ph_bf16_" not in emit_hip(_spec(name), math_mode="safe")


def _row_call(kernel, m=4, w=64, out=None, **kw):
    s = pl.BlockSpec((m, w), lambda i: (i, 0))
    return pa.hip_call(kernel, grid=(3,), in_specs=[s], out_specs=s, out_shape=pl.ShapeDtypeStruct((3 * m, w), F), **kw)


def _read_back(x_ref, o_ref):
    o_ref[...] = x_ref[...]
    o_ref[0, :] = o_ref[1, :] * 2.0


def _across_rows(x_ref, o_ref):
    o_ref[...] = x_ref[...] - jnp.sum(x_ref[...], axis=0, keepdims=True)


def _transposed(x_ref, o_ref):
    o_ref[...] = x_ref[...] + jnp.reshape(x_ref[...].T, (4, 64))


def _part(x_ref, o_ref):
    o_ref[0:2, :] = x_ref[0:2, :] * 2.0
    o_ref[2:4, :] = x_ref[2:4, :]


def _exchange(x_ref, o_ref):
    """A store that returns what the element held."""
    tree, leaves = o_ref._indexer((0, 0))
    (old,) = current_builder().add("swap", [o_ref._t, x_ref[0, 0] * 2.0, *leaves], [ShapedArray((), F)], tree=tree)
    o_ref[...] = x_ref[...] + old


@pytest.mark.parametrize("kernel", [_read_back, _across_rows, _transposed, _part, _exchange])
def test_other_forms_keep_their_lowering(kernel):
    """An output read where another lane wrote it, a reduction across rows,
    a transpose, part of a block, a store whose old value is used."""
    spec = trace(_row_call(kernel)._staged, np.zeros((12, 64), F))
    assert not isinstance(plan_of(spec), SpreadPlan)
    emit_hip(spec, math_mode="fast")


@pytest.mark.parametrize("name", sorted({**OVERWRITTEN, **OVERWRITTEN_WIDE, **CROSSED}))
def test_stores_of_one_element_stay_in_one_lane(name):
    """Lanes are not ordered: an element that two stores write has one lane."""
    call, args = {**OVERWRITTEN, **OVERWRITTEN_WIDE, **CROSSED}[name](np.random.default_rng(1))
    assert not isinstance(plan_of(trace(call._staged, *args)), SpreadPlan)


@pytest.mark.parametrize("mode", ["safe", "relaxed", "fast", "reproducible"])
@pytest.mark.parametrize("name", sorted(LANE_ROWS))
def test_lane_rows_are_synchronised_where_lanes_meet(name, mode):
    """Lane 0's stores, and what every lane reads, stand between barriers
    (of the wavefront, where it is the whole instance)."""
    call, args = LANE_ROWS[name](np.random.default_rng(1))
    spec = trace(call._staged, *args)
    plan = plan_of(spec)
    assert isinstance(plan, LanePlan)
    lines = emit_hip(spec, math_mode=mode).split('extern "C"')[-1].splitlines()
    sync = ("__syncthreads();",) if plan.lanes > 64 else ("__builtin_amdgcn_wave_barrier();",
                                                          '__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");')
    guards = [i for i, x in enumerate(lines) if x.lstrip().startswith("if (_lane == 0) {")]
    assert guards
    for i in guards:
        end = next(j for j in range(i, len(lines)) if lines[j] == lines[i].replace("if (_lane == 0) {", "}"))
        assert lines[i - 1].strip() in sync and lines[end + 1].strip() in sync


def test_lane_rows_of_their_own_need_no_barrier():
    def kernel(x_ref, o_ref, s_ref):
        x = x_ref[...]
        o_ref[...] = x
        o_ref[...] = o_ref[...] * 2.0
        s_ref[0] = 1.0
        s_ref[1] = 2.0

    s = pl.BlockSpec((128, 2), lambda i: (i, 0))
    call = pa.hip_call(kernel, grid=(4,), in_specs=[s], out_specs=(s, pl.BlockSpec((2,), lambda i: (i,))),
                       out_shape=(pl.ShapeDtypeStruct((512, 2), F), pl.ShapeDtypeStruct((8,), F)))
    spec = trace(call._staged, np.zeros((512, 2), F))
    assert isinstance(plan_of(spec), LanePlan)
    text = emit_hip(spec, math_mode="safe")
    assert "__syncthreads" not in text and "wave_barrier" not in text


def test_disjoint_stores_of_one_output_are_spread():
    def kernel(x_ref, o_ref):
        x = x_ref[...]
        o_ref[:, 0] = jnp.sum(x, axis=1)  # both by the first lane of a row
        o_ref[:, 1] = jnp.max(x, axis=1)
        o_ref[3, 2] = 3.0  # by lane 0, another column

    call = pa.hip_call(kernel, grid=(3,), in_specs=[pl.BlockSpec((4, 40), lambda i: (i, 0))],
                       out_specs=pl.BlockSpec((4, 3), lambda i: (i, 0)), out_shape=pl.ShapeDtypeStruct((12, 3), F))
    assert isinstance(plan_of(trace(call._staged, np.zeros((12, 40), F))), SpreadPlan)


@pytest.mark.parametrize("name, primitive", [("dense_64x21x17_f32", "dot_general"), ("dense_33x7x33_f16", "dot_general"),
                                             ("rows_8x128_f32", "reduce_max"), ("flat_1000_u32", "get")])
def test_a_rule_of_ones_own_keeps_its_say(name, primitive, monkeypatch):
    built_in = RULES[primitive]

    def own(env, cursor, eqn):
        cursor.emit("// the user's rule")
        built_in(env, cursor, eqn)

    spec = _spec(name)
    assert isinstance(plan_of(spec), SpreadPlan)
    monkeypatch.setitem(RULES, primitive, own)
    assert "// the user's rule" in emit_hip(spec, math_mode="fast")
    assert not isinstance(plan_of(spec), SpreadPlan)


@pytest.mark.parametrize("name, block, taken", [
    *((n, b, b) for n in ("rows_4x17_f32", "rows_8x128_f32", "rows_64x40_f32", "flat_1250_bf16", "dense_64x21x17_f32")
      for b in (64, 512, 1024)),
    ("rows_1x1000_f32", 64, 256), ("rows_1x1000_f32", 1024, 256),  # a team of 256 is a workgroup
    ("moments_64x900_3_f32", 1024, 256)])  # 230 KB of rows
def test_the_workgroup_asked_for(name, block, taken):
    call, args = {**CASES, **MOMENTS}[name](np.random.default_rng(1), threadgroup=block, math_mode="safe")
    diag = call.explain(*args)
    assert diag.block == taken and diag.blocks * diag.block >= trace(call._staged, *args).num_programs * diag.lanes
    assert diag.resources.lds_bytes <= ORDERED_LDS + 1024


def test_small_blocks_and_plain_gridless_calls_keep_one_lane():
    def double(x_ref, o_ref):
        o_ref[...] = x_ref[...] * 2.0

    s = pl.BlockSpec((15,), lambda i: (i,))
    small = pa.hip_call(double, grid=(4,), in_specs=[s], out_specs=s, out_shape=pl.ShapeDtypeStruct((60,), F))
    assert plan_of(trace(small._staged, np.zeros(60, F))) is None
    whole = pa.hip_call(double, out_shape=pl.ShapeDtypeStruct((4096,), F))
    assert plan_of(trace(whole._staged, np.zeros(4096, F))) is None
