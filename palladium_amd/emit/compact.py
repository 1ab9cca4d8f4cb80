"""Workgroup lane compaction for divergent `while_loop`s.

An adaptive solver's per-lane `while_loop` keeps a wavefront issuing until
its slowest lane finishes; on config 2 (Van der Pol, mu log-uniform) half
the lane-attempts of a wavefront do no work. When a kernel's loop runs one
program instance per lane with nothing lane-specific inside it, the
instance is only its loop state: the carries and the loop's operands. Then
the state of a live instance can move to another lane, and a workgroup (256
to 1,024 lanes, see `workgroup_for`) can repack its live instances into its
lowest wavefronts every `EPOCH` iterations, so emptied wavefronts stop
issuing:

    epoch:  run up to EPOCH predicated iterations (a wavefront leaves the
            epoch early once none of its lanes is live);
            lanes whose instance finished store its carries in LDS at the
            instance's own slot;
            count the live lanes per wavefront (ballot, popcount);
            if packing frees a wavefront, live lanes write their state to
            LDS at their rank among the live (prefix over wavefronts +
            mbcnt) and lanes [0, live) read it back;
            stop when no lane of the workgroup is live.
    after:  every lane reloads its own instance's final carries.

Two things bound such a kernel: the iterations issued, and the one instance
with the most of them, whose wavefront is latency-bound (BS3: a SIMD with w
waves takes 137 + 117 w ns for an iteration of each, a lone wave 290 ns, and
2,646 iterations lie between start and end of the longest instance). In
lockstep epochs a long instance runs at the pace of the four waves on its
SIMD while they last, and alone afterwards. Where the loop's condition tells
how far an instance is (a float carry that starts at a constant and stays
below a bound), each epoch ends with an estimate of its remaining iterations,
(bound - carry) / progress per iteration so far; a histogram of the estimates
in LDS gives the line above which the longest 256 lie, these move to the
first four wavefronts (one a SIMD) and get three epochs' iterations to the
others' one (four in SAFE). The estimate only places instances: a wrong one costs time and
changes no result.

Each instance runs exactly the operations it ran before, in the same
order: results are bit-identical with and without compaction. Wavefront w
of a 1,024-lane workgroup shares its SIMD with w ± 4, w ± 8 ... (measured
on MI355X: consecutive wavefronts land on the CU's four SIMDs in turn), so
packing into the lowest wavefronts keeps the four SIMDs evenly loaded.

The control flow around each barrier is uniform over the workgroup (the
epoch loop stops on a count read from LDS), and no lane returns early (a
grid that does not fill its last workgroup keeps the extra lanes, which
hold no instance), so every wavefront meets every barrier.
"""

from __future__ import annotations

import dataclasses
import os
import re
from typing import Any

import numpy as np

from palladium_amd.ir import KeyAval, Literal, Var

WORKGROUP = 1024
EPOCH = 64
# Loop iterations per pass of the epoch loop (see emit_compacting_while), by
# math mode. More iterations per pass spread the pass's counter and branch
# over more attempts; SAFE's deterministic pow makes its iteration about 2.5
# times FAST's code, and past 16 of them its loop no longer fits the
# instruction cache two CUs share (64 KiB). Measured on BS3: FAST 0.698 /
# 0.690 / 0.673 / 0.667 / 0.659 / 0.652 ms at 1 / 2 / 4 / 8 / 16 / 32, SAFE
# 2.14 / 2.13 / 2.10 / 2.08 / 2.07 / 2.08, SAFE 2.12 at 64.
EPOCH_UNROLL = {"safe": 16, "other": 32}


# A pass holds at most this many traced operations of the loop body, so that
# a large body is not copied 32 times (code size, compile time).
EPOCH_UNROLL_OPS = 4096


def _count_eqns(j: Any) -> int:
    n = 0
    for e in j.eqns:
        n += 1
        for v in e.params.values():
            for sub in (v if isinstance(v, tuple) else (v,)):
                if hasattr(getattr(sub, "jaxpr", sub), "eqns"):
                    n += _count_eqns(getattr(sub, "jaxpr", sub))
    return n


def iterations_per_pass(hip_source: str) -> int:
    """The iterations per machine-loop pass the emitter chose for a
    compacted while loop in `hip_source` (1 if it has none)."""
    import re

    m = re.search(r"// (\d+) iterations per pass", hip_source)
    return int(m.group(1)) if m else 1


def epoch_unroll(math_mode: Any = None, body: Any = None) -> int:
    """Iterations of a compacted while loop per pass of its machine loop:
    the math mode's default, halved until the pass holds at most
    EPOCH_UNROLL_OPS of `body`'s operations (`PALLADIUM_EPOCH_UNROLL`
    overrides both)."""
    from palladium_amd.runtime import math_mode_ordinal

    raw = os.environ.get("PALLADIUM_EPOCH_UNROLL")
    if raw is not None:
        u = int(raw)
        if u < 1 or EPOCH % u:
            raise ValueError(f"PALLADIUM_EPOCH_UNROLL={u} must divide the epoch of {EPOCH} iterations")
        return u
    safe = math_mode is None or math_mode_ordinal(math_mode) in (0, 3)
    u = EPOCH_UNROLL["safe" if safe else "other"]
    n = _count_eqns(getattr(body, "jaxpr", body)) if body is not None else 0
    while u > 1 and u * n > EPOCH_UNROLL_OPS:
        u //= 2
    return u
# LDS per workgroup the compaction may use (2 workgroups per CU fit in 160 KB).
LDS_BUDGET = 78 * 1024

_LANE_SPECIFIC = {"program_id", "num_programs", "get", "swap", "lane_index", "lane_reduce", "while"}
# dtype -> 32-bit LDS words per value
_STORABLE = {"float32": 1, "int32": 1, "uint32": 1, "bool": 1, "float64": 2}


@dataclasses.dataclass(frozen=True)
class CompactPlan:
    index: int  # position of the loop among the top-level eqns
    workgroup: int  # lanes that repack together


def _jaxpr(j: Any) -> Any:
    return getattr(j, "jaxpr", j)


def _lane_free(jaxpr: Any) -> bool:
    for e in _jaxpr(jaxpr).eqns:
        if e.primitive.name in _LANE_SPECIFIC:
            return False
        for v in e.params.values():
            for sub in (v if isinstance(v, tuple) else (v,)):
                if hasattr(_jaxpr(sub), "eqns") and not _lane_free(sub):
                    return False
    return True


def _storable(v: Any) -> bool:
    aval = getattr(v, "aval", None)
    if aval is None or isinstance(aval, KeyAval):
        return False
    if int(np.prod(aval.shape)) != 1:
        return False
    return np.dtype(aval.dtype).name in _STORABLE


def enabled() -> bool:
    return os.environ.get("PALLADIUM_WHILE_COMPACTION", "1") != "0"


def workgroup_for(instances: int) -> int:
    """Lanes that repack together. Above 131,072 instances (two wavefronts on
    each of the 1,024 SIMDs) whole 1,024-lane workgroups, whose four waves a
    SIMD pack best. Below, a large workgroup crowds its waves onto one CU
    while others stand empty: BS3 (REPRODUCIBLE, 2,646 attempts at most) in
    1,024 / 512 / 256 lanes takes 1,155 / 883 / 782 us at 65,536 instances and
    1,132 / 869 / 778 at 5,000; ranked by progress (`_ranking`) 1,024 / 512
    lanes take 882 / 803 us at 131,072 and 892 / 1,004 at 262,144. Up to 4,096
    instances the geometry is the documented one, 1,024 lanes, which is not the
    fastest (ranked, 1,000 instances take 792 us, 5,000 in 256 lanes 692)."""
    if instances <= 4096 or instances > 131_072:
        return WORKGROUP
    return 256 if instances <= 65_536 else 512


def plan_for(spec: Any, jaxpr: Any, lanes: int, block: int | None) -> CompactPlan | None:
    """The loop to compact, or None. Needs: one lane per instance, a 1-D
    grid, no explicit workgroup size other than 1,024, and exactly one
    top-level `while` whose condition and body touch no ref, program id or
    nested while, with scalar 4-byte-or-bool carries and operands. A grid
    that does not fill whole workgroups keeps its extra lanes: they read
    the last instance's data, never enter the loop and store nothing."""
    if not enabled() or lanes != 1 or len(spec.grid) != 1:
        return None
    if block not in (None, WORKGROUP):
        return None
    whiles = [k for k, e in enumerate(jaxpr.eqns) if e.primitive.name == "while"]
    if len(whiles) != 1:
        return None
    e = jaxpr.eqns[whiles[0]]
    if getattr(e.params["cond_jaxpr"], "consts", None) or getattr(e.params["body_jaxpr"], "consts", None):
        return None
    if not (_lane_free(e.params["cond_jaxpr"]) and _lane_free(e.params["body_jaxpr"])):
        return None
    if not all(_storable(v) for v in list(e.invars) + list(e.outvars)):
        return None
    used = {v for x in jaxpr.eqns for v in x.invars} | set(jaxpr.outvars)
    n_state = sum(_nwords(v) for v in e.invars) + 1  # operands and carries, plus the slot index
    n_kept = sum(_nwords(v) for v in e.outvars if v in used)  # final carries read after the loop
    if (n_state + n_kept) * WORKGROUP * 4 > LDS_BUDGET:
        return None
    return CompactPlan(whiles[0], block or workgroup_for(spec.num_programs))


def _nwords(v: Any) -> int:
    return _STORABLE[np.dtype(v.aval.dtype).name]


def _store(arr: str, j: int, pos: str, c: Any) -> tuple[list[str], int]:
    """Lines writing value `c` to rows j, j+1, ... of LDS array `arr` at
    column `pos`, and the next free row."""
    e, t = c.expr, c.ctype
    if t == "double":
        bits = f"(unsigned long long)__double_as_longlong({e})"
        return [f"{arr}[{j}][{pos}] = (unsigned int)({bits});",
                f"{arr}[{j + 1}][{pos}] = (unsigned int)(({bits}) >> 32);"], j + 2
    if t == "float":
        word = f"__float_as_uint({e})"
    elif t == "bool":
        word = f"({e} ? 1u : 0u)"
    else:
        word = f"(unsigned int)({e})"
    return [f"{arr}[{j}][{pos}] = {word};"], j + 1


def _load(arr: str, j: int, pos: str, c: Any) -> tuple[str, int]:
    """The line reading `c` back from rows j, ... of `arr`, and the next row."""
    e, t = c.expr, c.ctype
    if t == "double":
        return (f"{e} = __longlong_as_double((long long)(((unsigned long long){arr}[{j + 1}][{pos}] << 32)"
                f" | (unsigned long long){arr}[{j}][{pos}]));"), j + 2
    w = f"{arr}[{j}][{pos}]"
    if t == "float":
        return f"{e} = __uint_as_float({w});", j + 1
    if t == "bool":
        return f"{e} = ({w} != 0u);", j + 1
    return f"{e} = ({t})({w});", j + 1


def _progress(eqn: Any, producers: dict) -> tuple[int, Any, float] | None:
    """(carry, bound, start) when the loop runs while a float32 carry that
    starts at a literal stays below a bound (an integrator's time, say); the
    bound is a literal or one of the condition's operands."""
    cn, bn = int(eqn.params["cond_nconsts"]), int(eqn.params["body_nconsts"])
    cj = _jaxpr(eqn.params["cond_jaxpr"])
    made = {ov: e for e in cj.eqns for ov in e.outvars}
    todo, tests = [cj.outvars[0]], []
    while todo:
        v = todo.pop()
        e = made.get(v) if isinstance(v, Var) else None
        if e is None:
            continue
        if e.primitive.name == "and":
            todo.extend(e.invars)
        elif e.primitive.name in ("lt", "le"):
            tests.append((e.invars[0], e.invars[1]))
        elif e.primitive.name in ("gt", "ge"):
            tests.append((e.invars[1], e.invars[0]))
    carries = {v: k for k, v in enumerate(cj.invars[cn:])}
    for low, high in tests:
        if not isinstance(low, Var) or low not in carries or np.dtype(low.aval.dtype) != np.float32:
            continue
        if not isinstance(high, Literal) and high not in cj.invars[:cn]:
            continue
        start = eqn.invars[cn + bn + carries[low]]
        while isinstance(start, Var):
            e = producers.get(start)
            start = e.invars[0] if e is not None and e.primitive.name == "broadcast_in_dim" else None
        if isinstance(start, Literal):
            return carries[low], high, float(start.val)
    return None


def _rows(vals: list) -> int:
    return sum(2 if c.ctype == "double" else 1 for c in vals)


# Ranking by progress: bins of the estimate (eight an octave), waves that take
# the instances with the most to do, and their epochs in those of the others.
RANK_BINS = 256
RANK_WAVES = 4
# math mode -> epochs. BS3 in 2 / 3 / 4 of them: REPRODUCIBLE 946 / 851 / 865 us
# at 262,144 instances, 3,710 / 3,378 / 3,412 at 1,048,576; SAFE, whose lone
# wave is slower against four, 1,640 / 1,515 / 1,492 and 6,460 / 6,036 / 5,758.
RANK_TURNS = {0: 4, 1: 3, 3: 3}
# Ranked only while the estimates' quartiles lie this many bins apart: with
# trip counts within 10 % of each other two or one bins would rank as well, and
# cost 10-60 % (563 -> 637 us, 77 -> 129).
RANK_SPREAD = 3
# The smallest body (equations) that is ranked. The counting costs 6-15 us a
# kernel whatever the body holds: 135 -> 141 us with 18 equations, 201 -> 205
# with 34, 526 -> 522 with 130 (1,000 trips each, 262,144 instances), while
# trip counts spread over 100-3,000 gain from 18 equations on in SAFE
# (261 -> 248, 557 -> 507, 952 -> 841 us with 18, 66, 130).
RANK_OPS = 64


def _ranking(env: Any, eqn: Any, workgroup: int, rows: int) -> tuple | None:
    """`_progress(eqn)` where ranking pays, else None: in workgroups of more
    than 256 lanes, where a SIMD holds more than one wave, and with room in LDS
    for the counts. BS3 unranked / ranked, REPRODUCIBLE and SAFE: 991 / 792 and
    1,745 / 1,357 us at 1,000 instances, 782 / 692 and 1,343 / 1,149 at 131,072
    (workgroups of 512), 1,065 / 851 and 1,864 / 1,492 at 262,144, 4,210 /
    3,378 and 7,375 / 5,758 at 1,048,576. FAST keeps its order: its text is
    held as a snapshot (672 -> 533 us when it is ranked)."""
    from palladium_amd.runtime import math_mode_ordinal

    mode = getattr(env, "math_mode", None)
    if mode is None or math_mode_ordinal(mode) not in RANK_TURNS or workgroup <= 256:
        return None
    if rows * workgroup * 4 + RANK_BINS * 4 > LDS_BUDGET or _count_eqns(_jaxpr(eqn.params["body_jaxpr"])) < RANK_OPS:
        return None
    found = _progress(eqn, env.producers)
    return None if found is None else (*found, EPOCH * RANK_TURNS[math_mode_ordinal(mode)])


# Functions with a branch for operands off their common path, by math mode; a
# form without it adds the lanes that need it to a mask (emit/prelude.py). A
# body with two of these branches or more runs on the common paths, with one
# branch an iteration that leaves the state untaken; the rest of that epoch
# then runs the full functions. A branch costs the lone wave its latency and
# keeps the scheduler from overlapping what stands on both sides of it: BS3
# REPRODUCIBLE (five branches -> one) 774 -> 692 us at 5,000 instances, 902 ->
# 851 at 262,144, SAFE (three -> one) 1,184 -> 1,101 and 1,554 -> 1,515. With
# one branch in the body there is nothing to merge. FAST has none.
_CHECKED = {
    0: re.compile(r"\bph_(?:pow|pow_log|pow_with_log)\("),
    3: re.compile(r"\bph_(?:rdiv|rrcp|rpow|dlog2f|dexp2f|exp|log)\("),
}


def _checked(env: Any) -> Any:
    """The pattern of such functions in this math mode, or None."""
    from palladium_amd.runtime import math_mode_ordinal

    mode = getattr(env, "math_mode", None)
    return _CHECKED.get(math_mode_ordinal(mode)) if mode is not None else None


def _rank_in(mask: str) -> str:
    """This lane's place among the set bits of a wavefront's `mask`."""
    return (f"(int)__builtin_amdgcn_mbcnt_hi((unsigned int)({mask} >> 32), "
            f"__builtin_amdgcn_mbcnt_lo((unsigned int){mask}, 0u))")


RANK_PRELUDE = r"""
/* The smallest bin (of 256) from which on at most `most` of the `live`
   instances are counted, or 256 unless the quartiles lie at least `spread`
   bins apart. Lane l sums bins 4 l .. 4 l + 3, then those of
   the lanes above it; every wavefront gets the same answer. */
__device__ __forceinline__ int ph_rank_cut(const unsigned int* hist, int live, int most, int spread) {
    const int lane = (int)(threadIdx.x & 63u);
    int c[4], above = 0;
    for (int i = 0; i < 4; ++i) { c[i] = (int)hist[4 * lane + i]; above += c[i]; }
    int sum = -above;
    for (int off = 1; off < 64; off *= 2) {
        const int up = __shfl_down(above, off);
        above += lane + off < 64 ? up : 0;
    }
    sum += above;  /* in the bins of higher lanes */
    int cut = 256, upper = 256, lower = 256;
    for (int i = 3; i >= 0; --i) {
        sum += c[i];
        if (sum <= most) cut = 4 * lane + i;
        if (4 * sum <= live) upper = 4 * lane + i;
        if (4 * sum <= 3 * live) lower = 4 * lane + i;
    }
    for (int off = 32; off > 0; off /= 2) {
        const int c2 = __shfl_xor(cut, off), u2 = __shfl_xor(upper, off), l2 = __shfl_xor(lower, off);
        cut = c2 < cut ? c2 : cut;
        upper = u2 < upper ? u2 : upper;
        lower = l2 < lower ? l2 : lower;
    }
    return upper - lower >= spread ? cut : 256;
}
"""


def emit_compacting_while(env: Any, cursor: Any, eqn: Any, emit_jaxpr: Any, declare_carries: Any,
                          copy_back: Any) -> None:
    """Emit `eqn` (a top-level `while`) with workgroup lane compaction."""
    cn = int(eqn.params["cond_nconsts"])
    bn = int(eqn.params["body_nconsts"])
    cj = _jaxpr(eqn.params["cond_jaxpr"])
    bj = _jaxpr(eqn.params["body_jaxpr"])
    # The loop's operands move with their instance: private copies.
    consts = []
    for v in eqn.invars[: cn + bn]:
        src = env.val(v)
        name = cursor.fresh("_k")
        cursor.emit(f"{src.ctype} {name} = {src.at('0')};")
        consts.append(dataclasses.replace(src, expr=name, space="local", readonly=False))
    cond_consts, body_consts = consts[:cn], consts[cn:]
    carries = declare_carries(env, cursor, eqn.invars[cn + bn:], eqn.outvars)
    state = consts + carries
    kept = [(k, c) for k, (c, ov) in enumerate(zip(carries, eqn.outvars)) if env.used(ov)]
    workgroup = env.compact_workgroup
    nw = workgroup // 64
    buf, res, cnt = cursor.fresh("_cbuf"), cursor.fresh("_cres"), cursor.fresh("_ccnt")
    kept_vals = [c for _, c in kept]
    ranked = _ranking(env, eqn, workgroup, _rows(state) + _rows(kept_vals) + 2)
    if ranked is not None:
        done = cursor.fresh("_done")
        cursor.emit(f"unsigned int {done} = 0u;  // iterations this lane's instance has been given")
        state = state + [dataclasses.replace(carries[0], expr=done, shape=(), ctype="unsigned int")]
        hist, lcnt, limit, turn, due, look = (
            cursor.fresh(p) for p in ("_chist", "_clong", "_climit", "_cturn", "_cdue", "_clook"))
        cursor.emit(f"__shared__ unsigned int {hist}[{RANK_BINS}];")
        cursor.emit(f"__shared__ int {lcnt}[{nw}];")
        cursor.emit(f"if (threadIdx.x < {RANK_BINS}u) {hist}[threadIdx.x] = 0u;")
        cursor.emit("__syncthreads();")
        cursor.emit(f"int {limit} = {EPOCH}, {turn} = 0, {due} = 1;")
    n_rows = _rows(state)
    cursor.emit(f"__shared__ unsigned int {buf}[{n_rows + 1}][{workgroup}];")
    if kept:
        cursor.emit(f"__shared__ unsigned int {res}[{_rows(kept_vals)}][{workgroup}];")
    cursor.emit(f"__shared__ int {cnt}[{nw}];")
    slot, own = cursor.fresh("_slot"), cursor.fresh("_own")
    first = f"(_in ? (int)threadIdx.x : -1)" if getattr(env, "compact_in", None) else "(int)threadIdx.x"
    cursor.emit(f"int {slot} = {first};  // the instance this lane holds; -1: none")
    wave = cursor.fresh("_wv")
    cursor.emit(f"const int {wave} = (int)(threadIdx.x >> 6);")
    with cursor.block("while (true)"):
        ep = cursor.fresh("_ep")
        unroll = epoch_unroll(getattr(env, "math_mode", None), bj)
        cursor.emit(f"// {unroll} iterations per pass")
        from palladium_amd.emit.rules import select_guards

        def iteration(odd: str | None) -> list[str]:
            """One iteration, and its body's lines: with `odd`, on the common
            paths of its checked functions, left untaken where a live lane
            needs another."""
            (pred,) = emit_jaxpr(env, cursor, cj, cond_consts + carries)
            live = cursor.fresh("_live")
            cursor.emit(f"const bool {live} = ({pred.at('0')}) && {slot} >= 0;")
            # (the ballot of a bool tests the compare's own mask; __any goes
            # through an int and a second compare)
            none = f"!__any({live})" if odd is None else f"__builtin_amdgcn_ballot_w64({live}) == 0ull"
            with cursor.block(f"if ({none})"):
                cursor.emit("break;")
            first = len(cursor.lines)
            outs = emit_jaxpr(env, cursor, bj, body_consts + carries)
            body = cursor.lines[first:]
            if odd is not None:
                name = cursor.fresh(odd)
                cursor.lines[first:] = ["    " * cursor.indent + f"unsigned long long {name} = 0ull;",
                                        *(names.sub(rf"\g<0>{name}, ", line) for line in body)]
                with cursor.block(f"if (__builtin_expect(({name} & __builtin_amdgcn_ballot_w64({live})) != 0ull, 0))"):
                    cursor.emit(f"{odd} = true;")
                    cursor.emit("break;")
            copy_back(cursor, outs, carries, predicate=live, guards=select_guards(env, bj, bn))
            return body

        trips = EPOCH if ranked is None else limit
        names, odd, full = _checked(env), None, []
        if names is not None:
            # the rest of an epoch that met an odd lane
            first = len(cursor.lines)
            with cursor.block(f"for (; {ep} < {trips}; ++{ep})"):
                body = iteration(None)
            full = cursor.lines[first:]
            del cursor.lines[first:]
            if not any("{" in line for line in body) and sum(len(names.findall(line)) for line in body) >= 2:
                odd = cursor.fresh("_odd")
                cursor.emit(f"bool {odd} = false;")
                cursor.emit(f"int {ep} = 0;")
        # `unroll` iterations per pass, each with its own exit test (a break
        # in any of them leaves the epoch): the pass's counter and branch are
        # shared among them.
        with cursor.block(f"for ({'' if odd else f'int {ep} = 0'}; {ep} < {trips}; {ep} += {unroll})"):
            for _ in range(unroll):
                iteration(odd)
        if odd is not None:
            with cursor.block(f"if ({odd})"):
                cursor.lines.extend(full)
        # Epoch boundary: the same condition, on the state as it stands.
        (pred,) = emit_jaxpr(env, cursor, cj, cond_consts + carries)
        cursor.emit(f"bool {own} = ({pred.at('0')}) && {slot} >= 0;")
        with cursor.block(f"if (!{own} && {slot} >= 0)"):
            j = 0
            for c in kept_vals:
                lines, j = _store(res, j, slot, c)
                for line in lines:
                    cursor.emit(line)
            cursor.emit(f"{slot} = -1;")
        if ranked is not None:
            from palladium_amd.emit.core import literal_cval

            k, bound, start, long_epoch = ranked
            edge = env.val(bound) if isinstance(bound, Literal) else cond_consts[cj.invars.index(bound)]
            est, bin_ = cursor.fresh("_cest"), cursor.fresh("_cbin")
            v = carries[k].at("0")
            cursor.emit(f"{done} += (unsigned int){limit};")
            cursor.emit(f"const bool {look} = ++{turn} >= {due};")
            cursor.emit(f"int {bin_} = 0;")
            with cursor.block(f"if ({look})"):
                # Iterations left at the instance's average rate so far; NaN
                # and no progress yet go to the last bin.
                cursor.emit(f"const float {est} = ({edge.at('0')} - {v}) * (float){done}"
                            f" * __builtin_amdgcn_rcpf({v} - {literal_cval(start, np.float32).expr});")
                cursor.emit(f"{bin_} = {est} < 1.0f ? 0 : ({est} < {float(2 ** (RANK_BINS // 8 - 1)):.1f}f"
                            f" ? (int)(__float_as_uint({est}) >> 20) - {127 * 8} : {RANK_BINS - 1});")
                cursor.emit(f"if ({own}) atomicAdd(&{hist}[{bin_}], 1u);")
        mask, total, before, active = (cursor.fresh(p) for p in ("_cm", "_ctot", "_cbef", "_cact"))
        cursor.emit(f"const unsigned long long {mask} = __ballot({own});")
        with cursor.block("if ((threadIdx.x & 63u) == 0u)"):
            cursor.emit(f"{cnt}[{wave}] = (int)__popcll({mask});")
        cursor.emit("__syncthreads();")
        cursor.emit(f"int {total} = 0, {before} = 0, {active} = 0;")
        w = cursor.fresh("_cw")
        with cursor.block(f"for (int {w} = 0; {w} < {nw}; ++{w})"):
            cursor.emit(f"const int _c = {cnt}[{w}];")
            cursor.emit(f"{total} += _c; {before} += ({w} < {wave}) ? _c : 0; {active} += (_c > 0) ? 1 : 0;")
        with cursor.block(f"if ({total} == 0)"):
            cursor.emit("break;")
        # Repack only when it frees a wavefront (the decision is uniform).
        repack = f"({total} + 63) / 64 < {active}"
        place = f"{before} + {_rank_in(mask)}"
        if ranked is not None:
            rank, lmask, nlong, lbefore = (cursor.fresh(p) for p in ("_crank", "_clm", "_cnl", "_clb"))
            cursor.emit(f"bool {rank} = false;")
            cursor.emit(f"unsigned long long {lmask} = 0ull;")
            cursor.emit(f"int {nlong} = 0, {lbefore} = 0;")
            with cursor.block(f"if ({look} && {total} > {64 * RANK_WAVES})"):
                cut = cursor.fresh("_ccut")
                cursor.emit(f"const int {cut} = ph_rank_cut({hist}, {total}, {64 * RANK_WAVES}, {RANK_SPREAD});")
                cursor.emit(f"{rank} = {cut} < {RANK_BINS};")
                cursor.emit(f"{due} = {rank} ? {turn} + 1 : 4 * {turn};")
                with cursor.block(f"if ({rank})"):
                    cursor.emit(f"{lmask} = __ballot({own} && {bin_} >= {cut});")
                    cursor.emit(f"if ((threadIdx.x & 63u) == 0u) {lcnt}[{wave}] = (int)__popcll({lmask});")
                cursor.emit("__syncthreads();")  # also: every wave has read the histogram
                w2 = cursor.fresh("_cw")
                with cursor.block(f"for (int {w2} = 0; {rank} && {w2} < {nw}; ++{w2})"):
                    cursor.emit(f"{nlong} += {lcnt}[{w2}]; {lbefore} += ({w2} < {wave}) ? {lcnt}[{w2}] : 0;")
            with cursor.block("else"):
                cursor.emit(f"{due} = {look} ? 2147483647 : {due};")  # not again: the count only falls
            repack = f"{rank} || {repack}"
            slow = f"({mask} & ~{lmask})"
            place = (f"(({lmask} >> (threadIdx.x & 63u)) & 1ull) ? {lbefore} + {_rank_in(lmask)}"
                     f" : {nlong} + ({before} - {lbefore}) + {_rank_in(slow)}")
        with cursor.block(f"if ({repack})"):
            with cursor.block(f"if ({own})"):
                pos = cursor.fresh("_cpos")
                cursor.emit(f"const int {pos} = {place};")
                j = 0
                for c in state:
                    lines, j = _store(buf, j, pos, c)
                    for line in lines:
                        cursor.emit(line)
                cursor.emit(f"{buf}[{n_rows}][{pos}] = (unsigned int){slot};")
            cursor.emit("__syncthreads();")
            with cursor.block(f"if ((int)threadIdx.x < {total})"):
                j = 0
                for c in state:
                    line, j = _load(buf, j, "threadIdx.x", c)
                    cursor.emit(line)
                cursor.emit(f"{slot} = (int){buf}[{n_rows}][threadIdx.x];")
            with cursor.block("else"):
                cursor.emit(f"{slot} = -1;")
        if ranked is not None:
            # The first waves, one on each SIMD, hold the instances with the
            # most to do, and do more of their iterations an epoch.
            cursor.emit(f"if ({look} && threadIdx.x < {RANK_BINS}u) {hist}[threadIdx.x] = 0u;")
            cursor.emit(f"{limit} = {rank} && __builtin_amdgcn_readfirstlane({wave}) < {RANK_WAVES}"
                        f" ? {long_epoch} : {EPOCH};")
        # Nothing is written to LDS again before every lane has read.
        cursor.emit("__syncthreads();")
    # Every instance has finished: each lane takes its own back.
    j = 0
    for c in kept_vals:
        line, j = _load(res, j, "threadIdx.x", c)
        cursor.emit(line)
