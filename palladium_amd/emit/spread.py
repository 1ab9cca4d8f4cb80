"""Spreading a block of any size over lanes.

A program instance whose block holds more than a few values (a gridless
call over a whole array, `BlockSpec((1250,), ...)`, one row of a matrix, a
few rows of it) would otherwise keep its arrays in one lane: the loads of
neighbouring lanes lie a block apart, the arrays spill to scratch, and a
small grid leaves almost every lane of the chip without work. This pass
rewrites such a kernel so that a *team* of lanes shares each row:

    block (M, W)  ->  M x T lanes, lane (m, t) holds R slots of row m,
                      slot s of lane t is element ((s / V) T + t) V + s % V

so a team reads V T neighbouring elements at a time, and a lane's V
neighbouring elements move as one wide access. A value is described per
dimension: 'm' (differs along the rows), 'w' (differs along the row) or 'u'
(the same all along, broadcast or size 1); per lane it is R scalars if it
has a 'w' dimension, else one. Values without any of the block's dimensions
stay as they are and every lane computes them. Reductions along W combine a
lane's own slots, then the team: DPP and permlane swaps inside a wavefront,
LDS across wavefronts. A float sum keeps the traced order (element by
element) unless the mode is FAST, so SAFE and REPRODUCIBLE results do not
depend on how a block is spread.

A product of whole input blocks, (M, K) @ (K, W), is computed in 16 x 16
tiles by the matrix cores (`_tile_plan`): the block's elements then lie in
lanes as those leave them, and what follows is element-wise on that.

Nothing orders the lanes of an instance, which may lie in several workgroups.
So an element has one lane: a kernel of which two stores may meet in an
element from different lanes, or that reads an output where another lane wrote
it, is not taken.

Control flow is uniform within an instance, as in `lanes`: a loop condition
or switch index that varies along the block is not taken, neither is
anything else outside these forms (`spread_transform` returns None and the
kernel is lowered as before).

What bounds such a kernel is HBM: softmax over 8192 x 1000 float32, one row
per instance, takes 10.8 us (6.0 TB/s of the 65.5 MB it reads and writes,
against 433 us when one lane held a row: 20 KB of scratch per lane and a
loaded line per element), and element-wise arithmetic on 4 million bfloat16
in blocks of 1,250 6.1 us (925 us before).
"""

from __future__ import annotations

import dataclasses
import math
from typing import Any

import numpy as np

from palladium_amd.emit.core import CVal, Cursor, Environment, ctype_of, declare, rule
from palladium_amd.emit.lanes import _ELEMENTWISE, _REDUCE, _depends_on_grid
from palladium_amd.emit.rules import DOT_UNROLL_LIMIT, FLOAT_CTYPES
from palladium_amd.dtypes import name as dtype_name
from palladium_amd.errors import EmitError
from palladium_amd.ir import (
    ClosedJaxpr,
    Jaxpr,
    JaxprEqn,
    KeyAval,
    Literal,
    RefAval,
    ShapedArray,
    Slice,
    Var,
    primitive,
)
from palladium_amd.runtime import math_mode_ordinal
from palladium_amd.trace import KernelSpec

# Blocks of fewer elements stay in one lane's registers: element-wise float32
# blocks of 8 run at the same speed either way (8.2 against 7.9 us for 4
# million elements), blocks of 16 take 10.3 us in one lane and 7.9 spread,
# blocks of 32 12.2 and 7.9.
MIN_BLOCK = 16
# With fewer instances than this (a quarter of a wavefront on each of the
# 1,024 SIMDs) lanes are idle anyway, and work that a whole team repeats
# costs nothing.
FEW_INSTANCES = 16_384
# A call without a grid is documented as one instance on one lane, and
# `explain` names the fix (a grid and BlockSpecs): it keeps that form unless
# it loops over more elements than one lane can hold unrolled, or multiplies
# matrices. The form is kept for what it says, not for its time: a grid of one
# instance is spread, and 1,000 float32 values in one block took 147 us in one
# lane and take 5.4 over lanes (on the device; either call adds the launch).
MIN_SINGLE = 65
# A lane-parallel kernel (block rows across lanes) whose rows are this long
# is spread along the rows instead, so a wavefront reads whole lines and not
# 64 rows at once. Softmax of 4 million float32 in blocks of 64 rows, lane
# rows against spread: 6.1 / 4.4 us at 8 columns, 8.6 / 4.4 at 16, 16.4 / 5.0
# at 128 (SAFE, sums in order: 6.7 / 6.4, 9.3 / 6.6, 19.8 / 8.5); at 4 columns
# a lane's row is one 16-byte load and both take 4.4.
MIN_ROW = 8
# Spread values are in registers, where FAST (and RELAXED's contraction) would
# regroup bfloat16 arithmetic across operations: x * y + c * x becomes
# x * (y + c), the sum rounded to 16 bits. One lane that held this many values
# had them in memory, every operation rounded as the interpreter does, and
# blocks of them still round so (`ROUNDED_PRELUDE`), after a product in tiles
# too. Shorter ones were in
# registers then too, as are the rows of a lane-parallel kernel. Results of
# x * y + 0.1 x - y / (x^2 + 1) that differ from the one-lane form's, rounded /
# regrouped: 28.9 / 0 % of them in blocks of 16, 18.5 / 7.6 of 24, 11.6 / 15.5
# of 32, 0.4 / 26.2 of 48, 0 / 26.6 of 1,250, where the error against 64 bits is
# 3.54e-3 / 3.63e-3 and the time the same. (float16 keeps the compiler's forms:
# its error is no larger for them, 4.6e-4 against 5.5e-4 in blocks of 1,250.)
MIN_ROUNDED = 32
MAX_SLOTS = 64
MAX_LANES = 1024
WAVE = 64
TILE = 16
# Ordered sums stage a team's row in LDS: at most this much per workgroup.
ORDERED_LDS = 60 * 1024
STAGING = "_rows"
DEFAULT_WORKGROUP = 256


def row_stride(width: int) -> int:
    """Words between the rows an ordered sum stages in LDS: 16-byte rows
    (four elements a read) whose starts fall on different banks."""
    return -(-width // 4) * 4 + 4


def staged_rows(width: int, team: int, workgroup: int) -> int:
    """Bytes of the rows that a workgroup's teams stage."""
    return max(1, workgroup // team) * row_stride(width) * 4


# Element-wise primitives the rewrites of `optimize` add to the traced ones.
_POINTWISE = _ELEMENTWISE | {"fma", "alignbit", "pow_log", "pow_with_log"}
_CALLS = {"pjit", "jit", "closed_call", "core_call", "custom_jvp_call", "custom_vjp_call"}
# Computed by every lane when no operand varies along the block.
_PLAIN = {"program_id", "num_programs", "random_wrap", "random_unwrap", "random_fold_in", "random_bits", "iota",
          "dot_general", "transpose"}


class _Bail(Exception):
    pass


@dataclasses.dataclass(frozen=True)
class SpreadPlan:
    """How a block is spread: `rows` (M) x `team` (T) lanes per instance,
    `slots` (R) elements of the `width` (W) per lane in runs of `vec` (V).
    `reduces`: some reduction runs along W."""

    rows: int
    width: int
    team: int
    slots: int
    vec: int
    reduces: bool
    block: tuple[int, int]  # the block as traced (rows and width before flattening)
    tile: tuple[int, int] | None = None  # dots: 16 x 16 tiles down and across a wavefront's part
    rounded: bool = False  # bfloat16 operations round one by one in every mode (`MIN_ROUNDED`)

    @property
    def lanes(self) -> int:
        if self.tile:
            return -(-self.rows // (TILE * self.tile[0])) * WAVE
        return self.rows * self.team

    @property
    def chunks(self) -> int:
        return self.slots // self.vec

    def workgroup(self, block: int | None, default: int) -> int:
        """A reducing team wider than a wavefront is one workgroup (its lanes
        meet at barriers), whatever was asked for; narrower ones share the
        workgroup asked for as long as the rows of an ordered sum fit (the
        default's do)."""
        if not self.reduces:
            return block or default
        if self.team > WAVE:
            return self.team
        return block if block and staged_rows(self.width, self.team, block) <= ORDERED_LDS else default


Status = Any  # None (plain) or a tuple of 'm' / 'w' / 'u', one per dim


def _nontrivial(shape: tuple[int, ...]) -> tuple[int, ...]:
    return tuple(d for d in shape if d != 1)


def _sub(j: Any) -> Any:
    return getattr(j, "jaxpr", j)


class _Pass:
    """One walk over the kernel for a block of M x W with R slots a lane.
    The statuses do not depend on R, so a first walk (R = 1) tells which
    forms occur and a second one builds the jaxpr for the chosen layout."""

    def __init__(self, m: int, w: int, slots: int, outputs: set[int], tiles: bool = False):
        self.m, self.w, self.slots, self.tiles = m, w, slots, tiles
        self.deferred: dict[Var, Var] = {}  # dot operands: a whole block read by the dot itself
        self.dots: list[tuple[int, int, int]] = []  # (k, lhs and out itemsize)
        self.outputs = outputs
        self.refs: dict[Var, int] = {}
        self.env: dict[Var, Any] = {}
        self.st: dict[Var, Status] = {}
        self.wide: dict[tuple[int, Var], Var] = {}
        self.scopes: list[list] = []
        self.read: set[int] = set()  # output operands read back
        self.partial: set[int] = set()  # output operands not accessed element by own element
        self.used: set[Var] = set()  # values something reads
        self.written: dict[int, set] = {}  # output operand -> its stores: (which lane, fixed indices)
        self.reduces = False
        self.whole = True  # only full-block accesses, no lone 'm' or 'w'
        self.spread_eqns = 0  # weighted by loop trips
        self.plain_eqns = 0
        self.loops = False
        self.weight = 1
        self.stores = 0
        self.itemsizes: list[int] = []

    # -- statuses -----------------------------------------------------------
    def axis(self, shape: tuple[int, ...], d: int) -> str | None:
        """The block axis dimension d of a block-shaped value lies along."""
        big = [k for k, n in enumerate(shape) if n != 1]
        if d not in big:
            return "u"
        n = shape[d]
        if len(big) == 2:
            want = (self.m, self.w)[big.index(d)]
            return ("m", "w")[big.index(d)] if n == want else None
        if len(big) == 1:
            if n == self.w and (self.m == 1 or self.m != self.w or d == len(shape) - 1):
                return "w"
            return "m" if n == self.m else None
        return None

    def lane_aval(self, aval: Any, st: Status) -> Any:
        if st is None:
            return aval
        varies = "w" in st or (self.tiles and "m" in st)  # a tile's slots differ in row and column
        return ShapedArray((self.slots,) if varies and self.slots > 1 else (), aval.dtype, aval.weak_type)

    def status(self, x: Any) -> Status:
        return None if isinstance(x, Literal) else self.st[x]

    def atom(self, x: Any) -> Any:
        return x if isinstance(x, Literal) else self.env[x]

    def bind(self, v: Var, new: Any, st: Status) -> Any:
        self.env[v] = new
        self.st[v] = st
        if st is not None and any(s != "u" for s in st) and tuple(s for s in st if s != "u") not in (("m", "w"), ("w",), ("m",)):
            raise _Bail("row and column dims out of order")
        if st is not None and self.m > 1 and ("m" in st) != ("w" in st):
            self.whole = False
        return new

    def emit(self, eqns: list, invars: list, outvars: list, name: str, params: dict) -> None:
        eqns.append(JaxprEqn(invars, outvars, primitive(name), params))

    def size(self, x: Any) -> int:
        return 1 if isinstance(x, Literal) else math.prod(x.aval.shape)

    def join(self, a: Status, b: Status, what: str) -> Status:
        if a is None or b is None:
            return a if b is None else b
        if len(a) != len(b):
            raise _Bail(f"{what}: ranks differ")
        out = []
        for x, y in zip(a, b):
            if x != y and "u" not in (x, y):
                raise _Bail(f"{what}: rows against columns")
            out.append(y if x == "u" else x)
        return tuple(out)

    def widen(self, eqns: list, x: Any, shape: tuple[int, ...], dtype: Any) -> Any:
        """`x` (a per-lane atom) at the per-lane `shape`: a scalar operand of
        a slot array is broadcast explicitly, as the frontend does."""
        if isinstance(x, Literal) or tuple(x.aval.shape) == tuple(shape):
            return x
        if math.prod(x.aval.shape) != 1:
            raise _Bail("per-lane shapes differ")
        key = (id(eqns), x)
        w = self.wide.get(key)
        if w is None or tuple(w.aval.shape) != tuple(shape):
            w = Var(ShapedArray(shape, x.aval.dtype))
            if tuple(x.aval.shape):
                s = Var(ShapedArray((), x.aval.dtype))
                self.emit(eqns, [x], [s], "reshape", {"new_sizes": (), "dimensions": None})
                x = s
            self.emit(eqns, [x], [w], "broadcast_in_dim", {"shape": tuple(shape), "broadcast_dimensions": (),
                                                           "sharding": None})
            self.wide[key] = w
        return w

    # -- jaxprs ---------------------------------------------------------------
    def walk(self, j: Jaxpr, eqns: list) -> None:
        uses: dict[Var, list] = {}
        for e in j.eqns:
            for i, x in enumerate(e.invars):
                if isinstance(x, Var):
                    uses.setdefault(x, []).append((e.primitive.name, i))
        for o in j.outvars:
            if isinstance(o, Var):
                uses.setdefault(o, []).append(("out", 0))
        self.used.update(uses)
        for e in j.eqns:
            if e.primitive.name == "get" and uses.get(e.outvars[0]) and all(
                    n == "dot_general" for n, _ in uses[e.outvars[0]]) and self.whole_input(e):
                self.deferred[e.outvars[0]] = e.invars[0]
                self.env[e.outvars[0]], self.st[e.outvars[0]] = None, None
                continue
            self.eqn(e, eqns)

    def whole_input(self, e: JaxprEqn) -> bool:
        """A read of an input's whole rank-2 block."""
        shape = tuple(int(d) for d in e.invars[0].aval.shape)
        idx = e.params["tree"].unflatten(list(e.invars[1:]))
        return (self.refs[e.invars[0]] not in self.outputs and len(shape) == 2
                and all(isinstance(ix, Slice) and isinstance(ix.start, (int, np.integer)) and int(ix.start) == 0
                        and ix.size == n and ix.stride == 1 for ix, n in zip(idx[0].indices if idx else (), shape)))

    def dot(self, e: JaxprEqn, eqns: list) -> None:
        """(M, K) @ (K, W) -> the block, both operands whole inputs."""
        (lc, rc), (lb, rb) = e.params["dimension_numbers"]
        lhs, rhs = e.invars
        if not all(isinstance(x, Var) and x in self.deferred for x in (lhs, rhs)) or tuple(lb) or tuple(rb):
            raise _Bail("dot of computed operands")
        (lc,), (rc,) = tuple(lc), tuple(rc)
        ls, rs = tuple(lhs.aval.shape), tuple(rhs.aval.shape)
        out = e.outvars[0]
        if int(lc) != 1 or tuple(out.aval.shape) != (self.m, self.w) or self.m < 2:
            raise _Bail("dot of another shape than the block")
        names = {dtype_name(x.aval.dtype) for x in (lhs, rhs)}
        if len(names) != 1 or not names <= {"float32", "float16", "bfloat16"} or dtype_name(out.aval.dtype) not in names | {"float32"}:
            raise _Bail("dot of other types")
        k = int(ls[1])
        self.dots.append((k, np.dtype(lhs.aval.dtype).itemsize, np.dtype(out.aval.dtype).itemsize))
        self.whole = False
        self.spread_eqns += self.weight * k
        nv = Var(self.lane_aval(out.aval, ("m", "w")))
        self.emit(eqns, [self.env[self.deferred[lhs]], self.env[self.deferred[rhs]]], [nv], "spread_dot",
                  {"k": k, "rhs_strides": (int(rs[1]), 1) if int(rc) == 0 else (1, int(rs[1]))})
        self.bind(out, nv, ("m", "w"))

    def inner(self, j: Jaxpr, outer: list, status: list, weight: int) -> tuple[list[Var], list, list]:
        """Walk a sub-jaxpr whose invars take the statuses given (refs keep
        their operand); returns its new invars, eqns and out atoms."""
        new = []
        for v, o, s in zip(j.invars, outer, status):
            if isinstance(v.aval, RefAval):
                self.refs[v] = self.refs[o]
                nv = Var(v.aval)
                self.env[v], self.st[v] = nv, None
            else:
                nv = Var(self.lane_aval(v.aval, s))
                self.bind(v, nv, s)
            new.append(nv)
        eqns: list = []
        self.scopes.append(eqns)  # kept alive: `wide` goes by their identity
        old, self.weight = self.weight, self.weight * weight
        self.walk(j, eqns)
        self.weight = old
        return new, eqns, [self.atom(o) for o in j.outvars]

    def to_status(self, eqns: list, x: Any, aval: Any, st: Status) -> Any:
        """A loop's or branch's value as the status its result has."""
        if st is None:
            return x
        shape = self.lane_aval(aval, st).shape
        if isinstance(x, Literal):
            v = Var(ShapedArray(shape, x.aval.dtype))
            self.emit(eqns, [x], [v], "broadcast_in_dim", {"shape": shape, "broadcast_dimensions": (), "sharding": None})
            return v
        if shape == () and tuple(x.aval.shape) != ():
            v = Var(ShapedArray((), x.aval.dtype))
            self.emit(eqns, [x], [v], "reshape", {"new_sizes": (), "dimensions": None})
            return v
        return self.widen(eqns, x, shape, x.aval.dtype)

    def meet(self, aval: Any, a: Status, b: Status, xa: Any, xb: Any, what: str) -> Status:
        """Join of two values of one aval where either may be plain."""
        for s, x in ((a, xa), (b, xb)):
            if s is None and (a, b) != (None, None) and self.size(x) != 1:
                raise _Bail(f"{what}: plain array meets a spread value")
        if a is None and b is None:
            return None
        rank = len(aval.shape)
        return self.join(a if a is not None else ("u",) * rank, b if b is not None else ("u",) * rank, what)

    # -- equations --------------------------------------------------------------
    def eqn(self, e: JaxprEqn, eqns: list) -> None:
        name = e.primitive.name
        sts = [self.status(x) for x in e.invars]
        spread = any(s is not None for s in sts)
        if name in ("get", "swap"):
            self.access(e, eqns)
            return
        if any(isinstance(getattr(x, "aval", None), RefAval) for x in e.invars) and name not in _CALLS | {"scan", "while", "cond"}:
            raise _Bail(f"{name} on a ref")
        if name == "dot_general" and any(isinstance(x, Var) and x in self.deferred for x in e.invars):
            self.dot(e, eqns)
            return
        if name in _CALLS:
            inner = _sub(e.params.get("jaxpr") or e.params.get("call_jaxpr"))
            outer = list(e.invars)[-len(inner.invars):] if inner.invars else []
            for v, o in zip(inner.invars, outer):
                if isinstance(v.aval, RefAval):
                    self.refs[v] = self.refs[o]
                self.env[v], self.st[v] = self.atom(o), self.status(o)
            self.walk(inner, eqns)
            for ov, iv in zip(e.outvars, inner.outvars):
                self.env[ov], self.st[ov] = self.atom(iv), self.status(iv)
            return
        if name == "scan":
            self.scan(e, eqns)
            return
        if name == "while":
            self.while_(e, eqns)
            return
        if name == "cond":
            self.cond(e, eqns)
            return
        if name == "broadcast_in_dim":
            self.broadcast(e, eqns, sts[0])
            return
        if name == "iota" and not spread:
            shape = tuple(int(d) for d in e.params["shape"])
            dim = int(e.params["dimension"])
            if math.prod(shape) > 1 and all(self.axis(shape, d) is not None for d in range(len(shape))):
                st = tuple(self.axis(shape, d) if d == dim else "u" for d in range(len(shape)))
                nv = Var(self.lane_aval(e.outvars[0].aval, st))
                if st[dim] == "u":  # a dim of one: index 0
                    self.emit(eqns, [], [nv], "iota", {**e.params, "shape": (), "dimension": 0})
                else:
                    self.whole = False
                    self.emit(eqns, [], [nv], "spread_index", {"axis": st[dim]})
                self.bind(e.outvars[0], nv, st)
                return
        if name in _REDUCE and spread:
            self.reduce(e, eqns, sts[0])
            return
        if name in ("reshape", "squeeze", "expand_dims") and spread:
            if e.params.get("dimensions") is not None and name == "reshape":
                raise _Bail("reshape with dimensions")
            old, new = tuple(e.invars[0].aval.shape), tuple(e.outvars[0].aval.shape)
            if _nontrivial(old) != _nontrivial(new):
                raise _Bail("reshape of the block")
            kept = [s for s, n in zip(sts[0], old) if n != 1]
            st = tuple(kept.pop(0) if n != 1 else "u" for n in new)
            self.bind(e.outvars[0], self.atom(e.invars[0]), st)
            return
        if name in _POINTWISE:
            if not spread:
                self.plain(e, eqns)
                return
            st: Status = None
            rank = len(e.outvars[0].aval.shape)
            for x, s in zip(e.invars, sts):
                if s is None:
                    if self.size(x) != 1:
                        raise _Bail(f"{name}: plain array operand of a spread value")
                    continue
                if len(s) != rank:
                    raise _Bail(f"{name}: ranks differ")
                st = self.join(st, s, name)
            self.spread_eqns += self.weight
            outs = [Var(self.lane_aval(ov.aval, st)) for ov in e.outvars]
            shape = outs[0].aval.shape
            ins = [self.widen(eqns, self.atom(x), shape, None) for x in e.invars]
            self.emit(eqns, ins, outs, name, dict(e.params))
            for ov, nv in zip(e.outvars, outs):
                self.bind(ov, nv, st)
            return
        if spread or name not in _PLAIN | set(_REDUCE) | {"reshape", "squeeze", "expand_dims"}:
            raise _Bail(f"no spread rule for {name}")
        self.plain(e, eqns)

    def plain(self, e: JaxprEqn, eqns: list) -> None:
        self.plain_eqns += self.weight
        outs = [Var(ov.aval) for ov in e.outvars]
        self.emit(eqns, [self.atom(x) for x in e.invars], outs, e.primitive.name, dict(e.params))
        for ov, nv in zip(e.outvars, outs):
            self.bind(ov, nv, None)

    def broadcast(self, e: JaxprEqn, eqns: list, st: Status) -> None:
        src, out = e.invars[0], e.outvars[0]
        shape = tuple(int(d) for d in e.params["shape"])
        bd = tuple(int(d) for d in e.params["broadcast_dimensions"])
        if st is not None:
            new = ["u"] * len(shape)
            for sd, od in enumerate(bd):
                if src.aval.shape[sd] == shape[od]:
                    new[od] = st[sd]
            self.bind(out, self.atom(src), tuple(new))
            return
        if self.size(src) == 1 and math.prod(shape) > 1 and all(self.axis(shape, d) is not None for d in range(len(shape))):
            # one value for the whole block: one scalar per lane
            x = self.atom(src)
            nv = Var(ShapedArray((), out.aval.dtype))
            if not isinstance(x, Literal) and tuple(x.aval.shape) != ():
                self.emit(eqns, [x], [nv], "reshape", {"new_sizes": (), "dimensions": None})
            else:
                self.emit(eqns, [x], [nv], "broadcast_in_dim", {"shape": (), "broadcast_dimensions": (), "sharding": None})
            self.bind(out, nv, ("u",) * len(shape))
            return
        self.plain(e, eqns)

    def reduce(self, e: JaxprEqn, eqns: list, st: Status) -> None:
        src = e.invars[0]
        axes = {int(a) for a in e.params["axes"]}
        kind = _REDUCE[e.primitive.name]
        along = any(st[d] == "w" for d in axes)
        for d in axes:
            if st[d] == "m":
                raise _Bail("reduction across rows")
            if st[d] == "u" and src.aval.shape[d] != 1:
                raise _Bail("reduction over a broadcast dim")
        if kind == "sum" and not along:
            raise _Bail("sum of one value")  # 0 + x: not x when x is -0
        kept = tuple(s for d, s in enumerate(st) if d not in axes)
        x = self.atom(src)
        nst: Status = kept if kept else None
        if not along:
            self.bind(e.outvars[0], x, nst)
            return
        nv = Var(self.lane_aval(e.outvars[0].aval, nst))
        self.reduces = True
        self.spread_eqns += self.weight
        self.emit(eqns, [x], [nv], "spread_reduce", {"kind": kind})
        self.bind(e.outvars[0], nv, nst)

    def access(self, e: JaxprEqn, eqns: list) -> None:
        store = e.primitive.name == "swap"
        ref = e.invars[0]
        k = self.refs[ref]
        shape = tuple(int(d) for d in ref.aval.shape)
        if store and e.outvars[0] in self.used:
            raise _Bail("a store's value before it")
        idx = e.params["tree"].unflatten(list(e.invars[2 if store else 1:]))
        indices = list(idx[0].indices) if idx else [Slice(0, n, 1) for n in shape]
        kept = [d for d, ix in enumerate(indices) if isinstance(ix, Slice)]
        for ix in indices:
            if not isinstance(ix, Slice) and self.status(ix) is not None:
                raise _Bail("ref index varies along the block")
        axes: list[str | None] = []
        for d in kept:
            ix = indices[d]
            full = isinstance(ix.start, (int, np.integer)) and int(ix.start) == 0 and ix.size == shape[d] and ix.stride == 1
            axes.append(self.axis(shape, d) if full else None)
        vary = [a for a in axes if a in ("m", "w")]
        spread = bool(vary) and all(a is not None for a in axes)
        own = spread and len(vary) == len(_nontrivial(shape)) and ("m" in vary or self.m == 1) and "w" in vary
        if k in self.outputs:
            if not own:
                self.partial.add(k)
            if not store:
                self.read.add(k)
        if not spread:
            if vary or (store and self.status(e.invars[1]) is not None and any(s != "u" for s in self.status(e.invars[1]))):
                raise _Bail("part of the block")
            if store:
                self.stored(k, (), indices)
                used = e.outvars[0]
                self.env[used], self.st[used] = None, None
                v = e.invars[1]
                x = self.atom(v)
                if self.status(v) is not None and math.prod(v.aval.shape) != 1:
                    raise _Bail("broadcast value into a plain block")
                self.emit(eqns, [self.env[ref], x, *[self.atom(a) for a in e.invars[2:]]], [Var(e.outvars[0].aval)], "swap",
                          {**e.params, "lane0_only": True})
                self.stores += 1
                return
            self.plain(e, eqns)
            return
        strides = [math.prod(shape[d + 1:]) for d in range(len(shape))]
        terms, leaves = [], []
        for d, ix in enumerate(indices):
            if isinstance(ix, Slice):
                a = axes[kept.index(d)]
                if a != "u":
                    terms.append((a, strides[d]))
            elif isinstance(ix, (int, np.integer)):
                terms.append((int(ix), strides[d]))
            else:
                leaves.append(self.atom(ix))
                terms.append(("idx", strides[d]))
        if not own:
            self.whole = False
        self.spread_eqns += self.weight
        self.itemsizes.append(np.dtype(ref.aval.dtype).itemsize)
        params = {"terms": tuple(terms)}
        if not store:
            st = tuple(axes)
            nv = Var(self.lane_aval(e.outvars[0].aval, st))
            self.emit(eqns, [self.env[ref], *leaves], [nv], "spread_get", params)
            self.bind(e.outvars[0], nv, st)
            return
        self.stored(k, tuple((d, a) for d, a in zip(kept, axes) if a != "u"), indices)
        v = e.invars[1]
        s = self.status(v)
        x = self.atom(v)
        if s is None:
            if self.size(v) != 1:
                raise _Bail("plain array stored along the block")
        else:
            if len(s) != len(axes):
                raise _Bail("store of another rank")
            for a, b in zip(s, axes):
                if a != "u" and a != b:
                    raise _Bail("store across the block's axes")
        if not isinstance(x, Literal) and tuple(x.aval.shape) not in ((), (self.slots,)):
            y = Var(ShapedArray((), x.aval.dtype))
            self.emit(eqns, [x], [y], "reshape", {"new_sizes": (), "dimensions": None})
            x = y
        if "m" not in vary and self.m > 1:
            params["first_row"] = True
        if "w" not in vary:
            params["first_lane"] = True
        old = e.outvars[0]
        self.env[old], self.st[old] = None, None
        self.emit(eqns, [self.env[ref], x, *leaves], [], "spread_swap", params)
        self.stores += 1

    def stored(self, k: int, lane: tuple, indices: list) -> None:
        """Note a store. The lane that stores an element follows from the
        element and `lane`, the dims that lie along the block (none: lane 0
        stores them all)."""
        fixed = tuple(int(ix.val) if isinstance(ix, Literal) else int(ix) if isinstance(ix, (int, np.integer)) else None
                      for ix in indices)
        self.written.setdefault(k, set()).add((lane, fixed))

    def overwrites(self) -> bool:
        """Whether two lanes may store one element of an output. Nothing
        orders their stores (an instance's lanes may lie in several
        workgroups), so such a kernel keeps its program order in one lane."""
        return any(a != b and not any(i is not None and j is not None and i != j for i, j in zip(at, bt))
                   for stores in self.written.values() for a, at in stores for b, bt in stores)

    # -- control flow ---------------------------------------------------------
    def scan(self, e: JaxprEqn, eqns: list) -> None:
        body = _sub(e.params["jaxpr"])
        nc = len(e.outvars)
        nconst = len(e.invars) - nc
        if len(body.outvars) != nc or e.params.get("reverse", False):
            raise _Bail("scan with xs or ys")
        for iv, bv in zip(e.invars, body.invars):
            if tuple(getattr(iv.aval, "shape", ())) != tuple(getattr(bv.aval, "shape", ())):
                raise _Bail("scan with xs")
        self.loops = True
        trips = max(1, int(e.params["length"]))
        consts, inits = list(e.invars[:nconst]), list(e.invars[nconst:])
        carry, new, beqns, outs = self.fix(body, consts, inits, trips)
        ins = [self.atom(x) for x in consts] + [self.to_status(eqns, self.atom(x), v.aval, s)
                                                for x, v, s in zip(inits, body.invars[nconst:], carry)]
        self.finish(e, eqns, "scan", {**e.params, "jaxpr": ClosedJaxpr(Jaxpr([], new, outs, beqns), [])}, ins, carry)

    def fix(self, body: Jaxpr, consts: list, inits: list, trips: int) -> tuple:
        """Statuses of the carries of a loop, and its body under them."""
        n = len(consts)
        cvars = body.invars[n:]
        carry = [self.status(x) for x in inits]
        for _ in range(3 * len(carry) + 2):
            mark = (self.spread_eqns, self.plain_eqns)
            new, beqns, outs = self.inner(body, consts + inits, [self.status(c) for c in consts] + carry, trips)
            after = [self.status(o) for o in body.outvars]
            merged = [self.meet(v.aval, c, a, v, o, "loop carry") for v, c, a, o in zip(cvars, carry, after, body.outvars)]
            if merged == carry:
                break
            carry = merged
            self.spread_eqns, self.plain_eqns = mark
        else:
            raise _Bail("loop statuses do not settle")
        outs = [self.to_status(beqns, o, v.aval, s) for o, v, s in zip(outs, cvars, carry)]
        return carry, new, beqns, outs

    def finish(self, e: JaxprEqn, eqns: list, name: str, params: dict, ins: list, carry: list) -> None:
        outs = [Var(self.lane_aval(ov.aval, s)) for ov, s in zip(e.outvars, carry)]
        self.emit(eqns, ins, outs, name, params)
        for ov, nv, s in zip(e.outvars, outs, carry):
            self.bind(ov, nv, s)

    def while_(self, e: JaxprEqn, eqns: list) -> None:
        cn, bn = int(e.params["cond_nconsts"]), int(e.params["body_nconsts"])
        cj, bj = _sub(e.params["cond_jaxpr"]), _sub(e.params["body_jaxpr"])
        self.loops = True
        consts, inits = list(e.invars[cn:cn + bn]), list(e.invars[cn + bn:])
        carry, new, beqns, outs = self.fix(bj, consts, inits, 16)
        cnew, ceqns, (pred,) = self.inner(cj, list(e.invars[:cn]) + inits,
                                          [self.status(x) for x in e.invars[:cn]] + carry, 16)
        if self.status(cj.outvars[0]) is not None:
            raise _Bail("loop condition varies along the block")
        ins = [self.atom(x) for x in e.invars[:cn + bn]] + [self.to_status(eqns, self.atom(x), v.aval, s)
                                                            for x, v, s in zip(inits, bj.invars[bn:], carry)]
        self.finish(e, eqns, "while", {**e.params, "cond_jaxpr": ClosedJaxpr(Jaxpr([], cnew, [pred], ceqns), []),
                                       "body_jaxpr": ClosedJaxpr(Jaxpr([], new, outs, beqns), [])}, ins, carry)

    def cond(self, e: JaxprEqn, eqns: list) -> None:
        if self.status(e.invars[0]) is not None:
            raise _Bail("switch index varies along the block")
        ops = list(e.invars[1:])
        built = []
        sts: list[Status] = []
        for b, br in enumerate(e.params["branches"]):
            j = _sub(br)
            new, beqns, outs = self.inner(j, ops, [self.status(o) for o in ops], 1)
            got = [self.status(o) for o in j.outvars]
            sts = got if b == 0 else [self.meet(ov.aval, x, y, ov, o, "branches")
                                      for ov, x, y, o in zip(e.outvars, sts, got, j.outvars)]
            built.append((j, new, beqns, outs))
        branches = []
        for j, new, beqns, outs in built:
            outs = [self.to_status(beqns, o, ov.aval, s) for o, ov, s in zip(outs, e.outvars, sts)]
            branches.append(ClosedJaxpr(Jaxpr([], new, outs, beqns), []))
        self.finish(e, eqns, "cond", {**e.params, "branches": tuple(branches)}, [self.atom(x) for x in e.invars], sts)


# ---------------------------------------------------------------------------
# choosing the layout


def _candidates(spec: KernelSpec) -> list[tuple[int, int]]:
    """(M, W) of the blocks worth trying: the largest block that moves with
    the grid (any block of a gridless kernel), then the largest output."""
    operands = list(spec.inputs) + list(spec.outputs)
    moving = [o for o in operands if spec.num_programs == 1 or _depends_on_grid(o)]
    out: list[tuple[int, int]] = []
    for group in (moving, list(spec.outputs)):
        if not group:
            continue
        best = max(group, key=lambda o: math.prod(o.block_shape or (1,)))
        dims = _nontrivial(tuple(int(d) for d in best.block_shape))
        if len(dims) == 1:
            dims = (1, dims[0])
        if len(dims) == 2 and dims not in out and dims[0] <= MAX_LANES:
            out.append(dims)  # type: ignore[arg-type]
    return out


def _run(spec: KernelSpec, jaxpr: Jaxpr, m: int, w: int, slots: int, tiles: bool = False) -> tuple[_Pass, Jaxpr]:
    n_in = len(spec.inputs)
    p = _Pass(m, w, slots, set(range(n_in, n_in + len(spec.outputs))), tiles)
    new = []
    for k, v in enumerate(jaxpr.invars):
        p.refs[v] = k
        nv = Var(v.aval)
        p.env[v], p.st[v] = nv, None
        new.append(nv)
    eqns: list = []
    p.walk(jaxpr, eqns)
    if p.read & p.partial:
        raise _Bail("an output is read where another lane wrote it")
    if p.overwrites():
        raise _Bail("two lanes store one element of an output")
    return p, Jaxpr([], new, [], eqns)


def _tile_plan(p: _Pass, m: int, w: int, programs: int, lane_plan: Any) -> SpreadPlan | None:
    """A block that dots fill, in 16 x 16 tiles: a wavefront holds A x B of
    them (16 A rows, all W columns), lane l rows 4 (l / 16) .. + 3 and column
    l % 16 of each, as the matrix instructions leave their results; tile b's
    column c is the block's B c + b, so a lane's B columns lie side by side
    and move as one access."""
    if p.reduces or p.partial:
        return None
    across = -(-w // TILE)
    # Narrow products stay a row per lane: 262,144 rows of float32, lane rows
    # against tiles, 8 x 8 4.6 / 6.3 us, 32 x 8 18.6 / 9.1 but in order (SAFE)
    # 20.6 / 22.0, 64 x 8 73 / 14.7 (127 / 38 in order; past 32 the lane's
    # contraction is a loop over memory), 4 x 16 9.5 / 7.2, 16 x 16 32 / 7.1.
    if lane_plan is not None and w < TILE and (w < 4 or min(k for k, *_ in p.dots) <= DOT_UNROLL_LIMIT):
        return None
    if m < TILE or 4 * across > MAX_SLOTS:
        return None
    down = 2 if 8 * across <= MAX_SLOTS and programs * m >= 2048 * 2 * TILE else 1
    while -(-m // (TILE * down)) * WAVE > _lanes_max(programs):
        down *= 2
        if 4 * across * down > MAX_SLOTS:
            return None
    return SpreadPlan(m, w, WAVE, 4 * across * down, 1, False, (m, w), (down, across), _rounds(m, w, lane_plan))


def _rounds(m: int, w: int, lane_plan: Any) -> bool:
    return lane_plan is None and m * w >= MIN_ROUNDED


def _lanes_max(programs: int) -> int:
    """An instance's lanes: a launch has fewer than 2**31 of them in all."""
    return min(MAX_LANES, (2**31 - 1) // programs)


def _layout(p: _Pass, m: int, w: int, programs: int) -> tuple[int, int, int] | None:
    """(T, R, V) for M rows of W, or None."""
    limit = _lanes_max(programs) // m
    if limit < 1:
        return None
    item = max(p.itemsizes, default=4)
    vmax = max(1, 16 // max(item, 1))
    if not p.reduces:
        # Any team size will do. Programs with loops want one element a lane
        # (more wavefronts, shorter chains). The others want wide accesses as
        # long as the launch still puts four wavefronts on every SIMD: 4 a
        # lane is fastest or level throughout (element-wise, 16 million:
        # float32 27.9 / 27.4 / 26.9 / 27.4 us with 1 / 2 / 4 / 8 a lane,
        # bfloat16 26.0 / 21.0 / 15.9 / 16.6, float16 22.6 / 16.4 / 15.2 /
        # 14.4; 400,000: 2.0-2.2 us whatever the width).
        v = 1
        if not p.loops:
            v = min(vmax, 4)
            while v > 1 and (w % v or programs * m * w // v < 256 * 1024):
                v //= 2
        chunks = -(-w // (v * limit))
        team = -(-w // (v * chunks))
        return (team, v * chunks, v) if v * chunks <= MAX_SLOTS else None
    v = vmax
    while v > 1 and w % v:
        v //= 2
    if p.loops:
        v = 1
    # Teams of a power of two lie inside a wavefront or fill whole ones. A
    # lane takes up to 16 bytes of a row, 32 from half a wavefront on: fewer
    # leave lanes without an element, more make a team read short pieces of
    # lines. Softmax of 8 million float32, teams of 4 / 8 / 16 / 32 / 64:
    # rows of 33 18.0 / 13.6 / 11.3 / 16.5 / 28.6 us (16 taken; 20.7 with a
    # row in one lane), of 64 10.7 / 10.5 / 10.3 / 10.5 / 16.0 (16), of 200
    # - / 11.3 / 10.9 / 10.4 / 10.5 (32; 25.2 in one lane).
    team_max = min(limit, WAVE if m > 1 else MAX_LANES)
    team_max = 1 << (team_max.bit_length() - 1)
    team = 1
    while team < team_max and -(-w // (team * v)) * v * item > (1 if p.loops else 16 if team < 32 else 32):
        team *= 2
    # A launch of few rows spreads them wider.
    wide = team_max if m > 1 else min(team_max, 256)
    while team < wide and team * v < w and programs * m * team < 2048 * WAVE:
        team *= 2
    slots = -(-w // (team * v)) * v
    return (team, slots, v) if slots <= MAX_SLOTS else None


def staging(env: Environment) -> list[str]:
    """The kernel's array for the rows of ordered sums, if it has any."""
    n = getattr(env, "staged", 0)
    return [f"    __shared__ __attribute__((aligned(16))) unsigned char {STAGING}[{n}];"] if n else []


def own_rules(plan: SpreadPlan | None = None) -> bool:
    """Whether the rules this lowering stands in for are the built-in ones (a
    user's own rule for an access, a reduction or, in tiles, a product keeps
    its say)."""
    from palladium_amd.emit.core import RULES

    if plan is not None and plan.tile:
        return RULES["dot_general"].__module__ == "palladium_amd.emit.rules"
    return all(RULES[n].__module__ == "palladium_amd.emit.rules"
               for n in ("get", "swap", "iota", "broadcast_in_dim", "reshape", "squeeze", "expand_dims", *_REDUCE))


def spread_transform(spec: KernelSpec, lane_plan: Any = None) -> SpreadPlan | None:
    """The spread form of `spec`, or None where it is lowered otherwise.
    `lane_plan`: the lane-parallel plan `lanes.lane_transform` found."""
    if lane_plan is not None and lane_plan.rows is not None:
        return None  # a ragged tail
    programs = spec.num_programs
    gridless = programs == 1 and not any(b.index_map_jaxpr.jaxpr.invars for b in spec.inputs + spec.outputs)
    for m, w in _candidates(spec):
        if m * w < 2:
            continue
        if lane_plan is None and m * w < (MIN_SINGLE if gridless else MIN_BLOCK):
            continue
        try:
            p, _ = _run(spec, spec.jaxpr, m, w, 1)
        except _Bail:
            continue
        if not p.stores or p.spread_eqns == 0 or (gridless and not p.loops and not p.dots):
            continue
        if p.dots:
            plan = _tile_plan(p, m, w, programs, lane_plan)
            if plan is not None:
                return plan
            continue
        if p.plain_eqns > 8 * p.spread_eqns and programs > FEW_INSTANCES:
            continue  # mostly work that every lane of a team would repeat
        if lane_plan is not None and m > 1 and w < MIN_ROW:
            continue  # a short row a lane already
        if lane_plan is not None and m == 1 and (p.reduces or p.loops):
            continue  # one element a lane already
        if p.whole and not p.reduces:
            # element by element: one row of M W
            layout = _layout(p, 1, m * w, programs)
            rows, width = 1, m * w
        else:
            layout = _layout(p, m, w, programs)
            rows, width = m, w
        if layout is None or rows * layout[0] < 2:
            continue
        team, slots, vec = layout
        if lane_plan is not None and m == 1 and vec == 1:
            continue
        if p.reduces:
            if staged_rows(width, team, DEFAULT_WORKGROUP) > ORDERED_LDS:
                continue
        return SpreadPlan(rows, width, team, slots, vec, p.reduces, (m, w), rounded=_rounds(m, w, lane_plan))
    return None


def spread_jaxpr(spec: KernelSpec, plan: SpreadPlan, jaxpr: Jaxpr) -> Jaxpr:
    """`jaxpr` (the kernel's, as traced or rewritten by `optimize`) per lane.
    The rewrites come first: which products a mode fuses is decided on the
    traced program, where the interpreter decides it too."""
    m, w = plan.block
    try:
        _, j = _run(spec, jaxpr, m, w, plan.slots, plan.tile is not None)
    except _Bail as e:
        raise EmitError(f"internal: a rewritten kernel no longer spreads ({e})") from None
    return _flatten(j, m, w) if plan.rows != m and not plan.tile else j


def _flatten(j: Jaxpr, m: int, w: int) -> Jaxpr:
    """Accesses of a whole M x W block (rows W apart) as one run."""

    def eqn(e: JaxprEqn) -> JaxprEqn:
        params = {}
        for k, v in e.params.items():
            if isinstance(v, ClosedJaxpr):
                v = ClosedJaxpr(_flatten(v.jaxpr, m, w), v.consts)
            elif isinstance(v, tuple) and v and all(isinstance(b, ClosedJaxpr) for b in v):
                v = tuple(ClosedJaxpr(_flatten(b.jaxpr, m, w), b.consts) for b in v)
            params[k] = v
        if e.primitive.name in ("spread_get", "spread_swap"):
            params["terms"] = tuple(t for t in params["terms"] if t[0] != "m")
        return JaxprEqn(e.invars, e.outvars, e.primitive, params)

    return Jaxpr(j.constvars, j.invars, j.outvars, [eqn(e) for e in j.eqns])


# ---------------------------------------------------------------------------
# emission. Every kernel of a plan holds, per lane: `_m` (its row), `_t` (its
# place in the team) and per chunk q of V slots `_wq`, the first element, and
# `_kq`, whether the row has it (only where a row does not fill its chunks).


def spread_prologue(env: Environment, cursor: Cursor, plan: SpreadPlan, block: int) -> None:
    env.spread = plan  # type: ignore[attr-defined]
    env.spread_block = block  # type: ignore[attr-defined]
    if plan.tile:
        down, across = plan.tile
        cursor.emit(f"const int _c = _lane % {TILE};")
        cursor.emit(f"const int _h = _lane % {WAVE} / {TILE};")
        cursor.emit(f"const int _r = _lane / {WAVE} * {TILE * down};")
        for a in range(down):
            for i in range(4):
                cursor.emit(f"const int _m{a}_{i} = _r + {TILE * a + i} + 4 * _h;")
        for b in range(across):
            cursor.emit(f"const int _w{b} = _c * {across} + {b};" if across > 1 else "const int _w0 = _c;")
        return
    if plan.rows > 1:
        cursor.emit(f"const int _m = _lane / {plan.team};")
        cursor.emit(f"const int _t = _lane % {plan.team};")
    else:
        cursor.emit("const int _t = _lane;")
    for q in range(plan.chunks):
        first = f"({q * plan.team} + _t)" if q else "_t"
        cursor.emit(f"const int _w{q} = {first} * {plan.vec};")
        if _masked(plan, q):
            cursor.emit(f"const bool _k{q} = _w{q} < {plan.width};")


def _tile_slots(plan: SpreadPlan) -> list[tuple[int, int, int, str]]:
    """(A, B, register, condition under which the block has the element) of
    every slot of a tiled plan."""
    down, across = plan.tile  # type: ignore[misc]
    out = []
    for a in range(down):
        for b in range(across):
            for i in range(4):
                conds = []
                if plan.rows % (TILE * down):
                    conds.append(f"_m{a}_{i} < {plan.rows}")
                if across * TILE > plan.width:
                    conds.append(f"_w{b} < {plan.width}")
                out.append((a, b, i, " && ".join(conds)))
    return out


def _tile_slot(plan: SpreadPlan, a: int, b: int, i: int) -> int:
    """A row's neighbouring columns of one lane are neighbouring slots."""
    down, across = plan.tile  # type: ignore[misc]
    return (a * 4 + i) * across + b


def _tile_runs(plan: SpreadPlan, eqn: JaxprEqn) -> bool:
    """Whether a lane's columns of a row lie side by side in memory."""
    return _stride_w(eqn) == 1 and plan.tile[1] > 1  # type: ignore[index]


def _tile_offset(env: Environment, eqn: JaxprEqn, leaves: list, a: int, b: int, i: int) -> str:
    terms = []
    leaves = list(leaves)
    for what, stride in eqn.params["terms"]:
        if what in ("m", "w"):
            e = f"_m{a}_{i}" if what == "m" else f"_w{b}"
        elif what == "idx":
            e = f"({env.val(leaves.pop(0)).expr})"
        else:
            if what * stride:
                terms.append(str(what * stride))
            continue
        terms.append(f"{e} * {stride}" if stride != 1 else e)
    return " + ".join(terms) or "0"


def _masked(plan: SpreadPlan, q: int) -> bool:
    return (q + 1) * plan.team * plan.vec > plan.width


def _offset(env: Environment, eqn: JaxprEqn, leaves: list, chunk: int | None) -> str:
    """The element offset of an access in its block: of its row, and of
    chunk `chunk` along it."""
    terms = []
    leaves = list(leaves)
    for what, stride in eqn.params["terms"]:
        if what == "m":
            e = "_m"
        elif what == "w":
            e = f"_w{chunk}"
        elif what == "idx":
            e = f"({env.val(leaves.pop(0)).expr})"
        else:
            if what * stride:
                terms.append(str(what * stride))
            continue
        terms.append(f"{e} * {stride}" if stride != 1 else e)
    return " + ".join(terms) or "0"


def _stride_w(eqn: JaxprEqn) -> int | None:
    return next((s for what, s in eqn.params["terms"] if what == "w"), None)


def _tile_access(env: Environment, cursor: Cursor, plan: SpreadPlan, eqn: JaxprEqn, leaves: list, ref: CVal,
                 val: CVal, store: bool) -> None:
    """Every slot of a tiled block between memory and the array `val`, a
    row's neighbouring columns as one object where the row has them all.
    Slots past the block are not stored, and load as zero."""
    down, across = plan.tile  # type: ignore[misc]
    runs = _tile_runs(plan, eqn)
    rows_alike = not any(what == "m" for what, _ in eqn.params["terms"])  # one row serves all
    for a in range(down):
        for i in range(4):
            conds = {b: c for aa, b, ii, c in _tile_slots(plan) if (aa, ii) == (a, i)}
            first = _tile_slot(plan, a, 0, i)
            if rows_alike and not store and (a, i) != (0, 0):
                for b in range(across):
                    cursor.emit(f"{val.at(str(first + b))} = {val.at(str(b))};")
                continue

            def each() -> None:
                for b, cond in conds.items():
                    x = f"{ref.expr}[{_tile_offset(env, eqn, leaves, a, b, i)}]"
                    guard = f"if ({cond}) " if cond else ""
                    v = val.at(str(first + b))
                    cursor.emit(f"{guard}{f'{x} = {v}' if store else f'{v} = {x}'};")

            if not store and any(conds.values()):
                for b in range(across):
                    cursor.emit(f"{val.at(str(first + b))} = ({ref.ctype})0;")
            if not runs:
                each()
                continue
            mem, reg = f"{ref.expr} + {_tile_offset(env, eqn, leaves, a, 0, i)}", f"&{val.expr}[{first}]"
            to, frm = (mem, reg) if store else (reg, mem)
            copy = f"__builtin_memcpy({to}, {frm}, sizeof({ref.ctype}) * {across});"
            whole = conds[across - 1]  # the last column's condition is all of them
            cursor.emit(f"if ({whole}) {{ {copy} }}" if whole else copy)
            if whole and plan.width % across:
                cursor.emit("else {")
                each()
                cursor.emit("}")


@rule("spread_get")
def _rule_spread_get(env: Environment, cursor: Cursor, eqn: JaxprEqn) -> None:
    """Load this lane's part of a block. A lane's V neighbouring elements
    are copied as one object of the element's alignment, so the compiler
    makes one wide load of them where the hardware takes it unaligned;
    slots past the row's end hold zero."""
    plan = env.spread  # type: ignore[attr-defined]
    ref = env.val(eqn.invars[0])
    leaves = eqn.invars[1:]
    out = eqn.outvars[0]
    if plan.tile:
        dst = declare(env, cursor, out)
        _tile_access(env, cursor, plan, eqn, leaves, ref, dst, False)
        return
    stride = _stride_w(eqn)
    if stride is None:
        declare(env, cursor, out, init=f"{ref.expr}[{_offset(env, eqn, leaves, None)}]")
        return
    dst = declare(env, cursor, out, init=f"({ref.ctype})0") if plan.slots == 1 else declare(env, cursor, out)
    for q in range(plan.chunks):
        at = _offset(env, eqn, leaves, q)
        slots = range(q * plan.vec, (q + 1) * plan.vec)
        if plan.slots > 1 and _masked(plan, q):
            for s in slots:
                cursor.emit(f"{dst.at(str(s))} = ({ref.ctype})0;")
        if _masked(plan, q):
            cursor.emit(f"if (_k{q}) {{")
        if plan.vec > 1 and stride == 1:
            cursor.emit(f"__builtin_memcpy(&{dst.expr}[{q * plan.vec}], {ref.expr} + {at}, sizeof({ref.ctype}) * {plan.vec});")
        else:
            for v, s in enumerate(slots):
                cursor.emit(f"{dst.at(str(s))} = {ref.expr}[{at}{f' + {v * stride}' if v else ''}];")
        if _masked(plan, q):
            cursor.emit("}")


@rule("spread_swap")
def _rule_spread_swap(env: Environment, cursor: Cursor, eqn: JaxprEqn) -> None:
    """Store this lane's part of a block: its own elements; one value per
    row from the team's first lane, one row for all from the first row."""
    plan = env.spread  # type: ignore[attr-defined]
    ref = env.val(eqn.invars[0])
    value = env.val(eqn.invars[1])
    leaves = eqn.invars[2:]
    if ref.readonly:
        raise EmitError("cannot store into an input ref")
    if plan.tile:
        if value.size == 1 or value.ctype != ref.ctype:
            packed = cursor.fresh("_v")
            cursor.emit(f"{ref.ctype} {packed}[{plan.slots}];")
            for s in range(plan.slots):
                cursor.emit(f"{packed}[{s}] = {value.at(str(s))};")
            value = CVal(packed, (plan.slots,), ref.ctype)
        _tile_access(env, cursor, plan, eqn, leaves, ref, value, True)
        return
    guards = []
    if eqn.params.get("first_row") and plan.rows > 1:
        guards.append("_m == 0")
    if eqn.params.get("first_lane"):
        guards.append("_t == 0")
    if guards:
        cursor.emit(f"if ({' && '.join(guards)}) {{")
    stride = _stride_w(eqn)
    if stride is None:
        cursor.emit(f"{ref.expr}[{_offset(env, eqn, leaves, None)}] = {value.at('0')};")
    else:
        wide = plan.vec > 1 and stride == 1
        if wide and (value.size == 1 or value.ctype != ref.ctype):
            packed = cursor.fresh("_v")
            cursor.emit(f"{ref.ctype} {packed}[{plan.slots}];")
            for s in range(plan.slots):
                cursor.emit(f"{packed}[{s}] = {value.at(str(s))};")
            value = CVal(packed, (plan.slots,), ref.ctype)
        for q in range(plan.chunks):
            at = _offset(env, eqn, leaves, q)
            if _masked(plan, q):
                cursor.emit(f"if (_k{q}) {{")
            if wide:
                cursor.emit(f"__builtin_memcpy({ref.expr} + {at}, &{value.expr}[{q * plan.vec}], sizeof({ref.ctype}) * {plan.vec});")
            else:
                for v in range(plan.vec):
                    cursor.emit(f"{ref.expr}[{at}{f' + {v * stride}' if v else ''}] = {value.at(str(q * plan.vec + v))};")
            if _masked(plan, q):
                cursor.emit("}")
    if guards:
        cursor.emit("}")


@rule("spread_index")
def _rule_spread_index(env: Environment, cursor: Cursor, eqn: JaxprEqn) -> None:
    """`iota` along the block: the row, or each slot's element."""
    plan = env.spread  # type: ignore[attr-defined]
    out = eqn.outvars[0]
    ct = ctype_of(out.aval.dtype)
    cast = f"({ct})(float)" if ct == "__bf16" else f"({ct})"
    if plan.tile:
        dst = declare(env, cursor, out)
        for a, b, i, _ in _tile_slots(plan):
            cursor.emit(f"{dst.at(str(_tile_slot(plan, a, b, i)))} = {cast}{f'_m{a}_{i}' if eqn.params['axis'] == 'm' else f'_w{b}'};")
        return
    if eqn.params["axis"] == "m":
        declare(env, cursor, out, init=f"{cast}_m")
        return
    if plan.slots == 1:
        declare(env, cursor, out, init=f"{cast}_w0")
        return
    dst = declare(env, cursor, out)
    for s in range(plan.slots):
        cursor.emit(f"{dst.at(str(s))} = {cast}(_w{s // plan.vec} + {s % plan.vec});")


# Cross-lane steps that combine ever larger groups; each leaves every lane of
# the group with the same value, bit for bit (a + b and b + a are equal).
_DPP_STEPS = ((2, "0xB1"), (4, "0x4E"), (8, "0x141"), (16, "0x140"))


@rule("spread_reduce")
def _rule_spread_reduce(env: Environment, cursor: Cursor, eqn: JaxprEqn) -> None:
    """One value per row over the team; every lane gets it. FAST float sums
    accumulate in float32 and take each lane's slots first; float sums of
    the other modes are added element by element in the traced order, from
    a copy of the row in LDS that every lane reads (the reads are the same
    address for a whole team, so each is one broadcast)."""
    plan = env.spread  # type: ignore[attr-defined]
    mode = getattr(env, "math_mode", None)
    kind = eqn.params["kind"]
    src = env.val(eqn.invars[0])
    out = eqn.outvars[0]
    ct = ctype_of(out.aval.dtype)
    isf = ct in FLOAT_CTYPES
    if kind == "sum" and isf and (mode is None or math_mode_ordinal(mode) != 2):
        _ordered_sum(env, cursor, plan, src, out, ct)
        return
    wt = "float" if isf else ("int" if ct == "bool" else ct)
    init = {"sum": "0.0f" if isf else "0", "or": "0", "and": "1",
            "max": "(-__builtin_inff())" if isf else {"int": "(-2147483647 - 1)", "unsigned int": "0u", "bool": "0"}.get(ct),
            "min": "__builtin_inff()" if isf else {"int": "2147483647", "unsigned int": "0xFFFFFFFFu", "bool": "1"}.get(ct)}[kind]

    def comb(a: str, b: str) -> str:
        if kind == "sum":
            return f"({a} + {b})"
        if kind in ("max", "min"):
            return f"ph_f{kind}({a}, {b})" if isf else f"(({a} {'>' if kind == 'max' else '<'} {b}) ? {a} : {b})"
        return f"({a} {'|' if kind == 'or' else '&'} {b})"

    acc = cursor.fresh("_sr")
    cursor.emit(f"{wt} {acc} = {init};")
    for s in range(plan.slots):
        x = f"({wt})({src.at(str(s))})"
        if _masked(plan, s // plan.vec):
            x = f"(_k{s // plan.vec} ? {x} : {init})"
        cursor.emit(f"{acc} = {comb(acc, x)};")
    team = min(plan.team, WAVE)
    for group, ctrl in _DPP_STEPS:
        if team >= group:
            # named first: inside a conditional expression the exchange
            # would run on a part of the lanes only
            a = cursor.fresh("_sd")
            cursor.emit(f"const {wt} {a} = ph_dpp<{ctrl}>({acc});")
            cursor.emit(f"{acc} = {comb(acc, a)};")
    for group in (32, 64):
        if team >= group:
            a, b = cursor.fresh("_sa"), cursor.fresh("_sb")
            cursor.emit(f"{wt} {a}, {b};")
            cursor.emit(f"ph_swap{group // 2}({acc}, {a}, {b});")
            cursor.emit(f"{acc} = {comb(a, b)};")
    if plan.team > WAVE:
        waves = plan.team // WAVE
        sh = cursor.fresh("_lds")
        cursor.emit(f"__shared__ {wt} {sh}[{waves}];")
        cursor.emit(f"if ((_t & {WAVE - 1}) == 0) {sh}[_t / {WAVE}] = {acc};")
        cursor.emit("__syncthreads();")
        cursor.emit(f"{acc} = {sh}[0];")
        for k in range(1, waves):
            cursor.emit(f"{acc} = {comb(acc, f'{sh}[{k}]')};")
        cursor.emit("__syncthreads();")
    declare(env, cursor, out, init=f"({acc} != 0)" if ct == "bool" else f"({ct})({acc})")


def _ordered_sum(env: Environment, cursor: Cursor, plan: SpreadPlan, src: CVal, out: Any, ct: str) -> None:
    """init 0, then one add per element in index order, in the type a lane
    alone accumulates in (bfloat16 sums in float32, rounded once)."""
    act = "float" if ct == "__bf16" else ct
    # the same bytes a row in every type: teams of other wavefronts may be a sum ahead
    stride = row_stride(plan.width) * (2 if act == "_Float16" else 1)
    teams = max(1, env.spread_block // plan.team)  # type: ignore[attr-defined]
    row, acc = cursor.fresh("_rp"), cursor.fresh("_acc")
    sync = "__syncthreads();" if plan.team > WAVE else "ph_wave_sync();"
    # One array for all sums of a kernel (each ends with its reads done): the
    # compiler adds up those of a kernel, and three of 58 KB are past the CU's.
    env.staged = teams * row_stride(plan.width) * 4  # type: ignore[attr-defined]
    at = f"(threadIdx.x / {plan.team}u) * {stride}u" if teams > 1 else "0"
    cursor.emit(f"{act}* {row} = ({act}*){STAGING} + {at};")
    for s in range(plan.slots):
        q = s // plan.vec
        put = f"{row}[_w{q} + {s % plan.vec}] = ({act})({src.at(str(s))});"
        cursor.emit(f"if (_k{q}) {put}" if _masked(plan, q) else put)
    cursor.emit(sync)
    i = cursor.fresh("_i")
    cursor.emit(f"{act} {acc} = ({act})0;")
    cursor.emit("#pragma unroll 16")
    with cursor.block(f"for (int {i} = 0; {i} < {plan.width}; ++{i})"):
        cursor.emit(f"{acc} = {acc} + {row}[{i}];")
    cursor.emit(sync)
    declare(env, cursor, out, init=f"({ct})({acc})")


_VECTORS = {"float": "ph_f32x4", "__bf16": "ph_bf16x8", "_Float16": "ph_f16x8"}
# Instruction of a 16-bit operand pair (8 elements a lane, 32 per step).
_MFMA16 = {"__bf16": "__builtin_amdgcn_mfma_f32_16x16x32_bf16", "_Float16": "__builtin_amdgcn_mfma_f32_16x16x32_f16"}


@rule("spread_dot")
def _rule_spread_dot(env: Environment, cursor: Cursor, eqn: JaxprEqn) -> None:
    """Rows of `lhs` (M, K) times `rhs` (K, W) into the block's tiles.

    FAST: matrix instructions, float32 accumulators (16x16x4 for float32,
    16x16x32 for the 16-bit types, whose products are exact in float32). A
    lane of tile row l % 16 takes 16 neighbouring bytes of its row per step,
    at the same k for both operands, so their order within a step is free.
    Rows and columns past the block read its last ones (their results are
    not stored); k past the end is zero in both.

    Other modes: the traced sequence acc = acc + a * b in k order, each lane
    for its own elements (4 rows a tile, one column), four k at a time.

    Rows x (64, 32) + bias, tanh, 262,144 rows: float32 280 -> 22 us (4.6
    TB/s of the 101 MB it cannot do without), bfloat16 257 -> 12.7, in order
    547 -> 46; (128, 64) bfloat16 1,162 -> 28 us. A row per lane read its row
    from memory once per column. What is left is the way through the caches: a
    wavefront of 32 rows (8 KB there) loads all the weights (8 KB) again."""
    plan = env.spread  # type: ignore[attr-defined]
    mode = getattr(env, "math_mode", None)
    lhs, rhs = env.val(eqn.invars[0]), env.val(eqn.invars[1])
    out = eqn.outvars[0]
    ct = ctype_of(out.aval.dtype)
    k = int(eqn.params["k"])
    sk, sn = eqn.params["rhs_strides"]
    down, across = plan.tile
    dst = declare(env, cursor, out)
    ragged = across * TILE > plan.width
    cols = []
    for b in range(across):
        cols.append(cursor.fresh("_col"))
        cursor.emit(f"const int {cols[-1]} = {f'min(_w{b}, {plan.width - 1})' if ragged else f'_w{b}'};")
    # A lane's neighbouring columns come in one load, from the last place
    # where the row has them all.
    wide_cols = sn == 1 and across > 1 and plan.width >= across
    if wide_cols and ragged and plan.width % across:
        wide_cols = False
    first_col = cols[0]
    if wide_cols and ragged:
        first_col = cursor.fresh("_col")
        cursor.emit(f"const int {first_col} = min(_w0, {plan.width - across});")

    def at(row: str, col: str, kk: str) -> tuple[str, str]:
        r = f"{rhs.expr}[({kk}) * {sk} + {col}]" if sn == 1 else f"{rhs.expr}[{kk} + {col} * {sn}]"
        return f"{lhs.expr}[{row} * {k} + {kk}]", r

    if mode is not None and math_mode_ordinal(mode) == 2:
        per = 4 if lhs.ctype == "float" else 8  # elements a lane takes per step
        step = 4 * per
        rows, accs = [], []
        for a in range(down):
            rows.append(cursor.fresh("_row"))
            r = f"_r + {TILE * a} + _c"
            clip = plan.rows % (TILE * down)
            cursor.emit(f"const int {rows[-1]} = {f'min({r}, {plan.rows - 1})' if clip else r};")
            for b in range(across):
                accs.append(cursor.fresh("_acc"))
                cursor.emit(f"ph_f32x4 {accs[-1]} = {{0.0f, 0.0f, 0.0f, 0.0f}};")

        def one(k0: str, tail: bool) -> None:
            base = cursor.fresh("_k")
            cursor.emit(f"const int {base} = {k0} + {per} * _h;")
            # A tail takes the last elements there are and makes those of the
            # lane before it zero: no branch around a load. (64, 40) float16
            # blocks of k = 15, 177,664 rows 17.9 -> 13.5 us, k = 84 7.4 -> 6.4,
            # float32 k = 50 35.4 -> 33.0. Whole pieces of float32 stay behind
            # their one branch (k = 36 15.0 against 16.5 us, 100 22.1 / 25.0).
            first, short = base, tail and k < per
            if tail and (k % per or per == 8):
                tail = False
                if not short:
                    base = cursor.fresh("_k")
                    cursor.emit(f"const int {base} = min({first}, {k - per});")
            ks = [f"min({base} + {v}, {k - 1})" if short else f"{base} + {v}" for v in range(per)]
            names = []
            for row in rows:
                names.append(cursor.fresh("_fa"))
                _fragment(cursor, names[-1], lhs, [at(row, "0", x)[0] for x in ks], base, k, tail, not short)
            wide = []
            if wide_cols:
                vt = _VECTORS[rhs.ctype]
                wide = [cursor.fresh("_fb") for _ in range(across)]
                row = cursor.fresh("_wr")
                zero = ", ".join([f"({rhs.ctype})0"] * per)
                for x in wide:
                    cursor.emit(f"{vt} {x}{f' = {{{zero}}}' if tail else ''};")
                for v in range(per):
                    cursor.emit(f"{f'if ({base} + {v} < {k}) ' if tail else ''}{{ {rhs.ctype} {row}[{across}]; "
                                f"__builtin_memcpy({row}, &{at('0', first_col, ks[v])[1]}, sizeof({rhs.ctype}) * {across}); "
                                + " ".join(f"{x}[{v}] = {row}[{b}];" for b, x in enumerate(wide)) + " }")
            else:
                for col in cols:
                    wide.append(cursor.fresh("_fb"))
                    _fragment(cursor, wide[-1], rhs, [at("0", col, x)[1] for x in ks], base, k, tail, sk == 1 and not short)
            if first != base or short:
                for x, c in [*((x, lhs) for x in names), *((x, rhs) for x in wide)]:
                    for v in range(per):
                        test = f"{base} + {v} < {k}" if short else f"{base} + {v} >= {first}"
                        cursor.emit(f"{x}[{v}] = {test} ? {x}[{v}] : ({c.ctype})0;")
            for a in range(down):
                for b in range(across):
                    acc = accs[a * across + b]
                    if per == 4:
                        for v in range(4):
                            cursor.emit(f"{acc} = __builtin_amdgcn_mfma_f32_16x16x4f32({names[a]}[{v}], {wide[b]}[{v}], {acc}, 0, 0, 0);")
                    else:
                        cursor.emit(f"{acc} = {_MFMA16[lhs.ctype]}({names[a]}, {wide[b]}, {acc}, 0, 0, 0);")

        full = k // step
        if full:
            i = cursor.fresh("_s")
            cursor.emit("#pragma unroll")
            with cursor.block(f"for (int {i} = 0; {i} < {full * step}; {i} += {step})"):
                one(i, False)
        if k % step:
            cursor.emit("{")
            one(str(full * step), True)
            cursor.emit("}")
        for a, b, i, _ in _tile_slots(plan):
            cursor.emit(f"{dst.at(str(_tile_slot(plan, a, b, i)))} = ({ct}){accs[a * across + b]}[{i}];")
        return
    act = "float" if ct == "__bf16" else ct
    slots = [(_tile_slot(plan, a, b, i), a, b, i) for a, b, i, _ in _tile_slots(plan)]
    acc = cursor.fresh("_acc")
    cursor.emit(f"{act} {acc}[{plan.slots}];")
    for s in range(plan.slots):
        cursor.emit(f"{acc}[{s}] = ({act})0;")

    def conv(x: str, c: CVal) -> str:
        return x if c.ctype == act else f"(({act}){x})"

    def steps(k0: str, n: int) -> None:
        x, y = cursor.fresh("_x"), cursor.fresh("_y")
        cursor.emit(f"{lhs.ctype} {x}[{4 * down}][{n}];")
        cursor.emit(f"{rhs.ctype} {y}[{n}][{across}];")
        for a in range(down):
            for i in range(4):
                row = f"_m{a}_{i}"
                if plan.rows % (TILE * down):
                    row = f"min({row}, {plan.rows - 1})"
                cursor.emit(f"__builtin_memcpy({x}[{4 * a + i}], {lhs.expr} + {row} * {k} + {k0}, sizeof({lhs.ctype}) * {n});")
        for v in range(n):
            if wide_cols:
                cursor.emit(f"__builtin_memcpy({y}[{v}], &{at('0', first_col, f'{k0} + {v}')[1]}, sizeof({rhs.ctype}) * {across});")
                continue
            for b in range(across):
                cursor.emit(f"{y}[{v}][{b}] = {at('0', cols[b], f'{k0} + {v}')[1]};")
        for v in range(n):
            for s, a, b, i in slots:
                cursor.emit(f"{acc}[{s}] = {acc}[{s}] + {conv(f'{x}[{4 * a + i}][{v}]', lhs)} * {conv(f'{y}[{v}][{b}]', rhs)};")

    if k >= 4:
        i = cursor.fresh("_s")
        with cursor.block(f"for (int {i} = 0; {i} < {k // 4 * 4}; {i} += 4)"):
            steps(i, 4)
    if k % 4:
        cursor.emit("{")
        steps(str(k // 4 * 4), k % 4)
        cursor.emit("}")
    for s in range(plan.slots):
        cursor.emit(f"{dst.at(str(s))} = ({ct}){acc}[{s}];")


def _fragment(cursor: Cursor, name: str, ref: CVal, elements: list[str], base: str, k: int, tail: bool, run: bool) -> None:
    """Declare a lane's operand of a matrix instruction: `elements` in k
    order, from `base` on (zero past k in a `tail`, of whole operands);
    neighbours in memory if `run`, then read as one object of the element's
    alignment."""
    n = len(elements)
    vt = _VECTORS[ref.ctype]
    copy = f"__builtin_memcpy(&{name}, &{elements[0]}, sizeof({ref.ctype}) * {n});"
    if run and not tail:
        cursor.emit(f"{vt} {name};")
        cursor.emit(copy)
        return
    zero = ", ".join([f"({ref.ctype})0"] * n)
    if run:  # all of it or none (k a multiple of n)
        cursor.emit(f"{vt} {name} = {{{zero}}};")
        cursor.emit(f"if ({base} < {k}) {copy}")
        return
    cursor.emit(f"{vt} {name} = {{{zero}}};" if tail else f"{vt} {name};")
    for v, x in enumerate(elements):
        cursor.emit(f"if ({base} + {v} < {k}) {name}[{v}] = {x};" if tail else f"{name}[{v}] = {x};")
