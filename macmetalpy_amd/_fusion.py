"""Lazy fusion engine: expression DAG -> one HIP kernel (hiprtc), cached.

Reference: src/macmetalpy/_fusion.py.  The reference records unary ops (and
binary ops over already-lazy operands) as a DAG of ``InputNode`` /
``UnaryOpNode`` / ``BinaryOpNode`` (:37-71), limits depth to 16 (:24), and
on materialisation emits one MSL ``fused_op`` kernel over same-shape,
same-dtype, contiguous inputs (:297-409), caching the text by topology
(:408-436).  Scalars and broadcasts are materialised into full arrays
before they reach the DAG (ndarray.py:1026, 1062-1065).

This engine keeps the node names, the depth cap and the materialisation
triggers, and goes further:

* every elementwise op is lazy (binary roots too), scalars are ``ScalarNode``
  kernel arguments and broadcast operands are stride-0 views, so
  ``tanh(x*r + 1.0)`` with ``r`` of shape (1, N) reads ``x`` and ``r`` once;
* leaves may be strided views of any supported dtype; casts are nodes;
* a reduction over the last axis (or all axes) can be fused as an epilogue
  (``materialize_reduce``), accumulating in float64 per row;
* a DAG of a single op over contiguous operands runs the precompiled
  kernels of libmmp_hip.so (the reference's single-unary fast path,
  _fusion.py:452-464, generalised to binary and scalar forms);
* generated kernels evaluate the same csrc/mmp_ops.h functions with the same
  flags as the precompiled ones, so fused == unfused bit for bit.

Generated kernels are HBM-bound: each leaf is read once per output element
(a broadcast leaf is re-read from cache) and the output written once.
"""
from __future__ import annotations

import ctypes
import os
import threading
from typing import Optional

import numpy as np

from . import _abi
from ._backend import HipBackend
from ._config import get_config
from ._dtypes import ctype_name, dtype_code

__all__ = [
    "FusionNode", "InputNode", "ScalarNode", "UnaryOpNode", "BinaryOpNode", "CastNode",
    "WhereNode", "materialize", "materialize_reduce", "generate_source", "_MAX_DEPTH", "RTC_OPTIONS",
]

_MAX_DEPTH = 16
_MAX_LEAVES = 24
_BLOCK = 256
_UNROLL = 4
_ELEMS = 4  # consecutive elements per thread per unroll step (vector path)


def _map_unroll(kinds) -> int:
    """Unroll steps of a map kernel's workgroup tile (_BLOCK * _ELEMS
    elements each).  An expression with a single contiguous leaf and
    nothing else to read streams best in 1024-element tiles; two or more
    leaves (or a broadcast one) in 4096-element tiles.  Measured on MI355X
    at 2^28 elements (GB/s, two runs; tiles of 1024 / 2048 / 4096 / 8192):
    sqrt(|x|) + exp(-x*x) 6132-6487 / 6331-6400 / 6160-6214 / 5952-6066,
    x >> 3 (int32) 6355-6388 / 5886-5967 / 6001-6067 / 5431-5511, isnan
    6526-6581 / 6500-6518 / 6053-6191 / 6010-6074, clip 6373-6506 /
    6212-6275 / 6005-6033 / 6115-6145; a & b 6190-6203 / 6082-6126 /
    6354-6393 / 5798-5814, a * b + c 5938-5965 / 5998-6004 / 6100-6143 /
    5818-5830, X * r with a broadcast row 5951-6035 / 5854-5904 / 6023-6030
    / 5855-5912.  The native gate applies the same rule (native_gate.cpp,
    map_tile)."""
    return 1 if len(kinds) == 1 and kinds[0] == "c" else _UNROLL


def _map_tile(kinds) -> int:
    return _BLOCK * _ELEMS * _map_unroll(kinds)
# Workgroups of a row-sum launch, split over its rows (a row gets at most
# one per 4096 elements).  Measured on 2^28 float32 reduced whole:
# any(a > 3) / count_nonzero 6.7 TB/s at 1024, 5.9-6.0 at 2048, 5.7 at 512;
# sum(a * b) 6.8-6.9 at all three.
_SUM_BLOCKS = 1024
_SUM_UNROLL = 4     # vector steps per thread unrolled in the row-sum loop

_CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc")
# Same numerics flags as the precompiled library (csrc/build.py).
RTC_OPTIONS = ("-O3 -std=c++17 -ffp-contract=off "
               "-Xclang -target-feature -Xclang -packed-fp32-ops")

_ops_header_text: Optional[str] = None


def _ops_header() -> str:
    global _ops_header_text
    if _ops_header_text is None:
        with open(os.path.join(_CSRC, "mmp_ops.h")) as f:
            _ops_header_text = f.read().replace("#pragma once", "")
    return _ops_header_text


# ---------------------------------------------------------------- nodes
class FusionNode:
    __slots__ = ("_shape", "_dtype", "_depth", "_buffers", "_nleaves")


class InputNode(FusionNode):
    """A device-resident array view (buffer, element offset, strides)."""
    __slots__ = ("_buffer", "_offset", "_strides")

    def __init__(self, buffer, shape, dtype, strides, offset=0):
        self._buffer = buffer
        self._shape = tuple(shape)
        self._dtype = np.dtype(dtype)
        self._strides = tuple(strides)
        self._offset = int(offset)
        self._depth = 0
        self._buffers = (buffer,)
        self._nleaves = 1


class ScalarNode(FusionNode):
    """A scalar kernel argument: its value converted to ``dtype`` (NumPy's
    conversion), held as the little-endian bits of that value."""
    __slots__ = ("_bits",)

    def __init__(self, value, dtype):
        self._dtype = np.dtype(dtype)
        raw = np.array(value, dtype=self._dtype).tobytes()
        self._bits = int.from_bytes(raw.ljust(8, b"\0"), "little")
        self._shape = ()
        self._depth = 0
        self._buffers = ()
        self._nleaves = 0

    @property
    def _value(self):
        """The value as a 0-d array of ``dtype``."""
        raw = self._bits.to_bytes(8, "little")[:self._dtype.itemsize]
        return np.frombuffer(raw, dtype=self._dtype).reshape(())


def _merge_buffers(*nodes):
    seen, out = set(), []
    for n in nodes:
        for b in n._buffers:
            if id(b) not in seen:
                seen.add(id(b))
                out.append(b)
    return tuple(out)


class UnaryOpNode(FusionNode):
    __slots__ = ("_op_name", "_input")

    def __init__(self, op_name, input_node, shape, dtype):
        self._op_name = op_name
        self._input = input_node
        self._shape = tuple(shape)
        self._dtype = np.dtype(dtype)
        self._depth = input_node._depth + 1
        self._buffers = input_node._buffers
        self._nleaves = input_node._nleaves


class CastNode(FusionNode):
    __slots__ = ("_input",)

    def __init__(self, input_node, dtype):
        self._input = input_node
        self._shape = input_node._shape
        self._dtype = np.dtype(dtype)
        self._depth = input_node._depth  # free: folded into the consumer
        self._buffers = input_node._buffers
        self._nleaves = input_node._nleaves


class BinaryOpNode(FusionNode):
    __slots__ = ("_op_name", "_lhs", "_rhs")

    def __init__(self, op_name, lhs, rhs, shape, dtype):
        self._op_name = op_name
        self._lhs = lhs
        self._rhs = rhs
        self._shape = tuple(shape)
        self._dtype = np.dtype(dtype)
        self._depth = max(lhs._depth, rhs._depth) + 1
        self._buffers = _merge_buffers(lhs, rhs)
        self._nleaves = lhs._nleaves + rhs._nleaves


class WhereNode(FusionNode):
    """``cond ? x : y`` (reference where_shader, _kernels.py:984-1000);
    ``cond`` is a bool node, ``x`` and ``y`` have the result dtype."""
    __slots__ = ("_cond", "_x", "_y")

    def __init__(self, cond, x, y, shape, dtype):
        self._cond = cond
        self._x = x
        self._y = y
        self._shape = tuple(shape)
        self._dtype = np.dtype(dtype)
        self._depth = max(cond._depth, x._depth, y._depth) + 1
        self._buffers = _merge_buffers(cond, x, y)
        self._nleaves = cond._nleaves + x._nleaves + y._nleaves


# ---------------------------------------------------------- DAG analysis
def _c_contig_strides(shape):
    st, acc = [], 1
    for s in reversed(shape):
        st.append(acc)
        acc *= s
    return tuple(reversed(st))


def _bcast_strides(shape, strides, target):
    diff = len(target) - len(shape)
    out = [0] * diff
    for s, st, t in zip(shape, strides, target[diff:]):
        out.append(st if (s == t and s != 1) else 0)
    return out


class _Program:
    """Post-order linearisation of a DAG with deduplicated leaves."""

    def __init__(self, root):
        self.root = root
        self.arrays = []      # InputNode leaves (unique views)
        self.scalars = []     # ScalarNode leaves
        self.steps = []       # (kind, payload...) per SSA value
        self.dtypes = []      # dtype per SSA value
        self._memo = {}
        self._leaf_index = {}
        self.result = self._visit(root)

    def _visit(self, node):
        nid = id(node)
        idx = self._memo.get(nid)
        if idx is not None:
            return idx
        cls = type(node)
        if cls is InputNode:
            key = (id(node._buffer), node._offset, node._strides, node._shape, node._dtype)
            k = self._leaf_index.get(key)
            if k is None:
                k = len(self.arrays)
                self._leaf_index[key] = k
                self.arrays.append(node)
            step = ("load", k)
        elif cls is UnaryOpNode:
            step = ("unary", node._op_name, self._visit(node._input))
        elif cls is BinaryOpNode:
            step = ("binary", node._op_name, self._visit(node._lhs), self._visit(node._rhs))
        elif cls is ScalarNode:
            step = ("scalar", len(self.scalars))
            self.scalars.append(node)
        elif cls is CastNode:
            step = ("cast", self._visit(node._input))
        elif cls is WhereNode:
            step = ("where", self._visit(node._cond), self._visit(node._x),
                    self._visit(node._y))
        else:
            raise TypeError(f"unknown fusion node {cls.__name__}")
        self.steps.append(step)
        self.dtypes.append(node._dtype)
        idx = len(self.steps) - 1
        self._memo[nid] = idx
        return idx


def _collapse(shape, stride_lists, keep_last=False):
    """Merge adjacent dims contiguous for every operand; drop size-1 dims.
    Returns (shape, [strides per operand]).  With keep_last, the last dim
    is never merged with the dims before it."""
    n = len(shape)
    cshape, cstr = [], [[] for _ in stride_lists]
    for d in range(n):
        is_last = keep_last and d == n - 1
        if shape[d] == 1 and not is_last:
            continue
        mergeable = bool(cshape) and not is_last and all(
            sl[-1] == st[d] * shape[d] for sl, st in zip(cstr, stride_lists))
        if mergeable:
            cshape[-1] *= shape[d]
            for sl, st in zip(cstr, stride_lists):
                sl[-1] = st[d]
        else:
            cshape.append(shape[d])
            for sl, st in zip(cstr, stride_lists):
                sl.append(st[d])
    return cshape, cstr


# --------------------------------------------------------------- codegen
_ARG_FIELDS_CACHE: dict = {}


def _param_struct(n_in, n_sc, n_outer):
    key = (n_in, n_sc, n_outer)
    cls = _ARG_FIELDS_CACHE.get(key)
    if cls is None:
        fields = [
            ("ptr", ctypes.c_uint64 * max(1, n_in)),
            ("outp", ctypes.c_uint64),
            ("sbits", ctypes.c_uint64 * max(1, n_sc)),
            ("n", ctypes.c_int64),
            ("rows", ctypes.c_int64),
            ("cols", ctypes.c_int64),
            ("colblocks", ctypes.c_int64),
            ("oshape", ctypes.c_int64 * max(1, n_outer)),
            ("ostride", ctypes.c_int64 * max(1, n_in * n_outer)),
            ("lstride", ctypes.c_int64 * max(1, n_in)),
            ("scale", ctypes.c_double),
        ]
        cls = type(f"FusedParams_{n_in}_{n_sc}_{n_outer}", (ctypes.Structure,),
                   {"_fields_": fields})
        _ARG_FIELDS_CACHE[key] = cls
    return cls


_STRUCT_DECL = """
struct P {{
  unsigned long long ptr[{nin}];
  unsigned long long outp;
  unsigned long long sbits[{nsc}];
  long long n, rows, cols, colblocks;
  long long oshape[{nout}];
  long long ostride[{nio}];
  long long lstride[{nin}];
  double scale;
}};
"""

_BITS_T = {1: "unsigned char", 2: "unsigned short", 4: "unsigned int", 8: "unsigned long long"}


def _acc_type(dtype):
    """Accumulator of a fused sum: float64, uint64 for unsigned inputs,
    else int64 (NumPy sums bool and signed integers as int64)."""
    if dtype.kind == "f":
        return "double", np.dtype(np.float64)
    if dtype.kind == "u":
        return "mmp_u64", np.dtype(np.uint64)
    return "mmp_i64", np.dtype(np.int64)


_FAST_DTYPES = (np.dtype(np.float32), np.dtype(np.float16))


def _op_fn(table, op_name, dtype, fast):
    """mmp_ops.h function for ``op_name`` computing in ``dtype``; the
    ``_fast`` form under fast_math for float32 / float16."""
    fn = table[op_name]
    if fast and op_name in _abi.FAST_MATH_OPS and dtype in _FAST_DTYPES:
        return fn + "_fast"
    return fn


_NONNEG_UNARY = frozenset(("abs_op", "absolute_op", "fabs_op", "square_op", "sqrt_op", "exp_op",
                           "exp2_op", "cosh_op"))


def _sign_facts(prog: _Program):
    """Per SSA value, (never below zero, never above zero) as far as the
    expression shows it, NaN aside: |x|, x*x, exp(...) are >= 0, their
    negations <= 0, products and sums of known signs follow (scalar leaves
    count as unknown: kernels are cached by structure, and a scalar's value
    is a launch parameter).  Lets the
    code generator call the forms of exp and log1p without the cases their
    argument cannot reach (bit for bit the same results)."""
    facts, canon = [], []
    for i, step in enumerate(prog.steps):
        kind, f = step[0], (False, False)
        canon.append(("load", step[1]) if kind == "load" else i)
        if prog.dtypes[i].kind != "f":
            facts.append(f)
            continue
        if kind == "cast":
            f = facts[step[1]] if prog.dtypes[step[1]].kind == "f" else f
        elif kind == "unary":
            a = facts[step[2]]
            if step[1] in _NONNEG_UNARY:
                f = (True, False)
            elif step[1] in ("neg_op", "negative_op"):
                f = (a[1], a[0])
        elif kind == "where":
            a, b = facts[step[2]], facts[step[3]]
            f = (a[0] and b[0], a[1] and b[1])
        elif kind == "binary":
            op, a, b = step[1], facts[step[2]], facts[step[3]]
            if op == "mul_op":
                if canon[step[2]] == canon[step[3]]:
                    f = (True, False)
                else:
                    f = ((a[0] and b[0]) or (a[1] and b[1]), (a[0] and b[1]) or (a[1] and b[0]))
            elif op == "add_op":
                f = (a[0] and b[0], a[1] and b[1])
            elif op == "sub_op":
                f = (a[0] and b[1], a[1] and b[0])
        facts.append(f)
    return facts


_FLAT_UNROLL = 4  # 4-element vectors per thread of a flat kernel
# Outputs a flat launch is worth: smaller ones would be under 16 of its tiles,
# and the row launch spreads them over more CUs (1000 x 100: 5.6 us a call
# either way; 30,000 x 8: 14.3 by rows, 5.7 flat).
_FLAT_MIN = 1 << 16


def _flat_cols(kinds, cols, traffic, wide, spread, tile):
    """Whether rows of ``cols`` elements of at most ``wide`` bytes go flat;
    ``traffic``: bytes of the output and of the leaves as large as it.

    A vector of a flat launch reads four elements of a row vector (or of an odd
    row) one by one, which costs more than the row launch's scalar rows as long
    as the data stay in the caches; the vectors are worth it where memory
    streams.  Us by rows / flat for (x - r) * r with a row vector, (x - c) * c
    with a value per row, r * c.  float32, 12,000,000 elements: 511 columns 19.6 /
    19.5, 19.4 / 16.8, 17.2 / 16.8; 1023 16.9 / 19.5, 16.9 / 16.8, 12.8 / 16.8;
    3001 16.2 / 19.9, 16.1 / 16.9, 10.5 / 16.9; 4097 (a tile and one element)
    23.3 / 20.2, 23.3 / 16.7, 16.6 / 16.6; whole vectors: 900 17.7 / 16.7, 17.7 /
    17, 13.3 / 9.1; 3500 16.3 / 17.2, 16.3 / 17, 10.8 / 8.8.  70,000,000: 511 156 /
    97, 156 / 92, 89 / 76; 1023 132 / 97, 132 / 91, 66 / 76; 10,001 127 / 99, 127 /
    91, 60 / 77; 3500 125 / 93, 126 / 91, 59 / 52.
    float16, 12,000,000: 1023 14.2 / 13.8, 14.3 / 10.6, 11.1 / 11.4; 3001 12.4 /
    13.9, 12.4 / 10.6, 9.5 / 11.2; 70,000,000: 3001 88 / 72, 87 / 47, 37 / 48.
    float64 (32 bytes a thread), 12,000,000: 130 48 / 43, 48 / 42, 46 / 36; 200
    36.5 / 39, 36 / 38, 35 / 34; 1023 29 / 45, 29 / 42, 20 / 35; with padded rows
    ('v') 300 53 / 48, 700 48 / 49; with a transposed leaf (``spread``) 255 64 / 42;
    70,000,000: 300 246 / 225, 241 / 220, 215 / 240; 511 201 / 259, 200 / 244, 176 /
    246; 5001 335 / 266, 277 / 243, 159 / 239."""
    big = traffic >= 192 << 20  # float32 rows of 5001: 200 MB 38.8 / 37.6, 38.8 / 33, 26 / 28.7
    streams = "f" in kinds or "v" in kinds
    empty = -(-cols // tile) * tile / cols if cols > tile else 1.0  # the row launch's tiles
    if wide == 8:
        limit = (400 if "v" in kinds else 255 if spread else 160 if not big else
                 300 if streams else 200)
        return cols <= limit or (big and streams and empty >= 1.36)
    if cols % _ELEMS == 0:
        return big or wide < 4 or cols <= 2048
    if "p" not in kinds and "g" not in kinds:  # nothing read along an odd row
        return big or wide < 4 or cols <= 1024 or cols > tile
    if big and streams:
        return True
    return (cols <= (1024 if wide < 4 else 800 if big else 512)
            or empty >= (1.6 if wide < 4 else 1.7))


def _flat_kinds(outer, cols, leaf_str, ptrs, itemsizes, out_ptr, out_itemsize, tile):
    """Leaf classes of a flat launch, or None where the row launch stays.

    The row launch gives every row its own workgroups, so rows shorter than a
    workgroup's ``tile`` leave most of it idle, and a row length that is no
    multiple of 4 takes it element by element.  The flat launch cuts the
    output into tiles whatever its rows: a vector finds its row and column
    with one 32-bit division (hence fewer than 2^31 elements).  Classes: 'f'
    follows the output (read as vectors: its pointer and the output's must be
    aligned); where rows are whole aligned vectors, a row vector repeated down
    the rows is read as vectors ('q'), so are rows lying further apart ('v'),
    and a value per row once per vector ('w'); else by element ('p', 'r', and
    'g' for any other strides, whose loads are spread too wide to take long
    rows flat).  (x - m) / d of a
    2,000,000 x 50 float32 x and row vectors m, d: 655 us by rows,
    134 flat (6 TB/s); 12,000,000 x 8: 4965 and 126.  How long rows may be is
    _flat_cols's to say."""
    if len(outer) != 1 or (cols >= tile and cols % _ELEMS == 0):
        return None
    if not _FLAT_MIN <= outer[0] * cols < 1 << 31 or out_ptr % (_ELEMS * out_itemsize):
        return None
    whole = cols % _ELEMS == 0
    kinds = []
    for (row_st, col_st), ptr, isz in zip(leaf_str, ptrs, itemsizes):
        aligned = ptr % (_ELEMS * isz) == 0
        if row_st == cols and col_st == 1 and aligned:
            kinds.append("f")
        elif row_st == 0 and col_st == 1:
            kinds.append("q" if whole and aligned else "p")
        elif col_st == 0:
            kinds.append("w" if whole else "r")
        elif col_st == 1 and whole and aligned and row_st % _ELEMS == 0:
            kinds.append("v")
        elif cols < _BLOCK:
            kinds.append("g")
        else:
            return None
    wide = max(itemsizes + [out_itemsize])
    spread = any(k == "g" and st[1] != 1 for k, st in zip(kinds, leaf_str))
    traffic = outer[0] * cols * (out_itemsize + sum(s for k, s in zip(kinds, itemsizes) if k in "fvg"))
    return kinds if _flat_cols(kinds, cols, traffic, wide, spread, tile) else None


def _flat_body(kinds, ct, vtypes, out_ct, expr_lines, res):
    """Body of a flat kernel (see _flat_kinds) after the leaf and scalar
    declarations."""
    tile = _FLAT_UNROLL * _BLOCK * _ELEMS
    L = []
    L.append("  const unsigned n = (unsigned)p.n, cols = (unsigned)p.cols;")
    for k, kind in enumerate(kinds):
        if kind in "rwgv":
            L.append(f"  const long long rs{k} = p.ostride[{k}];")
        if kind == "g":
            L.append(f"  const long long cs{k} = p.lstride[{k}];")

    def at(k):
        """Leaf k at (row, col)."""
        return {"p": f"in{k}[col]", "q": f"in{k}[col]", "r": f"in{k}[(long long)row * rs{k}]",
                "w": f"in{k}[(long long)row * rs{k}]",
                "v": f"in{k}[(long long)row * rs{k} + col]",
                "g": f"in{k}[(long long)row * rs{k} + (long long)col * cs{k}]"}[kinds[k]]

    L.append(f"  const unsigned i0 = blockIdx.x * {tile}u;")
    L.append(f"  if (n - i0 >= {tile}u) {{")
    for k, kind in enumerate(kinds):
        if kind == "f":
            L.append(f"    {vtypes[ct[k]]} l{k}[{_FLAT_UNROLL}];")
    L.append(f"    #pragma unroll\n    for (int u = 0; u < {_FLAT_UNROLL}; ++u) {{")
    L.append(f"      const unsigned i = i0 + (u * {_BLOCK} + threadIdx.x) * {_ELEMS};")
    for k, kind in enumerate(kinds):
        if kind == "f":
            L.append(f"      l{k}[u] = __builtin_nontemporal_load((const {vtypes[ct[k]]}*)(in{k} + i));")
    L.append("    }")
    L.append(f"    #pragma unroll\n    for (int u = 0; u < {_FLAT_UNROLL}; ++u) {{")
    L.append(f"      const unsigned i = i0 + (u * {_BLOCK} + threadIdx.x) * {_ELEMS};")
    L.append("      unsigned row = i / cols, col = i - row * cols;")
    for k, kind in enumerate(kinds):
        if kind in "qv":
            L.append(f"      const {vtypes[ct[k]]} l{k} = *(const {vtypes[ct[k]]}*)&{at(k)};")
        elif kind == "w":
            L.append(f"      const {ct[k]} l{k} = {at(k)};")
        elif kind != "f":
            L.append(f"      {ct[k]} l{k}[{_ELEMS}];")
    if any(kind in "prg" for kind in kinds):
        # the elements' loads ahead of the arithmetic
        L.append(f"      #pragma unroll\n      for (int e = 0; e < {_ELEMS}; ++e) {{")
        for k, kind in enumerate(kinds):
            if kind in "prg":
                L.append(f"        l{k}[e] = {at(k)};")
        L.append("        if (++col == cols) { col = 0; ++row; }")
        L.append("      }")
    L.append(f"      {vtypes[out_ct]} o;")
    L.append(f"      #pragma unroll\n      for (int e = 0; e < {_ELEMS}; ++e) {{")

    def elem(k):
        if kinds[k] == "f":
            return f"({ct[k]})l{k}[u][e]"
        return f"l{k}" if kinds[k] == "w" else f"({ct[k]})l{k}[e]"
    L.extend(expr_lines(elem, "        "))
    L.append(f"        o[e] = {res};")
    L.append("      }")
    L.append(f"      __builtin_nontemporal_store(o, ({vtypes[out_ct]}*)(({out_ct}*)p.outp + i));")
    L.append("    }")
    L.append("    return;")
    L.append("  }")
    L.append(f"  for (unsigned i = i0 + threadIdx.x; i < n; i += {_BLOCK}) {{")
    L.append("    const unsigned row = i / cols, col = i - row * cols;")
    L.extend(expr_lines(lambda k: f"in{k}[i]" if kinds[k] == "f" else at(k), "    "))
    L.append(f"    (({out_ct}*)p.outp)[i] = {res};")
    L.append("  }")
    L.append("}")
    return L


_COL_UNROLL = 4  # rows in flight per lane of a column-sum kernel


def _col_kinds(outer, cols, leaf_str):
    """Leaf classes of a column-sum launch over (rows, cols), or None: 'v'
    rows of contiguous values (any row stride), 'p' a row vector (read once
    per lane), 'r' one value per row."""
    if len(outer) != 1 or cols < _ELEMS:
        return None
    kinds = []
    for row_st, col_st in leaf_str:
        if col_st == 1:
            kinds.append("p" if row_st == 0 else "v")
        elif col_st == 0:
            kinds.append("r")
        else:
            return None
    return kinds


def _col_body(kinds, ct, expr_lines, res):
    """Body of a column-sum kernel: partial sums over the splits of the rows,
    P[split][col] in float64.  Lanes lie on the columns as in the library's
    strided reduction: 4 adjacent columns each (the last lane of a row that 4
    does not divide on the row's last 4), 2^lg lanes side by side on a row,
    the wave's others on the rows below, four waves on rows in turn; lanes
    meet by shuffles, waves in LDS."""
    U = _COL_UNROLL
    L = []
    for k, kind in enumerate(kinds):
        if kind != "p":
            L.append(f"  const long long rs{k} = p.ostride[{k}];")
    L += ["  const int lg = (int)p.n, G = 1 << lg;",
          "  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;",
          "  const long long cols = p.cols, rows = p.rows;",
          "  const unsigned S = (unsigned)p.colblocks;",
          "  const unsigned cb = blockIdx.x / S, s = blockIdx.x - cb * S;",
          f"  const long long c0 = (long long)cb * G * {_ELEMS};",
          f"  const long long cn = c0 + (lane & (G - 1)) * {_ELEMS};",
          f"  const long long c = cn + {_ELEMS} <= cols ? cn : cols - {_ELEMS};",
          "  const long long per = (rows + S - 1) / S, b0 = s * per;",
          "  const long long b1 = b0 + per < rows ? b0 + per : rows;",
          "  const long long step = 4ll << (6 - lg);",
          f"  double acc[{_ELEMS}] = {{}};",
          "  if (cn < cols) {"]
    for k, kind in enumerate(kinds):
        if kind == "p":
            L.append(f"    {ct[k]} l{k}[{_ELEMS}];")
            L.append(f"    __builtin_memcpy(l{k}, in{k} + c, sizeof(l{k}));")

    def rows_of(n):
        """One step: n rows' loads, then their values."""
        out = []
        for k, kind in enumerate(kinds):
            if kind == "v":
                out.append(f"      {ct[k]} l{k}[{n}][{_ELEMS}];")
            elif kind == "r":
                out.append(f"      {ct[k]} l{k}[{n}];")
        out.append(f"      #pragma unroll\n      for (int u = 0; u < {n}; ++u) {{")
        for k, kind in enumerate(kinds):
            if kind == "v":
                out.append(f"        __builtin_memcpy(l{k}[u], in{k} + (l + step * u) * rs{k} + c, "
                           f"sizeof(l{k}[u]));")
            elif kind == "r":
                out.append(f"        l{k}[u] = in{k}[(l + step * u) * rs{k}];")
        out.append("      }")
        out.append(f"      #pragma unroll\n      for (int u = 0; u < {n}; ++u)")
        out.append(f"        #pragma unroll\n        for (int e = 0; e < {_ELEMS}; ++e) {{")
        load = {"v": "l{}[u][e]", "p": "l{}[e]", "r": "l{}[u]"}
        out.extend(expr_lines(lambda k: load[kinds[k]].format(k), "          "))
        out.append(f"          acc[e] += (double){res};")
        out.append("        }")
        return out

    L.append("    long long l = b0 + ((long long)wave << (6 - lg)) + (lane >> lg);")
    L.append(f"    for (; l + step * {U - 1} < b1; l += step * {U}) {{")
    L.extend(rows_of(U))
    L.append("    }")
    L.append("    for (; l < b1; l += step) {")
    L.extend(rows_of(1))
    L.append("    }")
    L.append("  }")
    L += ["  for (int m = G; m < 64; m <<= 1)",
          f"    for (int e = 0; e < {_ELEMS}; ++e) acc[e] += __shfl_xor(acc[e], m, 64);",
          f"  __shared__ double part[4][{64 * _ELEMS}];",
          "  if (lane < G && cn < cols)",
          f"    for (int e = 0; e < {_ELEMS}; ++e)",
          "      if (c + e >= cn) part[wave][c + e - c0] = acc[e];",
          "  __syncthreads();",
          "  const int t = threadIdx.x;",
          f"  if (t < G * {_ELEMS} && c0 + t < cols)",
          "    ((double*)p.outp)[s * cols + c0 + t] = "
          "(((part[0][t] + part[1][t]) + part[2][t]) + part[3][t]) * p.scale;",
          "}"]
    return L


def generate_source(prog: _Program, kinds, nouter, out_dtype, vec, mode, fast=False):
    """HIP source for ``prog``.

    kinds[k]: last-dim stride class of array leaf k ('c' unit, 'b' zero,
    's' general).  nouter: number of outer (row) dims (0 = 1-D launch).
    mode: 'map' (elementwise, contiguous output), 'flat' (the same over the
    flat index, for rows too short or too odd to be a workgroup's: kinds as
    _flat_kinds gives them), 'sum' (row-sum epilogue), 'colsum' (sums down
    the columns, kinds as _col_kinds gives them).
    fast: use the fast_math forms of the transcendentals.
    """
    nin, nsc = len(prog.arrays), len(prog.scalars)
    L = []
    L.append(_ops_header())
    L.append(_STRUCT_DECL.format(nin=max(1, nin), nsc=max(1, nsc), nout=max(1, nouter),
                                 nio=max(1, nin * nouter)))
    ct = [ctype_name(a._dtype) for a in prog.arrays]
    out_ct = ctype_name(out_dtype)
    if mode == "sum":
        acc_ct, _ = _acc_type(prog.dtypes[prog.result])
    # vector types for the vectorised path
    vtypes = {}
    if vec:
        for t in set(ct + ([out_ct] if mode != "sum" else [])):
            vt = "v4_" + t.replace(" ", "_")
            st = "unsigned char" if t == "bool" else t
            vtypes[t] = vt
            L.append(f"typedef {st} {vt} __attribute__((ext_vector_type(4)));")

    signs = _sign_facts(prog)

    def expr_lines(load_expr, indent):
        """Statements computing every SSA value; load_expr(k) -> leaf k."""
        out = []
        for i, step in enumerate(prog.steps):
            t = ctype_name(prog.dtypes[i])
            kind = step[0]
            if kind == "load":
                rhs = load_expr(step[1])
            elif kind == "scalar":
                rhs = f"s{step[1]}"
            elif kind == "cast":
                src_t = ctype_name(prog.dtypes[step[1]])
                rhs = f"mmp_convert<{t}, {src_t}>(t{step[1]})"
            elif kind == "unary":
                fn = _op_fn(_abi.UNARY_FN, step[1], prog.dtypes[i], fast)
                if fn == "op_exp" and signs[step[2]][1]:
                    fn = "op_exp_nonpos"
                elif fn == "op_log1p" and signs[step[2]][0]:
                    fn = "op_log1p_nonneg"
                rhs = f"{fn}(t{step[2]})"
            elif kind == "where":
                rhs = f"(t{step[1]} ? t{step[2]} : t{step[3]})"
            elif step[1] in _abi.COMPARE_OPS:
                rhs = f"(t{step[2]} {_abi.COMPARE_OPS[step[1]][1]} t{step[3]})"
            else:
                rhs = f"{_op_fn(_abi.BINARY_FN, step[1], prog.dtypes[i], fast)}(t{step[2]}, t{step[3]})"
            out.append(f"{indent}const {t} t{i} = {rhs};")
        return out

    L.append(f'extern "C" __global__ __launch_bounds__({_BLOCK}) void fused_op(P p) {{')
    for k in range(nin):
        L.append(f"  const {ct[k]}* __restrict__ in{k} = (const {ct[k]}*)p.ptr[{k}];")
    for j, sc in enumerate(prog.scalars):
        t = ctype_name(sc._dtype)
        bt = _BITS_T[sc._dtype.itemsize]
        if t == "bool":
            L.append(f"  const bool s{j} = (p.sbits[{j}] & 1ull) != 0;")
        else:
            L.append(f"  const {t} s{j} = __builtin_bit_cast({t}, ({bt})p.sbits[{j}]);")
    if mode == "colsum":
        L.extend(_col_body(kinds, ct, expr_lines, f"t{prog.result}"))
        return "\n".join(L) + "\n"
    if mode == "flat":
        L.extend(_flat_body(kinds, ct, vtypes, out_ct, expr_lines, f"t{prog.result}"))
        return "\n".join(L) + "\n"
    # row setup
    if nouter == 0:
        L.append("  const long long row = 0; const long long cb = blockIdx.x;")
        for k in range(nin):
            L.append(f"  const long long ro{k} = 0;")
    else:
        # workgroup ids, colblocks and the outer extents are below 2^31
        # (HIP's grid limit), so the index splits divide in 32 bits: a
        # 64-bit division is ~130 scalar instructions per wave
        L.append("  const unsigned cbk = (unsigned)p.colblocks;")
        L.append("  const unsigned rowu = blockIdx.x / cbk;")
        L.append("  const long long row = rowu;")
        L.append("  const long long cb = blockIdx.x - rowu * cbk;")
        for k in range(nin):
            L.append(f"  long long ro{k} = 0;")
        L.append("  { unsigned r = rowu;")
        for d in range(nouter - 1, -1, -1):
            L.append(f"    {{ const unsigned q = r / (unsigned)p.oshape[{d}]; "
                     f"const long long ix = r - q * (unsigned)p.oshape[{d}];")
            for k in range(nin):
                L.append(f"      ro{k} += ix * p.ostride[{k * nouter + d}];")
            L.append("      r = q; }")
        L.append("  }")
    L.append("  const long long cols = p.cols;")
    tile = _map_tile(kinds)
    unroll = _map_unroll(kinds)

    def scalar_load(k, col):
        if kinds[k] == "c":
            return f"in{k}[ro{k} + {col}]"
        if kinds[k] == "b":
            return f"in{k}[ro{k}]"
        return f"in{k}[ro{k} + {col} * p.lstride[{k}]]"

    res = f"t{prog.result}"
    if mode == "map":
        L.append("  const long long obase = row * cols;")
        L.append(f"  const long long c0 = cb * {tile}LL;")
        L.append(f"  const long long c1 = c0 + {tile}LL < cols ? c0 + {tile}LL : cols;")
        if vec:
            L.append(f"  if (c0 + {tile}LL <= cols) {{")
            for k in range(nin):
                if kinds[k] == "c":
                    L.append(f"    {vtypes[ct[k]]} l{k}[{unroll}];")
            L.append(f"    #pragma unroll\n    for (int u = 0; u < {unroll}; ++u) {{")
            L.append(f"      const long long c = c0 + ((long long)u * {_BLOCK} + threadIdx.x) * {_ELEMS};")
            for k in range(nin):
                if kinds[k] == "c":
                    L.append(f"      l{k}[u] = __builtin_nontemporal_load((const {vtypes[ct[k]]}*)(in{k} + ro{k} + c));")
            L.append("    }")
            for k in range(nin):
                if kinds[k] == "b":
                    L.append(f"    const {ct[k]} bc{k} = in{k}[ro{k}];")
            L.append(f"    #pragma unroll\n    for (int u = 0; u < {unroll}; ++u) {{")
            L.append(f"      const long long c = c0 + ((long long)u * {_BLOCK} + threadIdx.x) * {_ELEMS};")
            L.append(f"      {vtypes[out_ct]} r;")
            L.append(f"      #pragma unroll\n      for (int e = 0; e < {_ELEMS}; ++e) {{")

            def vload(k):
                if kinds[k] == "c":
                    return f"({ct[k]})l{k}[u][e]"
                return f"bc{k}"
            L.extend(expr_lines(vload, "        "))
            L.append(f"        r[e] = {res};")
            L.append("      }")
            L.append(f"      __builtin_nontemporal_store(r, ({vtypes[out_ct]}*)(({out_ct}*)p.outp + obase + c));")
            L.append("    }")
            L.append("    return;")
            L.append("  }")
        L.append(f"  for (long long c = c0 + threadIdx.x; c < c1; c += {_BLOCK}) {{")
        L.extend(expr_lines(lambda k: scalar_load(k, "c"), "    "))
        L.append(f"    (({out_ct}*)p.outp)[obase + c] = {res};")
        L.append("  }")
        L.append("}")
    else:  # row-sum epilogue
        L.append(f"  {acc_ct} acc = 0;")
        L.append("  const unsigned cbk_ = (unsigned)p.colblocks;")
        if vec:
            # column ranges are multiples of 4 elements, so every 16-byte
            # (or narrower) vector load of a contiguous leaf is aligned
            L.append("  const long long span = cols + p.colblocks - 1;")
            L.append("  const long long per = ((span < 0x100000000LL ? (long long)((unsigned)span / cbk_) "
                     ": span / p.colblocks) + 3) & ~3LL;")
        else:
            L.append("  const long long span = cols + p.colblocks - 1;")
            L.append("  const long long per = span < 0x100000000LL ? (long long)((unsigned)span / cbk_) "
                     ": span / p.colblocks;")
        L.append("  const long long c0 = cb * per;")
        L.append("  const long long c1 = c0 + per < cols ? c0 + per : cols;")
        if vec:
            for k in range(nin):
                if kinds[k] == "b":
                    L.append(f"  const {ct[k]} bc{k} = in{k}[ro{k}];")
            L.append(f"  #pragma unroll {_SUM_UNROLL}")
            L.append(f"  for (long long c = c0 + threadIdx.x * {_ELEMS}; c < c1; "
                     f"c += {_BLOCK * _ELEMS}) {{")
            for k in range(nin):
                if kinds[k] == "c":
                    L.append(f"    const {vtypes[ct[k]]} l{k} = __builtin_nontemporal_load("
                             f"(const {vtypes[ct[k]]}*)(in{k} + ro{k} + c));")
            L.append(f"    #pragma unroll\n    for (int e = 0; e < {_ELEMS}; ++e) {{")

            def vload_sum(k):
                if kinds[k] == "c":
                    return f"({ct[k]})l{k}[e]"
                return f"bc{k}"
            L.extend(expr_lines(vload_sum, "      "))
            L.append(f"      acc += ({acc_ct}){res};")
            L.append("    }")
            L.append("  }")
        else:
            L.append(f"  for (long long c = c0 + threadIdx.x; c < c1; c += {_BLOCK}) {{")
            L.extend(expr_lines(lambda k: scalar_load(k, "c"), "    "))
            L.append(f"    acc += ({acc_ct}){res};")
            L.append("  }")
        L.append("  // wave64 butterfly, then one value per wave through LDS")
        L.append("  #pragma unroll\n  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);")
        L.append(f"  __shared__ {acc_ct} red[{_BLOCK // 64}];")
        L.append("  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;")
        L.append("  __syncthreads();")
        L.append("  if (threadIdx.x == 0) {")
        L.append(f"    {acc_ct} s = red[0];")
        L.append(f"    for (int w = 1; w < {_BLOCK // 64}; ++w) s += red[w];")
        L.append("    if (p.colblocks == 1) {")
        if _acc_type(prog.dtypes[prog.result])[0] == "double":
            L.append(f"      (({out_ct}*)p.outp)[row] = mmp_convert<{out_ct}, double>(s * p.scale);")
            L.append("    } else {")
            L.append("      ((double*)p.outp)[row * p.colblocks + cb] = s * p.scale;")
        else:
            L.append(f"      (({out_ct}*)p.outp)[row] = mmp_convert<{out_ct}, {acc_ct}>(s);")
            L.append("    } else {")
            L.append(f"      (({acc_ct}*)p.outp)[row * p.colblocks + cb] = s;")
        L.append("    }")
        L.append("  }")
        L.append("}")
    return "\n".join(L) + "\n"


# ------------------------------------------------------------ execution
_kernel_cache: dict = {}
_cache_lock = threading.Lock()


def clear_kernel_caches() -> None:
    """Forget every compiled-kernel handle (by source and by structure)."""
    with _cache_lock:
        _kernel_cache.clear()
        _struct_cache.clear()


def _kernel_for(src: str) -> int:
    k = _kernel_cache.get(src)
    if k is None:
        k = HipBackend().compile(src, "fused_op", RTC_OPTIONS)
        with _cache_lock:
            _kernel_cache[src] = k
    return k


# Kernels by program structure: the generated source is a function of the
# SSA steps (op names and operand indices), the value dtypes, the leaves'
# dtypes and stride classes, the number of outer dimensions, the output
# dtype, the vector flag and the mode -- so a repeated expression skips
# source generation (about 30 us of Python per call) as well as compilation.
_struct_cache: dict = {}


def _kernel_for_program(prog, kinds, nouter, out_dtype, vec, mode) -> int:
    fast = get_config().fast_math
    key = (tuple(prog.steps), tuple(prog.dtypes), tuple(a._dtype for a in prog.arrays),
           tuple(kinds), nouter, out_dtype, vec, mode, fast)
    k = _struct_cache.get(key)
    if k is None:
        k = _kernel_for(generate_source(prog, kinds, nouter, out_dtype, vec, mode, fast))
        with _cache_lock:
            _struct_cache[key] = k
    return k


def _leaf_ptr(node: InputNode) -> int:
    return node._buffer.ptr + node._offset * node._dtype.itemsize


def _scalar_bits(sc: ScalarNode) -> int:
    return sc._bits


def _plan(prog: _Program, shape, keep_last):
    """Collapse the iteration space and classify leaves."""
    strides = [_bcast_strides(a._shape, a._strides, shape) for a in prog.arrays]
    out_st = list(_c_contig_strides(shape))
    cshape, cstr = _collapse(list(shape), strides + [out_st], keep_last=keep_last)
    leaf_str = cstr[:-1]
    if not cshape:
        cshape = [1]
        leaf_str = [[0] for _ in leaf_str]
    cols = cshape[-1]
    outer = cshape[:-1]
    kinds = []
    for st in leaf_str:
        ls = st[-1] if st else 0
        kinds.append("c" if ls == 1 else ("b" if ls == 0 else "s"))
    return cshape, outer, cols, leaf_str, kinds


def _fill_params(prog, P, outer, cols, leaf_str, out_ptr, colblocks, scale):
    nin, nouter = len(prog.arrays), len(outer)
    p = P()
    for k, a in enumerate(prog.arrays):
        p.ptr[k] = _leaf_ptr(a)
        p.lstride[k] = leaf_str[k][-1] if leaf_str[k] else 0
        for d in range(nouter):
            p.ostride[k * nouter + d] = leaf_str[k][d]
    for j, sc in enumerate(prog.scalars):
        p.sbits[j] = _scalar_bits(sc)
    rows = 1
    for d, s in enumerate(outer):
        p.oshape[d] = s
        rows *= s
    p.outp = out_ptr
    p.rows = rows
    p.cols = cols
    p.n = rows * cols
    p.colblocks = colblocks
    p.scale = scale
    return p, rows


def _vec_ok(prog, kinds, leaf_str, outer, cols, out_ptr, out_itemsize, mode):
    """Whether every leaf can be read (and, for 'map', the output written)
    4 elements at a time with aligned vector accesses."""
    if cols % _ELEMS:
        return False
    if mode == "map" and out_ptr % (_ELEMS * out_itemsize):
        return False
    for k, a in enumerate(prog.arrays):
        if kinds[k] == "s":
            return False
        if kinds[k] == "c":
            align = _ELEMS * a._dtype.itemsize
            if _leaf_ptr(a) % align:
                return False
            if any(st % _ELEMS for st in leaf_str[k][:-1]):
                return False
    return True


def _check_grid(nblocks: int) -> None:
    """HIP counts at most 2^32 - 1 work-items per grid dimension; the
    generated kernels also split workgroup ids in 32-bit arithmetic."""
    if nblocks * _BLOCK > 0xFFFFFFFF:
        raise ValueError("fused launch too large")


def run_map(root: FusionNode, out_buffer, out_ptr: int) -> None:
    """Evaluate ``root`` into the C-contiguous output at ``out_ptr``."""
    prog = _Program(root)
    shape = root._shape
    cshape, outer, cols, leaf_str, kinds = _plan(prog, shape, keep_last=False)
    out_dtype = root._dtype
    tile = _map_tile(kinds)
    flat = _flat_kinds(outer, cols, leaf_str, [_leaf_ptr(a) for a in prog.arrays],
                       [a._dtype.itemsize for a in prog.arrays], out_ptr, out_dtype.itemsize, tile)
    if flat is not None:
        kern = _kernel_for_program(prog, flat, 1, out_dtype, True, "flat")
        P = _param_struct(len(prog.arrays), len(prog.scalars), 1)
        p, rows = _fill_params(prog, P, outer, cols, leaf_str, out_ptr, 1, 1.0)
        nblocks = -(-rows * cols // (_FLAT_UNROLL * _BLOCK * _ELEMS))
        if nblocks:
            HipBackend().launch(kern, (nblocks, 1, 1), (_BLOCK, 1, 1), [p])
        return
    vec = _vec_ok(prog, kinds, leaf_str, outer, cols, out_ptr, out_dtype.itemsize, "map")
    kern = _kernel_for_program(prog, kinds, len(outer), out_dtype, vec, "map")
    colblocks = -(-cols // tile)
    P = _param_struct(len(prog.arrays), len(prog.scalars), len(outer))
    p, rows = _fill_params(prog, P, outer, cols, leaf_str, out_ptr, colblocks, 1.0)
    nblocks = rows * colblocks
    if nblocks == 0:
        return
    _check_grid(nblocks)
    HipBackend().launch(kern, (nblocks, 1, 1), (_BLOCK, 1, 1), [p])


def _run_sum_py(root: FusionNode, axis_last: bool, out_dtype, out_ptr: int, mean: bool):
    """Fused reduction epilogue: sum (or mean) of ``root`` over its last axis
    (axis_last=True) or over all elements, written to ``out_ptr``."""
    from ._backend import HipBackend as _HB
    be = _HB()
    prog = _Program(root)
    shape = tuple(root._shape)
    if not axis_last:
        # reduce everything: rows are the collapsed outer dims, then the
        # per-row partials are summed by the precompiled reduction.
        cshape, outer, cols, leaf_str, kinds = _plan(prog, shape, keep_last=False)
    else:
        cshape, outer, cols, leaf_str, kinds = _plan(prog, shape, keep_last=True)
    rows = 1
    for s in outer:
        rows *= s
    count = cols if axis_last else max(1, int(np.prod(shape)) if shape else 1)
    scale = (1.0 / count) if mean else 1.0
    acc_ct, acc_dt = _acc_type(root._dtype)
    # enough blocks to fill 256 CUs; at least 4K elements per block
    want = max(1, _SUM_BLOCKS // max(1, rows))
    colblocks = max(1, min(want, -(-cols // 4096)))
    final_direct = axis_last and colblocks == 1
    P = _param_struct(len(prog.arrays), len(prog.scalars), len(outer))
    vec = _vec_ok(prog, kinds, leaf_str, outer, cols, 0, 0, "sum")
    kern = _kernel_for_program(prog, kinds, len(outer), out_dtype if final_direct else acc_dt,
                               vec, "sum")
    if final_direct:
        p, rows = _fill_params(prog, P, outer, cols, leaf_str, out_ptr, 1, scale)
        _check_grid(rows)
        be.launch(kern, (rows, 1, 1), (_BLOCK, 1, 1), [p])
        return None
    _check_grid(rows * colblocks)
    part = be.create_buffer(rows * colblocks, acc_dt)
    p, rows = _fill_params(prog, P, outer, cols, leaf_str, part.ptr, colblocks, scale)
    be.launch(kern, (rows * colblocks, 1, 1), (_BLOCK, 1, 1), [p])
    outer_n, length = (rows, colblocks) if axis_last else (1, rows * colblocks)
    be.reduce(_abi.REDUCE_SUM, dtype_code(acc_dt), dtype_code(out_dtype), outer_n, length, 1,
              part.ptr, out_ptr)
    return part  # keep alive until the stream passes it (pool is stream-ordered)


# Elements a fused column sum is worth: below, the call's own work in Python
# (about 27 us) outlasts the pass over memory that it saves (100,000 x 45: 20 us
# through a temporary, 28 fused).
COL_SUM_MIN = 1 << 24


def run_col_sum(root: FusionNode, out_dtype, out_ptr: int, scale: float) -> bool:
    """Sum of a 2-D floating ``root`` down its columns, times ``scale``, into
    ``out_ptr`` without materialising it; False where the leaves' strides are
    not a column-sum launch's.  The mean of (x - m)**2 down the columns of a 2,000,000 x 50
    float32 x: 210 us through a temporary, 72 fused."""
    prog = _Program(root)
    _, outer, cols, leaf_str, _ = _plan(prog, root._shape, keep_last=True)
    kinds = _col_kinds(outer, cols, leaf_str)
    if kinds is None:
        return False
    be = HipBackend()
    rows, lg = outer[0], 0
    while lg < 6 and (_ELEMS << lg) < cols:
        lg += 1
    ncb = -(-cols // (_ELEMS << lg))
    # two workgroups a CU, each with some steps of rows to walk
    splits = max(1, min(512 // ncb, rows // ((4 << (6 - lg)) * _COL_UNROLL)))
    _check_grid(ncb * splits)
    kern = _kernel_for_program(prog, kinds, 1, np.dtype(out_dtype), False, "colsum")
    P = _param_struct(len(prog.arrays), len(prog.scalars), 1)
    part = be.create_buffer(splits * cols, np.dtype(np.float64))
    p, _ = _fill_params(prog, P, outer, cols, leaf_str, part.ptr, splits, scale)
    p.n = lg
    be.launch(kern, (ncb * splits, 1, 1), (_BLOCK, 1, 1), [p])
    be.reduce(_abi.REDUCE_SUM, dtype_code(np.dtype(np.float64)), dtype_code(np.dtype(out_dtype)), 1,
              splits, cols, part.ptr, out_ptr)
    return True


def is_precompiled_unary(node) -> bool:
    return (isinstance(node, UnaryOpNode) and _abi.precompiled_unary_ok(node._op_name, node._dtype)
            and isinstance(node._input, InputNode)
            and node._input._dtype == node._dtype
            and node._input._shape == node._shape
            and node._input._strides == _c_contig_strides(node._shape))


def _contig_leaf(n, shape, dtype):
    return (isinstance(n, InputNode) and n._dtype == dtype and n._shape == tuple(shape)
            and n._strides == _c_contig_strides(shape))


def materialize_node(node: FusionNode, out_ptr: int) -> None:
    """Compute ``node`` into the contiguous output at ``out_ptr``."""
    be = HipBackend()
    n = 1
    for s in node._shape:
        n *= s
    if n == 0:
        return
    if (get_config().fast_math and getattr(node, "_op_name", None) in _abi.FAST_MATH_OPS
            and node._dtype in _FAST_DTYPES):
        run_map(node, None, out_ptr)  # the generated kernel carries the fast form
        return
    if is_precompiled_unary(node):
        code = _abi.UNARY_OPS[node._op_name][0]
        be.unary(code, dtype_code(node._dtype), n, _leaf_ptr(node._input), out_ptr)
        return
    if isinstance(node, BinaryOpNode) and node._op_name in _abi.BINARY_OPS:
        a, b = node._lhs, node._rhs
        code = _abi.BINARY_OPS[node._op_name][0]
        dc = dtype_code(node._dtype)
        if _contig_leaf(a, node._shape, node._dtype) and _contig_leaf(b, node._shape, node._dtype):
            be.binary(code, dc, n, _leaf_ptr(a), _leaf_ptr(b), out_ptr)
            return
        if (_contig_leaf(a, node._shape, node._dtype) and isinstance(b, ScalarNode)
                and b._dtype == node._dtype):
            be.binary_scalar(code, dc, n, _leaf_ptr(a), b._value, 1, out_ptr)
            return
        if (isinstance(a, ScalarNode) and a._dtype == node._dtype
                and _contig_leaf(b, node._shape, node._dtype)):
            be.binary_scalar(code, dc, n, _leaf_ptr(b), a._value, 0, out_ptr)
            return
    if isinstance(node, CastNode) and isinstance(node._input, InputNode):
        src = node._input
        be.copy(dtype_code(src._dtype), dtype_code(node._dtype), src._shape, _leaf_ptr(src),
                src._strides, out_ptr)
        return
    run_map(node, None, out_ptr)


def compile_for_native(root, kinds, nouter, out_dtype, vec, mode="map") -> int:
    """Kernel handle of the generated kernel for ``root`` ('map', 'flat' or
    'sum' mode) with the iteration plan the native gate computed (leaf stride
    classes ``kinds``, ``nouter`` outer dims, output dtype, vector flag);
    the DAG is linearised here in the same order as there."""
    prog = _Program(root)
    return _kernel_for_program(prog, list(kinds), nouter, np.dtype(out_dtype), bool(vec), mode)


def _materialize_py(arr) -> None:
    """Evaluate a lazy ndarray in place (reference: _fusion.py:443-486):
    afterwards ``arr._buffer`` holds the result and ``arr._fusion_node`` is
    None.  The native gate (``_native.materialize``, bound to
    ``materialize`` by the package) handles the common cases and calls this
    for the rest."""
    node = arr._fusion_node
    if node is None:
        return
    be = HipBackend()
    buf = be.create_buffer(arr.size, arr._dtype)
    materialize_node(node, buf.ptr)
    arr._buffer = buf
    arr._fusion_node = None
    arr._np_data = None
    arr._offset = 0
    arr._strides = _c_contig_strides(arr._shape)


# Replaced by the native gate's versions when the package is set up.
materialize = _materialize_py
run_sum = _run_sum_py
