"""Generic lowering of graph nodes that no fused kernel pattern covers.

Elementwise and layout nodes are fused into *programs* for the
``nk_ew_program`` kernel.  A program is evaluated over the index space of
the value it produces; layout ops between a producer and its consumer are
affine index maps (broadcast, transpose, slice, reverse, size-1 reshapes),
so they compose into the load strides of the program's inputs instead of
being materialised.  Reductions and dots likewise read their operands
through composed strides.  Everything else (gather/scatter, cumsum,
concatenate, pad, dynamic-update-slice) has a small dedicated step.
"""

from __future__ import annotations

import ctypes
from typing import Dict, List, Optional, Sequence, Tuple

import numpy as np

from nkipy_amd.core import dtypes as dt
from nkipy_amd.core.backend.ir import Value
from nkipy_amd.dispatch.launchers import GemvArgs, Launch, LaunchError, _reduce_planes
from nkipy_amd.dispatch.plan import Slot, Step

# ---------------------------------------------------------------------------
# dtype codes and op codes shared with csrc/kernels/generic.hip
# ---------------------------------------------------------------------------
DT_CODE = {
    dt.float32: 0, dt.float16: 1, dt.bfloat16: 2, dt.float8_e4m3fn: 3, dt.int8: 4,
    dt.int16: 5, dt.int32: 6, dt.int64: 7, dt.uint8: 8, dt.uint16: 9, dt.uint32: 10,
    dt.uint64: 11, dt.bool_: 12, dt.float64: 13,
}

OP_LOAD, OP_CONST, OP_IOTA = 0, 1, 2
UNARY_CODES = {
    "negate": 10, "abs": 11, "exponential": 12, "log": 13, "sqrt": 14, "rsqrt": 15,
    "sine": 16, "cosine": 17, "tan": 18, "atan": 19, "tanh": 20, "ceil": 21, "floor": 22,
    "round_nearest_even": 23, "trunc": 24, "sign": 25, "not": 26, "log_plus_one": 27,
    "exponential_minus_one": 28, "is_finite": 29, "is_nan": 30, "logistic": 31, "log2": 32,
    "convert": 33, "copy": 33,
}
BINARY_CODES = {
    "add": 40, "subtract": 41, "multiply": 42, "divide": 43, "power": 44, "maximum": 45,
    "minimum": 46, "and": 47, "or": 48, "xor": 49, "remainder": 50, "floor_divide": 51,
    "atan2": 52,
}
COMPARE_CODES = {"EQ": 60, "NE": 61, "LT": 62, "LE": 63, "GT": 64, "GE": 65}
OP_SELECT = 70

EW_OPS = set(UNARY_CODES) | set(BINARY_CODES) | {"compare", "select", "iota"}
LAYOUT_OPS = {"broadcast_in_dim", "transpose", "slice", "reverse"}

EW_MAX_RANK = 6
EW_MAX_IN = 8
EW_MAX_INSTR = 40
EW_REGS = 16
RED_MAX_RANK = 6


def dtype_code(d) -> int:
    d = dt.canonical(d)
    if d not in DT_CODE:
        raise LaunchError(f"dtype {dt.name(d)} is not supported by the generic kernels")
    return DT_CODE[d]


def contiguous_strides(shape) -> np.ndarray:
    s = np.ones(len(shape), dtype=np.int64)
    for i in range(len(shape) - 2, -1, -1):
        s[i] = s[i + 1] * shape[i + 1]
    return s


# ---------------------------------------------------------------------------
# ctypes mirrors of the kernel argument structs
# ---------------------------------------------------------------------------
class EwInput(ctypes.Structure):
    _fields_ = [("ptr", ctypes.c_void_p), ("strides", ctypes.c_int64 * EW_MAX_RANK),
                ("dtype", ctypes.c_int32), ("pad", ctypes.c_int32)]


class EwInstr(ctypes.Structure):
    _fields_ = [("op", ctypes.c_int16), ("dst", ctypes.c_int8), ("a", ctypes.c_int8),
                ("b", ctypes.c_int8), ("c", ctypes.c_int8), ("dtype", ctypes.c_int8),
                ("flags", ctypes.c_int8), ("imm", ctypes.c_double)]


class EwArgs(ctypes.Structure):
    _fields_ = [
        ("out", ctypes.c_void_p), ("out_offset", ctypes.c_int64),
        ("out_strides", ctypes.c_int64 * EW_MAX_RANK), ("shape", ctypes.c_int64 * EW_MAX_RANK),
        ("total", ctypes.c_int64), ("rank", ctypes.c_int32), ("n_in", ctypes.c_int32),
        ("n_instr", ctypes.c_int32), ("out_dtype", ctypes.c_int32),
        ("result_reg", ctypes.c_int32), ("pad", ctypes.c_int32), ("nthreads", ctypes.c_int64),
        ("inp", EwInput * EW_MAX_IN), ("prog", EwInstr * EW_MAX_INSTR),
    ]


class EwfInput(ctypes.Structure):
    _fields_ = [("ptr", ctypes.c_void_p), ("strides", ctypes.c_int32 * EW_MAX_RANK),
                ("dtype", ctypes.c_int32), ("mode", ctypes.c_int32)]


class EwfInstr(ctypes.Structure):
    _fields_ = [(n, ctypes.c_uint8) for n in ("op", "dst", "a", "b", "c", "dtype")] + \
        [("pad", ctypes.c_uint8 * 2), ("imm", ctypes.c_float)]


class EwfArgs(ctypes.Structure):
    _fields_ = [
        ("out", ctypes.c_void_p), ("out_strides", ctypes.c_int32 * EW_MAX_RANK),
        ("shape", ctypes.c_uint32 * EW_MAX_RANK), ("total", ctypes.c_uint32), ("step", ctypes.c_uint32),
        ("rank", ctypes.c_int32), ("n_instr", ctypes.c_int32), ("out_dtype", ctypes.c_int32),
        ("out_mode", ctypes.c_int32), ("result_reg", ctypes.c_int32), ("rows4", ctypes.c_int32),
        ("inp", EwfInput * EW_MAX_IN), ("prog", EwfInstr * EW_MAX_INSTR),
    ]


# what nk_ew_f32 evaluates: values of these types, these operations
_EWF_TYPES = (dt.float32, dt.float16, dt.bfloat16, dt.bool_)
_EWF_CODES = {DT_CODE[d] for d in _EWF_TYPES}
_EWF_OPS = {OP_LOAD, OP_CONST, OP_SELECT} | set(COMPARE_CODES.values()) | {
    UNARY_CODES[n] for n in ("negate", "abs", "exponential", "log", "sqrt", "rsqrt", "tanh", "ceil", "floor",
                             "round_nearest_even", "trunc", "sign", "is_finite", "is_nan", "logistic", "copy")} | {
    BINARY_CODES[n] for n in ("add", "subtract", "multiply", "divide", "maximum", "minimum")}
_EWF_NOT = UNARY_CODES["not"]
# evaluated in double: a result of these in fp16 takes nk_ew_f32_f16fn, which
# narrows it in one rounding as the general kernel does
_EWF_FUNCTIONS = {UNARY_CODES[n] for n in ("exponential", "log", "rsqrt", "tanh", "logistic")}
EWF_RAGGED_MIN = 512 * 256  # a round of nk_ew_program: two workgroups per CU


def collapse_dims(shape, strides):
    """(shape, strides) with size-1 dimensions dropped and neighbours merged
    where every operand's strides (a list per operand) allow."""
    dims = [(int(n), [int(st[d]) for st in strides]) for d, n in enumerate(shape) if n != 1]
    out = []
    for n, st in dims:
        if out and all(a == b * n for a, b in zip(out[-1][1], st)):
            out[-1] = (out[-1][0] * n, st)
        else:
            out.append((n, st))
    out = out or [(1, [0] * len(strides))]
    return [n for n, _ in out], [[st[i] for _, st in out] for i in range(len(strides))]


class ReduceArgs(ctypes.Structure):
    _fields_ = [
        ("inp", ctypes.c_void_p), ("out", ctypes.c_void_p),
        ("out_shape", ctypes.c_int64 * RED_MAX_RANK), ("out_strides", ctypes.c_int64 * RED_MAX_RANK),
        ("red_shape", ctypes.c_int64 * RED_MAX_RANK), ("red_strides", ctypes.c_int64 * RED_MAX_RANK),
        ("n_out", ctypes.c_int64), ("n_red", ctypes.c_int64),
        ("out_rank", ctypes.c_int32), ("red_rank", ctypes.c_int32), ("op", ctypes.c_int32),
        ("in_dtype", ctypes.c_int32), ("out_dtype", ctypes.c_int32), ("acc_f32", ctypes.c_int32),
    ]


class DotArgs(ctypes.Structure):
    _fields_ = [
        ("A", ctypes.c_void_p), ("B", ctypes.c_void_p), ("C", ctypes.c_void_p),
        ("batch", ctypes.c_int64), ("M", ctypes.c_int64), ("N", ctypes.c_int64), ("K", ctypes.c_int64),
        ("sab", ctypes.c_int64), ("sam", ctypes.c_int64), ("sak", ctypes.c_int64),
        ("sbb", ctypes.c_int64), ("sbk", ctypes.c_int64), ("sbn", ctypes.c_int64),
        ("a_dtype", ctypes.c_int32), ("b_dtype", ctypes.c_int32), ("c_dtype", ctypes.c_int32),
        ("pad", ctypes.c_int32),
    ]


class GatherArgs(ctypes.Structure):
    _fields_ = [
        ("src", ctypes.c_void_p), ("idx", ctypes.c_void_p), ("out", ctypes.c_void_p),
        ("O", ctypes.c_int64), ("A", ctypes.c_int64), ("I", ctypes.c_int64), ("N", ctypes.c_int64),
        ("nthreads", ctypes.c_int64), ("mode", ctypes.c_int32), ("dtype", ctypes.c_int32),
    ]


class CumsumArgs(ctypes.Structure):
    _fields_ = [
        ("inp", ctypes.c_void_p), ("out", ctypes.c_void_p),
        ("O", ctypes.c_int64), ("A", ctypes.c_int64), ("N", ctypes.c_int64),
        ("in_dtype", ctypes.c_int32), ("out_dtype", ctypes.c_int32),
        ("acc_f32", ctypes.c_int32), ("pad", ctypes.c_int32),
    ]


class Copy16Args(ctypes.Structure):
    _fields_ = [("src", ctypes.c_void_p), ("dst", ctypes.c_void_p),
                ("n16", ctypes.c_int64), ("nthreads", ctypes.c_int64)]


def copy16(src_ptr: int, dst_ptr: int, nbytes: int) -> Launch:
    """Streaming device copy of ``nbytes`` (multiple of 16, 16-byte aligned)."""
    if nbytes % 16 or src_ptr % 16 or dst_ptr % 16:
        raise LaunchError("copy16 needs 16-byte aligned pointers and a multiple of 16 bytes")
    n16 = nbytes // 16
    grid = max(1, min((n16 + 255) // 256, 1 << 20))
    return Launch("generic", "nk_copy16", (grid, 1, 1), (256, 1, 1),
                  Copy16Args(src_ptr, dst_ptr, n16, grid * 256), bytes=2 * nbytes)


def copy_words(src_ptr: int, dst_ptr: int, nbytes: int) -> Launch:
    """Device copy of 16-bit elements at any address (a one-load program)."""
    total = nbytes // 2
    grid = _grid_for(total)
    a = EwArgs()
    a.out, a.total, a.rank, a.n_in, a.n_instr, a.nthreads = dst_ptr, total, 1, 1, 1, grid * 256
    a.shape[0], a.out_strides[0], a.out_dtype = total, 1, dtype_code(dt.uint16)
    a.inp[0].ptr, a.inp[0].strides[0], a.inp[0].dtype = src_ptr, 1, dtype_code(dt.uint16)
    a.prog[0].op, a.prog[0].dtype = OP_LOAD, dtype_code(dt.uint16)
    return Launch("generic", "nk_ew_program", (grid, 1, 1), (256, 1, 1), a, bytes=2 * nbytes)


class DecodeE4m3Args(ctypes.Structure):
    _fields_ = [("src", ctypes.c_void_p), ("dst", ctypes.c_void_p), ("n8", ctypes.c_int64),
                ("nthreads", ctypes.c_int64)]


def decode_e4m3(src_ptr: int, dst_ptr: int, n: int) -> Launch:
    """fp8 E4M3FN codes -> bf16 (``n`` a multiple of 8; 8- / 16-byte aligned)
    with the decode the GEMM kernel stages its fp8 operand through."""
    if n % 8 or src_ptr % 8 or dst_ptr % 16:
        raise LaunchError("decode_e4m3 needs n % 8 == 0, 8-byte aligned codes, 16-byte aligned output")
    n8 = n // 8
    grid = max(1, min((n8 + 255) // 256, 1 << 20))
    return Launch("generic", "nk_decode_e4m3_bf16", (grid, 1, 1), (256, 1, 1),
                  DecodeE4m3Args(src_ptr, dst_ptr, n8, grid * 256), bytes=3 * n)


def _grid_for(total: int, max_blocks: int = 16384) -> int:
    return max(1, min((total + 255) // 256, max_blocks))


# ---------------------------------------------------------------------------
# Affine index maps through layout nodes
# ---------------------------------------------------------------------------
def is_unit_reshape(src_shape, dst_shape) -> bool:
    """True if the reshape only inserts / removes size-1 dimensions."""
    return [s for s in src_shape if s != 1] == [s for s in dst_shape if s != 1]


def map_to_operand(node, A: np.ndarray, b: np.ndarray) -> Tuple[np.ndarray, np.ndarray]:
    """Given the affine map (A, b) from program index to the index of
    ``node.out``, return the map to the index of ``node.inputs[0]``."""
    op = node.op
    src = node.inputs[0]
    if op == "broadcast_in_dim":
        dims = list(node.attrs["broadcast_dimensions"])
        if not dims:
            return np.zeros((0, A.shape[1]), np.int64), np.zeros(0, np.int64)
        return A[dims, :].copy(), b[dims].copy()
    if op == "transpose":
        perm = node.attrs["permutation"]
        A2 = np.zeros((src.ndim, A.shape[1]), np.int64)
        b2 = np.zeros(src.ndim, np.int64)
        for k, p in enumerate(perm):
            A2[p] = A[k]
            b2[p] = b[k]
        return A2, b2
    if op == "slice":
        st = np.asarray(node.attrs["start_indices"], np.int64)
        sd = np.asarray(node.attrs["strides"], np.int64)
        return A * sd[:, None], st + sd * b
    if op == "reverse":
        A2, b2 = A.copy(), b.copy()
        for d in node.attrs["dimensions"]:
            A2[d] = -A[d]
            b2[d] = (src.shape[d] - 1) - b[d]
        return A2, b2
    if op == "reshape":
        out = node.out
        o_dims = [i for i, s in enumerate(out.shape) if s != 1]
        i_dims = [i for i, s in enumerate(src.shape) if s != 1]
        A2 = np.zeros((src.ndim, A.shape[1]), np.int64)
        b2 = np.zeros(src.ndim, np.int64)
        for od, idim in zip(o_dims, i_dims):
            A2[idim] = A[od]
            b2[idim] = b[od]
        return A2, b2
    # elementwise: same index space
    return A, b


def is_affine_layout(node) -> bool:
    if node.op in LAYOUT_OPS:
        return True
    if node.op == "reshape":
        return is_unit_reshape(node.inputs[0].shape, node.out.shape)
    return False


# ---------------------------------------------------------------------------
# Program builder
# ---------------------------------------------------------------------------
class ProgramTooLarge(Exception):
    pass


class Program:
    """Register program over the index space ``shape``."""

    def __init__(self, shape):
        self.shape = tuple(int(s) for s in shape)
        self.instrs: List[tuple] = []  # (op, dst, a, b, c, dtype, flags, imm)
        self.inputs: List[tuple] = []  # (value, strides over program dims, offset)
        self._next_reg = 0
        self._memo: Dict[tuple, int] = {}

    def _reg(self) -> int:
        if self._next_reg >= EW_REGS:
            raise ProgramTooLarge("register file exhausted")
        r = self._next_reg
        self._next_reg += 1
        return r

    def emit(self, op, a=0, b=0, c=0, dtype=dt.float32, flags=0, imm=0.0) -> int:
        if len(self.instrs) >= EW_MAX_INSTR:
            raise ProgramTooLarge("instruction budget exhausted")
        dst = self._reg()
        self.instrs.append((op, dst, a, b, c, dtype_code(dtype), flags, float(imm)))
        return dst

    def load(self, v: Value, strides, offset) -> int:
        key = ("load", v.id, tuple(int(s) for s in strides), int(offset))
        if key in self._memo:
            return self._memo[key]
        if len(self.inputs) >= EW_MAX_IN:
            raise ProgramTooLarge("too many inputs")
        self.inputs.append((v, tuple(int(s) for s in strides), int(offset)))
        r = self.emit(OP_LOAD, dtype=v.dtype, imm=len(self.inputs) - 1)
        self._memo[key] = r
        return r


def scalar_constant(v: Value) -> Optional[float]:
    if v.node is not None and v.node.op == "constant" and v.size == 1:
        payload = v.node.attrs["value"]
        if payload.dtype.fields is not None:  # bf16 / fp8 bit patterns
            return float(dt.to_float32(payload).reshape(-1)[0])
        return float(np.asarray(payload).reshape(-1)[0])
    return None


class ProgramBuilder:
    """Builds the program computing ``root`` with loads of materialised values."""

    def __init__(self, materialized):
        self.materialized = materialized  # callable(Value) -> bool

    def build(self, root: Value, shape=None) -> Program:
        shape = root.shape if shape is None else shape
        if len(shape) > EW_MAX_RANK:
            raise LaunchError(f"elementwise rank {len(shape)} exceeds {EW_MAX_RANK}")
        prog = Program(shape)
        R = len(shape)
        A = np.eye(len(root.shape), R, dtype=np.int64) if len(root.shape) == R else None
        if A is None:
            raise LaunchError("program shape must match the root rank")
        b = np.zeros(len(root.shape), np.int64)
        r = self._emit(prog, root, A, b, top=True)
        prog.result = r
        return prog

    def _emit(self, prog: Program, v: Value, A, b, top=False) -> int:
        key = ("val", v.id, A.tobytes(), b.tobytes())
        if key in prog._memo:
            return prog._memo[key]
        node = v.node
        c = scalar_constant(v)
        if c is not None:
            r = prog.emit(OP_CONST, dtype=v.dtype, imm=c)
        elif (self.materialized(v) and not top) or node is None or node.op == "constant":
            s = contiguous_strides(v.shape)
            strides = s @ A if v.ndim else np.zeros(A.shape[1], np.int64)
            offset = int(s @ b) if v.ndim else 0
            r = prog.load(v, strides, offset)
        elif node.op == "iota":
            d = node.attrs["dimension"]
            # index along dim d is row d of the map: only pure axis maps allowed
            row, off = A[d], b[d]
            nz = np.nonzero(row)[0]
            if len(nz) == 1 and row[nz[0]] == 1 and off == 0:
                r = prog.emit(OP_IOTA, dtype=v.dtype, imm=int(nz[0]))
            elif len(nz) == 0:
                r = prog.emit(OP_CONST, dtype=v.dtype, imm=float(off))
            else:
                raise ProgramTooLarge("iota through a non-trivial index map")
        elif is_affine_layout(node):
            A2, b2 = map_to_operand(node, A, b)
            r = self._emit(prog, node.inputs[0], A2, b2)
        elif node.op == "reshape":
            # a general reshape of a non-materialised value cannot be inlined
            raise ProgramTooLarge("reshape inside an elementwise chain")
        elif node.op in UNARY_CODES:
            x = self._emit(prog, node.inputs[0], A, b)
            flags = 1 if dt.is_int(node.inputs[0].dtype) else 0
            r = prog.emit(UNARY_CODES[node.op], a=x, dtype=v.dtype, flags=flags)
        elif node.op in BINARY_CODES:
            x = self._emit(prog, node.inputs[0], A, b)
            y = self._emit(prog, node.inputs[1], A, b)
            flags = 1 if (dt.is_int(v.dtype) or dt.is_bool(v.dtype)) else 0
            r = prog.emit(BINARY_CODES[node.op], a=x, b=y, dtype=v.dtype, flags=flags)
        elif node.op == "compare":
            x = self._emit(prog, node.inputs[0], A, b)
            y = self._emit(prog, node.inputs[1], A, b)
            r = prog.emit(COMPARE_CODES[node.attrs["comparison_direction"]], a=x, b=y, dtype=dt.bool_)
        elif node.op == "select":
            p = self._emit(prog, node.inputs[0], A, b)
            x = self._emit(prog, node.inputs[1], A, b)
            y = self._emit(prog, node.inputs[2], A, b)
            r = prog.emit(OP_SELECT, a=p, b=x, c=y, dtype=v.dtype)
        else:
            raise ProgramTooLarge(f"op {node.op} is not elementwise")
        prog._memo[key] = r
        return r


class ProgramStep(Step):
    """One launch writing ``shape`` elements of ``out``: a plain copy of a
    contiguous value takes the streaming copy kernel, a program over float
    types ``nk_ew_f32`` (the same bits as) the general ``nk_ew_program``."""

    kind = "elementwise"

    def __init__(self, desc, prog: Program, out: Value, out_dtype=None,
                 out_strides=None, out_offset: int = 0):
        ins = [v for v, _, _ in prog.inputs]
        super().__init__(desc, ins, [out])
        self.prog = prog
        self.out = out
        self.out_dtype = dt.canonical(out_dtype if out_dtype is not None else out.dtype)
        self.out_strides = (contiguous_strides(prog.shape) if out_strides is None
                            else np.asarray(out_strides, np.int64))
        self.out_offset = int(out_offset)

    def launches(self, addr):
        p = self.prog
        a = EwArgs()
        a.out = addr(self.out)
        a.out_offset = self.out_offset
        total = int(np.prod(p.shape)) if p.shape else 1
        rank = len(p.shape)
        for d in range(rank):
            a.shape[d] = p.shape[d]
            a.out_strides[d] = int(self.out_strides[d])
        a.total = total
        a.rank = rank
        a.n_in = len(p.inputs)
        a.n_instr = len(p.instrs)
        a.out_dtype = dtype_code(self.out_dtype)
        a.result_reg = p.result
        grid = _grid_for(total)
        a.nthreads = grid * 256
        for i, (v, strides, off) in enumerate(p.inputs):
            a.inp[i].ptr = addr(v) + off * v.dtype.itemsize
            for d in range(rank):
                a.inp[i].strides[d] = strides[d]
            a.inp[i].dtype = dtype_code(v.dtype)
        for k, (op, dst, x, y, z, dtc, flags, imm) in enumerate(p.instrs):
            I = a.prog[k]
            I.op, I.dst, I.a, I.b, I.c, I.dtype, I.flags, I.imm = op, dst, x, y, z, dtc, flags, imm
        if total == 0:
            return []
        if getattr(p, "flat_copy", False) and self.out_offset == 0 and self.out_dtype == p.inputs[0][0].dtype:
            src = a.inp[0].ptr
            nbytes = total * self.out_dtype.itemsize
            if nbytes % 16 == 0 and src % 16 == 0 and a.out % 16 == 0:
                return [copy16(src, a.out, nbytes)]
        fast = self._float_form(addr, total)
        if fast is not None:
            return [fast]
        return [Launch("generic", "nk_ew_program", (grid, 1, 1), (256, 1, 1), a,
                       bytes=total * self.out_dtype.itemsize)]


    def _float_form(self, addr, total: int) -> Optional[Launch]:
        """The ``nk_ew_f32`` (``_f16fn``) launch, or None where a type, an operation or
        an offset past 2^31 needs the general kernel."""
        p = self.prog
        if total >= 2**31 - 4096 or self.out_dtype not in _EWF_TYPES or any(
                v.dtype not in _EWF_TYPES for v, _, _ in p.inputs):
            return None
        for op, _, _, _, _, dtc, flags, _ in p.instrs:
            if dtc not in _EWF_CODES or flags or not (op in _EWF_OPS or (op == _EWF_NOT and dtc == DT_CODE[dt.bool_])):
                return None
        shape, strides = collapse_dims(p.shape, [self.out_strides] + [s for _, s, _ in p.inputs])
        span = max(sum(abs(st) * (n - 1) for n, st in zip(shape, ss)) for ss in strides)
        if span >= 2**31:
            return None
        # rows that are no multiple of four cost a thread four index
        # decompositions an operand: no gain before the general kernel's one
        # element per thread fills more than one round (us there / here: an
        # added row over 1000 x 33 9.0 / 9.9, four operands 11.0 / 12.0, a
        # transpose of 33 x 2 x 5 x 64 8.4 / 10.0; 4001 x 33 12.5 / 9.9)
        if len(shape) > 1 and shape[-1] % 4 and total <= EWF_RAGGED_MIN:
            return None

        def mode(ptr, st, isz):
            if st[-1] == 0:
                return 0
            whole = st[-1] == 1 and all(x % 4 == 0 for x in st[:-1]) and ptr % (4 * isz) == 0
            return 1 if whole else 2

        a = EwfArgs()
        a.out = addr(self.out) + self.out_offset * self.out_dtype.itemsize
        a.total, a.rank, a.n_instr = total, len(shape), len(p.instrs)
        a.out_dtype, a.result_reg = dtype_code(self.out_dtype), p.result
        a.rows4 = 1 if shape[-1] % 4 == 0 else 0
        a.out_mode = mode(a.out, strides[0], self.out_dtype.itemsize)
        for d, n in enumerate(shape):
            a.shape[d], a.out_strides[d] = n, strides[0][d]
        for i, (v, _, off) in enumerate(p.inputs):
            st = strides[1 + i]
            a.inp[i].ptr = addr(v) + off * v.dtype.itemsize
            for d in range(len(shape)):
                a.inp[i].strides[d] = st[d]
            a.inp[i].dtype, a.inp[i].mode = dtype_code(v.dtype), mode(a.inp[i].ptr, st, v.dtype.itemsize)
        for k, (op, dst, x, y, z, dtc, _, imm) in enumerate(p.instrs):
            I = a.prog[k]
            I.op, I.dst, I.a, I.b, I.c, I.dtype, I.imm = op, dst, x, y, z, dtc, float(np.float32(imm))
        grid = max(1, min(-(-total // 1024), 65536))
        a.step = grid * 1024
        half = any(op in _EWF_FUNCTIONS and dtc == DT_CODE[dt.float16] for op, _, _, _, _, dtc, _, _ in p.instrs)
        symbol = "nk_ew_f32_f16fn" if half else "nk_ew_f32"
        return Launch("generic", symbol, (grid, 1, 1), (256, 1, 1), a, bytes=total * self.out_dtype.itemsize)


def strided_access(v: Value, materialized) -> Tuple[Value, np.ndarray, int]:
    """Follow affine layout ops from ``v`` down to a materialised value.
    Returns (base value, strides over v's index space, element offset)."""
    A = np.eye(v.ndim, dtype=np.int64)
    b = np.zeros(v.ndim, np.int64)
    cur = v
    while not materialized(cur) and cur.node is not None and is_affine_layout(cur.node):
        A, b = map_to_operand(cur.node, A, b)
        cur = cur.node.inputs[0]
    s = contiguous_strides(cur.shape)
    strides = s @ A if cur.ndim else np.zeros(v.ndim, np.int64)
    off = int(s @ b) if cur.ndim else 0
    return cur, strides, off


REDUCE_CODES = {"add": 0, "maximum": 1, "minimum": 2, "multiply": 3, "and": 4, "or": 5}


class ReduceStep(Step):
    kind = "reduce"

    def __init__(self, node, base: Value, strides, offset: int):
        super().__init__(f"{node.op} {node.attrs.get('computation', '')} over "
                         f"{node.attrs.get('dimensions', node.attrs.get('axis'))}", [base], [node.out])
        self.node = node
        self.base = base
        self.strides = np.asarray(strides, np.int64)
        self.offset = offset
        src = node.inputs[0]
        if node.op in ("argmax", "argmin"):
            red = (node.attrs["axis"],)
            self.code = 6 if node.op == "argmax" else 7
        else:
            red = tuple(node.attrs["dimensions"])
            self.code = REDUCE_CODES[node.attrs["computation"]]
        keep = [d for d in range(src.ndim) if d not in red]
        if len(keep) > RED_MAX_RANK or len(red) > RED_MAX_RANK:
            raise LaunchError("reduction rank too large")
        self.out_shape = [src.shape[d] for d in keep]
        self.out_str = [int(self.strides[d]) for d in keep]
        self.red_shape = [src.shape[d] for d in red]
        self.red_str = [int(self.strides[d]) for d in red]
        acc = node.attrs.get("acc_dtype")
        self.acc_f32 = 1 if (acc is not None and dt.canonical(acc) == dt.float32) else 0

    def launches(self, addr):
        a = ReduceArgs()
        a.inp = addr(self.base) + self.offset * self.base.dtype.itemsize
        a.out = addr(self.node.out)
        for i, (s, st) in enumerate(zip(self.out_shape, self.out_str)):
            a.out_shape[i], a.out_strides[i] = s, st
        for i, (s, st) in enumerate(zip(self.red_shape, self.red_str)):
            a.red_shape[i], a.red_strides[i] = s, st
        n_out = int(np.prod(self.out_shape)) if self.out_shape else 1
        n_red = int(np.prod(self.red_shape)) if self.red_shape else 1
        a.n_out, a.n_red = n_out, n_red
        a.out_rank, a.red_rank = len(self.out_shape), len(self.red_shape)
        a.op = self.code
        a.in_dtype = dtype_code(self.base.dtype)
        a.out_dtype = dtype_code(self.node.out.dtype)
        a.acc_f32 = self.acc_f32
        if n_out == 0:
            return []
        if n_out >= 2**31:
            raise LaunchError("too many reduction outputs for one launch")
        return [Launch("generic", "nk_reduce", (n_out, 1, 1), (256, 1, 1), a)]


class DotF32Args(ctypes.Structure):
    _fields_ = [
        ("A", ctypes.c_void_p), ("B", ctypes.c_void_p), ("C", ctypes.c_void_p),
        ("batch", ctypes.c_int64), ("M", ctypes.c_int64), ("N", ctypes.c_int64), ("K", ctypes.c_int64),
        ("sab", ctypes.c_int64), ("sam", ctypes.c_int64), ("sak", ctypes.c_int64),
        ("sbb", ctypes.c_int64), ("sbk", ctypes.c_int64), ("sbn", ctypes.c_int64),
        ("a_dtype", ctypes.c_int32), ("b_dtype", ctypes.c_int32), ("c_dtype", ctypes.c_int32),
        ("a_mode", ctypes.c_int32), ("b_mode", ctypes.c_int32), ("ksplit", ctypes.c_int32),
        ("kc", ctypes.c_int32), ("c_vec", ctypes.c_int32),
        ("a_bytes", ctypes.c_int32), ("b_bytes", ctypes.c_int32),
    ]


_DOT_F32 = {dt.float32: 0, dt.float16: 1, dt.bfloat16: 2}
DOT_TILE = 128  # the larger side of a tile
DOT_TARGET_WGS = 768  # three workgroups per CU
DOT_MIN_RANGE = 128   # k per range


def dot_tile(M: int, N: int, fp32: bool) -> Tuple[int, int]:
    """Tile of :class:`DotStep`'s matrix-core form: 32 x 128 for fp32 pairs of
    up to 32 rows (feed-forwards of 2048 / 6144, us against 64 x 64: 1 row 63 /
    78, 9 rows 66 / 82; from 33 rows on they are no faster even where they pad
    less: 100 rows 133 / 132, 200 rows 236 / 225, 600 rows 569 / 517)."""
    return (32, 128) if fp32 and M <= 32 and N > 64 else (64, 64)


def dot_split(batch: int, M: int, N: int, K: int, tile: Tuple[int, int] = (64, 64)) -> Tuple[int, int]:
    """(ranges, k per range) of :class:`DotStep`'s matrix-core form: K ranges
    when the tiles alone do not give every CU three workgroups (us, one range
    / as many as do: 200 x 1024 x 3072 101 / 24, 200 x 6144 x 1024 45 / 38, 1
    x 2048 x 8192 276 / 24; 1024 x 3072 x 1024, 768 tiles, 59 in one, 66 in
    two), of 128 k at least."""
    tiles = batch * -(-M // tile[0]) * -(-N // tile[1])
    ks = max(1, min(DOT_TARGET_WGS // tiles, K // DOT_MIN_RANGE, 65535 // batch))
    while ks > 1 and 4 * ks * batch * M * N > 1 << 27:
        ks -= 1
    kc = -(-(-(-K // ks)) // 32) * 32 if K else 32
    return max(1, -(-K // kc)), kc


def _dot_mode(ptr: int, esz: int, s_row: int, s_k: int, s_batch: int, rows: int, K: int, batch: int) -> int:
    """Load mode of an operand: four elements at a time along k (1) or along
    its rows / columns (2) when they are contiguous and every such piece is
    whole and aligned, else one (0)."""
    if ptr % (4 * esz) or (batch > 1 and s_batch % 4):
        return 0
    if s_k == 1 and K % 4 == 0 and (s_row % 4 == 0 or rows == 1):
        return 1
    return 2 if s_row == 1 and rows % 4 == 0 and s_k % 4 == 0 else 0


def _dot_span(esz: int, s_row: int, s_k: int, rows: int, K: int) -> int:
    """Bytes from an operand's first element to the end of its last (one
    batch); negative strides, which a buffer resource cannot address, give
    no span."""
    if s_row < 0 or s_k < 0:
        return 1 << 62
    return ((max(rows, 1) - 1) * s_row + (max(K, 1) - 1) * s_k + 1) * esz


def dot_small(batch: int, M: int, N: int, K: int, half: bool, scalar: bool) -> bool:
    """Whether an unsplit product stays on nk_dot's 16 x 16 tiles: where the
    matrix-core tiles are mostly padding, or where the product ends within a
    few steps and nk_dot's shorter prologue wins (``half``: a 16-bit operand,
    ``scalar``: one loaded element by element).  us, nk_dot / nk_dot_f32:
    8192 of 16 x 16 x 16 11.7 / 30.7, 8192 of 17 x 17 x 4 34.5 / 40.4 (but of
    32 x 64 x 16 68.6 / 37.8); bf16 64 x 64 x 64 6.7 / 8.1, 512 of 16 x 200 x 8
    10.7 / 13.8, 512 of 33 x 33 x 17 11.3 / 8.6; fp32 16 of 33 x 33 x 33
    6.4 / 8.1, 128 of 33 x 33 x 33 7.7 / 8.2, 512 of 33 x 33 x 8 8.8 / 8.2,
    64 of 64 x 64 x 64 (vector loads) 8.2 / 6.9."""
    tiles = -(-M // 16) * -(-N // 16)
    steps = batch * tiles * -(-K // 16)
    if tiles == 1 or (tiles <= 4 and max(M, N) <= 64 and K <= 16):
        return True
    return (K <= 256 and steps <= 7168) if half else (scalar and K <= 128 and steps <= 3456)


class DotStep(Step):
    """Fallback batched dot with arbitrary operand strides (fp32 accumulate):
    fp32, fp16 and bf16 operands on the matrix cores (nk_dot_f32), other
    types and small products (:func:`dot_small`) on nk_dot."""

    kind = "dot"

    def __init__(self, node, lhs, rhs, plan=None):
        super().__init__("dot (generic)", [lhs[0], rhs[0]], [node.out])
        self.node = node
        a_v, a_s, a_o = lhs
        b_v, b_s, b_o = rhs
        at = node.attrs
        src_a, src_b = node.inputs
        lb, rb = list(at["lhs_batch"]), list(at["rhs_batch"])
        lc, rc = list(at["lhs_contract"]), list(at["rhs_contract"])
        lf = [i for i in range(src_a.ndim) if i not in lb and i not in lc]
        rf = [i for i in range(src_b.ndim) if i not in rb and i not in rc]
        if len(lc) != 1 or len(rf) > 1 or len(lb) != len(rb):
            raise LaunchError("generic dot supports one contracting dim and a rank<=2 rhs per batch")

        def collapse(dims, shape, strides, what):
            """(size, stride) of dims merged into one; LaunchError if the
            strides do not describe one uniform axis."""
            if not dims:
                return 1, 0
            st = int(strides[dims[-1]])
            expect = st
            for i in reversed(dims):
                if shape[i] != 1 and int(strides[i]) != expect:
                    raise LaunchError(f"generic dot: {what} dims are not collapsible")
                expect *= shape[i]
            return int(np.prod([shape[i] for i in dims])), st

        self.M, self.sam = collapse(lf, src_a.shape, a_s, "lhs free")
        self.batch, self.sab = collapse(lb, src_a.shape, a_s, "lhs batch")
        _, self.sbb = collapse(rb, src_b.shape, b_s, "rhs batch")
        self.sak = int(a_s[lc[0]])
        self.K = src_a.shape[lc[0]]
        self.N = src_b.shape[rf[0]] if rf else 1
        self.sbn = int(b_s[rf[0]]) if rf else 0
        self.sbk = int(b_s[rc[0]])
        self.a_v, self.a_o, self.b_v, self.b_o = a_v, a_o, b_v, b_o
        # (operands are addressed with 32-bit offsets, whole stages past their end)
        span = max(_dot_span(a_v.dtype.itemsize, self.sam, self.sak, self.M + DOT_TILE, self.K + 2 * DOT_TILE),
                   _dot_span(b_v.dtype.itemsize, self.sbn, self.sbk, self.N + DOT_TILE, self.K + 2 * DOT_TILE))
        self.f32 = all(v.dtype in _DOT_F32 for v in (a_v, b_v, node.out)) and span < 2**31
        self.split, self.planes = (1, self.K), None
        self.keep_planes = False  # the consumer adds them (SwigluPlanesStep)
        outputs = self.batch * self.M * self.N
        pair32 = a_v.dtype == dt.float32 and b_v.dtype == dt.float32
        self.tile = dot_tile(self.M, self.N, pair32)
        if self.f32 and outputs > 0:
            ranges = dot_split(self.batch, self.M, self.N, self.K, self.tile)[0] if node.out.dtype != dt.float16 else 1
            scalar = 0 in (_dot_mode(0, 1, self.sam, self.sak, self.sab, self.M, self.K, self.batch),
                           _dot_mode(0, 1, self.sbn, self.sbk, self.sbb, self.N, self.K, self.batch))
            self.f32 = ranges > 1 or not dot_small(self.batch, self.M, self.N, self.K, not pair32, scalar)
        if self.f32 and plan is not None and outputs > 0:
            # (the reduction writes fp32 or bf16)
            ks, kc = dot_split(self.batch, self.M, self.N, self.K, self.tile)
            if ks > 1 and node.out.dtype != dt.float16 and outputs < 2**31:
                self.split = ks, kc
                self.planes = Slot(plan.add_buffer(4 * ks * outputs, "temp", "dot.partials"))

    def _launches_f32(self, addr):
        ks, kc = self.split
        a = DotF32Args()
        a.A = addr(self.a_v) + self.a_o * self.a_v.dtype.itemsize
        a.B = addr(self.b_v) + self.b_o * self.b_v.dtype.itemsize
        out, ctype = addr(self.node.out), self.node.out.dtype
        a.C = addr(self.planes) if ks > 1 else out
        a.batch, a.M, a.N, a.K = self.batch, self.M, self.N, self.K
        a.sab, a.sam, a.sak = self.sab, self.sam, self.sak
        a.sbb, a.sbk, a.sbn = self.sbb, self.sbk, self.sbn
        a.a_dtype, a.b_dtype = _DOT_F32[self.a_v.dtype], _DOT_F32[self.b_v.dtype]
        a.c_dtype = 0 if ks > 1 else _DOT_F32[ctype]
        esa, esb = self.a_v.dtype.itemsize, self.b_v.dtype.itemsize
        a.a_mode = _dot_mode(a.A, esa, self.sam, self.sak, self.sab, self.M, self.K, self.batch)
        a.b_mode = _dot_mode(a.B, esb, self.sbn, self.sbk, self.sbb, self.N, self.K, self.batch)
        a.a_bytes = _dot_span(esa, self.sam, self.sak, self.M, self.K)
        a.b_bytes = _dot_span(esb, self.sbn, self.sbk, self.N, self.K)
        a.ksplit, a.kc = ks, kc if ks > 1 else -(-max(self.K, 1) // 32) * 32
        a.c_vec = 1 if a.c_dtype == 0 and self.N % 4 == 0 and a.C % 16 == 0 else 0
        sym = f"nk_dot_f32_{'f' if esa == 4 else 'h'}{a.a_mode}_{'f' if esb == 4 else 'h'}{a.b_mode}"
        tm, tn = self.tile
        sym += "_wide" if tm == 32 else ""
        ls = [Launch("dotf32", sym, (-(-self.N // tn), -(-self.M // tm), self.batch * ks),
                     (256, 1, 1), a, flops=2 * self.batch * self.M * self.N * self.K)]
        return ls + ([] if self.keep_planes else self.reduction(addr))

    def reduction(self, addr):
        ks, kc = self.split
        if ks == 1:
            return []
        red = GemvArgs(None, None, None, addr(self.node.out), None, None, None, None, addr(self.planes),
                       self.batch * self.M, self.N, self.K, self.K, self.K, self.N, ks, kc, 0, 0)
        return [_reduce_planes(red, self.node.out.dtype, False)]

    def launches(self, addr):
        if self.M * self.N * self.batch == 0:
            return []
        gx, gy = (self.N + 15) // 16, (self.M + 15) // 16
        if gy > 65535 or self.batch > 65535:
            raise LaunchError("generic dot grid too large")
        if self.f32:
            return self._launches_f32(addr)
        a = DotArgs()
        a.A = addr(self.a_v) + self.a_o * self.a_v.dtype.itemsize
        a.B = addr(self.b_v) + self.b_o * self.b_v.dtype.itemsize
        a.C = addr(self.node.out)
        a.batch, a.M, a.N, a.K = self.batch, self.M, self.N, self.K
        a.sab, a.sam, a.sak = self.sab, self.sam, self.sak
        a.sbb, a.sbk, a.sbn = self.sbb, self.sbk, self.sbn
        a.a_dtype = dtype_code(self.a_v.dtype)
        a.b_dtype = dtype_code(self.b_v.dtype)
        a.c_dtype = dtype_code(self.node.out.dtype)
        return [Launch("generic", "nk_dot", (gx, gy, self.batch), (256, 1, 1), a,
                       flops=2 * self.batch * self.M * self.N * self.K)]


class SwigluPlanesArgs(ctypes.Structure):
    _fields_ = [("P", ctypes.c_void_p), ("out", ctypes.c_void_p), ("plane", ctypes.c_int64)] + \
        [(n, ctypes.c_int32) for n in ("rows", "F", "N", "ks", "og", "ou")]


class SwigluPlanesStep(Step):
    """``(g * (1 / (1 + exp(-g)))) * u`` over two column blocks of a fp32
    product that nothing else reads, from the product's partial planes
    (nk_swiglu_planes_f32): one launch for the planes' reduction and the
    program, the same bits."""

    kind = "swiglu"

    def __init__(self, dot: DotStep, prog: ProgramStep, cols: Tuple[int, int]):
        super().__init__("SwiGLU of a product's planes", prog.inputs, prog.outputs)
        self.dot, self.prog, self.cols = dot, prog, cols

    def launches(self, addr):
        d = self.dot
        out, ks = addr(self.prog.out), d.split[0]
        part = addr(d.planes) if ks > 1 else addr(d.node.out)
        if out % 16 or part % 16:
            return d.reduction(addr) + self.prog.launches(addr)
        rows, F = d.batch * d.M, self.prog.prog.shape[-1]
        if rows * F == 0:
            return []
        a = SwigluPlanesArgs(part, out, rows * d.N, rows, F, d.N, ks, *self.cols)
        return [Launch("generic", "nk_swiglu_planes_f32", (-(-rows * F // 256), 1, 1), (64, 1, 1), a,
                       bytes=4 * rows * F * (2 * ks + 1))]


def _swiglu_columns(prog: Program, v: Value) -> Optional[Tuple[int, int]]:
    """(first gate column, first up column) when the program is the SwiGLU of
    two column blocks of ``v``, else None."""
    code = dtype_code(dt.float32)
    regs: Dict[int, tuple] = {}
    exp, neg = UNARY_CODES["exponential"], UNARY_CODES["negate"]
    add, mul, div = (BINARY_CODES[n] for n in ("add", "multiply", "divide"))
    for op, dst, x, y, _, dtc, flags, imm in prog.instrs:
        if dtc != code or flags:
            return None
        if op == OP_LOAD:
            regs[dst] = ("load", int(imm))
        elif op == OP_CONST:
            regs[dst] = ("const", imm)
        elif op in (exp, neg):
            regs[dst] = (op, regs[x])
        elif op in (add, mul, div):
            ab = (regs[x], regs[y])
            regs[dst] = (op,) + (ab if op == div else tuple(sorted(ab, key=repr)))
        else:
            return None
    pair = lambda op, *ab: (op,) + tuple(sorted(ab, key=repr))
    one = ("const", 1.0)
    silu = lambda g: pair(mul, g, (div, one, pair(add, one, (exp, (neg, g)))))
    if len(prog.inputs) != 2:
        return None
    lead = tuple(int(s) for s in contiguous_strides(v.shape))
    offs = []
    for w, strides, off in prog.inputs:
        if w.id != v.id or tuple(strides) != lead or off % 4 or off < 0 or off + prog.shape[-1] > v.shape[-1]:
            return None
        offs.append(off)
    for g, u in ((0, 1), (1, 0)):
        if regs[prog.result] == pair(mul, silu(("load", g)), ("load", u)):
            return offs[g], offs[u]
    return None


def fuse_swiglu_planes(plan):
    """Replace the programs that are a SwiGLU over a fp32 product's planes."""
    buffer = lambda v: plan.slots[v.id].buffer if v.id in plan.slots else None
    for i, st in enumerate(plan.steps):
        if not isinstance(st, ProgramStep) or not st.prog.inputs or st.out.dtype != dt.float32:
            continue
        v = st.prog.inputs[0][0]
        dots = [d for d in plan.steps[:i] if isinstance(d, DotStep) and d.node.out.id == v.id]
        if len(dots) != 1 or v.dtype != dt.float32 or buffer(v) is None:
            continue
        d, p = dots[0], st.prog
        if (plan.buffers[buffer(v)].kind != "temp" or d.N != v.shape[-1] or d.N % 4 or len(p.shape) != v.ndim
                or p.shape[:-1] != tuple(v.shape[:-1]) or p.shape[-1] % 4 or d.batch * d.M * d.N >= 2**31
                or st.out_offset or st.out_dtype != dt.float32
                or tuple(st.out_strides) != tuple(contiguous_strides(p.shape))):
            continue
        others = [w for s in plan.steps if s is not st and s is not d for w in list(s.inputs) + list(s.outputs)]
        if any(buffer(w) == buffer(v) for w in others):
            continue
        cols = _swiglu_columns(p, v)
        if cols is not None:
            d.keep_planes = True
            plan.steps[i] = SwigluPlanesStep(d, st, cols)


def axis_view(shape, axis) -> Tuple[int, int, int]:
    O = int(np.prod(shape[:axis])) if axis else 1
    N = int(np.prod(shape[axis + 1:])) if axis + 1 < len(shape) else 1
    return O, shape[axis], N


class GatherStep(Step):
    """take (0), take_along_axis (1), scatter (2), put_along_axis (3)."""

    kind = "gather"
    MODES = {"take": 0, "take_along_axis": 1, "scatter_along_axis": 2, "put_along_axis": 3}

    def __init__(self, node):
        mode = self.MODES[node.op]
        op = node.inputs
        src = op[0] if mode <= 1 else op[2]
        super().__init__(node.op, [src, op[1]], [node.out])
        self.node, self.mode, self.src, self.idx = node, mode, src, op[1]
        ax = node.attrs["axis"]
        operand = op[0]
        O, A, N = axis_view(operand.shape, ax)
        if mode in (0, 2):
            I = op[1].size
        else:
            I = op[1].shape[ax]
        self.dims = (O, A, I, N)

    def launches(self, addr):
        O, A, I, N = self.dims
        a = GatherArgs()
        a.src = addr(self.src)
        a.idx = addr(self.idx)
        a.out = addr(self.node.out)
        a.O, a.A, a.I, a.N = O, A, I, N
        total = O * I * N
        grid = _grid_for(total)
        a.nthreads = grid * 256
        a.mode = self.mode
        a.dtype = dtype_code(self.node.out.dtype)
        if total == 0:
            return []
        return [Launch("generic", "nk_gather", (grid, 1, 1), (256, 1, 1), a)]


class TopkArgs(ctypes.Structure):
    _fields_ = [("inp", ctypes.c_void_p), ("idx", ctypes.c_void_p), ("rows", ctypes.c_int64),
                ("n", ctypes.c_int64), ("k", ctypes.c_int32), ("largest", ctypes.c_int32),
                ("dtype", ctypes.c_int32), ("pad", ctypes.c_int32)]


class TopkSegArgs(ctypes.Structure):
    _fields_ = [("inp", ctypes.c_void_p), ("keys", ctypes.c_void_p), ("idx", ctypes.c_void_p),
                ("n", ctypes.c_int64), ("nseg", ctypes.c_int32), ("k", ctypes.c_int32),
                ("largest", ctypes.c_int32), ("dtype", ctypes.c_int32)]


TOPK_SEG = 4096        # elements per workgroup of the segment form
TOPK_SEG_MIN = 8192    # row length from which the segment form is taken
TOPK_SEG_MAX_K = 16


class TopkStep(Step):
    """Indices of the k largest (or smallest) elements of each row along the
    last axis, ordered by value, ties by index (nk_topk).  Rows of two
    segments and more of a float type take the segment form, up to 16 picks
    (each costs every workgroup a reduction): 8 rows of 151936 bf16, one
    pick, 5.4 + 4.0 us against 250."""

    kind = "topk"

    def __init__(self, node, plan=None):
        x = node.inputs[0]
        super().__init__("topk", [x], [node.out])
        self.node, self.x = node, x
        self.n = x.shape[-1] if x.ndim else 1
        self.rows = x.size // max(self.n, 1)
        self.nseg, self.keys = -(-self.n // TOPK_SEG), None
        k = int(node.attrs["k"])
        if (plan is not None and TOPK_SEG_MIN <= self.n < 2**32 and 0 < k <= TOPK_SEG_MAX_K and self.rows > 0
                and x.dtype in (dt.float32, dt.float16, dt.bfloat16) and self.rows * self.nseg < 2**31):
            self.keys = Slot(plan.add_buffer(8 * self.rows * self.nseg * k, "temp", "topk.keys"))

    def launches(self, addr):
        at = self.node.attrs
        if self.rows == 0:
            return []
        if self.rows >= 2**31:
            raise LaunchError("topk: too many rows")
        if self.keys is not None:
            k = int(at["k"])
            a = TopkSegArgs(addr(self.x), addr(self.keys), addr(self.node.out), self.n, self.nseg, k,
                            1 if at["largest"] else 0, dtype_code(self.x.dtype))
            return [Launch("generic", "nk_topk_segments", (self.rows * self.nseg, 1, 1), (256, 1, 1), a,
                           bytes=self.rows * self.n * self.x.dtype.itemsize),
                    Launch("generic", "nk_topk_merge", (self.rows, 1, 1), (256, 1, 1), a,
                           bytes=8 * self.rows * self.nseg * k)]
        a = TopkArgs(addr(self.x), addr(self.node.out), self.rows, self.n, int(at["k"]),
                     1 if at["largest"] else 0, dtype_code(self.x.dtype), 0)
        return [Launch("generic", "nk_topk", (self.rows, 1, 1), (256, 1, 1), a,
                       bytes=self.rows * self.n * self.x.dtype.itemsize * int(at["k"]))]


class CumsumStep(Step):
    kind = "cumsum"

    def __init__(self, node):
        super().__init__("cumsum", [node.inputs[0]], [node.out])
        self.node = node

    def launches(self, addr):
        n = self.node
        O, A, N = axis_view(n.inputs[0].shape, n.attrs["axis"])
        a = CumsumArgs()
        a.inp, a.out = addr(n.inputs[0]), addr(n.out)
        a.O, a.A, a.N = O, A, N
        a.in_dtype, a.out_dtype = dtype_code(n.inputs[0].dtype), dtype_code(n.out.dtype)
        acc = n.attrs.get("acc_dtype")
        a.acc_f32 = 1 if acc is not None and dt.canonical(acc) == dt.float32 else 0
        lines = O * N
        if lines == 0 or A == 0:
            return []
        return [Launch("generic", "nk_cumsum", ((lines + 255) // 256, 1, 1), (256, 1, 1), a)]


def flat_copy_program(src: Value) -> Program:
    """Program copying a contiguous value element by element (rank 1)."""
    prog = Program((src.size,))
    r = prog.load(src, (1,), 0)
    prog.result = r
    prog.flat_copy = True
    return prog

