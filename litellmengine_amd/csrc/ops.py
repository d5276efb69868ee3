"""Python face of the HIP kernels: checks operands on the host, then launches
on the current stream.  Tensors are torch tensors on the GPU (torch is the
allocator and the stream owner; the arithmetic is in `*.hip`).  There is no
CPU path: without a GPU or without the compiled libraries these raise.
"""
from __future__ import annotations

import ctypes
import threading
from typing import Optional

import torch

from ..parts.base import Injected, PartialSums, Prenormed, ScaledSum, Written, is_own_function
from . import build
from .record import LaunchRecord
from .tuning import ProductTuning
from .limits import (MAX_DELTA_HEAD_DIM, MAX_GLA_HEAD_DIM, MAX_HEAD_DIM, MAX_SSD_DIM, MAX_SUMMED_NORM_WIDTH,
                     MAX_WKV_HEAD_DIM)

F32, BF16 = 0, 1
_P = ctypes.c_void_p
_I = ctypes.c_int
_L = ctypes.c_int64
_F = ctypes.c_float
_TYPES = {"P": _P, "I": _I, "L": _L, "F": _F}


class KernelError(RuntimeError):
    pass


class _Recording(threading.local):
    to: Optional[LaunchRecord] = None  # the record that this thread's launches go into (record.py)


_recording = _Recording()
_of_kind = {}  # (dtype, device) -> a tensor of no elements: its new_empty() takes the host 0.25 us less than torch.empty() with a type and a device


def _made(shape, dtype, device) -> torch.Tensor:
    kind = _of_kind.get((dtype, device))
    if kind is None:
        kind = torch.empty((0,), dtype=dtype, device=device)
        if type(kind) is torch.Tensor:  # (a tracing mode's own kind would be found long after the mode)
            _of_kind[dtype, device] = kind
    t = kind.new_empty(shape)
    if _recording.to is not None:
        _recording.to.made.append(t)
    return t


def _made_like(x: torch.Tensor) -> torch.Tensor:
    t = torch.empty_like(x)
    if _recording.to is not None:
        _recording.to.made.append(t)
    return t


def dtype_code(dtype: torch.dtype) -> int:
    if dtype == torch.float32:
        return F32
    if dtype == torch.bfloat16:
        return BF16
    raise KernelError(f"kernels take float32 or bfloat16 tensors, not {dtype}")


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def _need(cond: bool, msg: str) -> None:
    if not cond:
        raise KernelError(msg)


def _dev(t: torch.Tensor, name: str, dtype=None) -> None:
    # (on every operand of every launch: the messages are made only when they are needed)
    if not t.is_cuda:
        raise KernelError(f"{name} must live on the GPU")
    if not t.is_contiguous():
        raise KernelError(f"{name} must be contiguous")
    if dtype is not None and t.dtype != dtype:
        raise KernelError(f"{name} must be {dtype}, is {t.dtype}")


def _rows(t: torch.Tensor, name: str, dtype=None) -> None:
    """A matrix whose rows may lie apart (some columns of a wider one): elements of a row are neighbours."""
    if not t.is_cuda:
        raise KernelError(f"{name} must live on the GPU")
    if t.dim() != 2 or (t.shape[1] > 1 and t.stride(1) != 1):
        raise KernelError(f"{name} must be a matrix with contiguous rows")
    if dtype is not None and t.dtype != dtype:
        raise KernelError(f"{name} must be {dtype}, is {t.dtype}")


# the current stream's handle without the Stream object around it (a launch is a few microseconds
# of Python as it is; torch.cuda.current_stream() alone costs as much again)
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


_raw_device = getattr(torch._C, "_cuda_getDevice", None)


def _stream_handle() -> int:
    if _raw_stream is not None and _raw_device is not None:
        return _raw_stream(_raw_device())
    return torch.cuda.current_stream().cuda_stream


def _library_product(x, weight, out):
    torch.mm(x, weight.t(), out=out)


class HipOps:
    """The operations a model part may call.  One instance per process is enough."""

    MAX_HEAD_DIM = MAX_HEAD_DIM

    def __init__(self, tuning: Optional[ProductTuning] = None):
        if not torch.cuda.is_available():
            raise KernelError("litellmengine_amd needs a GPU: its kernels have no CPU form")
        self._fn = {}
        self._forms = {}  # by sizes: the form in which a delta of the residual stream is taken (_form_of_delta) ...
        self._forms_tuning = None  # ... with these numbers
        self._wide = {}  # by sizes: wide_form
        self._rows = {}  # by sizes: rows_tile
        self._gated_f32 = {}  # by sizes: gated_f32_tiles
        self.tuning = tuning or ProductTuning()  # which kernel takes a product (never what it gives, beyond the order of its sums)

    # -- plumbing ---------------------------------------------------------
    def _get(self, lib: str, name: str, argtypes, restype=_I):
        """`argtypes`: ctypes' types, or a letter for each (a text is no list that every launch makes anew)."""
        key = (lib, name)
        fn = self._fn.get(key)
        if fn is None:
            fn = getattr(build.load_library(lib), name)
            fn.argtypes = [_TYPES[t] for t in argtypes] if isinstance(argtypes, str) else argtypes
            fn.restype = restype
            self._fn[key] = fn
        return fn

    def _run(self, lib: str, name: str, argtypes, *args):
        fn = self._fn.get((lib, name)) or self._get(lib, name, argtypes)
        stream = _raw_stream(_raw_device()) if _raw_stream is not None and _raw_device is not None else _stream_handle()
        code = fn(*args, stream)
        if code != 0:
            self._failed(lib, name, code)
        if _recording.to is not None:
            _recording.to.launch(fn, lib, name, args, stream)

    @staticmethod
    def _failed(lib: str, name: str, code: int):
        msg = build.load_library(lib).lle_error_string(code).decode()
        raise KernelError(f"{name} failed to launch: {msg} (hip error {code})")

    # -- the launches of a layer for the layers that are alike (record.py) ------------------
    def may_record(self) -> bool:
        """Whether what this object launches may be launched again for another layer: not where a caller has put a method of
        its own in the place of one, which would not be called then."""
        return (type(self) is HipOps and _recording.to is None and _written.unchanged()
                and all(is_own_function(self, k, v) for k, v in vars(self).items() if callable(v)))

    def record(self) -> LaunchRecord:
        """From here until end_record() this thread's launches are kept."""
        _recording.to = LaunchRecord(_stream_handle())
        return _recording.to

    @staticmethod
    def end_record() -> None:
        _recording.to = None

    def replay(self, replay, operands, addresses) -> None:
        failed = replay.run(operands, addresses)
        if failed is not None:
            self._failed(*failed)

    @staticmethod
    def _library(take, x, weight, result):
        record = _recording.to
        if record is not None:
            record.product(take, x, weight, result)
        return result

    @staticmethod
    def _not_recorded() -> None:
        record = _recording.to
        if record is not None:
            record.whole = False

    # -- embedding -----------------------------------------------------------
    def embedding(self, ids: torch.Tensor, table: torch.Tensor, feedback=None, token_seq=None,
                  seq_slots=None, scale: float = 1.0) -> torch.Tensor:
        """ids int32 [N], table [V, H] -> float32 [N, H] (the residual stream), times `scale`.  With `feedback`
        (int32, indexed by request slot), `token_seq` [N] and `seq_slots`: an id below zero is
        replaced by feedback[seq_slots[token_seq[n]]], the token that argmax(..., scatter=...) left there."""
        _dev(ids, "ids", torch.int32)
        _dev(table, "embedding table")
        _need(ids.dim() == 1 and table.dim() == 2, "embedding wants ids [N] and a table [V, H]")
        N, H = ids.shape[0], table.shape[1]
        if feedback is not None:
            for t, name in ((feedback, "feedback"), (token_seq, "token_seq"), (seq_slots, "seq_slots")):
                _need(t is not None, "feedback, token_seq and seq_slots come together")
                _dev(t, name, torch.int32)
            _need(token_seq.shape == (N,), "token_seq must be [N]")
        out = _made((N, H), dtype=torch.float32, device=table.device)
        self._run("elementwise", "lle_embedding_scaled", "PPPIIIPPPFP",
                  _ptr(ids), _ptr(table), _ptr(out), N, H, dtype_code(table.dtype), _ptr(feedback),
                  _ptr(token_seq) if feedback is not None else None, _ptr(seq_slots) if feedback is not None else None,
                  float(scale))
        return out

    def embedding_rmsnorm(self, ids, table, weight, eps: float, feedback=None, token_seq=None, seq_slots=None):
        """embedding() and the RMSNorm of its rows in one launch: (float32 [N, H] residual stream,
        [N, H] normed rows in the table's type)."""
        _dev(ids, "ids", torch.int32)
        _dev(table, "embedding table")
        _dev(weight, "norm weight")
        _need(ids.dim() == 1 and table.dim() == 2, "embedding wants ids [N] and a table [V, H]")
        N, H = ids.shape[0], table.shape[1]
        _need(weight.shape == (H,), f"norm weight must be [{H}], is {list(weight.shape)}")
        if feedback is not None:
            for t, name in ((feedback, "feedback"), (token_seq, "token_seq"), (seq_slots, "seq_slots")):
                _need(t is not None, "feedback, token_seq and seq_slots come together")
                _dev(t, name, torch.int32)
            _need(token_seq.shape == (N,), "token_seq must be [N]")
        hidden = _made((N, H), dtype=torch.float32, device=table.device)
        out = _made((N, H), dtype=table.dtype, device=table.device)
        self._run("norm", "lle_embedding_rmsnorm", "PPPPIPIIFIPPPP",
                  _ptr(ids), _ptr(table), _ptr(hidden), _ptr(weight), dtype_code(weight.dtype), _ptr(out), N, H,
                  float(eps), dtype_code(table.dtype), _ptr(feedback),
                  _ptr(token_seq) if feedback is not None else None, _ptr(seq_slots) if feedback is not None else None)
        return hidden, out

    def embedding_norm(self, ids, table, scale: float, positions, pos_table, weight, eps: float, next_weight, next_eps: float,
                       out_dtype, feedback=None, token_seq=None, seq_slots=None):
        """The first rows of the residual stream where they are more than the embedding's: float32 [N, H]
        h[n] = RMSNorm(table[ids[n]] * scale + pos_table[positions[n]]) * weight (`pos_table` None: no position vectors;
        `weight` None: without that norm), and RMSNorm(h) * next_weight in `out_dtype` from the same launch (None where
        `next_weight` is None).  The caller has checked ids and positions."""
        _dev(ids, "ids", torch.int32)
        _dev(table, "embedding table")
        _need(ids.dim() == 1 and table.dim() == 2, "embedding wants ids [N] and a table [V, H]")
        N, H = ids.shape[0], table.shape[1]
        if pos_table is not None:
            _dev(pos_table, "position table")
            _dev(positions, "positions", torch.int32)
            _need(pos_table.dim() == 2 and pos_table.shape[1] == H and pos_table.shape[0] > 0, f"the position table must be [P, {H}]")
            _need(positions.shape == (N,), "positions must be [N]")
        for t, name in ((weight, "norm weight"), (next_weight, "next norm weight")):
            if t is not None:
                _dev(t, name)
                _need(t.shape == (H,), f"{name} must be [{H}]")
        if feedback is not None:
            for t, name in ((feedback, "feedback"), (token_seq, "token_seq"), (seq_slots, "seq_slots")):
                _need(t is not None, "feedback, token_seq and seq_slots come together")
                _dev(t, name, torch.int32)
            _need(token_seq.shape == (N,), "token_seq must be [N]")
        hidden = _made((N, H), dtype=torch.float32, device=table.device)
        out = _made((N, H), dtype=out_dtype, device=table.device) if next_weight is not None else None
        code = lambda t: F32 if t is None else dtype_code(t.dtype)
        self._run("norm", "lle_embedding_norm",
                  "PPIFPPPPIIPPIFPPIFPIIIP",
                  _ptr(ids), _ptr(table), dtype_code(table.dtype), float(scale), _ptr(feedback),
                  _ptr(token_seq) if feedback is not None else None, _ptr(seq_slots) if feedback is not None else None,
                  _ptr(pos_table), code(pos_table), pos_table.shape[0] if pos_table is not None else 0,
                  _ptr(positions) if pos_table is not None else None, _ptr(weight), code(weight), float(eps), _ptr(hidden),
                  _ptr(next_weight), code(next_weight), float(next_eps), _ptr(out), N, H, dtype_code(out_dtype))
        return hidden, out

    # -- norms ---------------------------------------------------------------
    def add_rmsnorm(self, hidden, delta, weight, eps: float, out_dtype, rows=None) -> torch.Tensor:
        """hidden float32 [N, H] (+ delta [N, H] of out_dtype, or float32 partial sums
        [slices, N, H], bare or as PartialSums, that are added in slice order) -> norm * weight, out_dtype.
        Without `rows` the sum is written back to `hidden` and every row is normed;
        with `rows` (int32 [R]) only those rows are read and nothing is written back."""
        _dev(hidden, "hidden", torch.float32)
        _dev(weight, "norm weight")
        N, H = hidden.shape
        _need(weight.shape == (H,), f"norm weight must be [{H}], is {list(weight.shape)}")
        if isinstance(delta, PartialSums):
            delta = delta.sums
        sums = delta is not None and delta.dim() == 3  # partial sums of a product taken in slices of K
        if sums:
            _dev(delta, "partial sums", torch.float32)
            _need(delta.shape[1:] == hidden.shape and H % 4 == 0 and H <= MAX_SUMMED_NORM_WIDTH,
                  f"partial sums {list(delta.shape)} do not fit the residual stream {list(hidden.shape)}")
        elif delta is not None:
            _dev(delta, "delta", out_dtype)
            _need(delta.shape == hidden.shape, "delta must have the shape of hidden")
        if rows is not None:
            _dev(rows, "rows", torch.int32)
            R = rows.shape[0]
        else:
            R = N
        out = _made((R, H), dtype=out_dtype, device=hidden.device)
        if sums:
            self._run("norm", "lle_add_rmsnorm_sums", "PPILPPIPIIFIP",
                      _ptr(hidden), _ptr(delta), delta.shape[0], delta.stride(0), _ptr(rows), _ptr(weight),
                      dtype_code(weight.dtype), _ptr(out), R, H, float(eps), dtype_code(out_dtype))
            return out
        self._run("norm", "lle_add_rmsnorm", "PPPPIPIIFIP",
                  _ptr(hidden), _ptr(delta), _ptr(rows), _ptr(weight), dtype_code(weight.dtype), _ptr(out),
                  R, H, float(eps), dtype_code(out_dtype))
        return out

    def rmsnorm(self, x, weight, eps: float, out_dtype=None) -> torch.Tensor:
        """x [R, H] -> x * rsqrt(mean(x^2) + eps) * weight, same type (`out_dtype` bfloat16 for float32 rows: the
        result in bfloat16 from the same launch)."""
        _dev(x, "x")
        _dev(weight, "norm weight")
        R, H = x.shape
        _need(weight.shape == (H,), f"norm weight must be [{H}], is {list(weight.shape)}")
        if out_dtype is not None and out_dtype != x.dtype:
            _need(x.dtype == torch.float32 and out_dtype == torch.bfloat16, "a norm hands float32 rows on as they are or in bfloat16")
            out = _made((R, H), dtype=out_dtype, device=x.device)
            self._run("norm", "lle_rmsnorm_f32_to_bf16", "PPIPIIFP",
                      _ptr(x), _ptr(weight), dtype_code(weight.dtype), _ptr(out), R, H, float(eps))
            return out
        out = _made_like(x)
        self._run("norm", "lle_rmsnorm", "PPIPIIFIP",
                  _ptr(x), _ptr(weight), dtype_code(weight.dtype), _ptr(out), R, H, float(eps), dtype_code(x.dtype))
        return out

    # -- matrix products -------------------------------------------------------
    def can_fold_norm(self, rows: int, width: int, dtype) -> bool:
        """Whether an RMSNorm over `width` of a step of `rows` tokens can be done by the
        products before and after it (the weight-streaming kernel's few-rows forms)."""
        most = 32 if width <= self.tuning.skinny_small_width else self.tuning.skinny_max_rows
        return dtype == torch.bfloat16 and 0 < rows <= most and width % 8 == 0 and not self.force_library_gemm

    def can_fold_norm_f32(self, rows: int, width: int) -> bool:
        """The same for a float32 model: as many rows as the weight-streaming products take (which of two ways a row's norm goes
        follows the width alone, so its bits do not depend on the number of rows among those; and the model folds no norm that only some
        kinds of steps could fold, the final one), where the products after it go by way of LDS."""
        return (0 < rows <= self.tuning.skinny_f32_max_rows and width % 32 == 0 and width >= 512
                and not self.force_library_gemm and not self.force_simt_gemm)

    def norm_sum_parts(self, width: int) -> int:
        """Into how many column ranges the product before a folded norm over `width` splits the
        sums of squares (one per tile of its launch; the kernel library decides the tiles)."""
        return self._get("gemm", "lle_gemm_skinny_resid_parts", "I")(int(width))

    def _linear_folded(self, x, weight, fold, gated: bool, out_dtype=torch.bfloat16):
        """The forms of the weight-streaming product around a folded norm: `x` a Prenormed
        (its row factors are applied to the result), `fold` a NormFold (the result goes
        into the residual stream and comes back as the next Prenormed)."""
        pre = x if isinstance(x, Prenormed) else None
        xin = pre.xw if pre is not None else x
        _dev(xin, "x", torch.bfloat16)
        _dev(weight, "weight", torch.bfloat16)
        M, K = xin.shape
        N = weight.shape[0]
        _need(weight.shape[1] == K, f"weight [{N}, {weight.shape[1]}] does not fit x [{M}, {K}]")
        _need(K % 8 == 0, f"the weight-streaming product needs a multiple of 8 columns, not {K}")
        _need(pre is None or fold is None, "a product takes a Prenormed or makes one, not both")
        if pre is not None:
            _need(self.can_fold_norm(M, K, xin.dtype), f"a norm over {K} cannot be folded for {M} rows")
            _dev(pre.sums, "sums", torch.float32)
            parts = pre.sums.shape[1]
            _need(pre.sums.shape == (16 if M <= 16 else 32, parts) and pre.xw.shape[1] == K,
                  "sums of squares do not fit")
            _need(not gated or N % 2 == 0, "a gated weight has an even number of rows")
            _need(out_dtype == torch.bfloat16 or (out_dtype == torch.float32 and not gated),
                  "the product after a folded norm writes bfloat16, or float32 where it is not gated")
            out = _made((M, N // 2 if gated else N), dtype=out_dtype, device=xin.device)
            self._run("gemm", "lle_gemm_skinny_scaled_bf16", "PPPPIFIIIIIP",
                      _ptr(xin), _ptr(weight), _ptr(out), _ptr(pre.sums), parts, float(pre.eps), M, N, K, int(gated),
                      dtype_code(out_dtype))
            return out
        _dev(fold.hidden, "hidden", torch.float32)
        _dev(fold.weight, "norm weight")
        _need(not gated and fold.hidden.shape == (M, N) and fold.weight.shape == (N,),
              f"residual stream {list(fold.hidden.shape)} does not fit a product [{M}, {N}]")
        _need(self.can_fold_norm(M, N, xin.dtype), f"a norm over {N} cannot be folded for {M} rows")
        xw = _made((M, N), dtype=torch.bfloat16, device=xin.device)
        sums = _made((16 if M <= 16 else 32, self.norm_sum_parts(N)), dtype=torch.float32, device=xin.device)
        self._run("gemm", "lle_gemm_skinny_resid_bf16", "PPPPIPPIIIP",
                  _ptr(xin), _ptr(weight), _ptr(fold.hidden), _ptr(fold.weight), dtype_code(fold.weight.dtype),
                  _ptr(xw), _ptr(sums), M, N, K)
        return Prenormed(xw, sums, fold.eps)

    def _linear_folded_f32(self, x, weight, fold, gated: bool):
        """_linear_folded of float32 operands (up to 64 rows).  A gated product of more rows than its kernel takes, and where two launches
        are faster, is the plain one and silu_mul: the same bits."""
        pre = x if isinstance(x, Prenormed) else None
        xin = pre.xw if pre is not None else x
        _dev(xin, "x", torch.float32)
        _dev(weight, "weight", torch.float32)
        M, K = xin.shape
        N = weight.shape[0]
        _need(weight.shape[1] == K and K % 4 == 0, f"weight [{N}, {weight.shape[1]}] does not fit x [{M}, {K}]")
        _need(pre is None or fold is None, "a product takes a Prenormed or makes one, not both")
        if pre is not None:
            _need(self.can_fold_norm_f32(M, K), f"a norm over {K} cannot be folded for {M} rows")
            _dev(pre.sums, "sums", torch.float32)
            parts = pre.sums.shape[1]
            _need(pre.sums.shape[0] == -(-M // 16) * 16, "sums of squares do not fit")
            _need(not gated or N % 2 == 0, "a gated weight has an even number of rows")
            in_one = gated and self._gated_f32_in_one(M, N, K)
            out = _made((M, N // 2 if in_one else N), dtype=torch.float32, device=xin.device)
            self._run("gemm", "lle_gemm_skinny_scaled_f32", "PPPPIFIIIIP", _ptr(xin), _ptr(weight),
                      _ptr(out), _ptr(pre.sums), parts, float(pre.eps), M, N, K, int(in_one))
            return self.silu_mul(out) if gated and not in_one else out
        _dev(fold.hidden, "hidden", torch.float32)
        _dev(fold.weight, "norm weight")
        _need(not gated and fold.hidden.shape == (M, N) and fold.weight.shape == (N,),
              f"residual stream {list(fold.hidden.shape)} does not fit a product [{M}, {N}]")
        _need(self.can_fold_norm_f32(M, N), f"a norm over {N} cannot be folded for {M} rows")
        xw = _made((M, N), dtype=torch.float32, device=xin.device)
        sums = _made((-(-M // 16) * 16, self.norm_sum_parts(N)), dtype=torch.float32, device=xin.device)
        self._run("gemm", "lle_gemm_skinny_resid_f32", "PPPPIPPIIIP", _ptr(xin), _ptr(weight),
                  _ptr(fold.hidden), _ptr(fold.weight), dtype_code(fold.weight.dtype), _ptr(xw), _ptr(sums), M, N, K)
        return Prenormed(xw, sums, fold.eps)

    def linear(self, x, weight, out_dtype=None, fold=None, sums_ok=False):
        """x [M, K] . weight [N, K]^T -> [M, N].  With `sums_ok` the caller takes the result also as
        PartialSums (float32 [slices, M, N], what add_rmsnorm adds into the residual stream).  float32 operands take a
        32-bit product: few rows the weight-streaming kernel (float32 matrix instruction), more rows a tiled kernel
        (operands split exactly into three bfloat16 parts); the plain-FMA kernel where K is no multiple of 4.  bfloat16 operands: few rows take the
        weight-streaming matrix-core kernel, more rows the library product; both
        accumulate in 32-bit and write either result type.  `x` a Prenormed or `fold`
        a NormFold: see _linear_folded."""
        if fold is not None or isinstance(x, Prenormed):
            if weight.dtype == torch.float32:
                _need(out_dtype in (None, torch.float32), "a float32 product has a float32 result")
                return self._linear_folded_f32(x, weight, fold, gated=False)
            _need(out_dtype in (None, torch.bfloat16) or (fold is None and out_dtype == torch.float32),
                  "a product that makes a folded norm's input writes bfloat16")
            return self._linear_folded(x, weight, fold, gated=False, out_dtype=out_dtype or torch.bfloat16)
        _dev(x, "x")
        _dev(weight, "weight", x.dtype)
        M, K = x.shape
        N = weight.shape[0]
        _need(weight.shape[1] == K, f"weight [{N}, {weight.shape[1]}] does not fit x [{M}, {K}]")
        out_dtype = out_dtype or x.dtype
        if x.dtype == torch.bfloat16:
            if sums_ok and out_dtype == torch.bfloat16:
                form, slices = self._form_of_delta(x.dtype, M, N, K)
                if form == "tiles":
                    return PartialSums(self.linear_tile_sums(x, weight, slices))
                if form == "slices":
                    return PartialSums(self.linear_slices(x, weight, slices))
                if form == "library":
                    # one batched library product over the slices of K, partial sums left in 32-bit
                    def take(x, weight, out=None):
                        xs = x.view(M, slices, K // slices).permute(1, 0, 2)
                        ws = weight.view(N, slices, K // slices).permute(1, 2, 0)
                        return torch.bmm(xs, ws, out_dtype=torch.float32) if out is None else torch.bmm(xs, ws, out_dtype=torch.float32, out=out)

                    return PartialSums(self._library(take, x, weight, take(x, weight)))
            t = self.tuning
            skinny = K % 8 == 0 and not self.force_library_gemm and (
                M <= t.skinny_max_rows
                or (M <= 32 and K <= t.skinny_small_width and N * K <= t.skinny_small_weight)
                # 17 to 32 rows against a weight with many rows for every CU: the streaming kernel with two
                # tiles of X rows in its registers (K a multiple of 1024 up to 4096)
                or (M <= 32 and K % 1024 == 0 and K <= 4096 and N >= t.stream_32_rows_min_share * self.compute_units()))
            if skinny:
                out = _made((M, N), dtype=out_dtype, device=x.device)
                self._run("gemm", "lle_gemm_skinny_bf16", "PPPIIIIP",
                          _ptr(x), _ptr(weight), _ptr(out), M, N, K, dtype_code(out_dtype))
                return out
            tile = self.rows_tile(x, weight, gated=False) if 32 < M <= 128 and out_dtype == torch.bfloat16 else 0
            if tile:
                return self.linear_rows(x, weight, tile)
            # the library product accumulates in 32-bit and can leave the result so
            if out_dtype == torch.bfloat16:
                return self._library(_library_product, x, weight, torch.mm(x, weight.t()))
            self._not_recorded()
            return torch.mm(x, weight.t(), out_dtype=out_dtype)
        _need(out_dtype == torch.float32, "a float32 product has a float32 result")
        # (up to 16 columns are one step of one of the weight-streaming kernel's sixteen wavefronts: nothing to stream, and in
        # the tiles' kernel a row's result does not depend on how many rows there are)
        if M <= self.tuning.skinny_f32_max_rows and K % 4 == 0 and K > 16 and not self.force_library_gemm:
            slices = self._form_of_delta(x.dtype, M, N, K)[1] if sums_ok else 1
            if slices > 1:
                return PartialSums(self.linear_f32_slices(x, weight, slices))
            out = _made((M, N), dtype=out_dtype, device=x.device)
            # few rows: W streamed once, float32 matrix instruction
            self._run("gemm", "lle_gemm_skinny_f32", "PPPIIIP", _ptr(x), _ptr(weight), _ptr(out),
                      M, N, K)
            return out
        if K % 4 == 0 and not self.force_simt_gemm:
            slices = self._form_of_delta(x.dtype, M, N, K)[1] if sums_ok else 1
            out = self.linear_f32_tiles(x, weight, slices)
            return PartialSums(out) if slices > 1 else out[0]
        out = _made((M, N), dtype=out_dtype, device=x.device)
        self._run("gemm", "lle_gemm_nt_simt", "PPPIIILLLIIP",
                  _ptr(x), _ptr(weight), _ptr(out), M, N, K, K, K, N, dtype_code(x.dtype), dtype_code(out_dtype))
        return out

    def _form_of_delta(self, dtype, M: int, N: int, K: int):
        """(form, slices of K) in which a product is taken whose reader adds up partial sums.  The choice is made from the sizes
        alone and kept for the next product of the same sizes: made anew each time it costs the host as much as the launch."""
        if self._forms_tuning is not self.tuning:  # (other numbers choose anew)
            self._forms, self._forms_tuning = {}, self.tuning
        key = (dtype, M, N, K, self.force_library_gemm)
        form = self._forms.get(key)
        if form is None:
            if dtype == torch.float32:
                form = ("f32", self.f32_slices_for(M, N, K))
            else:
                for name, choose in (("tiles", self.tile_slices_for), ("slices", self.slices_for), ("library", self.library_slices_for)):
                    form = (name, choose(M, N, K))
                    if form[1]:
                        break
                else:
                    form = ("whole", 0)
            if len(self._forms) >= 4096:
                self._forms.clear()
            self._forms[key] = form
        return form

    _F32_TILES = "PPPIIILLLIIP"

    def f32_slices_for(self, M: int, N: int, K: int) -> int:
        """In how many slices of K a float32 product is cut whose reader adds up partial sums, so that the CUs have work and no
        workgroup reads more of x than it has to (the kernel library says how many, from N and K: M only decides which
        of the two kernels it is, so beyond those rows, and up to them, a row's sums do not depend on how many rows there are);
        1 for the whole product, and where the reader (add_rmsnorm) takes no partial sums of that width."""
        if N > MAX_SUMMED_NORM_WIDTH or N % 4 != 0:
            return 1
        if M <= self.tuning.skinny_f32_max_rows:
            fn = getattr(build.load_library("gemm_f32"), "lle_gemm_slices_f32_count")
            fn.argtypes, fn.restype = [_I, _I], _I
            return int(fn(N, K))
        fn = getattr(build.load_library("gemm_f32"), "lle_gemm_nt_f32_slices")
        fn.argtypes, fn.restype = [_I, _I], _I
        return int(fn(N, K))

    def linear_f32_slices(self, x, weight, slices: int) -> torch.Tensor:
        """x [M, K] . weight [N, K]^T, float32, up to 64 rows, as partial sums over `slices` parts of K: [slices, M, N], to be
        added up by the reader in slice order."""
        _dev(x, "x", torch.float32)
        _dev(weight, "weight", torch.float32)
        M, K = x.shape
        N = weight.shape[0]
        _need(weight.shape[1] == K and K % 4 == 0 and M <= 64, f"weight [{N}, {weight.shape[1]}] does not fit x [{M}, {K}]")
        out = _made((slices, M, N), dtype=torch.float32, device=x.device)
        self._run("gemm_f32", "lle_gemm_slices_f32", "PPPIIIIP", _ptr(x), _ptr(weight), _ptr(out), M, N, K,
                  slices)
        return out

    def linear_f32_tiles(self, x, weight, slices: int = 1, tiles: int = -1) -> torch.Tensor:
        """x [M, K] . weight [N, K]^T, float32, in tiles: [slices, M, N], the sums over `slices` parts of K (whole steps of
        32 columns) to be added up by the reader.  `tiles`: which tile shape (below zero: the one that takes the least time)."""
        _dev(x, "x", torch.float32)
        _dev(weight, "weight", torch.float32)
        M, K = x.shape
        N = weight.shape[0]
        _need(weight.shape[1] == K and K % 4 == 0, f"weight [{N}, {weight.shape[1]}] does not fit x [{M}, {K}]")
        out = _made((slices, M, N), dtype=torch.float32, device=x.device)
        self._run("gemm_f32", "lle_gemm_nt_f32", self._F32_TILES, _ptr(x), _ptr(weight), _ptr(out), M, N, K, K, K, N, slices,
                  tiles)
        return out

    def gated_f32_tiles(self, x, weight) -> int:
        """In which tiles (0 or 1) a float32 product of gate and up of more rows than stream the weight takes the activation with it, or -1
        where the product and a pass for the activation stay (the same bits): the kernel library says, from the sizes."""
        M, K = x.shape
        if M <= self.tuning.skinny_f32_max_rows or K % 4 != 0 or self.force_library_gemm or self.force_simt_gemm:
            return -1
        key = (M, weight.shape[0], K, self.compute_units())
        tiles = self._gated_f32.get(key)
        if tiles is None:
            fn = getattr(build.load_library("gemm_f32"), "lle_gemm_nt_gated_f32_tiles")
            fn.argtypes, fn.restype = [_I, _I, _I], _I
            tiles = int(fn(*key[:3])) - 1
            if len(self._gated_f32) >= 4096:
                self._gated_f32.clear()
            self._gated_f32[key] = tiles
        return tiles

    def gated_f32(self, x, weight, tiles: int, activation: str, bias=None, limit: float = 0.0) -> torch.Tensor:
        """x [M, K], weight [N, K] (gate rows, then up rows), float32, in those tiles (see gated_f32_tiles) -> [M, N / 2]:
        silu(gate) * up, or ("clamp") what gate_up_clamped says."""
        _dev(x, "x", torch.float32)
        _dev(weight, "weight", torch.float32)
        M, K = x.shape
        N = weight.shape[0]
        _need(weight.shape[1] == K and K % 4 == 0 and N % 2 == 0, f"weight [{N}, {weight.shape[1]}] does not fit x [{M}, {K}]")
        _need(activation in ("silu", "clamp"), f"unknown activation {activation!r}")
        if bias is not None:
            _dev(bias, "bias", torch.float32)
            _need(activation == "clamp" and bias.shape == (N,), "bias must cover the whole weight of a clamped product")
        out = _made((M, N // 2), dtype=torch.float32, device=x.device)
        self._run("gemm_f32", "lle_gemm_nt_gated_f32", "PPPFPIIIIIP", _ptr(x), _ptr(weight), _ptr(bias),
                  float(limit), _ptr(out), M, N, K, ("silu", "clamp").index(activation) + 1, tiles)
        return out

    SLICED_MIN_ROWS, SLICED_MAX_ROWS = 17, 128  # (lle_gemm_mid_slices_max_rows)
    SLICED_UNIT = 1024  # columns of K that a slice is a multiple of (lle_gemm_mid_slices_unit)

    def slices_for(self, M: int, N: int, K: int) -> int:
        """In how many slices of K the product of 17 to 128 rows with a weight [N, K] is taken
        (see linear_slices), or 0 where the library product stays.  Weights with rows enough for
        every CU need no slices.  For the others the slice count is the one that a small model of
        the kernel's time likes best (rounds of N / 64 x slices workgroups over the CUs, each
        taking in its W and X at what a CU takes in, plus the way of the partial sums to the norm
        and back), and it is used where the workgroups fill the CUs in whole rounds (at least
        0.85 of them: o_proj, down_proj of the 8B sizes), or where K is at least twice N and the
        weight is not small: there the library's tiles are too few for the CUs and it does not
        split K (measured at 64 rows: down_proj of the 32B sizes, 5120 x 25600, in 5 slices 76 us
        against the library's 158; of the 14B sizes, 5120 x 17408, in 17 slices 70 against 132)."""
        if not (self.SLICED_MIN_ROWS <= M <= self.SLICED_MAX_ROWS) or N % 64 != 0 or self.force_library_gemm:
            return 0
        if N > MAX_SUMMED_NORM_WIDTH:  # the only reader of the partial sums (add_rmsnorm) takes no wider rows
            return 0
        units, t = self.compute_units(), self.tuning
        groups = N // 64
        if groups > units // 2 or K % self.SLICED_UNIT != 0:  # (rows enough for the library's own tiles)
            return 0
        parts = K // self.SLICED_UNIT
        rows = 32 if M <= 32 else 64 if M <= 64 else 96 if M <= 96 else 128  # the kernel's tiles of X
        best, best_time, best_fill = 0, 0.0, 0.0
        for slices in range(1, min(parts, 32) + 1):
            if parts % slices != 0:
                continue
            rounds = -(-groups * slices // units)
            taken_in = (64 + rows) * (K // slices) * 2  # bytes of W and X through a CU
            seconds = (rounds * (t.sliced_round_seconds + taken_in / t.cu_intake_bytes_per_s)
                       + slices * M * N * 8 / t.partial_sums_bytes_per_s)
            if best == 0 or seconds < best_time:
                best, best_time, best_fill = slices, seconds, groups * slices / (rounds * units)
        if best_fill >= t.sliced_min_fill or (K >= 2 * N and N * K >= t.sliced_long_k_min_weight):
            return best
        return 0

    def tile_slices_for(self, M: int, N: int, K: int) -> int:
        """In how many slices of K the tiled product takes a delta of the residual stream (linear_tile_sums), or 0 where another
        form stays.  It is taken where the whole product has too few tiles for the CUs and neither the sliced kernel of up to
        128 rows nor the library's batched slices have better ones.  Measured with the norm at 17 to 2048 rows of 73
        weights, 512 to 8192 wide, other form -> this one in us:
        * up to 32 rows weights that the sliced kernel does not take (5120 x 8192 31.0 -> 26.9; at most 8 % slower, 3072 x 2048
          at 17 rows 11.3 -> 12.3) and large ones (5120 x 25600 68 -> 56); up to 128 rows also K >= 2 N (4096 x 12288 at 96 rows
          40.4 -> 32.7; 4096 x 4096 gains nothing);
        * beyond, weights of small models (1024 x 2048 at 1000 rows 24.1 -> 17.0); over 512 rows the library's four slices are
          better for long K (1024 x 4096 at 1536 rows 27.9 -> 32.1, not taken; 1024 x 3072 25.6 -> 27.5 there, at 600 and 2048
          18.8 -> 16.6 and 32.6 -> 30.9; 512 x 2048 at 1536 rows 0.77 of it);
        * others with K < 2 N up to 256 rows (4096 x 4096 at 160 rows 33.5 -> 23.4, 5120 x 8192 57.8 -> 38.7), and up to 512 rows
          where 128 x 128 tiles of the whole product leave a third of the CUs without work (4096 x 4096 at 512 rows 37.7 ->
          35.5, 5120 x 8192 78 -> 64; 6144 x 4096 at 400 rows, three quarters, 43.2 -> 49.6, not taken) and K is long enough for
          slices (5120 x 2048 at 512 rows 29.6 -> 32.4, not taken)."""
        if K % 64 != 0 or N % 4 != 0 or N > MAX_SUMMED_NORM_WIDTH or self.force_library_gemm or N * K < 1 << 20:
            return 0
        if M <= 32:
            taken = M > 16 and (N * K >= 1 << 26 or self.slices_for(M, N, K) == 0)
        elif M <= 128:
            taken = K >= 2 * N or self.slices_for(M, N, K) == 0
        elif N <= 1024 and N * K <= 1 << 22:
            taken = M <= 512 or (M <= 2048 and (K <= 3 * N or N * K <= 1 << 20))
        else:
            whole_tiles = -(-M // 128) * -(-N // 128)
            taken = K < 2 * N and (M <= 256 or (M <= 512 and 3 * whole_tiles <= 2 * self.compute_units() and 4 * K >= 3 * N))
        if not taken:
            return 0
        fn = getattr(build.load_library("gemm_tile"), "lle_gemm_tile_sums_slices")
        fn.argtypes, fn.restype = [_I, _I, _I], _I
        return int(fn(M, N, K))

    def linear_tile_sums(self, x, weight, slices: int, tiles: int = -1) -> torch.Tensor:
        """x [M, K] . weight [N, K]^T, bfloat16, as float32 partial sums over `slices` equal parts of K (whole stages of 64
        columns): [slices, M, N], to be added up by the reader in slice order.  `tiles`: which tile shape (below zero: the one
        that takes the least time)."""
        _dev(x, "x", torch.bfloat16)
        _dev(weight, "weight", torch.bfloat16)
        M, K = x.shape
        N = weight.shape[0]
        _need(weight.shape[1] == K and K % 64 == 0, f"weight [{N}, {weight.shape[1]}] does not fit x [{M}, {K}]")
        out = _made((slices, M, N), dtype=torch.float32, device=x.device)
        self._run("gemm_tile", "lle_gemm_tile_sums_bf16", "PPPIIIIIP", _ptr(x), _ptr(weight), _ptr(out),
                  M, N, K, slices, tiles)
        return out

    def library_slices_for(self, M: int, N: int, K: int) -> int:
        """In how many slices of K the LIBRARY takes a product of more than 128 rows whose result is a
        delta of the residual stream, or 0 for the whole product.  The library cuts the result into
        tiles of up to 256 x 256 and does not split K: a weight with few rows and a long K
        (down_proj) leaves CUs without a tile or gets small tiles.  Slices are tiles as well (one
        batched product), up to 4 while the CUs have room for them; the residual add + norm then
        reads float32 partial sums, which costs part of the gain.  Measured at 4096 x 12288 against
        the whole product, both with the norm: 512 rows 90 -> 65 us (4 slices), 1024 rows 126 -> 106
        (4), 2048 rows 214 -> 205 (2), 4096 rows slower (not taken); square weights (o_proj) gain nothing."""
        if M <= self.SLICED_MAX_ROWS or self.force_library_gemm or K < 2 * N:
            return 0
        if N > MAX_SUMMED_NORM_WIDTH or N % 4 != 0:
            return 0
        tiles = -(-M // 256) * -(-N // 256)
        slices = min(self.tuning.library_max_slices, self.compute_units() // tiles)
        while slices > 1 and K % (8 * slices) != 0:
            slices -= 1
        return slices if slices > 1 else 0

    def wide_form(self, x, weight) -> int:
        """In which tiles (one of eleven) the tiled product of many rows takes gate and up (gated_wide), or -1 where the library and a
        pass for the activation stay: from the sizes alone, but for operands that do not begin at 16 bytes, which only the
        library takes."""
        M, K = x.shape
        if M <= 128 or self.force_library_gemm:
            return -1
        key = (M, weight.shape[0], K, self.compute_units())
        form = self._wide.get(key)
        if form is None:
            fn = getattr(build.load_library("gemm_wide"), "lle_gemm_wide_form")
            fn.argtypes, fn.restype = [_I, _I, _I, _I], _I
            form = int(fn(*key)) - 1
            if len(self._wide) >= 4096:
                self._wide.clear()
            self._wide[key] = form
        return form if (x.data_ptr() | weight.data_ptr()) % 16 == 0 else -1

    def rows_tile(self, x, weight, gated: bool) -> int:
        """How many rows of the weight a workgroup takes where a product of 33 to 256 rows is linear_rows' (the kernel library says which
        are, from the sizes), or 0 where it is not; operands that do not begin at 16 bytes are never."""
        M, K = x.shape
        if not 32 < M <= 256 or self.force_library_gemm:
            return 0
        key = (M, weight.shape[0], K, int(gated), self.compute_units())
        tile = self._rows.get(key)
        if tile is None:
            fn = getattr(build.load_library("gemm_rows"), "lle_gemm_rows_tile")
            fn.argtypes, fn.restype = [_I] * 5, _I
            tile = int(fn(*key))
            if len(self._rows) >= 4096:
                self._rows.clear()
            self._rows[key] = tile
        return tile if (x.data_ptr() | weight.data_ptr()) % 16 == 0 else 0

    def linear_rows(self, x, weight, tile: int, activation: Optional[str] = None, bias=None, limit: float = 0.0) -> torch.Tensor:
        """x [M, K], weight [N, K], bfloat16, up to 128 rows (with `activation` 256), `tile` rows of the weight (or gate rows) a workgroup: x weight^T [M, N], or with
        `activation` what gated_wide gives, [M, N / 2]."""
        _dev(x, "x", torch.bfloat16)
        _dev(weight, "weight", torch.bfloat16)
        M, K = x.shape
        N = weight.shape[0]
        _need(weight.shape[1] == K and K % 256 == 0 and M <= (256 if activation else 128), f"weight [{N}, {weight.shape[1]}] does not fit x [{M}, {K}]")
        _need(activation in (None, "silu", "clamp"), f"unknown activation {activation!r}")
        if bias is not None:
            _dev(bias, "bias", torch.bfloat16)
            _need(activation == "clamp" and bias.shape == (N,), "bias must cover the whole weight of a clamped product")
        out = _made((M, N // 2 if activation else N), dtype=torch.bfloat16, device=x.device)
        self._run("gemm_rows", "lle_gemm_rows_bf16", "PPPFPIIIIIP", _ptr(x), _ptr(weight), _ptr(bias),
                  float(limit), _ptr(out), M, N, K, (None, "silu", "clamp").index(activation), tile)
        return out

    def gated_wide(self, x, weight, form: int, activation: str, bias=None, limit: float = 0.0) -> torch.Tensor:
        """x [M, K], weight [N, K] (gate rows, then up rows), bfloat16, in tiles of that form (see wide_form) -> [M, N / 2]:
        silu(gate) * up, or ("clamp") what gate_up_clamped says."""
        _dev(x, "x", torch.bfloat16)
        _dev(weight, "weight", torch.bfloat16)
        M, K = x.shape
        N = weight.shape[0]
        _need(weight.shape[1] == K and K % 64 == 0, f"weight [{N}, {weight.shape[1]}] does not fit x [{M}, {K}]")
        _need(activation in ("silu", "clamp"), f"unknown activation {activation!r}")
        if bias is not None:
            _dev(bias, "bias", torch.bfloat16)
            _need(bias.shape == (N,), "bias must cover the whole weight")
        out = _made((M, N // 2), dtype=torch.bfloat16, device=x.device)
        self._run("gemm_wide", "lle_gemm_wide_bf16", "PPPFPIIIIIP", _ptr(x), _ptr(weight), _ptr(bias),
                  float(limit), _ptr(out), M, N, K, 1 + ("silu", "clamp").index(activation), form)
        return out

    def linear_slices(self, x, weight, slices: int) -> torch.Tensor:
        """x [M, K] . weight [N, K]^T as float32 partial sums over `slices` equal parts of K:
        [slices, M, N], to be added up by the reader in slice order (M <= 128)."""
        _dev(x, "x", torch.bfloat16)
        _dev(weight, "weight", torch.bfloat16)
        M, K = x.shape
        N = weight.shape[0]
        _need(weight.shape[1] == K, f"weight [{N}, {weight.shape[1]}] does not fit x [{M}, {K}]")
        _need(0 < M <= self.SLICED_MAX_ROWS and N % 64 == 0 and slices > 0 and K % (self.SLICED_UNIT * slices) == 0,
              f"no product in {slices} slices for [{M}, {K}] x [{N}, {K}]")
        out = _made((slices, M, N), dtype=torch.float32, device=x.device)
        self._run("gemm", "lle_gemm_mid_slices_bf16", "PPPIIIIP", _ptr(x), _ptr(weight), _ptr(out),
                  M, N, K, slices)
        return out

    # (which of these kernels takes a product is decided by the numbers in self.tuning)
    force_library_gemm = False
    force_simt_gemm = False  # tests flip this to reach the plain-FMA kernel at sizes the matrix instruction takes

    # -- attention ---------------------------------------------------------------
    def rope_table(self, positions, inv_freq) -> torch.Tensor:
        """cos and sin of float(position) * inv_freq for every token: float32 [N, len(inv_freq), 2].
        Made once per step; every head of every layer with this rotation reads it."""
        _dev(positions, "positions", torch.int32)
        _dev(inv_freq, "inv_freq", torch.float32)
        N, half = positions.shape[0], inv_freq.shape[0]
        out = _made((N, half, 2), dtype=torch.float32, device=positions.device)
        self._run("rope_kv", "lle_rope_table", "PPPIIP", _ptr(positions), _ptr(inv_freq), _ptr(out),
                  N, half)
        return out

    def qk_norm_rope_write(self, qkv, slots, q_weight, k_weight, cos_sin, rotary_dim: int, eps: float, kv_layer,
                           num_q_heads: int, num_kv_heads: int, head_dim: int, write_kv: bool = True) -> torch.Tensor:
        """qkv [N, (nq + 2 nkv) d] -> q [N, nq, d] normed and rotated; K (normed, rotated)
        and V go to the pages `kv_layer` [pages, 2, nkv, page_size, d] at `slots` [N].
        `cos_sin` is rope_table()'s [N, rotary_dim / 2, 2] (None when rotary_dim is 0)."""
        _dev(qkv, "qkv")
        _dev(slots, "slots", torch.int32)
        _dev(kv_layer, "kv_layer", qkv.dtype)
        nq, nkv, d = num_q_heads, num_kv_heads, head_dim
        N = qkv.shape[0]
        _need(qkv.shape == (N, (nq + 2 * nkv) * d), "qkv has the wrong width")
        _need(slots.shape == (N,), "slots must be [N]")
        _need(kv_layer.dim() == 5 and kv_layer.shape[1] == 2 and kv_layer.shape[2] == nkv
              and kv_layer.shape[4] == d, "kv_layer must be [pages, 2, nkv, page_size, d]")
        _need(0 <= rotary_dim <= d and rotary_dim % 2 == 0, "rotary_dim must be even and <= head_dim")
        wd = F32
        for w, name in ((q_weight, "q_norm weight"), (k_weight, "k_norm weight")):
            if w is not None:
                _dev(w, name)
                _need(w.shape == (d,), f"{name} must be [{d}]")
                wd = dtype_code(w.dtype)
        if q_weight is not None and k_weight is not None:
            _need(q_weight.dtype == k_weight.dtype, "q_norm and k_norm weights must share a type")
        if rotary_dim > 0:
            _dev(cos_sin, "cos_sin", torch.float32)
            _need(cos_sin.shape == (N, rotary_dim // 2, 2), "cos_sin must be [N, rotary_dim / 2, 2]")
        page_size = kv_layer.shape[3]
        q_out = _made((N, nq, d), dtype=qkv.dtype, device=qkv.device)
        self._run("rope_kv", "lle_qk_norm_rope_write",
                  "PPPPIPIFPPIIIIILIIP",
                  _ptr(qkv), _ptr(slots), _ptr(q_weight), _ptr(k_weight), wd,
                  _ptr(cos_sin) if rotary_dim > 0 else None, rotary_dim, float(eps), _ptr(q_out), _ptr(kv_layer),
                  N, nq, nkv, d, page_size, kv_layer.stride(0), 1 if write_kv else 0, dtype_code(qkv.dtype))
        return q_out

    def paged_attention(self, q, kv_layer, block_table, seq_slots, cu_tokens, kv_lens, token_seq,
                        window: Optional[int], scale: float, min_q_len: int = 0, max_q_len: int = 0,
                        max_kv_len: int = 0, sinks=None, keep_first: int = 0, softcap: Optional[float] = None) -> torch.Tensor:
        """q [N, nq, d] against the pages -> [N, nq * d].  `softcap`: the scores pass through
        softcap * tanh(score / softcap) (None: not).  `keep_first`: beside a window the first so many keys stay
        in sight too.  `sinks` (float32 [nq], or None): every head's
        softmax has one more place, with that score and no value: p_j = exp(s_j) / (exp(sink) + sum exp(s_j)).
        `min_q_len`, `max_q_len`
        and `max_kv_len` are host-side bounds of this batch; they choose the kernels
        and the number of key splits, never the result.  bfloat16 with head_dim a
        multiple of 32 and a page size a multiple of 16 runs on the matrix cores;
        everything else takes the generic kernel."""
        _dev(q, "q")
        _dev(kv_layer, "kv_layer", q.dtype)
        for t, name in ((block_table, "block_table"), (seq_slots, "seq_slots"), (cu_tokens, "cu_tokens"),
                        (kv_lens, "kv_lens"), (token_seq, "token_seq")):
            _dev(t, name, torch.int32)
        N, nq, d = q.shape
        nkv, page_size = kv_layer.shape[2], kv_layer.shape[3]
        _need(kv_layer.shape[4] == d and kv_layer.shape[1] == 2, "kv_layer must be [pages, 2, nkv, page_size, d]")
        _need(nq % nkv == 0, "q heads must be a multiple of kv heads")
        _need(d <= self.MAX_HEAD_DIM, f"head_dim {d} is larger than the attention kernels take ({self.MAX_HEAD_DIM})")
        _need(token_seq.shape == (N,), "token_seq must be [N]")
        S = seq_slots.shape[0]
        _need(cu_tokens.shape == (S + 1,) and kv_lens.shape == (S,), "cu_tokens [S + 1], kv_lens [S]")
        _need(block_table.dim() == 2, "block_table must be [slots, pages]")
        if sinks is not None:
            _dev(sinks, "sinks", torch.float32)
            _need(sinks.shape == (nq,), "sinks must be [nq]")
        out = _made((N, nq * d), dtype=q.dtype, device=q.device)
        win = int(window) if window else 0
        keep = int(keep_first) if win else 0
        _need(keep >= 0, "keep_first must not be negative")
        cap = float(softcap) if softcap else 0.0
        _need(cap >= 0.0, "a cap must be positive")
        both = keep > 0 and cap > 0.0  # (only the generic kernel knows kept keys and capped scores together)
        mfma = (q.dtype == torch.bfloat16 and d % 32 == 0 and page_size % 16 == 0 and max_q_len > 0
                and max_kv_len > 0 and S <= 65535 and not both and not self.force_generic_attention)
        group = nq // nkv
        if (q.dtype == torch.float32 and d % 16 == 0 and page_size % 16 == 0 and max_q_len > 0 and max_kv_len > 0
                and S <= 65535 and not both and not self.force_generic_attention):
            # float32 on the matrix cores (float32 operands, products and sums; many rows of 128: operands in three bfloat16 parts)
            rows = max_q_len * group
            span = min(max_kv_len, win + max_q_len) if win else max_kv_len
            tiles, paired, rounds = self.f32_attention_form(N, nq, nkv, d, keep == 0 and cap == 0.0, max_q_len, span)
            part_steps = self.f32_attention_part_steps(N, S, nq, nkv, d, keep == 0 and cap == 0.0, max_q_len, span)
            if part_steps:
                ns, row_blocks = self.f32_attention_parts(part_steps, rows, group, max_kv_len, span)
                tiles, paired = 3, part_steps
            else:
                row_blocks = 1 if rows <= 16 else -(-rows // (64 * tiles))
                ns = self.f32_attention_splits(S, nkv, row_blocks, max_q_len, max_kv_len, win, rounds)
            ws_o = ws_ml = None
            if ns > 1:
                ws_o = _made((N * nq * ns * d,), dtype=torch.float32, device=q.device)
                ws_ml = _made((N * nq * ns * 2,), dtype=torch.float32, device=q.device)
            self._run("attention", "lle_paged_attention_mfma_f32",
                      "PPPPPPPPPIIIIIILIIIFIIIIPFP",
                      _ptr(q), _ptr(kv_layer), _ptr(block_table), _ptr(seq_slots), _ptr(cu_tokens), _ptr(kv_lens),
                      _ptr(out), _ptr(ws_o), _ptr(ws_ml), N, S, nq, nkv, d, page_size, kv_layer.stride(0),
                      block_table.shape[1], win, keep, float(scale), row_blocks, tiles, paired, ns, _ptr(sinks), cap)
            return out
        if not mfma:
            self._run("attention", "lle_paged_attention_generic",
                      "PPPPPPPPIIIIILIIIFIPFP",
                      _ptr(q), _ptr(kv_layer), _ptr(block_table), _ptr(seq_slots), _ptr(cu_tokens), _ptr(kv_lens),
                      _ptr(token_seq), _ptr(out), N, nq, nkv, d, page_size, kv_layer.stride(0), block_table.shape[1],
                      win, keep, float(scale), dtype_code(q.dtype), _ptr(sinks), cap)
            return out
        min_q_len = min_q_len or 1
        run_decode = min_q_len * group <= 16
        run_prefill = max_q_len * group > 16
        ns_decode = self.decode_splits(S, nkv, max_kv_len, win) if run_decode else 1
        ns_prefill = self.prefill_splits(S, nkv, group, d, max_q_len, max_kv_len, win) if run_prefill else 1
        row_tiles = (self.prefill_form(S, nkv, group, d, max_q_len, max_kv_len, win, ns_prefill, q.device)
                     if run_prefill else 0)
        ns = max(ns_decode, ns_prefill)
        ws_o = ws_ml = None
        if ns > 1:
            ws_o = _made((N * nq * ns * d,), dtype=torch.float32, device=q.device)
            ws_ml = _made((N * nq * ns * 2,), dtype=torch.float32, device=q.device)
        self._run("attention", "lle_paged_attention_mfma",
                  "PPPPPPPPPPIIIIIILIIFIIIIIIPIFP",
                  _ptr(q), _ptr(kv_layer), _ptr(block_table), _ptr(seq_slots), _ptr(cu_tokens), _ptr(kv_lens),
                  _ptr(token_seq), _ptr(out), _ptr(ws_o), _ptr(ws_ml), N, S, nq, nkv, d, page_size,
                  kv_layer.stride(0), block_table.shape[1], win, float(scale), int(run_decode), ns_decode,
                  int(run_prefill), ns_prefill, max_q_len, row_tiles, _ptr(sinks), keep, cap)
        return out

    def can_fuse_rope_attention(self, dtype, head_dim: int, rotary_dim: int, page_size: int, group: int,
                                max_q_len: int, max_kv_len: int, num_seqs: int, kv_heads: int = 0) -> bool:
        """Whether qk_norm_rope_attention takes this step: bfloat16, a rotation over the whole head
        of a multiple of 64 elements, and only requests of at most 16 / group tokens (decode steps); float32: one token and few
        keys a request, heads of 64 or 128."""
        if dtype == torch.float32:
            # past 176 keys a wavefront has two steps: then only where a workgroup a request and kv head reach as many CUs as the key
            # splits of the two launches do (256 keys, 8 kv heads: 8 requests 11.4 us in two launches and 12.5 in one, 12 14.0 and
            # 12.5, 16 16.4 and 12.9; 140 keys, 8 requests: 12.9 and 9.3)
            workgroups, units = num_seqs * kv_heads, self.compute_units()
            if max_kv_len > 176 and workgroups < 96:
                return False
            # one workgroup fits a CU: two rounds of them, or nearly three (8 kv heads, 97 / 256 keys: 64 requests 19.6 / 29.6 us in
            # two launches and 17.5 / 28.5 in one, 80 24.4 / 36.5 and 23.0 / 37.8, 96 27.2 / 43.2 and 24.4 / 40.4, 128 30.7 / 50.5
            # and 31.3 / 53.7, 256 52 / 118 and 58 / 130)
            if not (workgroups <= 2 * units or 2.75 * units <= workgroups <= 3 * units):
                return False
            return (head_dim in (64, 128) and rotary_dim == head_dim and page_size % 16 == 0 and max_q_len == 1 and group <= 16
                    and 0 < max_kv_len <= self._get("attention", "lle_short_decode_max_keys_f32", [])()
                    and 48 * group * head_dim + 1536 <= 65536 and num_seqs <= 65535 and not self.force_generic_attention
                    and not self.force_separate_rope)
        return (dtype == torch.bfloat16 and head_dim % 64 == 0 and head_dim <= self.MAX_HEAD_DIM
                and rotary_dim == head_dim and page_size % 16 == 0 and 0 < max_q_len and max_q_len * group <= 16
                and max_kv_len > 0 and num_seqs <= 65535 and not self.force_generic_attention
                and not self.force_separate_rope)

    def qk_norm_rope_attention(self, qkv, slots, q_weight, k_weight, cos_sin, eps: float, kv_layer, nq: int,
                               nkv: int, d: int, write_kv: bool, block_table, seq_slots, cu_tokens, kv_lens,
                               token_seq, window: Optional[int], scale: float, max_kv_len: int, order=None) -> torch.Tensor:
        """qk_norm_rope_write and paged_attention of a decode step in one launch (see
        can_fuse_rope_attention): the workgroup whose keys include a new token's position writes
        its K and V, every workgroup norms and rotates the q rows it multiplies.  `order` (int32 [S], or None):
        the requests in the order in which they are started, see decode_order.  `max_kv_len`: a bound on kv_lens; it chooses the
        kernel and its key splits, never the result (a request longer than it says may lose keys).  `token_seq` None: every
        request has one token; with few keys then, and always in float32, it is the launch of a wavefront for every few keys."""
        f32 = qkv.dtype == torch.float32
        _dev(qkv, "qkv", torch.float32 if f32 else torch.bfloat16)
        _dev(kv_layer, "kv_layer", qkv.dtype)
        _dev(cos_sin, "cos_sin", torch.float32)
        for t, name in ((slots, "slots"), (block_table, "block_table"), (seq_slots, "seq_slots"),
                        (cu_tokens, "cu_tokens"), (kv_lens, "kv_lens")):
            _dev(t, name, torch.int32)
        if token_seq is not None:
            _dev(token_seq, "token_seq", torch.int32)
        N = qkv.shape[0]
        page_size = kv_layer.shape[3]
        _need(qkv.shape[1] == (nq + 2 * nkv) * d, "qkv must be [N, (nq + 2 nkv) * d]")
        _need(tuple(kv_layer.shape[1:]) == (2, nkv, page_size, d), "kv_layer must be [pages, 2, nkv, page_size, d]")
        _need(slots.shape == (N,) and (token_seq is None or token_seq.shape == (N,)), "slots and token_seq must be [N]")
        _need(cos_sin.shape == (N, d // 2, 2), f"cos_sin must be [{N}, {d // 2}, 2]")
        _need((q_weight is None) == (k_weight is None), "q and k norm weights come together")
        wcode = 0
        if q_weight is not None:
            _dev(q_weight, "q_weight")
            _dev(k_weight, "k_weight", q_weight.dtype)
            _need(q_weight.shape == (d,) and k_weight.shape == (d,), f"q/k norm weights must be [{d}]")
            wcode = dtype_code(q_weight.dtype)
        S = seq_slots.shape[0]
        _need(cu_tokens.shape == (S + 1,) and kv_lens.shape == (S,), "cu_tokens [S + 1], kv_lens [S]")
        _need(token_seq is not None or N == S, "without token_seq every request has one token")
        _need(nq % nkv == 0 and d % 64 == 0 and page_size % 16 == 0 and S <= 65535,
              "the fused decode attention does not take these sizes")
        if order is not None:
            _dev(order, "order", torch.int32)
            _need(order.shape == (S,), "order must be [S]")
        win = int(window) if window else 0
        if f32:
            _need(token_seq is None and order is None and d in (64, 128), "in float32 every request has one token and heads are of 64 or 128")
            out = _made((N, nq * d), dtype=torch.float32, device=qkv.device)
            self._run("attention", "lle_qk_norm_rope_attention_decode_f32",
                      "PPPPIPFIPPPPPPIIIIILIIFIP",
                      _ptr(qkv), _ptr(slots), _ptr(q_weight), _ptr(k_weight), wcode, _ptr(cos_sin), float(eps), int(bool(write_kv)),
                      _ptr(kv_layer), _ptr(block_table), _ptr(seq_slots), _ptr(cu_tokens), _ptr(kv_lens), _ptr(out), S, nq, nkv, d,
                      page_size, kv_layer.stride(0), block_table.shape[1], win, float(scale), int(max_kv_len))
            return out
        ns = self.decode_splits(S, nkv, max_kv_len, win)
        out = _made((N, nq * d), dtype=torch.bfloat16, device=qkv.device)
        ws_o = ws_ml = None
        if ns > 1:
            ws_o = _made((N * nq * ns * d,), dtype=torch.float32, device=qkv.device)
            ws_ml = _made((N * nq * ns * 2,), dtype=torch.float32, device=qkv.device)
        self._run("attention", "lle_qk_norm_rope_attention_decode",
                  "PPPPIPFIPPPPPPPPPIIIIIILIIFIPIP",
                  _ptr(qkv), _ptr(slots), _ptr(q_weight), _ptr(k_weight), wcode, _ptr(cos_sin), float(eps),
                  int(bool(write_kv)), _ptr(kv_layer), _ptr(block_table), _ptr(seq_slots), _ptr(cu_tokens),
                  _ptr(kv_lens), _ptr(token_seq), _ptr(out), _ptr(ws_o), _ptr(ws_ml), N, S, nq, nkv, d, page_size,
                  kv_layer.stride(0), block_table.shape[1], win, float(scale), ns, _ptr(order), int(max_kv_len))
        return out

    def can_fuse_pair_rope_attention(self, u, dim: int, vdim: int, rot: int, kv_layer, num_q_heads: int, max_q_len: int, max_kv_len: int,
                                     num_seqs: int) -> bool:
        """Whether pair_rope_attention takes this step: bfloat16, one token a request and few keys, heads of 64 or 128 of q, k, v
        and cache alike."""
        D, nkv, page_size = kv_layer.shape[4], kv_layer.shape[2], kv_layer.shape[3]
        return (u.dtype == torch.bfloat16 and max_q_len == 1 and u.shape[0] == num_seqs and 0 < max_kv_len <= self.short_decode_max_keys()
                and dim == vdim == D and D in (64, 128) and rot % 8 == 0 and u.shape[1] % 8 == 0 and u.data_ptr() % 16 == 0
                and page_size % 16 == 0 and num_q_heads // nkv * D * 36 + 1152 <= 65536 and num_q_heads // nkv <= 16 and num_seqs <= 65535
                and not self.force_generic_attention and not self.force_separate_rope)

    def short_decode_max_keys(self) -> int:
        return self._get("attention", "lle_short_decode_max_keys", [])()

    def pair_rope_attention(self, u, slots, cos_sin, kv_layer, nq: int, nkv: int, d: int, write_kv: bool, block_table, seq_slots, cu_tokens,
                            kv_lens, window: Optional[int], scale: float, max_kv_len: int, softcap: Optional[float] = None) -> torch.Tensor:
        """pair_rope_write (without biases and value rotation) and paged_attention of a decode step in one launch, see
        can_fuse_pair_rope_attention: u [S, cols] holds q, k, v and columns that are left alone -> [S, nq * d]."""
        _dev(u, "u", torch.bfloat16)
        _dev(kv_layer, "kv_layer", torch.bfloat16)
        for t, name in ((slots, "slots"), (block_table, "block_table"), (seq_slots, "seq_slots"), (cu_tokens, "cu_tokens"),
                        (kv_lens, "kv_lens")):
            _dev(t, name, torch.int32)
        S, cols = u.shape
        page_size = kv_layer.shape[3]
        _need(cols >= (nq + 2 * nkv) * d, "u has too few columns")
        _need(tuple(kv_layer.shape[1:]) == (2, nkv, page_size, d), "kv_layer must be [pages, 2, nkv, page_size, d]")
        _need(slots.shape == (S,) and seq_slots.shape == (S,) and cu_tokens.shape == (S + 1,) and kv_lens.shape == (S,),
              "slots, seq_slots, kv_lens [S], cu_tokens [S + 1]")
        _need(block_table.dim() == 2, "block_table must be [slots, pages]")
        rot = 0
        if cos_sin is not None:
            _dev(cos_sin, "cos_sin", torch.float32)
            rot = 2 * cos_sin.shape[1]
            _need(cos_sin.shape == (S, rot // 2, 2) and rot <= d, "cos_sin must be [S, pairs, 2]")
        out = _made((S, nq * d), dtype=torch.bfloat16, device=u.device)
        self._run("attention", "lle_pair_rope_attention_decode",
                  "PIPPIIPPPPPPIIIIILIIFFIP",
                  _ptr(u), cols, _ptr(slots), _ptr(cos_sin), rot, int(bool(write_kv)), _ptr(kv_layer), _ptr(block_table), _ptr(seq_slots),
                  _ptr(cu_tokens), _ptr(kv_lens), _ptr(out), S, nq, nkv, d, page_size, kv_layer.stride(0), block_table.shape[1],
                  int(window) if window else 0, float(scale), float(softcap) if softcap else 0.0, int(max_kv_len))
        return out

    # Keys that a workgroup of the decode kernel asks for at its start (two steps of 32 for each of four wavefronts): up to so many
    # the longest request takes about as long as the shortest and an order is only one more thing to wait for.  (64 requests,
    # 8 key heads, as they come / longest first: of 64 to 256 keys 19.0 / 19.5 us, of 96 to 384 23.9 / 23.0, of 256 to 1024
    # 41.4 / 37.5; 96 of 2 key heads alike.)
    DECODE_KEYS_AT_ONCE = 256

    def decode_order(self, kv_lens, num_kv_heads: int):
        """The requests of a decode step by falling length (int32 [S], on the device), for qk_norm_rope_attention; None where its
        workgroups, one for every request and key head, all start at once or there are over 1024 requests.  (A CU holds one
        of them.  64 requests of 1000 to 4096 keys, 8 key heads: 130 us as they come, shortest first; 112 longest first.)"""
        _dev(kv_lens, "kv_lens", torch.int32)
        S = kv_lens.shape[0]
        if S > 1024 or S * num_kv_heads <= self.compute_units():
            return None
        order = _made((S,), dtype=torch.int32, device=kv_lens.device)
        self._run("attention", "lle_decode_order", "PPIP", _ptr(kv_lens), _ptr(order), S)
        return order

    force_generic_attention = False  # tests flip this to compare the two families of kernels
    force_prefill_form = 0           # tests set 1, 2 or 3 to reach every shape of the prompt-portion workgroups
    force_separate_rope = False      # tests flip this to compare the fused decode step with its two halves
    # measured on MI355X: about one workgroup per CU and at least 8 32-key steps (two per
    # wavefront) per split are best; more splits cost more in partial results than they gain
    DECODE_MIN_STEPS_PER_SPLIT = 8
    DECODE_MIN_STEPS_TO_SPLIT = 32

    PREFILL_MIN_STEPS_PER_SPLIT = 8

    def prefill_splits(self, num_seqs: int, num_kv_heads: int, group: int, head_dim: int, max_q_len: int,
                       max_kv_len: int, window: int) -> int:
        """Key splits of the prompt-portion kernel: 1 unless the portions are short and come after a
        long past, when their row blocks alone leave most of the chip idle.  Only the keys that
        every row sees count (the past; a prompt from an empty cache is never split: measured
        twice as slow at 512 tokens).  A split keeps at least 8 steps of 32 keys while the row
        blocks fill less than half the CUs and 32 otherwise, the splits fill the CUs once, and
        twice where every split still keeps 32 steps, at least two row blocks share the keys of a
        head and the row blocks alone fill at most half the CUs (measured: 128 tokens after 1 k keys 26 -> 20 us with 4 splits, 512 tokens after 16 k
        keys 289 -> 149 us with 4, 512 tokens after 1 k keys best unsplit; row blocks that fill the
        CUs by themselves are never split: 2048 tokens after 2048 keys 115 us unsplit, 151 in two;
        four requests of 32 tokens after 16 k keys 57 us in 8 splits, one workgroup a CU, 70 in 16)."""
        units = self.compute_units()
        rows_per_block = 128 if head_dim <= 128 else 64
        blocks = ((max_q_len * group + rows_per_block - 1) // rows_per_block) * num_kv_heads * max(1, num_seqs)
        past = max_kv_len - max_q_len
        if window:
            past = min(past, window)
        steps = max(0, past) // 32
        by_work = max(1, steps // (self.PREFILL_MIN_STEPS_PER_SPLIT if 2 * blocks < units else 32))
        by_fill = max(1, units // blocks)
        splits = min(by_work, by_fill)
        shared_keys = max_q_len * group >= 2 * rows_per_block  # else the keys' way from memory bounds the launch
        if splits == by_fill and 2 * blocks <= units and shared_keys and steps // (2 * splits) >= 32:
            splits *= 2
        return int(min(splits, 64))

    _compute_units: dict = {}

    def compute_units(self, device=None) -> int:
        """CUs of `device` (the current one if not given), asked once per device."""
        key = device.index if device is not None and device.index is not None else torch.cuda.current_device()
        if key not in self._compute_units:
            self._compute_units[key] = torch.cuda.get_device_properties(key).multi_processor_count
        return self._compute_units[key]

    def prefill_form(self, num_seqs: int, num_kv_heads: int, group: int, head_dim: int, max_q_len: int,
                     max_kv_len: int, window: int, nsplit: int, device) -> int:
        """The shape of the prompt-portion kernel's workgroups:
          1: four wavefronts of one 16-row tile each (64 rows a workgroup),
          2: four wavefronts of two tiles each (128 rows; every operand read from LDS serves both tiles),
          3: eight wavefronts of one tile each (128 rows; four wavefronts a SIMD; heads of 128 only).
        The low form when its workgroups all fit the chip at once (a short portion; at heads of 128
        at most one workgroup a CU, or one prompt from an empty cache); else the tall ones, which share a pass over the keys between more
        rows: form 3 at heads of 128, form 2 below.  Measured on MI355X at heads of 128 (forms 1 / 2 / 3): 2048 tokens from an empty cache
        60 / 65 / 57 us, 2048 tokens after 2048 keys 148 / 128 / 118 us, 49 tokens after 2048 keys
        17 / 21 / 19 us."""
        if head_dim > 128:
            return 1
        if self.force_prefill_form:
            return self.force_prefill_form if head_dim == 128 or self.force_prefill_form < 3 else 2
        resident = 2 * self.compute_units(device)
        rows = max_q_len * group
        low = -(-rows // 64) * num_kv_heads * max(1, num_seqs) * max(1, nsplit)
        if head_dim == 128:
            # (measured: a launch of at most one low workgroup a CU is about 1 us, up to 10 %, faster in
            # the low form, whatever its past and however many requests; so is one prompt from an empty
            # cache while the low form fits the chip at once; else form 3 wins by 5-15 %)
            units = resident // 2
            return 1 if low <= units or (low <= resident and max_kv_len <= max_q_len and num_seqs <= 1) else 3
        return 1 if low <= resident else 2

    def f32_attention_part_steps(self, N: int, S: int, nq: int, num_kv_heads: int, d: int, plain: bool, max_q_len: int, span: int) -> int:
        """The most steps of 32 keys that a workgroup of the float32 kernel of many rows (operands in three bfloat16 parts, blocks of 128
        rows, heads of 128) takes, or 0 where the float32 instruction's kernel stays.  Two workgroups a CU: as many steps as make one
        round of all blocks' parts, each block having half a part less than whole ones on average, and a tenth more; whole blocks
        where there are two a CU.  At 32 / 8 heads, the other kernel -> this one: prompts of 512 / 1024 / 2048 / 4096 tokens 55 -> 40, 116 -> 78,
        385 -> 246, 1375 -> 700 us, 300 tokens behind 4000 231 -> 131, 1000 behind 5000 914 -> 477, 512 behind 2048 beside 20 decoded
        tokens 468 -> 183.  Below two steps for every one of those workgroups, counted in whole blocks, a launch is the chain of one
        workgroup, which is longer here: 200 tokens 23 / 28, eight prompts of 100 23 / 24, 16 tokens behind 6000 34 / 39; 64 behind 2000,
        at the line, 40 / 38.
        The longest request's keys stand for every row's, those of a short prompt beside long decoded requests too, whose own are not known here.
        Measured at 32 / 8 heads, the other kernel -> this one: 32 tokens from an empty cache beside 4 / 20 / 63 decoded at 4096 46 -> 32, 178 -> 128,
        371 -> 370; 200 beside 20 at 4096 236 -> 143; 200 behind 1000 beside 63 at 1000 184 -> 162.  It loses where the portion's own keys are few and the decoded
        requests fill the chip, or are few: 200 from an empty cache beside 63 at 1000 117 -> 131, 32 behind 1000 beside 4 at 4096 46 -> 58 (the worst of
        130 such steps; five lose over 3 %)."""
        group = nq // num_kv_heads
        if not plain or d != 128 or max_q_len * group <= 16:
            return 0
        slots, length = 2 * self.compute_units(), (span - min(span, max_q_len) / 2) / 32
        if num_kv_heads * (N - S) * group / 128 * length < 1.9 * slots:  # (a token of each request left out: those that decode have no more)
            return 0
        blocks = num_kv_heads * max(S, -(-N * group // 128))
        if blocks >= slots:
            return 1 << 20
        return max(4, int(1.1 * blocks * length / (slots - blocks / 2)))

    @staticmethod
    def f32_attention_parts(part_steps: int, rows: int, group: int, max_kv_len: int, span: int) -> tuple:
        """(the most parts of a block of 128 rows, workgroups enough for the parts of all blocks of any request) in parts of at most `part_steps`
        steps of 32 keys (of equal parts where that makes more than 64).  A block's keys lie in one step more than they fill at most, and without a
        window block j from the end sees at least j - 1 blocks' tokens less than the last one; every block may have a part that is not whole."""
        steps, blocks = -(-min(span, max_kv_len) // 32) + 1, -(-rows // 128)
        most = min(64, -(-steps // part_steps))
        fewer = (128 // group) / 32 * (blocks - 1) * (blocks - 2) / 2 if span >= max_kv_len else 0.0
        return most, max(1, min(blocks * most, int((blocks * (steps + 1) - fewer) / part_steps) + blocks + 1))

    def f32_attention_form(self, N: int, nq: int, num_kv_heads: int, d: int, plain: bool, max_q_len: int,
                           span: int) -> tuple:
        """(tiles of 16 rows that a wavefront of the float32 matrix-core kernel takes, whether its long
        and short row blocks are paired, rounds of the CUs that key splits may fill).
        Two tiles share what is loaded of K and V, but half as many workgroups are left: from one and a
        half blocks of 128 rows per CU on (measured, 32 / 8 heads of 128: a 2048-token prompt 372 us, in
        one tile 481; a 1024-token one 184 and 126), and for portions with at least as much behind them,
        2048 keys or more, which key splits spread instead (300 tokens behind 4000: 239 us, in one tile
        469; 512 behind 2048: 220 and 285; 128 behind 1000: 53 and 44).  Splits fill two rounds where each has
        14 steps of 16 keys left, else one where it has 10; with fewer, or where half of the second tiles
        would be empty, one tile is faster: in one tile / two tiles and one round / two rounds 128 tokens behind
        2000 71.5 / 62.0 / 70.9 us, 200 behind 2000 131 / 108 / 101, 64 behind 2000 43 / 43 / 51; of 8 / 1 heads
        64 behind 4000 28.6 / 36.4 / 36.5, 128 behind 2000 28.9 / 30.1 / 40.4, 300 behind 2000 54 / 48 / 56.
        Between four thirds and two blocks per CU all of them start at once and nothing evens out what the CUs
        got: the second one of a CU is the shortest left (a 2048-token prompt 480 -> 372 us, a 1024-token
        one 178 -> 126); otherwise the longest first (4096 tokens: 1386 us, paired 1584; with 304 to 336 blocks
        most CUs get no second one, and the pairs' first half has its longest there: 1300 tokens of 16 / 8 heads
        173, paired 189, 600 and 60 tokens of 32 / 8 heads 80 and 99, under a window of 256 47 and 68)."""
        cus, group = self.compute_units(), nq // num_kv_heads
        if max_q_len * group <= 16:  # decoding: a block a request and key split
            return 1, 0, 1

        def blocks(tiles):  # (the rows of several requests share no block: a few more than this)
            return num_kv_heads * -(-N * group // (64 * tiles))

        tiles = 1
        if plain and d in (64, 128):
            if max_q_len * group > 64 and span >= max(2048, 2 * max_q_len) and 2 * blocks(2) < 3 * cus:
                steps = (span + 15) // 16  # (of a split, once the splits fill `rounds` rounds)
                for rounds, least in ((2, 14), (1, 10)):
                    if 5 * blocks(2) <= 3 * blocks(1) and steps >= least * (rounds * cus // blocks(2)):
                        return 2, 0, rounds
            elif 2 * blocks(2) >= 3 * cus:
                tiles = 2
        return tiles, int(4 * cus <= 3 * blocks(tiles) <= 6 * cus), 1

    def f32_attention_splits(self, num_seqs: int, num_kv_heads: int, row_blocks: int, max_q_len: int,
                             max_kv_len: int, window: int, rounds: int = 1) -> int:
        """Key splits of the float32 matrix-core kernel: enough workgroups for `rounds` rounds of the
        CUs (decoding: one; measured at 1000 keys, batch 16: 29 us, two rounds 30, three 39), at least 4
        of its 16-key steps each (measured at 512 keys: batch 1 in 2 / 8 splits 20 / 12 us, batch 8 in
        2 / 4 splits 22 / 18 us)."""
        span = min(max_kv_len, window + max_q_len) if window else max_kv_len
        by_work = max(1, (span + 15) // 16 // 4)
        by_fill = max(1, rounds * self.compute_units() // max(1, num_seqs * num_kv_heads * row_blocks))
        return int(min(by_work, by_fill, 64))

    def decode_splits(self, num_seqs: int, num_kv_heads: int, max_kv_len: int, window: int) -> int:
        """Key splits of the decode kernel: enough workgroups to fill the chip, but
        at least DECODE_MIN_STEPS_PER_SPLIT 32-key steps each, and none below DECODE_MIN_STEPS_TO_SPLIT steps: the merge
        that splits need is a launch of its own and costs what those steps take (measured at 512 keys:
        batch 16 unsplit 12.1 us, in two 14.2; batch 1 the same either way)."""
        span = min(max_kv_len, window + 32) if window else max_kv_len
        steps = (span + 31) // 32 + (1 if window else 0)
        by_work = max(1, steps // self.DECODE_MIN_STEPS_PER_SPLIT) if steps >= self.DECODE_MIN_STEPS_TO_SPLIT else 1
        by_fill = max(1, self.compute_units() // max(1, num_seqs * num_kv_heads))
        return int(min(by_work, by_fill, 64))

    def add_bias(self, x, bias) -> torch.Tensor:
        """x [M, N] += bias [N], in place (the sum in 32-bit); returns x."""
        _dev(x, "x")
        _dev(bias, "bias")
        _need(x.dim() == 2 and bias.shape == (x.shape[1],), f"bias {list(bias.shape)} does not fit x {list(x.shape)}")
        self._run("elementwise", "lle_add_bias", "PPIIIIP", _ptr(x), _ptr(bias), x.shape[0],
                  x.shape[1], dtype_code(x.dtype), dtype_code(bias.dtype))
        return x

    # -- feed-forward --------------------------------------------------------------
    def silu_mul(self, gate_up) -> torch.Tensor:
        """gate_up [N, 2 I] (gate columns first) -> silu(gate) * up, [N, I]."""
        _dev(gate_up, "gate_up")
        N, two_i = gate_up.shape
        _need(two_i % 2 == 0, "gate_up must have an even width")
        out = _made((N, two_i // 2), dtype=gate_up.dtype, device=gate_up.device)
        self._run("elementwise", "lle_silu_mul", "PPIIIP",
                  _ptr(gate_up), _ptr(out), N, two_i // 2, dtype_code(gate_up.dtype))
        return out

    def gate_up_silu(self, x, weight) -> torch.Tensor:
        """x [M, K], weight [2 I, K] (gate rows, then up rows) -> silu(x gate^T) * (x up^T), [M, I].
        Few rows run as ONE weight-streaming launch with the activation in its epilogue (float32: where _gated_f32_in_one says so), more as
        one launch where rows_tile, wide_form or, in float32, gated_f32_tiles says so; otherwise the product and silu_mul."""
        if isinstance(x, Prenormed):
            folded = self._linear_folded_f32 if weight.dtype == torch.float32 else self._linear_folded
            return folded(x, weight, None, gated=True)
        _dev(x, "x")
        _dev(weight, "weight", x.dtype)
        M, K = x.shape
        N2 = weight.shape[0]
        _need(weight.shape[1] == K and N2 % 2 == 0, f"weight {list(weight.shape)} does not fit x [{M}, {K}]")
        few = M <= self.tuning.skinny_max_rows or (M <= 32 and N2 * K <= self.tuning.skinny_small_weight)
        if x.dtype == torch.bfloat16 and few and K % 8 == 0 and not self.force_library_gemm:
            out = _made((M, N2 // 2), dtype=x.dtype, device=x.device)
            self._run("gemm", "lle_gemm_skinny_gated_bf16", "PPPIIIP",
                      _ptr(x), _ptr(weight), _ptr(out), M, N2, K)
            return out
        if x.dtype == torch.float32 and K % 4 == 0 and self._gated_f32_in_one(M, N2, K) and not self.force_library_gemm:
            out = _made((M, N2 // 2), dtype=x.dtype, device=x.device)
            self._run("gemm", "lle_gemm_skinny_gated_f32", "PPPIIIP",
                      _ptr(x), _ptr(weight), _ptr(out), M, N2, K)
            return out
        tile = self.rows_tile(x, weight, gated=True) if 32 < M <= 256 and x.dtype == torch.bfloat16 else 0
        if tile:
            return self.linear_rows(x, weight, tile, "silu")
        form = self.wide_form(x, weight) if x.dtype == torch.bfloat16 else -1
        if form >= 0:
            return self.gated_wide(x, weight, form, "silu")
        tiles = self.gated_f32_tiles(x, weight) if x.dtype == torch.float32 else -1
        if tiles >= 0:
            return self.gated_f32(x, weight, tiles, "silu")
        return self.silu_mul(self.linear(x, weight))

    def _gated_f32_in_one(self, M: int, N2: int, K: int) -> bool:
        """Whether the float32 product of gate and up and its activation are one launch (the same sums either way).  Not
        * over 32 rows, and up to 16 rows with more than 2560 columns but where the streaming kernel's gated form takes them: 3072 and
          4096 columns (beyond 2560 it has forms of six and of eight rounds of 512 columns), more than 16 gate rows for every CU in tiles of 16, the last of them at least half full (in two launches / in one at 8
          rows, shares of 20, 24, 28, 32, 33, 35, 40, 48, 49, 52 and 65 gate rows: 4096 columns 37.0 / 38.2, 41.2 / 40.4, 48.5 / 44.2, 52.8 / 49.9, 57.8 / 59.1,
          59.0 / 59.5, 64.7 / 63.6, 75.8 / 73.2, 81.7 / 84.7, 84.0 / 85.9, 104.9 / 108.3 us; 3072 columns 27.9 / 28.6, 30.3 / 28.9, 35.1 / 32.7,
          39.1 / 36.9, 42.1 / 43.1, 42.9 / 43.5, 47.1 / 45.3, 57.3 / 55.5, 61.4 / 59.8, 60.6 / 60.8, 78.9 / 79.8);
        * where the plain product's tiles of 16 rows are one for a CU at most: a gated one is two of them, so half of the CUs have
          work or all of them low tiles, which costs more than a launch saves but for short rows and 9 to 16 rows of x (in two
          launches / in one at 1, 8, 16 and 17 rows: 4096 x 1024 7.9, 8.4, 8.9, 9.5 / 6.4, 6.6, 7.3, 9.2 us; 2048 x 1536 7.9, 8.3,
          9.4, 10.7 / 8.3, 8.9, 9.0, 12.5; 4096 x 2560 13.9, 15.8, 18.1, 19.2 / 15.0, 15.1, 17.3, 21.4; 4096 x 4096 at 17 rows
          26.0 / 30.4; 5120 x 1536, over one round of tiles, 13.1, 13.4, 15.1, 18.0 / 10.3, 10.8, 11.8, 14.6)."""
        if M > 32 or (M <= 16 and not 16 < K <= 2560):
            share = -(-(N2 // 2) // self.compute_units())
            return M <= 16 and K in (3072, 4096) and share > 16 and (share - 1) % 16 >= 7
        return K <= 1024 or N2 > 16 * self.compute_units() or 8 < M <= 16

    def gate_up_clamped(self, x, weight, bias, limit: float) -> torch.Tensor:
        """x [M, K], weight [2 I, K] (gate rows, then up rows), bias [2 I] or None -> [M, I]: with g = min(x gate^T + b,
        limit) and u = clamp(x up^T + b, -limit, limit) the result is g sigmoid(1.702 g) (u + 1).  Few bfloat16 rows run as
        ONE weight-streaming launch with the activation in its epilogue, more as one launch where rows_tile, wide_form or, in float32,
        gated_f32_tiles says so; otherwise the product and bias_act."""
        _dev(x, "x")
        _dev(weight, "weight", x.dtype)
        M, K = x.shape
        N2 = weight.shape[0]
        _need(weight.shape[1] == K and N2 % 2 == 0, f"weight {list(weight.shape)} does not fit x [{M}, {K}]")
        if bias is not None:
            _dev(bias, "bias", x.dtype)
            _need(bias.shape == (N2,), "bias must cover the whole weight")
        few = M <= self.tuning.skinny_max_rows or (M <= 32 and N2 * K <= self.tuning.skinny_small_weight)
        if x.dtype == torch.bfloat16 and few and K % 8 == 0 and not self.force_library_gemm:
            _need(limit > 0.0, "a clamped activation has a positive limit")
            out = _made((M, N2 // 2), dtype=x.dtype, device=x.device)
            self._run("gemm", "lle_gemm_skinny_clamped_bf16", "PPPFPIIIP",
                      _ptr(x), _ptr(weight), _ptr(bias), float(limit), _ptr(out), M, N2, K)
            return out
        aligned = bias is None or bias.data_ptr() % 8 == 0
        tile = self.rows_tile(x, weight, gated=True) if 32 < M <= 256 and x.dtype == torch.bfloat16 and limit > 0.0 and aligned else 0
        if tile:
            return self.linear_rows(x, weight, tile, "clamp", bias, limit)
        form = self.wide_form(x, weight) if x.dtype == torch.bfloat16 and limit > 0.0 else -1
        if form >= 0 and aligned:
            return self.gated_wide(x, weight, form, "clamp", bias, limit)
        tiles = self.gated_f32_tiles(x, weight) if x.dtype == torch.float32 and limit > 0.0 else -1
        if tiles >= 0:
            return self.gated_f32(x, weight, tiles, "clamp", bias, limit)
        return self.bias_act(self.linear(x, weight), "clamp", True, bias=bias, limit=limit)

    # -- arrangements that norm a sublayer's output ------------------------------------
    def cast(self, x, dtype) -> torch.Tensor:
        """x in `dtype` (x itself where it has that type already)."""
        if x.dtype == dtype:
            return x
        _dev(x, "x")
        out = _made(x.shape, dtype=dtype, device=x.device)
        self._run("elementwise", "lle_cast", "PPLIIP", _ptr(x), _ptr(out), x.numel(),
                  dtype_code(x.dtype), dtype_code(dtype))
        return out

    def scale_(self, x, factor: float) -> torch.Tensor:
        """float32 x *= factor, in place."""
        _dev(x, "x", torch.float32)
        self._run("elementwise", "lle_scale", "PLFP", _ptr(x), x.numel(), float(factor))
        return x

    def rmsnorm_add(self, hidden, y, weight, eps: float, out_dtype, extra=None) -> torch.Tensor:
        """hidden float32 [N, H] += RMSNorm(y [+ extra]) * weight, in place and in 32-bit; returns the new
        rows in `out_dtype` (`hidden` itself for float32).  `y`, `extra`: [N, H], float32 or bfloat16 each."""
        _dev(hidden, "hidden", torch.float32)
        _dev(weight, "norm weight")
        N, H = hidden.shape
        _need(weight.shape == (H,), f"norm weight must be [{H}], is {list(weight.shape)}")
        for t, name in ((y, "y"), (extra, "extra")):
            if t is not None:
                _dev(t, name)
                _need(t.shape == hidden.shape, f"{name} must have the shape of hidden")
        out = None if out_dtype == torch.float32 else _made((N, H), dtype=out_dtype, device=hidden.device)
        self._run("norm", "lle_rmsnorm_add", "PPIPIPIPIIFIP",
                  _ptr(hidden), _ptr(y), dtype_code(y.dtype), _ptr(extra), dtype_code(extra.dtype) if extra is not None else 0,
                  _ptr(weight), dtype_code(weight.dtype), _ptr(out), N, H, float(eps), dtype_code(out_dtype))
        return hidden if out is None else out

    # -- gated recurrence -------------------------------------------------------------
    MINGRU_PIECE = 16  # tokens of one request that one thread walks before the walk is cut into pieces

    def mingru_scan(self, zxg, z_bias, x_bias, state, seq_slots, cu_tokens, out_dtype, max_q_len: int = 0):
        """zxg [N, 3 W] (update-gate, candidate and output-gate inputs side by side; float32 or bfloat16),
        biases float32 [W], state float32 [slots + 1, W] (read and advanced per request) -> [N, W] in
        `out_dtype`: S <- (1 - z) S + z c per token, out = S * silu(gate).  `max_q_len` (a host-side
        bound of the longest request of the step) only decides into how many pieces a walk is cut."""
        _dev(zxg, "zxg")
        _dev(z_bias, "z_bias", torch.float32)
        _dev(x_bias, "x_bias", torch.float32)
        _dev(state, "state", torch.float32)
        _dev(seq_slots, "seq_slots", torch.int32)
        _dev(cu_tokens, "cu_tokens", torch.int32)
        W = z_bias.shape[0]
        N, S = zxg.shape[0], seq_slots.shape[0]
        _need(zxg.shape == (N, 3 * W) and x_bias.shape == (W,), "zxg must be [N, 3 W] and the biases [W]")
        _need(state.dim() == 2 and state.shape[1] == W, "state must be [slots, W]")
        _need(cu_tokens.shape == (S + 1,), "cu_tokens must be [S + 1]")
        out = _made((N, W), dtype=out_dtype, device=zxg.device)
        pieces = max(1, min(1024, -(-max(1, max_q_len) // self.MINGRU_PIECE)))
        part = _made((S * pieces * 3 * W,), dtype=torch.float32, device=zxg.device) if pieces > 1 else None
        self._run("recurrent", "lle_mingru_scan", "PIPPPPPPIPIIIP",
                  _ptr(zxg), dtype_code(zxg.dtype), _ptr(z_bias), _ptr(x_bias), _ptr(state), _ptr(seq_slots),
                  _ptr(cu_tokens), _ptr(out), dtype_code(out_dtype), _ptr(part), S, W, pieces)
        return out

    # -- latent attention -------------------------------------------------------------
    def latent_kv_write(self, dkv, norm_w, eps: float, cos_sin, rot_dims: int, slots, pages, page_size: int,
                        rank: int, rot: int) -> None:
        """dkv [N, rank + rot] -> the pages: c = RMSNorm(first rank) * norm_w and the rest with its first
        `rot_dims` elements rotated in neighbouring pairs by cos_sin [N, rot_dims / 2, 2].  A page
        (one row of `pages`) is the latents [page_size][rank], the same transposed [rank][page_size],
        then the rotated parts [page_size][rot]; slots[n] < 0 writes nothing."""
        _dev(dkv, "dkv")
        _dev(norm_w, "latent norm weight")
        _dev(slots, "slots", torch.int32)
        N = dkv.shape[0]
        _need(dkv.shape == (N, rank + rot) and norm_w.shape == (rank,) and slots.shape == (N,), "dkv [N, rank + rot]")
        _need(pages.is_cuda and pages.dtype == dkv.dtype and pages.dim() == 2 and pages.stride(1) == 1
              and pages.shape[1] >= page_size * (2 * rank + rot), "pages must be [pages, page_size * (2 rank + rot)]")
        if rot_dims:
            _dev(cos_sin, "cos_sin", torch.float32)
            _need(cos_sin.shape == (N, rot_dims // 2, 2), "cos_sin must be [N, rot_dims / 2, 2]")
        self._run("latent", "lle_latent_kv_write", "PPIFPIPPLIIIIIP",
                  _ptr(dkv), _ptr(norm_w), dtype_code(norm_w.dtype), float(eps), _ptr(cos_sin) if rot_dims else None,
                  int(rot_dims), _ptr(slots), _ptr(pages), pages.stride(0), int(page_size), N, rank, rot,
                  dtype_code(dkv.dtype))

    def latent_q_rope(self, q, cos_sin, rot_dims: int, heads: int, dim: int, rot: int) -> torch.Tensor:
        """q [N, heads * (dim + rot)] -> the last `rot` elements of every head, rotated, float32 [N, heads, rot]."""
        _dev(q, "q")
        N = q.shape[0]
        _need(q.shape == (N, heads * (dim + rot)), "q must be [N, heads * (dim + rot)]")
        if rot_dims:
            _dev(cos_sin, "cos_sin", torch.float32)
            _need(cos_sin.shape == (N, rot_dims // 2, 2), "cos_sin must be [N, rot_dims / 2, 2]")
        out = _made((N, heads, rot), dtype=torch.float32, device=q.device)
        self._run("latent", "lle_latent_q_rope", "PPIPIIIIIP",
                  _ptr(q), _ptr(cos_sin) if rot_dims else None, int(rot_dims), _ptr(out), N, heads, dim, rot,
                  dtype_code(q.dtype))
        return out

    def heads_linear(self, x, heads: int, col0: int, K: int, weight, out_dtype) -> torch.Tensor:
        """x [N, heads * xw] (or [N, heads, xw]) and weight [heads, out, K]: for every head the columns
        col0 .. col0 + K of its part times weight[h]^T -> [N, heads, out].  bfloat16: one batched
        library product (32-bit accumulation, either result type); float32: the true 32-bit kernels, head by head."""
        _dev(x, "x")
        _dev(weight, "weight", x.dtype)
        N = x.shape[0]
        x3 = x.view(N, heads, -1)
        xw, O = x3.shape[2], weight.shape[1]
        _need(weight.shape == (heads, O, K) and 0 <= col0 and col0 + K <= xw, "weight must be [heads, out, K]")
        if x.dtype == torch.bfloat16:
            a = x3[:, :, col0 : col0 + K].transpose(0, 1)  # [heads, N, K]
            b = weight.transpose(1, 2)  # [heads, K, out]
            self._not_recorded()
            y = torch.bmm(a, b) if out_dtype == torch.bfloat16 else torch.bmm(a, b, out_dtype=out_dtype)
            return y.transpose(0, 1)  # [N, heads, out], strided
        _need(out_dtype == torch.float32, "a float32 product has a float32 result")
        out = _made((N, heads, O), dtype=torch.float32, device=x.device)
        quick = K % 4 == 0 and xw % 4 == 0 and col0 % 4 == 0 and not self.force_simt_gemm
        for h in range(heads):
            a_ptr = x.data_ptr() + 4 * (h * xw + col0)
            b_ptr = weight.data_ptr() + 4 * h * O * K
            c_ptr = out.data_ptr() + 4 * h * O
            if quick:
                self._run("gemm_f32", "lle_gemm_nt_f32", self._F32_TILES, a_ptr, b_ptr, c_ptr, N, O, K, heads * xw, K,
                          heads * O, 1, -1)
            else:
                self._run("gemm", "lle_gemm_nt_simt", "PPPIIILLLIIP",
                          a_ptr, b_ptr, c_ptr, N, O, K, heads * xw, K, heads * O, F32, F32)
        return out

    LATENT_GROUPS_PER_CU = 1
    force_generic_latent = False  # tests flip this to compare the two kernels
    last_latent_kernel = None  # (which kernel, key ranges) of the last latent_attention call: for tests

    def latent_query_dtype(self, cache_dtype, page_size: int, rank: int, rot: int):
        """The type in which latent_attention wants q_lat: the cache's where the matrix-core kernel takes the
        sizes (bfloat16, rank a multiple of 16 up to 512, rot a multiple of 8 up to 64, pages of a multiple of
        16 tokens), float32 otherwise."""
        mfma = (cache_dtype == torch.bfloat16 and rank % 16 == 0 and rank <= 512 and rot % 8 == 0 and rot <= 64
                and page_size % 16 == 0 and not self.force_generic_latent)
        return torch.bfloat16 if mfma else torch.float32

    def latent_row_tiles(self, heads: int, max_q_len: int) -> int:
        """16-row tiles per workgroup of the matrix-core kernel: two for prompt portions (a step's operands then
        serve 32 rows: measured at rank 512, 2048 tokens, 388 -> 325 us at 16 heads and 758 -> 629 us at 32), one for
        decoded tokens (two cost a wavefront a SIMD and 2 us of 22 at 32 heads)."""
        return self.force_latent_row_tiles or (2 if max_q_len >= 4 and max_q_len * heads >= 64 else 1)

    force_latent_row_tiles = 0  # tests set 1 or 2

    def latent_splits(self, num_seqs: int, heads: int, max_q_len: int, max_kv_len: int, window: int) -> int:
        """Key ranges per 16-row tile of the matrix-core kernel: enough workgroups (of four wavefronts) for
        LATENT_GROUPS_PER_CU on every CU, at least two 64-key steps each, at most 64."""
        tiles = max(1, num_seqs) * -(-max(1, max_q_len) * heads // (16 * self.latent_row_tiles(heads, max_q_len)))
        span = min(max_kv_len, window + max_q_len) if window else max_kv_len
        steps = -(-max(1, span) // 64)
        return int(max(1, min(-(-self.LATENT_GROUPS_PER_CU * self.compute_units() // tiles), steps // 2, 64)))

    def latent_attention(self, q_lat, q_rot, pages, page_size: int, rank: int, rot: int, block_table, seq_slots,
                         cu_tokens, kv_lens, token_seq, sink, window: Optional[int], scale: float, max_q_len: int,
                         max_kv_len: int, out_dtype) -> torch.Tensor:
        """All heads of every token against the cached latents: q_lat [N, H, rank] (float32 or the
        cache's type; any strides over N and H), q_rot float32 [N, H, rot], sink float32 [H] (None: an ordinary
        softmax, nothing but the keys in its sum) ->
        sum_j p_j c_j, [N, H, rank] in the cache's type.  `max_q_len` and `max_kv_len` are host-side
        bounds; they choose kernels, never results."""
        _dev(q_rot, "q_rot", torch.float32)
        if sink is not None:
            _dev(sink, "sink", torch.float32)
        for t, name in ((block_table, "block_table"), (seq_slots, "seq_slots"), (cu_tokens, "cu_tokens"),
                        (kv_lens, "kv_lens"), (token_seq, "token_seq")):
            _dev(t, name, torch.int32)
        N, H, _ = q_lat.shape
        S = seq_slots.shape[0]
        _need(q_lat.is_cuda and q_lat.shape == (N, H, rank) and q_lat.stride(2) == 1, "q_lat must be [N, H, rank]")
        _need(q_lat.dtype in (torch.float32, pages.dtype), "q_lat is float32 or of the cache's type")
        _need(q_rot.shape == (N, H, rot) and (sink is None or sink.shape == (H,)), "q_rot [N, H, rot], sink [H]")
        _need(pages.is_cuda and pages.dim() == 2 and pages.stride(1) == 1 and pages.dtype == out_dtype
              and pages.shape[1] >= page_size * (2 * rank + rot), "pages must be [pages, page_size * (2 rank + rot)]")
        _need(token_seq.shape == (N,) and cu_tokens.shape == (S + 1,) and kv_lens.shape == (S,), "the step's arrays")
        _need(block_table.dim() == 2, "block_table must be [slots, pages]")
        _need(rank <= 1024, f"a latent of {rank} elements is wider than the attention kernels take (1024)")
        out = _made((N, H, rank), dtype=out_dtype, device=pages.device)
        win = int(window) if window else 0
        if (q_lat.dtype == torch.bfloat16 and self.latent_query_dtype(pages.dtype, page_size, rank, rot) == torch.bfloat16
                and q_lat.stride(0) % 8 == 0 and q_lat.stride(1) % 8 == 0 and pages.stride(0) % 8 == 0
                and max_q_len > 0 and max_kv_len > 0):
            ns = self.latent_splits(S, H, max_q_len, max_kv_len, win)
            rt = self.latent_row_tiles(H, max_q_len)
            self.last_latent_kernel = ("matrix cores", ns)
            ws_o = ws_ml = None
            if ns > 1:
                ws_o = _made((N * H * ns * rank,), dtype=torch.float32, device=pages.device)
                ws_ml = _made((N * H * ns * 2,), dtype=torch.float32, device=pages.device)
            self._run("latent", "lle_latent_attention_mfma",
                      "PLLPPLIIIPIPPPPIFPPPIIIIIIP",
                      _ptr(q_lat), q_lat.stride(0), q_lat.stride(1), _ptr(q_rot), _ptr(pages), pages.stride(0),
                      int(page_size), rank, rot, _ptr(block_table), block_table.shape[1], _ptr(seq_slots),
                      _ptr(cu_tokens), _ptr(kv_lens), _ptr(sink), win, float(scale), _ptr(out), _ptr(ws_o), _ptr(ws_ml),
                      N, S, H, -(-max_q_len * H // (16 * rt)), ns, rt)
            return out
        self.last_latent_kernel = ("generic", 1)
        self._run("latent", "lle_latent_attention_generic",
                  "PILLPPLIIIPIPPPPPIFPIIIP",
                  _ptr(q_lat), dtype_code(q_lat.dtype), q_lat.stride(0), q_lat.stride(1), _ptr(q_rot), _ptr(pages),
                  pages.stride(0), int(page_size), rank, rot, _ptr(block_table), block_table.shape[1], _ptr(seq_slots),
                  _ptr(cu_tokens), _ptr(kv_lens), _ptr(token_seq), _ptr(sink), int(window) if window else 0,
                  float(scale), _ptr(out), N, H, dtype_code(out_dtype))
        return out

    # -- routed feed-forward ----------------------------------------------------------
    def moe_route(self, logits, bias, top: int, score: str = "softmax_chosen", experts: Optional[int] = None):
        """float32 logits [N, >= E] (+ bias [E], or None) -> (int32 ids [N, top] of the largest among the first
        E = `experts` columns (default: all), the lower index first among equals; float32 gains [N, top]).
        `score`: "softmax_chosen": the softmax over the chosen alone; "sigmoid": the sigmoid of every chosen
        value, as it is."""
        _dev(logits, "router logits", torch.float32)
        N, cols = logits.shape
        E = cols if experts is None else int(experts)
        _need(0 < E <= cols and 0 < top <= min(E, 32), "a router picks between 1 and 32 of its experts")
        _need(score in ("softmax_chosen", "sigmoid"), f"unknown router score {score!r}")
        if bias is not None:
            _dev(bias, "router bias", torch.float32)
            _need(bias.shape == (E,), "the router's bias must be [E]")
        ids = _made((N, top), dtype=torch.int32, device=logits.device)
        gains = _made((N, top), dtype=torch.float32, device=logits.device)
        self._run("moe", "lle_moe_route", "PPPPIIIIIP", _ptr(logits), _ptr(bias), _ptr(ids),
                  _ptr(gains), N, E, top, cols, 1 if score == "sigmoid" else 0)
        return ids, gains

    def moe_route_grouped(self, logits, correction, top: int, groups: int = 1, keep: int = 1, score: str = "softmax",
                          group_top: int = 1):
        """float32 logits [N, E] -> (int32 ids [N, top], float32 gains [N, top]).  Scores are the softmax over
        all E (`score` "sigmoid": every logit's own sigmoid); the choice is made on score + correction [E] (None:
        on the scores), among the experts of the `keep` of `groups` equal groups of neighbours whose `group_top`
        largest choice scores add up to most (the lower index wins a tie); gains are the chosen scores, without
        the correction, divided by their sum (+ 1e-20)."""
        _dev(logits, "router logits", torch.float32)
        N, E = logits.shape
        if correction is not None:
            _dev(correction, "router correction", torch.float32)
            _need(correction.shape == (E,), "the router's correction must be [E]")
        _need(score in ("softmax", "sigmoid") and group_top >= 1, f"unknown router score {score!r}")
        _need(0 < top <= min(E, 32), "a router picks between 1 and 32 of its experts")
        _need(groups > 0 and E % groups == 0 and 0 < keep <= groups and top <= keep * (E // groups),
              "the experts form equal groups, and the kept groups hold at least `top` experts")
        _need(2 * E + groups <= 4096, "the router's kernel keeps its scores in LDS: at most about 2000 experts")
        ids = _made((N, top), dtype=torch.int32, device=logits.device)
        gains = _made((N, top), dtype=torch.float32, device=logits.device)
        self._run("moe", "lle_moe_route_grouped", "PPPPIIIIIIIP", _ptr(logits),
                  _ptr(correction), _ptr(ids), _ptr(gains), N, E, top, int(groups), int(keep),
                  1 if score == "sigmoid" else 0, int(group_top))
        return ids, gains

    MOE_TILED_MIN_PAIRS = 129  # (token, choice) pairs from which the sorted, tiled kernels take a bfloat16 step

    EXPERT_FORMS = {"gated_silu": 0, "relu2": 1, "gated_clamp": 2}

    def moe_experts(self, x, ids, gains, gate_up, down, form: str = "gated_silu", gain_on_input: bool = False,
                    limit: float = 0.0) -> torch.Tensor:
        """x [N, K]; ids, gains [N, top]; gate_up [E, 2 F, K] (gate rows, then up rows); down [E, H, F] ->
        float32 [N, H]: sum_k gains[n, k] * down[e] (silu(gate[e] x) * (up[e] x)), e = ids[n, k].  An id from E on
        names an identity expert, whose result is x itself (then H = K).
        `form` "relu2": experts without a gate, down[e] relu(up[e] x)^2, `gate_up` is up [E, F, K].
        `form` "gated_clamp": g = min(gate[e] x, limit), u = clamp(up[e] x, -limit, limit), down[e] (g sigmoid(1.702 g) (u + 1)).
        `gain_on_input`: the result is sum_k expert_e(gains[n, k] * x) instead; the gain is applied to the first
        products' results, in 32-bit, before the activation.
        Few pairs, or float32: every pair streams its expert's rows.  Many bfloat16 pairs: sorted by expert
        on the device, then tiles of 128 pairs of one expert on the matrix cores."""
        _dev(x, "x")
        _dev(ids, "ids", torch.int32)
        _dev(gains, "gains", torch.float32)
        _dev(gate_up, "gate_up", x.dtype)
        _dev(down, "down", x.dtype)
        N, K = x.shape
        top = ids.shape[1]
        _need(form in self.EXPERT_FORMS, f"unknown expert form {form!r}")
        _need(form != "gated_clamp" or limit > 0.0, "clamped experts need a positive limit")
        plain = form == "relu2"
        E, F2, _ = gate_up.shape
        H = down.shape[1]
        F = F2 if plain else F2 // 2
        _need(ids.shape == (N, top) and gains.shape == (N, top), "ids and gains must be [N, top]")
        _need(gate_up.shape == (E, F2, K) and (plain or F2 % 2 == 0) and down.shape == (E, H, F), "expert weights do not fit")
        act = _made((N * top, F), dtype=x.dtype, device=x.device)
        out = _made((N, H), dtype=torch.float32, device=x.device)
        code, on_input = self.EXPERT_FORMS[form], (1 if gain_on_input else 0)
        if (x.dtype == torch.bfloat16 and N * top >= self.MOE_TILED_MIN_PAIRS and E <= 256 and K % 8 == 0 and F % 8 == 0
                and H % 4 == 0):
            plan = _made((4 * E + 1,), dtype=torch.int32, device=x.device)
            order = _made((2, N * top), dtype=torch.int32, device=x.device)
            y = _made((N * top, H), dtype=torch.float32, device=x.device)
            self._run("moe", "lle_moe_experts_tiled",
                      "PPPPPPPPPPPIIIIIIIIFP",
                      _ptr(x), _ptr(ids), _ptr(gains), _ptr(gate_up), _ptr(down), _ptr(plan), order[0].data_ptr(),
                      order[1].data_ptr(), _ptr(act), _ptr(y), _ptr(out), N, top, E, F, K, H, code, on_input, float(limit))
            return out
        self._run("moe", "lle_moe_experts", "PPPPPPPIIIIIIIIIFP",
                  _ptr(x), _ptr(ids), _ptr(gains), _ptr(gate_up), _ptr(down), _ptr(act), _ptr(out), N, top, E, F,
                  K, H, dtype_code(x.dtype), code, on_input, float(limit))
        return out

    # -- projections normed as a whole, sinks' attention gates -------------------------------
    def proj_norm_rope_write(self, qkv, bias, slots, q_weight, k_weight, cos_sin, rotary_dim: int, eps: float, kv_layer,
                             num_q_heads: int, num_kv_heads: int, dim: int, vdim: int, has_kv: bool = True,
                             write_kv: bool = True, per_head: bool = False) -> torch.Tensor:
        """A row of qkv holds q [nq dim], then (`has_kv`) k [nkv dim] and v [nkv vdim], then columns that are
        left alone; `bias` (or None) covers the whole row.  q and k are divided by the root mean square of their
        whole projection (`per_head`: every head by its own), times q_weight [nq dim] / k_weight [nkv dim] (None:
        times one), then the first `rotary_dim` elements of
        every head are rotated (half-split) by cos_sin [N, rotary_dim / 2, 2].  Returns q [N, nq, D] with
        D = kv_layer.shape[4] >= max(dim, vdim), zeros past dim; K and V^T go to the pages `kv_layer`
        [pages, 2, nkv, page_size, D] at `slots` [N] with zeros past dim and vdim."""
        _dev(qkv, "qkv")
        _dev(slots, "slots", torch.int32)
        _dev(kv_layer, "kv_layer", qkv.dtype)
        nq, nkv = num_q_heads, num_kv_heads
        N, cols = qkv.shape
        need = nq * dim + (nkv * (dim + vdim) if has_kv else 0)
        _need(cols >= need, "qkv has too few columns")
        _need(slots.shape == (N,), "slots must be [N]")
        _need(kv_layer.dim() == 5 and kv_layer.shape[1] == 2 and kv_layer.shape[2] == nkv, "kv_layer must be [pages, 2, nkv, page_size, D]")
        D, page_size = kv_layer.shape[4], kv_layer.shape[3]
        _need(D >= max(dim, vdim), "the cache's heads are smaller than the model's")
        _need(0 <= rotary_dim <= dim and rotary_dim % 2 == 0, "rotary_dim must be even and <= dim")
        if bias is not None:
            _dev(bias, "bias", qkv.dtype)
            _need(bias.shape == (cols,), "bias must cover the whole row")
        if q_weight is not None:
            _dev(q_weight, "q norm weight")
            _need(q_weight.shape == (nq * dim,), f"q norm weight must be [{nq * dim}]")
        if has_kv and k_weight is not None:
            _need(q_weight is not None, "both norms have weights, or neither")
            _dev(k_weight, "k norm weight", q_weight.dtype)
            _need(k_weight.shape == (nkv * dim,), f"k norm weight must be [{nkv * dim}]")
        _need(not per_head or nq + nkv <= 512, "heads normed one by one: at most 512 query and key heads together")
        if rotary_dim > 0:
            _dev(cos_sin, "cos_sin", torch.float32)
            _need(cos_sin.shape == (N, rotary_dim // 2, 2), "cos_sin must be [N, rotary_dim / 2, 2]")
        q_out = _made((N, nq, D), dtype=qkv.dtype, device=qkv.device)
        self._run("rope_kv", "lle_proj_norm_rope_write",
                  "PIPPPPIPIFPPIIIIIIILIIIIP",
                  _ptr(qkv), cols, _ptr(bias), _ptr(slots), _ptr(q_weight), _ptr(k_weight) if has_kv else None,
                  dtype_code(q_weight.dtype) if q_weight is not None else F32, _ptr(cos_sin) if rotary_dim > 0 else None,
                  rotary_dim, float(eps), _ptr(q_out), _ptr(kv_layer), N, nq, nkv, dim, vdim, D, page_size,
                  kv_layer.stride(0), 1 if has_kv else 0, 1 if write_kv else 0, 1 if per_head else 0,
                  dtype_code(qkv.dtype))
        return q_out

    def head_gate(self, a, gates, col0: int, heads: int, vdim: int) -> torch.Tensor:
        """a [N, heads * D], D >= vdim -> [N, heads * vdim]: head h's first vdim elements times
        sigmoid(gates[n, col0 + h])."""
        _dev(a, "a")
        _dev(gates, "gates", a.dtype)
        N = a.shape[0]
        _need(a.dim() == 2 and a.shape[1] % heads == 0 and a.shape[1] // heads >= vdim, "a must be [N, heads * D], D >= vdim")
        _need(gates.dim() == 2 and gates.shape[0] == N and 0 <= col0 and col0 + heads <= gates.shape[1], "gates [N, >= col0 + heads]")
        out = _made((N, heads * vdim), dtype=a.dtype, device=a.device)
        self._run("elementwise", "lle_head_gate", "PPIIPIIIIIP", _ptr(a), _ptr(gates),
                  gates.shape[1], int(col0), _ptr(out), N, heads, a.shape[1] // heads, vdim, dtype_code(a.dtype))
        return out

    def tanh_(self, x) -> torch.Tensor:
        """x = tanh(x), in place."""
        _dev(x, "x")
        self._run("elementwise", "lle_tanh", "PLIP", _ptr(x), x.numel(), dtype_code(x.dtype))
        return x

    def scaled_add_rmsnorm(self, hidden, a, b, mult: float, weight, eps: float, out_dtype, rows=None,
                           mult_b: Optional[float] = None) -> torch.Tensor:
        """hidden float32 [N, H] += mult * a + mult_b * b in 32-bit and in place (`b` may be None; a, b [N, H],
        float32 or bfloat16 each; `mult_b` None: mult), then RMSNorm(hidden) * weight in `out_dtype`.  With `rows` (int32 [R]) only
        those rows are read, row rows[r] gives row r of the result, and `hidden` is left alone."""
        _dev(hidden, "hidden", torch.float32)
        _dev(weight, "norm weight")
        N, H = hidden.shape
        _need(weight.shape == (H,), f"norm weight must be [{H}]")
        for t, name in ((a, "a"), (b, "b")):
            if t is not None:
                _dev(t, name)
                _need(t.shape == hidden.shape, f"{name} must have the shape of hidden")
        R = N
        if rows is not None:
            _dev(rows, "rows", torch.int32)
            R = rows.shape[0]
        out = _made((R, H), dtype=out_dtype, device=hidden.device)
        self._run("norm", "lle_scaled_add_rmsnorm", "PPIPIFFPPIPIIFIP",
                  _ptr(hidden), _ptr(a), dtype_code(a.dtype), _ptr(b), dtype_code(b.dtype) if b is not None else 0,
                  float(mult), float(mult if mult_b is None else mult_b), _ptr(rows), _ptr(weight), dtype_code(weight.dtype), _ptr(out), R, H, float(eps),
                  dtype_code(out_dtype))
        return out

    # -- recurrence with a matrix state ------------------------------------------------------
    def shift_mix(self, x, state, prev_offset: int, mu, token_seq, cu_tokens, seq_slots) -> torch.Tensor:
        """x [N, W] -> [M, N, W]: out[m, n] = x[n] + (prev - x[n]) * mu[m], prev = x[n - 1], or for the first
        token of a request's portion state[slot, prev_offset : prev_offset + W] (float32; what the step before
        left there).  mu float32 [M, W]."""
        _dev(x, "x")
        _rows(state, "state", torch.float32)
        _dev(mu, "mu", torch.float32)
        for t, name in ((token_seq, "token_seq"), (cu_tokens, "cu_tokens"), (seq_slots, "seq_slots")):
            _dev(t, name, torch.int32)
        N, W = x.shape
        M = mu.shape[0]
        _need(mu.shape == (M, W) and state.dim() == 2 and prev_offset + W <= state.shape[1], "mu [M, W]; the state row holds W saved elements")
        out = _made((M, N, W), dtype=x.dtype, device=x.device)
        self._run("wkv", "lle_shift_mix", "PPLIPPPPPIIIIP", _ptr(x), _ptr(state),
                  state.stride(0), int(prev_offset), _ptr(mu), _ptr(token_seq), _ptr(cu_tokens), _ptr(seq_slots), _ptr(out),
                  N, W, M, dtype_code(x.dtype))
        return out

    WKV_PIECE = 64  # tokens of one request that are walked in a row before the walk is cut into pieces
    WKV_MAX_DIM = MAX_WKV_HEAD_DIM

    def wkv_scan(self, r, k, v, wraw, w0, u, g, norm_w, eps: float, x, state, heads: int, dim: int, seq_slots,
                 cu_tokens, out_dtype, max_q_len: int = 0) -> torch.Tensor:
        """Per head, with the matrix state S [dim, dim] of the request (float32, `state[slot, : heads dim dim]`):
            o_t = (S + diag(u) k_t v_t^T)^T r_t;   S <- diag(exp(-exp(wraw_t + w0))) S + k_t v_t^T
        and the result [N, heads * dim] in `out_dtype` is o_t / rms(o_t) (per head, eps inside the root)
        * norm_w * silu(g_t).  r, k, v, wraw float32 [N, heads * dim]; w0, u float32 [heads * dim]; g, x in
        `out_dtype`.  The last row of every request's x [N, W] is saved behind the matrix state.
        `max_q_len` (a host-side bound) only decides into how many pieces a walk is cut."""
        HD = heads * dim
        for t, name in ((r, "r"), (k, "k"), (v, "v"), (wraw, "wraw"), (w0, "w0"), (u, "u")):
            _dev(t, name, torch.float32)
        _rows(state, "state", torch.float32)
        _dev(g, "g", out_dtype)
        _dev(x, "x", out_dtype)
        _dev(norm_w, "norm weight")
        _dev(seq_slots, "seq_slots", torch.int32)
        _dev(cu_tokens, "cu_tokens", torch.int32)
        N, W = x.shape
        S = seq_slots.shape[0]
        _need(0 < dim <= self.WKV_MAX_DIM, f"a head of the recurrence holds at most {self.WKV_MAX_DIM} channels")
        for t in (r, k, v, wraw, g):
            _need(t.shape == (N, HD), "r, k, v, wraw and g must be [N, heads * dim]")
        _need(w0.shape == (HD,) and u.shape == (HD,) and norm_w.shape == (HD,), "w0, u and the norm weight must be [heads * dim]")
        _need(state.dim() == 2 and state.shape[1] >= HD * dim + W, "a state row holds heads * dim * dim + W floats")
        _need(cu_tokens.shape == (S + 1,), "cu_tokens must be [S + 1]")
        out = _made((N, HD), dtype=out_dtype, device=x.device)
        piece = self.WKV_PIECE
        pieces = -(-max_q_len // piece) if max_q_len > 2 * piece else 1
        part = None
        if pieces > 1:
            part = _made((S * pieces * heads * (dim * dim + dim),), dtype=torch.float32, device=x.device)
        else:
            piece = 1 << 30
        self._run("wkv", "lle_wkv_scan",
                  "PPPPPPPPIFPPLIPPPIIIIIIPIP",
                  _ptr(r), _ptr(k), _ptr(v), _ptr(wraw), _ptr(w0), _ptr(u), _ptr(g), _ptr(norm_w),
                  dtype_code(norm_w.dtype), float(eps), _ptr(x), _ptr(state), state.stride(0), HD * dim, _ptr(seq_slots),
                  _ptr(cu_tokens), _ptr(out), S, heads, dim, W, pieces, piece, _ptr(part), dtype_code(out_dtype))
        return out

    # -- what enters the stream between two blocks ------------------------------------------------
    def inject_rmsnorm(self, hidden, delta, vector, again, weight, eps: float, out_dtype, rows=None) -> torch.Tensor:
        """hidden float32 [N, H] += delta + vector + the embedding's rows, in 32-bit and in place, then
        RMSNorm(hidden) * weight in `out_dtype`.  `delta`: [N, H] in either type, PartialSums, a ScaledSum with a
        factor of one, or None (any other delta is added up first); `vector` float32 [H] or None; `again` a
        parts.base.EmbeddedRows or None.  With `rows` (int32 [R]) only those rows are read, row rows[r] gives row r of
        the result, and `hidden` is left alone."""
        _dev(hidden, "hidden", torch.float32)
        _dev(weight, "norm weight")
        N, H = hidden.shape
        _need(weight.shape == (H,), f"norm weight must be [{H}]")
        a, b, slices, stride = delta, None, 1, 0
        if isinstance(delta, PartialSums):
            a = delta.sums
            slices, stride = a.shape[0], a.stride(0)
            _dev(a, "partial sums", torch.float32)
            _need(a.dim() == 3 and a.shape[1:] == hidden.shape, "partial sums must be [slices, N, H]")
        elif isinstance(delta, ScaledSum):
            a, b = delta.a, delta.b
            if delta.mult != 1.0 or (delta.b is not None and delta.mult_b not in (None, 1.0)):
                a, b = delta.total(), None
        elif isinstance(delta, Injected):
            a = delta.total()
        if a is not None and not isinstance(delta, PartialSums):
            for t, name in ((a, "delta"), (b, "delta's second summand")):
                if t is not None:
                    _dev(t, name)
                    _need(t.shape == hidden.shape, f"{name} must have the shape of hidden")
        if vector is not None:
            _dev(vector, "vector", torch.float32)
            _need(vector.shape == (H,), f"vector must be [{H}]")
        ids = table = feedback = token_seq = seq_slots = None
        scale = 1.0
        if again is not None:
            ids, table, scale = again.ids, again.table, float(again.scale)
            feedback, token_seq, seq_slots = again.feedback, again.token_seq, again.seq_slots
            _dev(ids, "ids", torch.int32)
            _dev(table, "embedding table")
            _need(ids.shape == (N,) and table.dim() == 2 and table.shape[1] == H, "the embedding's rows must fit hidden")
            if feedback is not None:
                for t, name in ((feedback, "feedback"), (token_seq, "token_seq"), (seq_slots, "seq_slots")):
                    _need(t is not None, "feedback, token_seq and seq_slots come together")
                    _dev(t, name, torch.int32)
                _need(token_seq.shape == (N,), "token_seq must be [N]")
        R = N
        if rows is not None:
            _dev(rows, "rows", torch.int32)
            R = rows.shape[0]
        out = _made((R, H), dtype=out_dtype, device=hidden.device)
        code = lambda t: 0 if t is None else dtype_code(t.dtype)
        self._run("norm", "lle_inject_rmsnorm",
                  "PPIILPIPPPIFPPPPPIPIIFIP",
                  _ptr(hidden), _ptr(a), code(a), slices, stride, _ptr(b), code(b), _ptr(vector), _ptr(ids), _ptr(table),
                  code(table), scale, _ptr(feedback), _ptr(token_seq) if feedback is not None else None,
                  _ptr(seq_slots) if feedback is not None else None, _ptr(rows), _ptr(weight), dtype_code(weight.dtype),
                  _ptr(out), R, H, float(eps), dtype_code(out_dtype))
        return out

    # -- attention gated element by element, heads' weights mixed ----------------------------------
    def pair_rope_write(self, u, bias, slots, cos_sin, v_cos_sin, kv_layer, num_q_heads: int, num_kv_heads: int, dim: int,
                        vdim: int, write_kv: bool = True) -> torch.Tensor:
        """A row of u holds q [nq dim], k [nkv dim], v [nkv vdim], then columns that are left alone; `bias` (or None)
        covers those three.  The first elements of every q and k head turn in neighbouring pairs by cos_sin
        [N, rot / 2, 2] (None: not), whole values by v_cos_sin [N, vdim / 2, 2] (None: not).  Returns q [N, nq, D] with
        D = kv_layer.shape[4] >= max(dim, vdim), zeros past dim; K and V^T go to the pages `kv_layer`
        [pages, 2, nkv, page_size, D] at `slots` [N] with zeros past dim and vdim."""
        _dev(u, "u")
        _dev(slots, "slots", torch.int32)
        _dev(kv_layer, "kv_layer", u.dtype)
        nq, nkv = num_q_heads, num_kv_heads
        N, cols = u.shape
        used = nq * dim + nkv * (dim + vdim)
        _need(cols >= used, "u has too few columns")
        _need(slots.shape == (N,), "slots must be [N]")
        _need(kv_layer.dim() == 5 and kv_layer.shape[1] == 2 and kv_layer.shape[2] == nkv, "kv_layer must be [pages, 2, nkv, page_size, D]")
        D, page_size = kv_layer.shape[4], kv_layer.shape[3]
        _need(D >= max(dim, vdim) and D % 2 == 0, "the cache's heads are smaller than the model's, or odd")
        if bias is not None:
            _dev(bias, "bias", u.dtype)
            _need(bias.shape == (used,), "bias must cover q, k and v")
        rot = 0
        for t, name, most in ((cos_sin, "cos_sin", dim), (v_cos_sin, "v_cos_sin", vdim)):
            if t is not None:
                _dev(t, name, torch.float32)
                _need(t.dim() == 3 and t.shape[0] == N and t.shape[2] == 2 and 2 * t.shape[1] <= most, f"{name} must be [N, pairs, 2]")
        if cos_sin is not None:
            rot = 2 * cos_sin.shape[1]
        _need(v_cos_sin is None or 2 * v_cos_sin.shape[1] == vdim, "v_cos_sin must cover the whole value")
        q_out = _made((N, nq, D), dtype=u.dtype, device=u.device)
        self._run("rope_kv", "lle_pair_rope_write",
                  "PIPPPIPPPIIIIIIILIIP",
                  _ptr(u), cols, _ptr(bias), _ptr(slots), _ptr(cos_sin), rot, _ptr(v_cos_sin), _ptr(q_out), _ptr(kv_layer), N,
                  nq, nkv, dim, vdim, D, page_size, kv_layer.stride(0), 1 if write_kv else 0, dtype_code(u.dtype))
        return q_out

    def turn_back_gate(self, a, u, gate_col: int, heads: int, vdim: int, v_cos_sin, out_scale: float = 1.0) -> torch.Tensor:
        """a [N, heads * D], D >= vdim -> [N, heads * vdim]: every head's first vdim elements, turned back in
        neighbouring pairs by v_cos_sin [N, vdim / 2, 2] (None: not), times sigmoid(u[n, gate_col + ...]) element by
        element, times out_scale."""
        _dev(a, "a")
        _dev(u, "u", a.dtype)
        N = a.shape[0]
        _need(a.dim() == 2 and a.shape[1] % heads == 0 and a.shape[1] // heads >= vdim, "a must be [N, heads * D], D >= vdim")
        _need(u.dim() == 2 and u.shape[0] == N and 0 <= gate_col and gate_col + heads * vdim <= u.shape[1], "u [N, >= gate_col + heads * vdim]")
        if v_cos_sin is not None:
            _dev(v_cos_sin, "v_cos_sin", torch.float32)
            _need(v_cos_sin.shape == (N, vdim // 2, 2) and vdim % 2 == 0, "v_cos_sin must cover the whole value")
        out = _made((N, heads * vdim), dtype=a.dtype, device=a.device)
        self._run("rope_kv", "lle_turn_back_gate", "PPIIPPIIIIFIP", _ptr(a), _ptr(u),
                  u.shape[1], int(gate_col), _ptr(v_cos_sin), _ptr(out), N, heads, a.shape[1] // heads, vdim, float(out_scale),
                  dtype_code(a.dtype))
        return out

    def talking_attention(self, q, kv_layer, block_table, seq_slots, cu_tokens, kv_lens, token_seq, chunk: Optional[int],
                          scale: float, slopes, talk, min_q_len: int = 0, max_q_len: int = 0,
                          max_kv_len: int = 0) -> torch.Tensor:
        """q [N, H, D] against the pages -> [N, H * D].  Position p sees the keys p // chunk * chunk .. p (chunk None:
        all from 0 on); scores (q . k) * scale - slopes[h] * (p - j) (slopes float32 [H] or None), softmax, then the
        heads' weights mixed, w_h <- sum_g talk[h, g] w_g (talk float32 [H, H]), head h on its own key/value head's
        values.  `min_q_len`, `max_q_len` and `max_kv_len` are host-side bounds of this batch; they choose the
        kernels, never the result."""
        _dev(q, "q")
        _dev(kv_layer, "kv_layer", q.dtype)
        for t, name in ((block_table, "block_table"), (seq_slots, "seq_slots"), (cu_tokens, "cu_tokens"),
                        (kv_lens, "kv_lens"), (token_seq, "token_seq")):
            _dev(t, name, torch.int32)
        N, H, D = q.shape
        G, P = kv_layer.shape[2], kv_layer.shape[3]
        _need(kv_layer.dim() == 5 and kv_layer.shape[4] == D and kv_layer.shape[1] == 2, "kv_layer must be [pages, 2, G, page_size, D]")
        _need(H % G == 0, "query heads must be a multiple of key/value heads")
        _need(token_seq.shape == (N,), "token_seq must be [N]")
        S = seq_slots.shape[0]
        _need(cu_tokens.shape == (S + 1,) and kv_lens.shape == (S,), "cu_tokens [S + 1], kv_lens [S]")
        _need(block_table.dim() == 2, "block_table must be [slots, pages]")
        _need(chunk is None or chunk > 0, "a chunk must be positive")
        _dev(talk, "talk", torch.float32)
        _need(talk.shape == (H, H), "talk must be [H, H]")
        if slopes is not None:
            _dev(slopes, "slopes", torch.float32)
            _need(slopes.shape == (H,), "slopes must be [H]")
        out = _made((N, H * D), dtype=q.dtype, device=q.device)
        run_decode, run_prefill = min_q_len <= 1, max_q_len > 1
        if (q.dtype == torch.bfloat16 and D % 32 == 0 and D <= 128 and P % 16 == 0 and max_q_len > 0 and max_kv_len > 0
                and S <= 65535 and (H <= 32 if run_prefill else H <= 128) and not self.force_generic_attention):
            K = splits = 0
            ws_s = ws_ml = None
            if run_decode:
                seen = min(chunk, max_kv_len) if chunk else max_kv_len  # keys that a query sees at most
                K = -(-(seen + 15) // 16) * 16
                # a wavefront should have a tile of 16 keys or two, and the workgroups fill the CUs once or twice
                splits = int(max(1, min(-(-K // 64), 2 * self.compute_units() // max(1, S * G))))
                ws_s = _made((S * H * K,), dtype=torch.float32, device=q.device)
                ws_ml = _made((S * H * (K // 16) * 2,), dtype=torch.float32, device=q.device)
            ws_sums = _made((N * H,), dtype=torch.float32, device=q.device) if run_prefill else None
            # one output head a wavefront: twice the workgroups, which make all scores again; where the tiles leave CUs idle
            out_heads = 1 if -(-max_q_len // 16) * S * 2 <= self.compute_units() else 2
            self._run("talking", "lle_talking_mfma",
                      "PPPPPPPPIIIIILIIFPPIIIPPIIIPP",
                      _ptr(q), _ptr(kv_layer), _ptr(block_table), _ptr(seq_slots), _ptr(cu_tokens), _ptr(kv_lens),
                      _ptr(token_seq), _ptr(out), S, H, G, D, P, kv_layer.stride(0), block_table.shape[1], int(chunk or 0),
                      float(scale), _ptr(slopes), _ptr(talk), int(run_decode), splits, K, _ptr(ws_s), _ptr(ws_ml),
                      int(run_prefill), max_q_len, out_heads, _ptr(ws_sums))
            return out
        self._run("talking", "lle_talking_generic",
                  "PPPPPPPPIIIIILIIFPPIP",
                  _ptr(q), _ptr(kv_layer), _ptr(block_table), _ptr(seq_slots), _ptr(cu_tokens), _ptr(kv_lens), _ptr(token_seq),
                  _ptr(out), N, H, G, D, P, kv_layer.stride(0), block_table.shape[1], int(chunk or 0), float(scale),
                  _ptr(slopes), _ptr(talk), dtype_code(q.dtype))
        return out

    # -- gated linear attention -----------------------------------------------------------------------
    GLA_PIECE = 64  # tokens of one request that are walked in a row before the walk is cut into pieces

    def gla_decay(self, low, a2, bias, tau: float) -> torch.Tensor:
        """sigmoid(low @ a2 + bias)^(1 / tau), all float32: low [N, R], a2 [R, C], bias [C] -> [N, C]."""
        for t, name in ((low, "low"), (a2, "a2"), (bias, "bias")):
            _dev(t, name, torch.float32)
        N, R = low.shape
        C = bias.shape[0]
        _need(a2.shape == (R, C), "a2 must be [R, C]")
        out = _made((N, C), dtype=torch.float32, device=low.device)
        self._run("gla", "lle_gla_decay", "PPPPIIIFP", _ptr(low), _ptr(a2), _ptr(bias), _ptr(out), N, R,
                  C, float(tau))
        return out

    def gla_scan(self, u, decay, q_scale: float, norm_w, eps: float, state, heads: int, dim: int, vdim: int, seq_slots,
                 cu_tokens, max_q_len: int = 0) -> torch.Tensor:
        """Per head, with the matrix state S [dim, vdim] of the request (float32, `state[slot, : heads dim vdim]`):
            S <- diag(decay_t) S + k_t v_t^T;   o_t = S^T (q_scale q_t)
        and the result [N, heads * vdim] is o_t / rms(o_t) (per head, eps inside the root) * norm_w [vdim] * silu(g_t).
        A row of u holds q [heads dim], k [heads dim], v [heads vdim], g [heads vdim]; decay float32 [N, heads * dim].
        `max_q_len` (a host-side bound) only decides into how many pieces a walk is cut."""
        _dev(u, "u")
        _dev(decay, "decay", torch.float32)
        _dev(norm_w, "norm weight", torch.float32)
        _rows(state, "state", torch.float32)
        _dev(seq_slots, "seq_slots", torch.int32)
        _dev(cu_tokens, "cu_tokens", torch.int32)
        N, cols = u.shape
        S = seq_slots.shape[0]
        _need(0 < dim <= MAX_GLA_HEAD_DIM and 0 < vdim <= MAX_GLA_HEAD_DIM, f"a head of the recurrence holds at most {MAX_GLA_HEAD_DIM} channels")
        _need(cols >= 2 * heads * (dim + vdim), "u has too few columns")
        _need(decay.shape == (N, heads * dim), "decay must be [N, heads * dim]")
        _need(norm_w.shape == (vdim,), "the norm weight must be [vdim]")
        _need(state.dim() == 2 and state.shape[1] >= heads * dim * vdim, "a state row holds heads * dim * vdim floats")
        _need(cu_tokens.shape == (S + 1,), "cu_tokens must be [S + 1]")
        out = _made((N, heads * vdim), dtype=u.dtype, device=u.device)
        piece = self.GLA_PIECE
        pieces = -(-max_q_len // piece) if max_q_len > 2 * piece else 1
        part = None
        if pieces > 1:
            part = _made((S * pieces * heads * (dim * vdim + dim),), dtype=torch.float32, device=u.device)
        else:
            piece = 1 << 30
        self._run("gla", "lle_gla_scan",
                  "PIPFPFPLPPPIIIIIIPIP",
                  _ptr(u), cols, _ptr(decay), float(q_scale), _ptr(norm_w), float(eps), _ptr(state), state.stride(0),
                  _ptr(seq_slots), _ptr(cu_tokens), _ptr(out), S, heads, dim, vdim, pieces, piece, _ptr(part),
                  dtype_code(u.dtype))
        return out

    # -- activations, caps, chained norms ---------------------------------------------------------
    ACT_CODES = {"silu": 0, "relu": 1, "relu2": 2, "gelu_tanh": 3, "clamp": 4}

    def bias_act(self, z, kind: str, gated: bool, bias=None, row_gate=None, limit: float = 0.0) -> torch.Tensor:
        """gated: z [N, 2 F] (gate columns first) -> act(gate + b) * (up + b), [N, F]; else z [N, F] -> act(z + b).
        `kind`: silu, relu, relu2 (the square of relu), gelu_tanh (gelu in its tanh form), or, gated only, clamp: with
        g = min(gate + b, limit) and u = clamp(up + b, -limit, limit) the result is g sigmoid(1.702 g) (u + 1); `bias` (or None) covers z's row; `row_gate` = (t, col), t
        float32 [N, any]: row n is multiplied by sigmoid(t[n, col]).  Everything in 32-bit."""
        _dev(z, "z")
        _need(kind in self.ACT_CODES, f"unknown activation {kind!r}")
        N, cols = z.shape
        _need(not gated or cols % 2 == 0, "a gated input has an even width")
        _need(kind != "clamp" or (gated and limit > 0.0), "a clamped activation is gated and has a positive limit")
        F = cols // 2 if gated else cols
        if bias is not None:
            _dev(bias, "bias", z.dtype)
            _need(bias.shape == (cols,), "bias must cover the whole row")
        gate_t, stride, col = None, 0, 0
        if row_gate is not None:
            gate_t, col = row_gate
            _dev(gate_t, "row gate", torch.float32)
            _need(gate_t.dim() == 2 and gate_t.shape[0] == N and 0 <= col < gate_t.shape[1], "row gate [N, > col]")
            stride = gate_t.shape[1]
        out = _made((N, F), dtype=z.dtype, device=z.device)
        self._run("elementwise", "lle_bias_act", "PPPIIPIIIIFIP", _ptr(z), _ptr(bias),
                  _ptr(gate_t), stride, int(col), _ptr(out), N, F, 1 if gated else 0, self.ACT_CODES[kind],
                  float(limit), dtype_code(z.dtype))
        return out

    def softcap_(self, x, cap: float) -> torch.Tensor:
        """float32 x = cap * tanh(x / cap), in place."""
        _dev(x, "x", torch.float32)
        _need(cap > 0.0, "a cap must be positive")
        self._run("elementwise", "lle_softcap", "PLFP", _ptr(x), x.numel(), float(cap))
        return x

    def rmsnorm_add_rmsnorm(self, hidden, y, weight, eps: float, next_weight, next_eps: float, out_dtype,
                            extra=None) -> torch.Tensor:
        """hidden float32 [N, H] += RMSNorm(y [+ extra]) * weight, in place and in 32-bit; returns
        RMSNorm(the new hidden) * next_weight in `out_dtype`: the norm after one sublayer and the norm before
        the next in one launch.  `y`, `extra`: [N, H], float32 or bfloat16 each."""
        _dev(hidden, "hidden", torch.float32)
        _dev(weight, "norm weight")
        _dev(next_weight, "next norm weight", weight.dtype)
        N, H = hidden.shape
        _need(weight.shape == (H,) and next_weight.shape == (H,), f"norm weights must be [{H}]")
        for t, name in ((y, "y"), (extra, "extra")):
            if t is not None:
                _dev(t, name)
                _need(t.shape == hidden.shape, f"{name} must have the shape of hidden")
        out = _made((N, H), dtype=out_dtype, device=hidden.device)
        self._run("norm", "lle_rmsnorm_add_rmsnorm", "PPIPIPPIPIIFFIP",
                  _ptr(hidden), _ptr(y), dtype_code(y.dtype), _ptr(extra), dtype_code(extra.dtype) if extra is not None else 0,
                  _ptr(weight), _ptr(next_weight), dtype_code(weight.dtype), _ptr(out), N, H, float(eps), float(next_eps),
                  dtype_code(out_dtype))
        return out

    # -- attention behind a short convolution --------------------------------------------------------
    def conv_norm_rope_write(self, u, taps, state, token_seq, cu_tokens, seq_slots, slots, q_weight, k_weight, cos_sin,
                             rotary_dim: int, eps: float, kv_layer, num_q_heads: int, num_kv_heads: int, dim: int,
                             vdim: int, write_kv: bool = True) -> torch.Tensor:
        """A row of u holds q [nq dim], k [nkv dim], v [nkv vdim] of one token.  Every channel is convolved over
        time with its J taps (float32 [cols, J]; the last tap meets the token itself), reading the rows of the
        same request ahead of it in this step and, before those, the request's state row (float32
        [slots + 1, (J - 1) cols], the last J - 1 rows of u that earlier steps brought, oldest first; None for
        J = 1).  Then every head of q and k is divided by its root mean square times q_weight / k_weight
        (float32 [dim], one for all heads), the first `rotary_dim` elements of every head are rotated (half-split)
        by cos_sin [N, rotary_dim / 2, 2].  Returns q [N, nq, D], D = kv_layer.shape[4] >= max(dim, vdim), zeros
        past dim; K and V^T go to the pages at `slots` with zeros past dim and vdim.  The state is left as it
        is: conv_state_update advances it."""
        _dev(u, "u")
        _dev(taps, "taps", torch.float32)
        _dev(slots, "slots", torch.int32)
        _dev(kv_layer, "kv_layer", u.dtype)
        for t, name in ((token_seq, "token_seq"), (cu_tokens, "cu_tokens"), (seq_slots, "seq_slots")):
            _dev(t, name, torch.int32)
        nq, nkv = num_q_heads, num_kv_heads
        N, cols = u.shape
        J = taps.shape[1]
        S = seq_slots.shape[0]
        _need(cols == (nq + nkv) * dim + nkv * vdim, "a row of u holds q, k and v")
        _need(taps.shape == (cols, J) and J >= 1, "taps must be [cols, J]")
        _need(slots.shape == (N,) and token_seq.shape == (N,) and cu_tokens.shape == (S + 1,), "slots, token_seq [N]; cu_tokens [S + 1]")
        _need(kv_layer.dim() == 5 and kv_layer.shape[1] == 2 and kv_layer.shape[2] == nkv, "kv_layer must be [pages, 2, nkv, page_size, D]")
        D, page_size = kv_layer.shape[4], kv_layer.shape[3]
        _need(D >= max(dim, vdim), "the cache's heads are smaller than the model's")
        _need(0 <= rotary_dim <= dim and rotary_dim % 2 == 0, "rotary_dim must be even and <= dim")
        if J > 1:
            _need(state is not None, "a convolution of several taps needs the requests' state rows")
            _rows(state, "state", torch.float32)
            _need(state.shape[1] >= (J - 1) * cols, "a state row holds J - 1 rows of u")
        _dev(q_weight, "q norm weight", torch.float32)
        _dev(k_weight, "k norm weight", torch.float32)
        _need(q_weight.shape == (dim,) and k_weight.shape == (dim,), f"the heads' norm weights must be [{dim}]")
        if rotary_dim > 0:
            _dev(cos_sin, "cos_sin", torch.float32)
            _need(cos_sin.shape == (N, rotary_dim // 2, 2), "cos_sin must be [N, rotary_dim / 2, 2]")
        q_out = _made((N, nq, D), dtype=u.dtype, device=u.device)
        self._run("rope_kv", "lle_conv_norm_rope_write",
                  "PIPIPLPPPPPPPIFPPIIIIIIILIIP",
                  _ptr(u), cols, _ptr(taps), J, _ptr(state) if J > 1 else None, state.stride(0) if J > 1 else 0,
                  _ptr(token_seq), _ptr(cu_tokens), _ptr(seq_slots), _ptr(slots), _ptr(q_weight), _ptr(k_weight),
                  _ptr(cos_sin) if rotary_dim > 0 else None, rotary_dim, float(eps), _ptr(q_out), _ptr(kv_layer), N, nq, nkv,
                  dim, vdim, D, page_size, kv_layer.stride(0), 1 if write_kv else 0, dtype_code(u.dtype))
        return q_out

    def conv_state_update(self, u, state, kept: int, cu_tokens, seq_slots) -> None:
        """state row of every request of the step <- the last `kept` rows of (the `kept` rows it held, then the
        request's rows of u in this step); state float32 [slots + 1, >= kept * cols], u [N, cols]."""
        _dev(u, "u")
        _rows(state, "state", torch.float32)
        _dev(cu_tokens, "cu_tokens", torch.int32)
        _dev(seq_slots, "seq_slots", torch.int32)
        N, cols = u.shape
        S = seq_slots.shape[0]
        _need(kept > 0 and state.shape[1] >= kept * cols and cu_tokens.shape == (S + 1,), "a state row holds `kept` rows of u")
        self._run("rope_kv", "lle_conv_state_update", "PIPLIPPIIP", _ptr(u), cols, _ptr(state),
                  state.stride(0), int(kept), _ptr(cu_tokens), _ptr(seq_slots), S, dtype_code(u.dtype))

    # -- the gated delta rule --------------------------------------------------------------
    DELTA_MAX_DIM = MAX_DELTA_HEAD_DIM
    DELTA_MAX_ADVANCE = 8  # (lle_delta_conv_max_advance)

    def delta_conv(self, u, taps, state, token_seq, cu_tokens, seq_slots, kv_heads: int, dim: int, heads: int, vdim: int,
                   unit_eps: float, q_scale: float, advance: bool = False):
        """A row of u holds q [G dim], k [G dim], v [H vdim] of one token (G = kv_heads, H = heads).  Every channel is
        convolved over time with its J taps (float32 [cols, J]; the last tap meets the token itself), reading the
        rows of the same request ahead of it in this step and, before those, the request's state row (float32
        [slots + 1, >= (J - 1) cols], the last J - 1 rows of u that earlier steps brought, oldest first; None for
        J = 1), then passes silu; every head of q and k becomes x / sqrt(sum x^2 + unit_eps), q times q_scale.
        Returns float32 q [N, G dim], k [N, G dim], v [N, H vdim].  The state is left as it is (conv_state_update
        advances it), or with `advance` moves on in the same launch (see can_advance_conv)."""
        _dev(u, "u")
        _dev(taps, "taps", torch.float32)
        for t, name in ((token_seq, "token_seq"), (cu_tokens, "cu_tokens"), (seq_slots, "seq_slots")):
            _dev(t, name, torch.int32)
        N, cols = u.shape
        J = taps.shape[1]
        S = seq_slots.shape[0]
        G, H = int(kv_heads), int(heads)
        _need(cols == 2 * G * dim + H * vdim, "a row of u holds q, k and v")
        _need(taps.shape == (cols, J) and J >= 1, "taps must be [cols, J]")
        _need(token_seq.shape == (N,) and cu_tokens.shape == (S + 1,), "token_seq [N]; cu_tokens [S + 1]")
        _need(0 < dim <= self.DELTA_MAX_DIM and 0 < vdim <= self.DELTA_MAX_DIM,
              f"a head of the delta rule holds at most {self.DELTA_MAX_DIM} channels")
        if J > 1:
            _need(state is not None, "a convolution of several taps needs the requests' state rows")
            _rows(state, "state", torch.float32)
            _need(state.shape[1] >= (J - 1) * cols, "a state row holds J - 1 rows of u")
        q = _made((N, G * dim), dtype=torch.float32, device=u.device)
        k = _made((N, G * dim), dtype=torch.float32, device=u.device)
        v = _made((N, H * vdim), dtype=torch.float32, device=u.device)
        _need(not advance or (1 < J <= self.DELTA_MAX_ADVANCE and N == S), "the state moves on in this launch for single tokens")
        self._run("delta", "lle_delta_conv", "PIPIPLPPPPPPIIIIIFFIIP",
                  _ptr(u), cols, _ptr(taps), J, _ptr(state) if J > 1 else None, state.stride(0) if J > 1 else 0,
                  _ptr(token_seq), _ptr(cu_tokens), _ptr(seq_slots), _ptr(q), _ptr(k), _ptr(v), N, G, dim, H, vdim,
                  float(unit_eps), float(q_scale), int(advance), dtype_code(u.dtype))
        return q, k, v

    def can_advance_conv(self, taps: int, max_q_len: int) -> bool:
        """Whether delta_conv can move the kept rows on itself: a step of single tokens, few taps."""
        return max_q_len == 1 and 1 < taps <= self.DELTA_MAX_ADVANCE

    def low_rank_gates(self, low, a_col: int, a2, a_log, dt_bias, dim: int, g_col: int = 0, g2=None):
        """low float32 [N, cols], a2 float32 [CA, RA], a_log float32 [CA / dim], dt_bias float32 [CA] ->
        decay float32 [N, CA]: exp(-exp(a_log[c // dim]) softplus(low[:, a_col : a_col + RA] @ a2[c] + dt_bias[c])); and with
        g2 [CG, RG] gate float32 [N, CG] = low[:, g_col : g_col + RG] @ g2^T (else None).  RA and RG are multiples of 16 (pad
        weights and columns with zeros), columns start at multiples of 4."""
        for t, name in ((low, "low"), (a2, "a2"), (a_log, "a_log"), (dt_bias, "dt_bias")):
            _dev(t, name, torch.float32)
        N, cols = low.shape
        CA, RA = a2.shape
        CG, RG = (0, 0) if g2 is None else g2.shape
        if g2 is not None:
            _dev(g2, "g2", torch.float32)
        _need(CA % dim == 0 and a_log.shape == (CA // dim,) and dt_bias.shape == (CA,), "a2 [heads * dim, R], a_log [heads], dt_bias [heads * dim]")
        _need(RA % 16 == 0 and RG % 16 == 0 and cols % 4 == 0 and a_col % 4 == 0 and g_col % 4 == 0, "ranks are multiples of 16, columns start at multiples of 4")
        _need(0 <= a_col and a_col + RA <= cols and 0 <= g_col and g_col + RG <= cols, "low has too few columns")
        decay = _made((N, CA), dtype=torch.float32, device=low.device)
        gate = _made((N, CG), dtype=torch.float32, device=low.device) if g2 is not None else None
        self._run("delta", "lle_low_rank_gates", "PIIIPIIPIIPPIPPIP",
                  _ptr(low), cols, int(a_col), int(g_col), _ptr(a2), RA, CA, _ptr(g2), RG, CG, _ptr(a_log), _ptr(dt_bias), int(dim),
                  _ptr(decay), _ptr(gate), N)
        return decay, gate

    DELTA_GATES_AHEAD = 64  # tokens of a step from which decays and betas are made by a launch of their own

    # Long requests of heads of 64 or 128 key channels go in chunks where their workgroups (one for a head and sixteen value channels) are no
    # more than the CUs: the walk's wavefronts, which share their SIMDs with one another well, are as fast or faster from there on (32
    # heads of 64 x 64, chunks / walk in us: one request of 128, 256, 2048 tokens 15 / 17, 24 / 29, 88 / 209; two of 192, 1024 23 / 23,
    # 64 / 108; four of 256, 1024 41 / 38, 134 / 129; 32 heads of 128 x 128: one of 128, 192, 2048 25 / 25, 29 / 33, 162 / 291; two of 512
    # 95 / 96, four 194 / 175).  A request's sums run in another order in chunks than walked: its last bits follow from how its prompt is cut and from how
    # many long requests stand beside it; single tokens are always walked.
    DELTA_WALK = 160  # most tokens of a request that are always walked
    DELTA_CHUNK_FLOATS = 1 << 28  # of what the chunks of a step keep, 1 GiB (30000 tokens of 32 heads of 64 x 64); steps of more tokens are walked

    def delta_scan(self, q, k, v, ba, a_log, dt_bias, state, heads: int, kv_heads: int, dim: int, vdim: int, seq_slots,
                   cu_tokens, decay=None) -> torch.Tensor:
        """Per head h, with the matrix state S [dim, vdim] of the request (float32; `state[slot]` holds the heads'
        states transposed, [heads][vdim][dim]) and the q, k of head h // (heads // kv_heads), token by token:
            beta = sigmoid(ba[t, h]);  g = exp(-exp(a_log[h]) softplus(ba[t, heads + h] + dt_bias[h]))
            S <- g S;  w = beta (v_t - S^T k_t);  S <- S + k_t w^T;  o_t = S^T q_t
        q, k float32 [N, kv_heads dim]; v float32 [N, heads vdim]; ba float32 [N, 2 heads]; a_log, dt_bias float32
        [heads].  With `decay` (float32 [N, heads dim], one of every key channel) S <- diag(decay_t) S instead; ba
        [N, >= heads] then begins with beta's inputs, and a_log and dt_bias are not used (None).
        Returns o float32 [N, heads vdim]; the states are advanced in place."""
        for t, name in ((q, "q"), (k, "k"), (v, "v"), (ba, "ba")) + (((a_log, "a_log"), (dt_bias, "dt_bias")) if decay is None
                                                                      else ((decay, "decay"),)):
            _dev(t, name, torch.float32)
        _rows(state, "state", torch.float32)
        _dev(seq_slots, "seq_slots", torch.int32)
        _dev(cu_tokens, "cu_tokens", torch.int32)
        N = v.shape[0]
        S = seq_slots.shape[0]
        H, G = int(heads), int(kv_heads)
        _need(G > 0 and H % G == 0, "the value heads are a multiple of the query/key heads")
        _need(0 < dim <= self.DELTA_MAX_DIM, f"a head of the delta rule holds at most {self.DELTA_MAX_DIM} key channels")
        _need(q.shape == (N, G * dim) and k.shape == (N, G * dim) and v.shape == (N, H * vdim),
              "q, k [N, kv_heads dim]; v [N, heads vdim]")
        if decay is None:
            _need(ba.shape == (N, 2 * H), "ba must be [N, 2 heads]")
            _need(a_log.shape == (H,) and dt_bias.shape == (H,), "a_log and dt_bias must be [heads]")
        else:
            _need(ba.dim() == 2 and ba.shape[0] == N and ba.shape[1] >= H and decay.shape == (N, H * dim),
                  "ba [N, >= heads]; decay [N, heads dim]")
        _need(state.shape[1] >= H * vdim * dim, "a state row holds heads * vdim * dim floats")
        _need(cu_tokens.shape == (S + 1,), "cu_tokens must be [S + 1]")
        out = _made((N, H * vdim), dtype=torch.float32, device=v.device)
        # steps with portions: the exponentials of decay and beta leave the walk (a step of single tokens keeps them there:
        # one launch less).  The number of tokens is known on the host and fixed inside a graph.
        args = (_ptr(q), _ptr(k), _ptr(v), _ptr(ba), ba.shape[1], _ptr(decay), _ptr(a_log), _ptr(dt_bias), _ptr(state), state.stride(0),
                _ptr(seq_slots), _ptr(cu_tokens), _ptr(out), S, H, G, dim, vdim)
        types = "PPPPIPPPPLPPPIIIII"
        few = 0  # requests that may go in chunks
        if N - S + 1 > self.DELTA_WALK * (1 if S == 1 else 4):  # (so many tokens may be one request's)
            few = self.compute_units(v.device) // (H * -(-int(vdim) // 16))
            if S > few and N > S * self.DELTA_WALK:  # (about all of them are long)
                few = 0
            floats = self._get("delta", "lle_delta_chunk_floats", "IIIII")(N, S, H, dim, vdim) if few > 0 else 0
            if 0 < floats <= self.DELTA_CHUNK_FLOATS and not any(t is not None and t.data_ptr() % 16 for t in (q, k, decay)):
                work = _made((floats,), dtype=torch.float32, device=v.device)
                # (a single request goes in chunks whatever cu_tokens says it has of the N tokens: nothing else is launched for it)
                self._run("delta", "lle_delta_chunks", types + "IIIPP", *args, N, self.DELTA_WALK if S > 1 else 0, few, _ptr(work))
                if S == 1:
                    return out
            else:
                few = 0
        gates = _made((N, 2 * H), dtype=torch.float32, device=v.device) if decay is None and N >= max(self.DELTA_GATES_AHEAD, 2 * S) else None
        self._run("delta", "lle_delta_scan", types + "PIIIP", *args, _ptr(gates), N, self.DELTA_WALK, few)
        return out

    def delta_out_norm(self, o, gate, norm_w, eps: float, heads: int, vdim: int, act: str = "silu", out_dtype=None) -> torch.Tensor:
        """o float32 [N, heads vdim], gate [N, heads vdim] in the activation type (or float32, with `out_dtype` saying
        the activation type) -> every head of o divided by its root mean square (eps inside the root) times norm_w [vdim]
        times act(gate), act silu or sigmoid."""
        _dev(o, "o", torch.float32)
        _dev(gate, "gate")
        _dev(norm_w, "norm weight")
        _need(act in ("silu", "sigmoid"), f"a gate's activation is silu or sigmoid, not {act!r}")
        N = o.shape[0]
        _need(o.shape == (N, heads * vdim) and gate.shape == o.shape and norm_w.shape == (vdim,),
              "o and gate [N, heads vdim]; norm weight [vdim]")
        out = _made(o.shape, dtype=out_dtype or gate.dtype, device=o.device)
        _need(gate.dtype in (torch.float32, out.dtype), "the gate is float32 or of the result's type")
        self._run("delta", "lle_delta_out_norm", "PPIIPIFPIIIIP", _ptr(o), _ptr(gate),
                  dtype_code(gate.dtype), 1 if act == "sigmoid" else 0, _ptr(norm_w), dtype_code(norm_w.dtype), float(eps),
                  _ptr(out), N, int(heads), int(vdim), dtype_code(out.dtype))
        return out

    # -- the state-space recurrence of Mamba-2 ----------------------------------------------------
    SSD_MAX_DIM = MAX_SSD_DIM
    SSD_CHUNK = 64  # tokens of a chunk (lle_ssd_chunk)
    SSD_WALK = 32  # most tokens of a request that are walked one by one (lle_ssd_walk)

    def ssd_conv(self, u, col0: int, taps, bias, state, token_seq, cu_tokens, seq_slots, single: bool = False, x=None,
                 dt_w=None):
        """The columns col0 .. col0 + C - 1 of u [N, cols] convolved over time channel by channel with J taps (float32
        [C, J]; the last tap meets the token itself) + bias (float32 [C] or None), then silu -> float32 [N, C].  Tokens
        ahead of the step come from the request's state row (float32 [slots + 1, >= (J - 1) C]: the last J - 1 inputs of
        earlier steps, oldest first; None for J = 1), which moves on by the step's tokens.  `single`: every request of the
        step has one token (the row then moves on in the same launch).  With x [N, K] and dt_w [H, K] the result is (that,
        x dt_w^T float32 [N, H]): in the same launch for single tokens and up to 8 taps, else a product of its own."""
        if x is not None and not (single and taps.shape[1] <= 8):
            return self.ssd_conv(u, col0, taps, bias, state, token_seq, cu_tokens, seq_slots, single), self.linear(x, dt_w, torch.float32)
        _dev(u, "u")
        _dev(taps, "taps", torch.float32)
        for t, name in ((token_seq, "token_seq"), (cu_tokens, "cu_tokens"), (seq_slots, "seq_slots")):
            _dev(t, name, torch.int32)
        N, cols = u.shape
        C, J = taps.shape
        S = seq_slots.shape[0]
        _need(0 <= col0 and col0 + C <= cols and J >= 1, "u has too few columns")
        _need(token_seq.shape == (N,) and cu_tokens.shape == (S + 1,), "token_seq [N]; cu_tokens [S + 1]")
        if bias is not None:
            _dev(bias, "bias", torch.float32)
            _need(bias.shape == (C,), "the convolution's bias must be [C]")
        if J > 1:
            _need(state is not None, "a convolution of several taps needs the requests' state rows")
            _rows(state, "state", torch.float32)
            _need(state.shape[1] >= (J - 1) * C, "a state row holds J - 1 inputs")
        out = _made((N, C), dtype=torch.float32, device=u.device)
        dt, K, H = None, 0, 0
        if x is not None:
            _dev(x, "x", u.dtype)
            _dev(dt_w, "dt_w", u.dtype)
            K, H = x.shape[1], dt_w.shape[0]
            _need(x.shape[0] == N and dt_w.shape == (H, K), "x must be [N, K], dt_w [H, K]")
            dt = _made((N, H), dtype=torch.float32, device=u.device)
        self._run("ssd", "lle_ssd_conv",
                  "PIIPIPPLPPPPIIIIPPPIIIP",
                  _ptr(u), cols, int(col0), _ptr(taps), J, _ptr(bias), _ptr(state) if J > 1 else None,
                  state.stride(0) if J > 1 else 0, _ptr(token_seq), _ptr(cu_tokens), _ptr(seq_slots), _ptr(out), N, S, C,
                  1 if single else 0, _ptr(x), _ptr(dt_w), _ptr(dt), K, H, dtype_code(u.dtype))
        return out if x is None else (out, dt)

    def ssd_heads_a_group(self, heads: int, groups: int, chunks: int) -> int:
        """Heads of a group that one workgroup of the chunks' second pass takes (they share C . B): as many as leave
        two workgroups for every CU."""
        most, share = max(1, heads * chunks // (2 * self.compute_units())), heads // groups
        return max(k for k in range(1, share + 1) if share % k == 0 and (k <= most or k == 1))

    def ssd_streams(self, num_tokens: int, heads: int, vdim: int, n: int, longest: int) -> bool:
        """Whether the chunks of long requests go one after the other, the state in registers (ssd_stream_kernel): up to 512 tokens, and beyond
        where the long requests' workgroups (a head and sixteen value channels each) are as many as the CUs.  With fewer the chain of the chunks
        is what takes the time: 32 heads of 64 x 128, chunks side by side / one after the other, one request of 256, 512, 1024, 2048 tokens
        34 / 24, 39 / 36, 54 / 59, 76 / 101 us; two of 1024 77 / 64; 64 heads, one request of 1024, 2048, 4096 tokens 76 / 63, 120 / 107, 224 / 189.
        Where those workgroups are fewer than 128 the chunks side by side catch up earlier, the more so the smaller a head (one request of 256, 320, 448, 512
        tokens, side by side / one after the other: 4 heads of 16 23 / 23, 23 / 25, 23 / 30, 23 / 33; 32 of 32 in 16 groups 27 / 29, 29 / 33, 30 / 39, 30 / 41;
        8 of 64 30 / 23, 30 / 26, 31 / 31, 32 / 34; 64 of 16 25 / 23, 30 / 26, 31 / 31, 31 / 34).  Heads that share no group read four times as much and gain
        less: 64 heads of 64 in 64 groups, four requests of 256, 512 tokens 109 / 101, 194 / 204.
        Requests of 32768 tokens and more have not been measured and stay as they were."""
        workgroups = max(1, num_tokens // max(1, longest)) * heads * (vdim // 16)  # (of as many long requests as there can be)
        few = 512 if workgroups >= 128 else 448 if vdim >= 64 else 256
        return n == 128 and vdim % 16 == 0 and longest < 1 << 15 and (longest <= few or workgroups >= self.compute_units())

    def ssd_scan(self, c, dt_in, dt_bias, a_log, D, state, heads: int, groups: int, vdim: int, n: int, seq_slots, cu_tokens,
                 min_q_len: int = 0, max_q_len: int = 0) -> torch.Tensor:
        """Per head h, with the matrix state S [n, vdim] of the request (float32; `state[slot]` begins with the heads'
        states transposed, [heads][vdim][n]) and the B, C of group h // (heads // groups), token by token:
            dt = softplus(dt_in[t, h] + dt_bias[h]);  S <- exp(-exp(a_log[h]) dt) S + dt B_t x_t^T;  y_t = S^T C_t + D[h] x_t
        A row of c (float32) holds x [heads vdim], B [groups n], C [groups n]; dt_in float32 [N, >= heads].  Returns y float32
        [N, heads vdim]; the states are advanced in place.  `min_q_len` and `max_q_len` are host-side bounds of the
        requests' tokens in this step (0: not known); they choose kernels, never results."""
        for t, name in ((c, "c"), (dt_in, "dt_in"), (dt_bias, "dt_bias"), (a_log, "a_log"), (D, "D")):
            _dev(t, name, torch.float32)
        _rows(state, "state", torch.float32)
        _dev(seq_slots, "seq_slots", torch.int32)
        _dev(cu_tokens, "cu_tokens", torch.int32)
        N, CC = c.shape
        S = seq_slots.shape[0]
        H, G = int(heads), int(groups)
        _need(G > 0 and H % G == 0, "the heads are a multiple of the groups")
        _need(0 < vdim <= self.SSD_MAX_DIM and 0 < n <= self.SSD_MAX_DIM, f"a head of the recurrence holds at most {self.SSD_MAX_DIM} channels")
        _need(CC == H * vdim + 2 * G * n, "a row of c holds x, B and C")
        _need(dt_in.dim() == 2 and dt_in.shape[0] == N and dt_in.shape[1] >= H, "dt_in must be [N, >= heads]")
        _need(dt_bias.shape == (H,) and a_log.shape == (H,) and D.shape == (H,), "dt_bias, a_log and D must be [heads]")
        _need(state.shape[1] >= H * vdim * n and cu_tokens.shape == (S + 1,), "a state row holds heads * vdim * n floats")
        longest = min(max_q_len or N, N)
        pieces = -(-longest // self.SSD_CHUNK) if longest > self.SSD_WALK else 0
        y = _made((N, H * vdim), dtype=torch.float32, device=c.device)
        part = part_decay = None
        together, stream_floats = 1, 0
        if pieces:
            slots = N // self.SSD_CHUNK + S
            # (a chunk's bytes of c are counted in 32 bits there)
            if S <= 65535 and CC < 1 << 23 and self.ssd_streams(N, H, int(vdim), int(n), longest) and (c.data_ptr() | y.data_ptr()) % 16 == 0:
                stream_floats = self._get("ssd", "lle_ssd_stream_floats", "IIII", _L)(N, S, H, G)
                part = _made((stream_floats,), dtype=torch.float32, device=c.device)
            else:
                part = _made((slots * H * vdim * n,), dtype=torch.float32, device=c.device)
                part_decay = _made((slots * H,), dtype=torch.float32, device=c.device)
                together = self.ssd_heads_a_group(H, G, -(-N // self.SSD_CHUNK))
        self._run("ssd", "lle_ssd_scan",
                  "PIPIPPPPLPPPIIIIIIIIPPILP",
                  _ptr(c), CC, _ptr(dt_in), dt_in.shape[1], _ptr(dt_bias), _ptr(a_log), _ptr(D), _ptr(state), state.stride(0),
                  _ptr(seq_slots), _ptr(cu_tokens), _ptr(y), S, H, G, int(vdim), int(n),
                  1 if (min_q_len or 1) <= self.SSD_WALK else 0, pieces, together, _ptr(part), _ptr(part_decay), N, stream_floats)
        return y

    def ssd_gate_norm(self, y, u, z_col: int, norm_w, eps: float, groups: int) -> torch.Tensor:
        """y float32 [N, inner], z = u[:, z_col : z_col + inner] -> y * silu(z), every one of `groups` equal parts of a row
        divided by its own root mean square (eps inside the root), times norm_w (float32 [inner]), in u's type."""
        _dev(y, "y", torch.float32)
        _dev(u, "u")
        _dev(norm_w, "norm weight", torch.float32)
        N, inner = y.shape
        _need(u.shape[0] == N and 0 <= z_col and z_col + inner <= u.shape[1], "u has too few columns")
        _need(norm_w.shape == (inner,) and groups > 0 and inner % groups == 0, "the norm weight must be [inner], cut into equal parts")
        out = _made((N, inner), dtype=u.dtype, device=u.device)
        self._run("ssd", "lle_ssd_gate_norm", "PPIIPFPIIIIP", _ptr(y), _ptr(u), u.shape[1],
                  int(z_col), _ptr(norm_w), float(eps), _ptr(out), N, inner, int(groups), dtype_code(u.dtype))
        return out

    # -- picking tokens --------------------------------------------------------------
    def argmax(self, logits, scatter=None) -> torch.Tensor:
        """float32 [R, V] -> int32 [R], first maximum wins.  `scatter` = (dst int32, index int32 [R]):
        the pick of row r is also written to dst[index[r]] (the host has made sure that index is in range)."""
        _dev(logits, "logits", torch.float32)
        R, V = logits.shape
        out = _made((R,), dtype=torch.int32, device=logits.device)
        chunks = max(1, min(64, V // 2048))  # enough workgroups to stream a long row from all CUs
        part_val = _made((R * chunks,), dtype=torch.float32, device=logits.device)
        part_idx = _made((R * chunks,), dtype=torch.int32, device=logits.device)
        dst = index = None
        if scatter is not None:
            dst, index = scatter
            _dev(dst, "scatter destination", torch.int32)
            _dev(index, "scatter index", torch.int32)
            _need(index.shape == (R,), "one scatter index for every row")
        self._run("sampling", "lle_argmax_rows_scatter", "PPPPIIIPPP",
                  _ptr(logits), _ptr(out), _ptr(part_val), _ptr(part_idx), R, V, chunks, _ptr(dst), _ptr(index))
        return out

    def sample(self, logits, temperature, uniform) -> torch.Tensor:
        """float32 logits [R, V], temperature [R] (<= 0: greedy), uniform [R] in [0, 1) -> int32 [R]."""
        _dev(logits, "logits", torch.float32)
        _dev(temperature, "temperature", torch.float32)
        _dev(uniform, "uniform", torch.float32)
        R, V = logits.shape
        _need(temperature.shape == (R,) and uniform.shape == (R,), "temperature and uniform must be [R]")
        out = _made((R,), dtype=torch.int32, device=logits.device)
        self._run("sampling", "lle_sample_rows", "PPPPIIP",
                  _ptr(logits), _ptr(temperature), _ptr(uniform), _ptr(out), R, V)
        return out


    # -- measured peaks (the benchmark's rooflines) ---------------------------------------------
    def probe_read_stream(self, data: torch.Tensor, blocks: int) -> None:
        """Launch a kernel that only reads `data` (any type, a multiple of 16 bytes), `blocks` workgroups."""
        _dev(data, "data")
        nbytes = data.numel() * data.element_size()
        _need(nbytes % 16 == 0 and nbytes > 0, "the read probe takes a multiple of 16 bytes")
        self._run("probe", "lle_probe_read_stream", "PLIPP", _ptr(data), nbytes, int(blocks), None)

    def probe_mfma(self, dtype, blocks: int, iters: int) -> float:
        """Launch a kernel of nothing but matrix instructions on registers; returns its flops."""
        self._run("probe", "lle_probe_mfma", "IIIPP", dtype_code(dtype), int(blocks), int(iters), None)
        per_instruction = 2.0 * 16 * 16 * (32 if dtype == torch.bfloat16 else 4)
        return per_instruction * 16 * iters * 4 * blocks


_written = Written(HipOps, free=("record", "end_record", "replay"))  # (these launch nothing of a layer's own)
_default: Optional[HipOps] = None


def default_ops() -> HipOps:
    global _default
    if _default is None:
        _default = HipOps()
    return _default
