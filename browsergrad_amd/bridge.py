"""HipRealizerBridge: the reference bridge protocol over libbghip (HIP, gfx950).

Python twin of the TypeScript ``createHipRealizerBridge`` (browsergrad_amd/node).
It implements the structural ``WebGpuBridge`` Protocol of the reference
(packages/browsergrad-jit/src/python/_bridge.py:61-289) method for method, so
the reference's walker (``_realize_webgpu.realize_webgpu``) and this package's
walker (``browsergrad_amd.realize``) can drive it unchanged:

    upload / materialize / release         realizer.ts:1007-1041
    matmul                                 realizer.ts:1043-1060
    fused_elementwise                      realizer.ts:1062-1085
    cast                                   realizer.ts:1087-1120
    flash_attention                        realizer.ts:1122-1151
    run_tensor_plan[_resident][_semantic]  realizer.ts:1557-1652
    aliveHandleCount / resourceSnapshot / flushProfiles  realizer.ts:275-279

Differences from the reference bridge are additive: float16 / bfloat16 are
accepted where the reference only takes float32 (realizer.ts:310-317), and
the ``*_ex`` methods expose strided / fused variants used by the walker.
Handles are plain ints minted by the library (from 1, never reused).
"""
from __future__ import annotations

import ctypes as C
import json
from typing import Any, Dict, Optional, Sequence, Tuple

import numpy as np

from . import _native as N
from .errors import JitNotImplementedError, KernelError

_REF_OPCODES = ("ADD", "MUL", "DIV", "NEG", "EXP", "LOG")  # fused_elementwise.ts:83-90


def _dtype_code(dtype: str, op: str) -> int:
    code = N.DTYPE_CODES.get(str(dtype))
    if code is None:
        raise KernelError(f"HIP bridge: {op} does not know dtype {dtype!r}")
    return code


def _shape(shape: Sequence[int]) -> Tuple[int, ...]:
    return tuple(int(d) for d in shape)


class HipRealizerBridge:
    """One HIP context (device + stream).  Not thread-shared (realizer.ts:894-897)."""

    def __init__(self, device: int = 0, profiling: bool = False) -> None:
        self._lib = N.load_library()
        ctx = N.ctx_p()
        rc = self._lib.bg_ctx_create(int(device), 1 if profiling else 0, C.byref(ctx))
        if rc != N.BG_OK or not ctx.value:
            raise KernelError(
                f"HIP bridge: cannot open HIP device {device} (status {rc}); "
                f"the HIP realizer has no CPU fallback",
                rc,
            )
        self._ctx = ctx
        self.device = device
        self.profiling = profiling
        self.counters = {"upload": 0, "materialize": 0, "release": 0, "matmul": 0}
        self._semantic_traces: dict = {}
        self._fused_descs: dict = {}

    # -- lifecycle -----------------------------------------------------------
    def close(self) -> None:
        if getattr(self, "_ctx", None) and self._ctx.value:
            self._lib.bg_ctx_destroy(self._ctx)
            self._ctx = N.ctx_p()

    def __del__(self) -> None:  # pragma: no cover - interpreter shutdown order
        try:
            self.close()
        except Exception:
            pass

    def __enter__(self) -> "HipRealizerBridge":
        return self

    def __exit__(self, *exc: Any) -> None:
        self.close()

    def _check(self, rc: int) -> None:
        if rc != N.BG_OK:
            msg = self._lib.bg_last_error(self._ctx)
            raise KernelError(msg.decode() if msg else f"HIP bridge error {rc}", rc)

    # -- buffer lifecycle (realizer.ts:1007-1041) -------------------------------
    def upload(self, data: Any, shape: Sequence[int], dtype: str) -> int:
        code = _dtype_code(dtype, "upload")
        if isinstance(data, np.ndarray):
            buf = np.ascontiguousarray(data)
            ptr, nbytes = buf.ctypes.data, buf.nbytes
            keep = buf
        else:
            keep = bytes(data) if not isinstance(data, (bytes, bytearray)) else data
            nbytes = len(keep)
            cbuf = C.create_string_buffer(keep, nbytes) if nbytes else None
            ptr = C.addressof(cbuf) if cbuf is not None else None
            keep = cbuf
        shp = _shape(shape)
        out = N.handle_t()
        self._check(self._lib.bg_upload(self._ctx, ptr, nbytes, N.i64_array(shp), len(shp), code,
                                        C.byref(out)))
        del keep
        self.counters["upload"] += 1
        return int(out.value)

    def upload_array(self, arr: np.ndarray) -> int:
        name = "bfloat16" if arr.dtype == np.uint16 and getattr(arr, "_bg_bf16", False) else arr.dtype.name
        return self.upload(arr, arr.shape, name)

    def materialize_into(self, handle: int, out: np.ndarray) -> np.ndarray:
        self._check(self._lib.bg_materialize(self._ctx, int(handle), out.ctypes.data, out.nbytes))
        self.counters["materialize"] += 1
        return out

    def materialize(self, handle: int, shape: Sequence[int], dtype: str) -> bytes:
        info = self.handle_info(handle)
        buf = (C.c_char * max(1, info["nbytes"]))()
        self._check(self._lib.bg_materialize(self._ctx, int(handle), buf, info["nbytes"]))
        self.counters["materialize"] += 1
        return bytes(buf)[: info["nbytes"]]

    def to_numpy(self, handle: int) -> np.ndarray:
        """Materialize a handle as an ndarray of its own shape and dtype
        (bfloat16 is returned as its uint16 bit pattern)."""
        info = self.handle_info(handle)
        np_dtype = {"bfloat16": np.uint16}.get(info["dtype"], info["dtype"])
        out = np.empty(info["shape"], dtype=np_dtype)
        return self.materialize_into(handle, out)

    def release(self, handle: Any) -> None:
        if handle is None:
            return
        self._check(self._lib.bg_release(self._ctx, int(handle)))
        self.counters["release"] += 1

    def handle_info(self, handle: int) -> dict:
        shp = (C.c_int64 * N.BG_MAX_RANK)()
        rank = C.c_int()
        dt = C.c_int()
        nb = C.c_int64()
        self._check(self._lib.bg_handle_info(self._ctx, int(handle), shp, C.byref(rank), C.byref(dt),
                                             C.byref(nb)))
        return {"shape": tuple(shp[i] for i in range(rank.value)), "dtype": N.DTYPE_NAMES[dt.value],
                "nbytes": int(nb.value)}

    # -- compute (realizer.ts:1043-1151) ------------------------------------------
    def matmul(self, a: int, b: int, m: int, k: int, n: int, dtype: str) -> int:
        self.counters["matmul"] += 1
        out = N.handle_t()
        self._check(self._lib.bg_matmul(self._ctx, int(a), int(b), int(m), int(k), int(n),
                                        _dtype_code(dtype, "matmul"), C.byref(out)))
        return int(out.value)

    def fused_elementwise(self, inputs: list, ops: list, shape: Sequence[int], dtype: str) -> int:
        for op in ops:
            name = op[0]
            if name not in _REF_OPCODES:
                raise KernelError(f"fused_elementwise: unsupported opcode {name!r}")
        arr = (N.FusedOp * max(1, len(ops)))(
            *[N.FusedOp(N.OPS[o[0]], int(o[1]), int(o[2]) if o[2] is not None else 0, 0) for o in ops])
        shp = _shape(shape)
        out = N.handle_t()
        self._check(self._lib.bg_fused_elementwise(
            self._ctx, N.handle_array(inputs), len(inputs), arr, len(ops), N.i64_array(shp), len(shp),
            _dtype_code(dtype, "fused_elementwise"), C.byref(out)))
        return int(out.value)

    def cast(self, handle: int, src_dtype: str, dst_dtype: str, shape: Sequence[int]) -> int:
        shp = _shape(shape)
        out = N.handle_t()
        self._check(self._lib.bg_cast(self._ctx, int(handle), _dtype_code(src_dtype, "cast"),
                                      _dtype_code(dst_dtype, "cast"), N.i64_array(shp), len(shp),
                                      C.byref(out)))
        return int(out.value)

    def flash_attention(self, q: int, k: int, v: int, mask: Optional[int], b: int, h: int, sq: int,
                        sk: int, d: int, scale: float, dtype: str) -> int:
        out = N.handle_t()
        self._check(self._lib.bg_flash_attention(
            self._ctx, int(q), int(k), int(v), int(mask or 0), int(b), int(h), int(sq), int(sk), int(d),
            float(scale), _dtype_code(dtype, "flash_attention"), C.byref(out)))
        return int(out.value)

    # -- extensions --------------------------------------------------------------------
    def matmul_ex(self, a: int, b: int, *, m: int, n: int, k: int, batch: int = 1,
                  lda: Optional[int] = None, ldb: Optional[int] = None, ldc: Optional[int] = None,
                  stride_a: Optional[int] = None, stride_b: Optional[int] = None,
                  stride_c: Optional[int] = None, offset_a: int = 0, offset_b: int = 0,
                  trans_b: bool = False, in_dtype: str = "float32", out_dtype: Optional[str] = None,
                  bias: Optional[int] = None, round_out: bool = False, act: int = N.ACT_NONE,
                  residual: Optional[int] = None, a_dtype: Optional[str] = None,
                  b_dtype: Optional[str] = None, f32_unsplit: bool = False) -> int:
        """bg_matmul_ex; ``f32_unsplit`` forms every float32 product by a
        float32 matrix instruction (BG_MATMUL_F32_UNSPLIT); with ``residual``
        (f32 [batch, m, n] added after the epilogue) or ``a_dtype`` /
        ``b_dtype`` (the dtypes the operands are stored in, cast to
        ``in_dtype`` in a pre-pass) it calls bg_matmul_ex2."""
        d = N.MatmulDesc()
        d.a, d.b, d.bias = int(a), int(b), int(bias or 0)
        d.batch, d.m, d.n, d.k = int(batch), int(m), int(n), int(k)
        d.lda = int(lda if lda is not None else k)
        d.ldb = int(ldb if ldb is not None else (k if trans_b else n))
        d.ldc = int(ldc if ldc is not None else n)
        d.stride_a = int(stride_a if stride_a is not None else m * d.lda)
        d.stride_b = int(stride_b if stride_b is not None else (n if trans_b else k) * d.ldb)
        d.stride_c = int(stride_c if stride_c is not None else m * d.ldc)
        d.offset_a, d.offset_b = int(offset_a), int(offset_b)
        d.trans_b = 1 if trans_b else 0
        d.in_dtype = _dtype_code(in_dtype, "matmul")
        d.out_dtype = _dtype_code(out_dtype or in_dtype, "matmul")
        d.round_f16 = 1 if round_out else 0
        d.act = int(act)
        if f32_unsplit:  # (a field's store is about 0.1 us of a call's 5)
            d.reserved = N.MATMUL_F32_UNSPLIT
        out = N.handle_t()
        if residual is None and a_dtype is None and b_dtype is None:
            self._check(self._lib.bg_matmul_ex(self._ctx, C.byref(d), C.byref(out)))
            return int(out.value)
        e = N.MatmulExt()
        e.residual = int(residual or 0)
        e.a_dtype = -1 if a_dtype is None else _dtype_code(a_dtype, "matmul")
        e.b_dtype = -1 if b_dtype is None else _dtype_code(b_dtype, "matmul")
        self._check(self._lib.bg_matmul_ex2(self._ctx, C.byref(d), C.byref(e), C.byref(out)))
        return int(out.value)

    def fused_ex(self, inputs: Sequence[int], ops: Sequence[Tuple[str, int, int, int]],
                 shape: Sequence[int], out_dtype: str, *, in_strides: Optional[Sequence[Sequence[int]]] = None,
                 imms: Sequence[float] = (), reduce: int = N.RED_NONE, keepdims: bool = False) -> int:
        # The ctypes descriptor depends only on the program's structure, so it
        # is built once per structure and reused with this call's handles
        # (building it costs ~20 us of Python, comparable to a whole
        # bandwidth-bound [4096, 4096] launch).
        key = (tuple(tuple(o) for o in ops), tuple(shape), out_dtype, tuple(imms), int(reduce),
               bool(keepdims), len(inputs),
               None if in_strides is None else tuple(tuple(s) for s in in_strides))
        entry = self._fused_descs.get(key)
        if entry is None:
            entry = self._fused_desc(len(inputs), ops, shape, out_dtype, in_strides, imms, reduce, keepdims)
            if len(self._fused_descs) >= 256:
                self._fused_descs.pop(next(iter(self._fused_descs)))
            self._fused_descs[key] = entry
        d, hs = entry[0], entry[1]
        for i, h in enumerate(inputs):
            hs[i] = int(h)
        out = N.handle_t()
        self._check(self._lib.bg_fused_ex(self._ctx, C.byref(d), C.byref(out)))
        return int(out.value)

    def _fused_desc(self, n_inputs: int, ops: Sequence[Tuple[str, int, int, int]], shape: Sequence[int],
                    out_dtype: str, in_strides: Optional[Sequence[Sequence[int]]], imms: Sequence[float],
                    reduce: int, keepdims: bool) -> tuple:
        """A bg_fused_desc for one program structure, with every array it
        points to (kept alive together in the returned tuple)."""
        shp = _shape(shape)
        d = N.FusedDesc()
        d.n_inputs = n_inputs
        hs = (N.handle_t * max(1, n_inputs))()
        d.inputs = C.cast(hs, C.POINTER(N.handle_t))
        sa = None
        if in_strides is not None:
            flat = [int(s) for st in in_strides for s in st]
            sa = N.i64_array(flat)
            d.in_strides = C.cast(sa, C.POINTER(C.c_int64))
        oparr = (N.FusedOp * max(1, len(ops)))(
            *[N.FusedOp(N.OPS[o[0]] if isinstance(o[0], str) else int(o[0]), int(o[1]), int(o[2]), int(o[3]))
              for o in ops])
        d.n_ops = len(ops)
        d.ops = C.cast(oparr, C.POINTER(N.FusedOp))
        imm_arr = (C.c_double * max(1, len(imms)))(*[float(x) for x in imms])
        d.n_imms = len(imms)
        d.imms = C.cast(imm_arr, C.POINTER(C.c_double))
        sarr = N.i64_array(shp)
        d.rank = len(shp)
        d.shape = C.cast(sarr, C.POINTER(C.c_int64))
        d.out_dtype = _dtype_code(out_dtype, "fused_elementwise")
        d.reduce_op = int(reduce)
        d.reduce_keepdims = 1 if keepdims else 0
        return (d, hs, sa, oparr, imm_arr, sarr)

    def attention_ex(self, q: int, k: int, v: int, *, batch: int, heads: int, sq: int, sk: int, d: int,
                     scale: float, causal: bool = False, in_dtype: str = "float16",
                     out_dtype: Optional[str] = None, round_scores: bool = False,
                     q_view: Tuple[int, int, int, int] = (0, 0, 0, 0),
                     k_view: Tuple[int, int, int, int] = (0, 0, 0, 0),
                     v_view: Tuple[int, int, int, int] = (0, 0, 0, 0),
                     o_strides: Tuple[int, int, int] = (0, 0, 0), tiled: bool = False) -> int:
        """q/k/v_view = (offset, batch stride, head stride, seq stride); zeros
        mean contiguous [B, H, S, D].  ``tiled``: the tiled kernels also for
        a few query rows, and float32 products by float32 matrix instructions
        (BG_ATTENTION_TILED)."""
        a = N.AttentionDesc()
        a.q, a.k, a.v = int(q), int(k), int(v)
        a.batch, a.heads, a.sq, a.sk, a.d = int(batch), int(heads), int(sq), int(sk), int(d)
        a.q_off, a.q_sb, a.q_sh, a.q_ss = (int(x) for x in q_view)
        a.k_off, a.k_sb, a.k_sh, a.k_ss = (int(x) for x in k_view)
        a.v_off, a.v_sb, a.v_sh, a.v_ss = (int(x) for x in v_view)
        a.o_sb, a.o_sh, a.o_ss = (int(x) for x in o_strides)
        a.scale = float(scale)
        a.causal = 1 if causal else 0
        a.in_dtype = _dtype_code(in_dtype, "flash_attention")
        a.out_dtype = _dtype_code(out_dtype or in_dtype, "flash_attention")
        a.round_scores = 1 if round_scores else 0
        if tiled:
            a.reserved = N.ATTENTION_TILED
        out = N.handle_t()
        self._check(self._lib.bg_attention_ex(self._ctx, C.byref(a), C.byref(out)))
        return int(out.value)

    def layer_norm(self, x: int, weight: int, bias: int, rows: int, cols: int, eps: float,
                   out_dtype: str = "float32") -> int:
        out = N.handle_t()
        self._check(self._lib.bg_layer_norm(self._ctx, int(x), int(weight), int(bias), int(rows), int(cols),
                                            float(eps), _dtype_code(out_dtype, "layer_norm"), C.byref(out)))
        return int(out.value)

    def layer_norm_backward_input(self, dy: int, x: int, weight: int, rows: int, cols: int,
                                  eps: float = 1e-5) -> int:
        """dX of LayerNorm (the plan op LAYER_NORM_BACKWARD_INPUT,
        tensor_plan.ts:2209-2255), f32 [rows, cols]."""
        out = N.handle_t()
        self._check(self._lib.bg_layer_norm_backward_input(self._ctx, int(dy), int(x), int(weight), int(rows),
                                                           int(cols), float(eps), C.byref(out)))
        return int(out.value)

    def layer_norm_backward_weight(self, dy: int, x: int, rows: int, cols: int, eps: float = 1e-5) -> int:
        """dW of LayerNorm (LAYER_NORM_BACKWARD_WEIGHT, tensor_plan.ts:2257-2295), f32 [cols]."""
        out = N.handle_t()
        self._check(self._lib.bg_layer_norm_backward_weight(self._ctx, int(dy), int(x), int(rows), int(cols),
                                                            float(eps), C.byref(out)))
        return int(out.value)

    def layer_norm_backward_bias(self, dy: int, rows: int, cols: int) -> int:
        """dB of LayerNorm (LAYER_NORM_BACKWARD_BIAS, tensor_plan.ts:2297-2321), f32 [cols]."""
        out = N.handle_t()
        self._check(self._lib.bg_layer_norm_backward_bias(self._ctx, int(dy), int(rows), int(cols),
                                                          C.byref(out)))
        return int(out.value)

    def optimizer_update(self, op: str, inputs: Sequence[int], n: int, *, lr: float = 0.0,
                         beta1: float = 0.9, beta2: float = 0.999, eps: float = 1e-8,
                         weight_decay: float = 0.0, step: int = 1) -> int:
        """One optimizer step over n f32 elements; `op` is the reference's plan
        op name (SGD_UPDATE, ADAMW_UPDATE_{M,V,PARAM}, ADAM_UPDATE_{M,V,PARAM};
        tensor_plan.ts:2000-2168) and `inputs` its input handles in the
        plan's order."""
        kind = N.OPTIM_KINDS.get(op)
        if kind is None:
            raise ValueError(f"optimizer_update: unknown op {op!r}")
        hs = (N.handle_t * max(len(inputs), 1))(*[int(h) for h in inputs])
        args = N.OptimArgs(float(lr), float(beta1), float(beta2), float(eps), float(weight_decay), int(step))
        out = N.handle_t()
        self._check(self._lib.bg_optimizer_update(self._ctx, kind, hs, len(inputs), C.byref(args), int(n),
                                                  C.byref(out)))
        return int(out.value)

    # -- convolutions (realizer.ts:114-238, 1153-1521) ------------------------------------
    def conv1d(self, input: int, weight: int, bias: Optional[int], n: int, cIn: int, lIn: int,  # noqa: N803
               cOut: int, k: int, stride: int, padding: int, dilation: int, groups: int, lOut: int,  # noqa: N803
               dtype: str = "float32") -> int:
        out = N.handle_t()
        self._check(self._lib.bg_conv1d(self._ctx, int(input), int(weight), int(bias or 0), n, cIn, lIn, cOut, k,
                                        stride, padding, dilation, groups, lOut, _dtype_code(dtype, "conv1d"),
                                        C.byref(out)))
        return int(out.value)

    def conv1d_backward_input(self, dy: int, weight: int, n: int, cIn: int, lIn: int, cOut: int,  # noqa: N803
                              k: int, stride: int, padding: int, dilation: int, groups: int, lOut: int,  # noqa: N803
                              dtype: str = "float32") -> int:
        out = N.handle_t()
        self._check(self._lib.bg_conv1d_backward_input(
            self._ctx, int(dy), int(weight), n, cIn, lIn, cOut, k, stride, padding, dilation, groups, lOut,
            _dtype_code(dtype, "conv1d_backward_input"), C.byref(out)))
        return int(out.value)

    def conv1d_backward_weight(self, dy: int, input: int, n: int, cIn: int, lIn: int, cOut: int,  # noqa: N803
                               k: int, stride: int, padding: int, dilation: int, groups: int, lOut: int,  # noqa: N803
                               dtype: str = "float32") -> int:
        out = N.handle_t()
        self._check(self._lib.bg_conv1d_backward_weight(
            self._ctx, int(dy), int(input), n, cIn, lIn, cOut, k, stride, padding, dilation, groups, lOut,
            _dtype_code(dtype, "conv1d_backward_weight"), C.byref(out)))
        return int(out.value)

    def conv1d_backward_bias(self, dy: int, n: int, cOut: int, lOut: int, dtype: str = "float32") -> int:  # noqa: N803
        out = N.handle_t()
        self._check(self._lib.bg_conv1d_backward_bias(self._ctx, int(dy), n, cOut, lOut,
                                                      _dtype_code(dtype, "conv1d_backward_bias"), C.byref(out)))
        return int(out.value)

    def conv2d(self, input: int, weight: int, bias: Optional[int], n: int, cIn: int, h: int, w: int,  # noqa: N803
               cOut: int, kh: int, kw: int, strideH: int, strideW: int, padH: int, padW: int,  # noqa: N803
               dilationH: int, dilationW: int, groups: int, outH: int, outW: int,  # noqa: N803
               dtype: str = "float32") -> int:
        out = N.handle_t()
        self._check(self._lib.bg_conv2d(self._ctx, int(input), int(weight), int(bias or 0), n, cIn, h, w, cOut, kh,
                                        kw, strideH, strideW, padH, padW, dilationH, dilationW, groups, outH, outW,
                                        _dtype_code(dtype, "conv2d"), C.byref(out)))
        return int(out.value)

    def conv2d_backward_input(self, dy: int, weight: int, n: int, cIn: int, h: int, w: int, cOut: int,  # noqa: N803
                              kh: int, kw: int, strideH: int, strideW: int, padH: int, padW: int,  # noqa: N803
                              dilationH: int, dilationW: int, groups: int, outH: int, outW: int,  # noqa: N803
                              dtype: str = "float32") -> int:
        out = N.handle_t()
        self._check(self._lib.bg_conv2d_backward_input(
            self._ctx, int(dy), int(weight), n, cIn, h, w, cOut, kh, kw, strideH, strideW, padH, padW, dilationH,
            dilationW, groups, outH, outW, _dtype_code(dtype, "conv2d_backward_input"), C.byref(out)))
        return int(out.value)

    def conv2d_backward_weight(self, dy: int, input: int, n: int, cIn: int, h: int, w: int, cOut: int,  # noqa: N803
                               kh: int, kw: int, strideH: int, strideW: int, padH: int, padW: int,  # noqa: N803
                               dilationH: int, dilationW: int, groups: int, outH: int, outW: int,  # noqa: N803
                               dtype: str = "float32") -> int:
        out = N.handle_t()
        self._check(self._lib.bg_conv2d_backward_weight(
            self._ctx, int(dy), int(input), n, cIn, h, w, cOut, kh, kw, strideH, strideW, padH, padW, dilationH,
            dilationW, groups, outH, outW, _dtype_code(dtype, "conv2d_backward_weight"), C.byref(out)))
        return int(out.value)

    def conv2d_backward_bias(self, dy: int, n: int, cOut: int, outH: int, outW: int,  # noqa: N803
                             dtype: str = "float32") -> int:
        out = N.handle_t()
        self._check(self._lib.bg_conv2d_backward_bias(self._ctx, int(dy), n, cOut, outH, outW,
                                                      _dtype_code(dtype, "conv2d_backward_bias"), C.byref(out)))
        return int(out.value)

    def conv_ex(self, op: str, a: int, b: int = 0, bias: int = 0, *, n: int, c_in: int, c_out: int,
                in_size: Sequence[int], out_size: Sequence[int], k: Sequence[int], stride: Sequence[int],
                pad: Sequence[int], dilation: Sequence[int], groups: int = 1, transposed: bool = False,
                output_pad: Optional[Sequence[int]] = None) -> int:
        """bg_conv_ex: `op` is forward / backward_input / backward_weight /
        backward_bias; spatial arrays have one entry per spatial dim."""
        r = len(in_size)
        d = N.ConvDesc()
        d.op = N.CONV_OPS[op]
        d.transposed = 1 if transposed else 0
        d.spatial = r
        d.n, d.c_in, d.c_out, d.groups = int(n), int(c_in), int(c_out), int(groups)
        for name, vals in (("in_", in_size), ("out", out_size), ("k", k), ("stride", stride), ("pad", pad),
                           ("dilation", dilation), ("output_pad", output_pad or [0] * r)):
            if len(vals) != r:
                raise ValueError(f"conv_ex: {name.strip('_')} needs {r} entries")
            arr = getattr(d, name)
            for i, v in enumerate(vals):
                arr[i] = int(v)
        d.a, d.b, d.bias = int(a), int(b or 0), int(bias or 0)
        out = N.handle_t()
        self._check(self._lib.bg_conv_ex(self._ctx, C.byref(d), C.byref(out)))
        return int(out.value)

    def copy_strided(self, src: int, offset: int, shape: Sequence[int], strides: Sequence[int]) -> int:
        shp = _shape(shape)
        out = N.handle_t()
        self._check(self._lib.bg_copy_strided(self._ctx, int(src), int(offset), N.i64_array(shp),
                                              N.i64_array(strides), len(shp), C.byref(out)))
        return int(out.value)

    def reshape(self, handle: int, shape: Sequence[int]) -> int:
        shp = _shape(shape)
        out = N.handle_t()
        self._check(self._lib.bg_reshape(self._ctx, int(handle), N.i64_array(shp), len(shp), C.byref(out)))
        return int(out.value)

    def reduce_last(self, x: int, rows: int, cols: int, op: int, keepdims: bool = False) -> int:
        out = N.handle_t()
        self._check(self._lib.bg_reduce_last(self._ctx, int(x), int(rows), int(cols), int(op),
                                             1 if keepdims else 0, C.byref(out)))
        return int(out.value)

    def softmax_last(self, x: int, rows: int, cols: int, out_dtype: str = "float32") -> int:
        out = N.handle_t()
        self._check(self._lib.bg_softmax_last(self._ctx, int(x), int(rows), int(cols),
                                              _dtype_code(out_dtype, "softmax"), C.byref(out)))
        return int(out.value)

    # -- tensor-plan route (realizer.ts:1557-1652) -------------------------------------
    def _plan_inputs(self, plan: dict, inputs: Sequence[Any]) -> Tuple[list, list, list]:
        """normalizeTensorPlanInputs (realizer.ts:857-892): each input is
        {value_id|valueId, data: bytes} (uploaded here, released after the
        run) or {value_id|valueId, handle} (resident, borrowed)."""
        steps = {int(st.get("value_id", st.get("valueId"))): st for st in plan.get("steps", [])}
        ids, handles, temps = [], [], []
        try:
            for i, inp in enumerate(inputs):
                if not isinstance(inp, dict):
                    raise KernelError(f"HIP bridge: tensor plan input {i} must be an object")
                raw_id = inp.get("valueId", inp.get("value_id"))
                if not isinstance(raw_id, (int, np.integer)) or isinstance(raw_id, bool):
                    raise KernelError(f"HIP bridge: tensor plan input {i}.valueId must be an integer")
                vid = int(raw_id)
                if inp.get("handle") is not None:
                    h = inp["handle"]
                    if not isinstance(h, (int, np.integer)) or isinstance(h, bool):
                        raise KernelError(f"HIP bridge: tensor plan input {i}.handle must be an integer")
                    ids.append(vid)
                    handles.append(int(h))
                    continue
                data = inp.get("data")
                if not isinstance(data, (bytes, bytearray, memoryview)):
                    raise KernelError(f"HIP bridge: tensor plan input {i}.data must be bytes")
                step = steps.get(vid)
                dtype = str(step["dtype"]) if step is not None else "float32"
                width = N.DTYPE_SIZES[_dtype_code(dtype, "tensor plan input")]
                nbytes = len(memoryview(data).cast("B"))
                if nbytes % width:
                    raise KernelError(
                        f"HIP bridge: tensor plan input {i}.data byte length must be divisible by {width}")
                shape = (nbytes // width,)
                if step is not None and int(np.prod(step["shape"], dtype=np.int64)) == nbytes // width:
                    shape = _shape(step["shape"])
                h = self.upload(data, shape, dtype)
                temps.append(h)
                ids.append(vid)
                handles.append(h)
        except BaseException:
            for h in temps:
                self.release(h)
            raise
        return ids, handles, temps

    @staticmethod
    def _plan_json(plan: Any) -> Tuple[dict, bytes]:
        """(parsed plan for input binding, wire text).  Text that does not
        parse here still goes to the library, whose reader reports it."""
        if isinstance(plan, (str, bytes)):
            text = plan.decode() if isinstance(plan, bytes) else plan
            try:
                obj = json.loads(text)
            except ValueError:
                obj = {}
            return (obj if isinstance(obj, dict) else {}), text.encode()
        return plan, json.dumps(plan, separators=(",", ":")).encode()

    def _run_plan(self, plan: Any, requests: Optional[Any], inputs: Sequence[Any], dtype: str,
                  resident: bool) -> Any:
        plan_obj, plan_text = self._plan_json(plan)
        if requests is None:
            req_text = None
        elif isinstance(requests, bytes):
            req_text = requests
        elif isinstance(requests, str):
            req_text = requests.encode()
        else:
            req_text = json.dumps(requests).encode()
        code = _dtype_code(dtype, "run_tensor_plan")
        ids, handles, temps = self._plan_inputs(plan_obj, inputs)
        try:
            root = N.handle_t()
            if resident or "steps" not in plan_obj:
                dst, nbytes = None, 0
            else:
                root_id = plan_obj.get("root_id", plan_obj.get("rootId"))
                root_step = next((st for st in plan_obj["steps"]
                                  if st.get("value_id", st.get("valueId")) == root_id), None)
                if root_step is None:  # malformed plan: let the library name the problem
                    raise KernelError(f"HIP bridge: tensor plan root {root_id} missing from steps")
                shape = _shape(root_step["shape"])
                n = int(np.prod(shape, dtype=np.int64)) if shape else 1
                nbytes = n * N.DTYPE_SIZES[_dtype_code(root_step["dtype"], "run_tensor_plan")]
                buf = C.create_string_buffer(max(nbytes, 1))
                dst = C.cast(buf, C.c_void_p)
            args = (N.i64_array(ids), N.handle_array(handles), len(ids), code, dst, nbytes, C.byref(root))
            if req_text is None:
                self._check(self._lib.bg_run_tensor_plan(self._ctx, plan_text, *args))
            else:
                self._check(self._lib.bg_run_tensor_plan_semantic(self._ctx, plan_text, req_text, *args))
        finally:
            for h in temps:
                self.release(h)
        if resident:
            return int(root.value)
        return bytes(buf.raw[:nbytes])

    def run_tensor_plan(self, plan: Any, inputs: Sequence[Any], dtype: str) -> bytes:
        return self._run_plan(plan, None, inputs, dtype, resident=False)

    def run_tensor_plan_resident(self, plan: Any, inputs: Sequence[Any], dtype: str) -> int:
        return self._run_plan(plan, None, inputs, dtype, resident=True)

    def run_tensor_plan_semantic(self, plan: Any, semantic_requests: Any, inputs: Sequence[Any],
                                 dtype: str) -> bytes:
        return self._run_plan(plan, semantic_requests, inputs, dtype, resident=False)

    def run_tensor_plan_resident_semantic(self, plan: Any, semantic_requests: Any, inputs: Sequence[Any],
                                          dtype: str) -> int:
        h = self._run_plan(plan, semantic_requests, inputs, dtype, resident=True)
        req = json.loads(semantic_requests) if isinstance(semantic_requests, (str, bytes)) else semantic_requests
        self._semantic_traces[h] = {"preparation": req}
        return h

    def semanticTensorPlanExecutionTrace(self, handle: int) -> dict:  # noqa: N802 - reference name
        """realizer.ts:1654-1667: the preparation bound to a resident semantic root."""
        trace = self._semantic_traces.get(int(handle))
        if trace is None:
            raise KernelError(f"HIP bridge: handle {handle} has no semantic tensor-plan execution trace")
        return trace

    def synchronize(self) -> None:
        self._check(self._lib.bg_synchronize(self._ctx))

    def device_ptr(self, handle: int) -> int:
        p = C.c_void_p()
        self._check(self._lib.bg_device_ptr(self._ctx, int(handle), C.byref(p)))
        return int(p.value or 0)

    def stream_ptr(self) -> int:
        p = C.c_void_p()
        self._check(self._lib.bg_stream(self._ctx, C.byref(p)))
        return int(p.value or 0)

    # -- diagnostics (realizer.ts:275-279, 287-298) -------------------------------------
    def aliveHandleCount(self) -> int:  # noqa: N802 - reference name
        n = C.c_int64()
        self._check(self._lib.bg_alive_handles(self._ctx, C.byref(n)))
        return int(n.value)

    alive_handle_count = aliveHandleCount

    def resourceSnapshot(self) -> dict:  # noqa: N802 - reference name
        s = N.Snapshot()
        self._check(self._lib.bg_resource_snapshot(self._ctx, C.byref(s)))
        return {
            "timingMode": "hip-event" if s.timing_mode == 1 else "unavailable",
            "timestampQueryAvailable": bool(s.timestamp_query_available),
            "currentOwnedGpuBytes": s.current_owned_bytes,
            "peakOwnedGpuBytes": s.peak_owned_bytes,
            "totalAllocatedGpuBytes": s.total_allocated_bytes,
            "totalReleasedGpuBytes": s.total_released_bytes,
            "aliveHandleCount": s.alive_handle_count,
            "pendingProfileCount": s.pending_profile_count,
            "passProfileCount": s.pass_profile_count,
            "poolCachedBytes": s.pool_cached_bytes,
            "poolHits": s.pool_hits,
            "poolMisses": s.pool_misses,
        }

    resource_snapshot = resourceSnapshot

    def flushProfiles(self) -> dict:  # noqa: N802 - reference name
        n = C.c_int()
        self._check(self._lib.bg_flush_profiles(self._ctx, None, 0, C.byref(n)))
        arr = (N.PassProfile * max(1, n.value))()
        got = C.c_int()
        self._check(self._lib.bg_flush_profiles(self._ctx, arr, n.value, C.byref(got)))
        snap = self.resourceSnapshot()
        snap["passProfiles"] = [
            {"label": arr[i].label.decode(), "gpuMs": arr[i].gpu_ms, "bytes": arr[i].bytes,
             "flops": arr[i].flops}
            for i in range(min(n.value, got.value))
        ]
        return snap

    flush_profiles = flushProfiles

    def set_launch_log(self, on: bool) -> None:
        """Record every kernel launch of this context (bg_set_launch_log)."""
        self._check(self._lib.bg_set_launch_log(self._ctx, 1 if on else 0))

    def take_launch_log(self) -> list:
        """The launches recorded since the last call, oldest first: kernel
        symbol, grid, block, LDS bytes and the kernel's register / scratch
        footprint (bg_take_launch_log)."""
        n = C.c_int()
        self._check(self._lib.bg_take_launch_log(self._ctx, None, 0, C.byref(n)))
        arr = (N.LaunchRecord * max(1, n.value))()
        got = C.c_int()
        self._check(self._lib.bg_take_launch_log(self._ctx, arr, n.value, C.byref(got)))
        return [{"kernel": arr[i].kernel.decode(errors="replace"), "grid": list(arr[i].grid),
                 "block": list(arr[i].block), "dynamicLds": int(arr[i].dynamic_lds),
                 "staticLds": int(arr[i].static_lds), "vgprs": int(arr[i].vgprs),
                 "scratchBytesPerLane": int(arr[i].scratch), "maxThreads": int(arr[i].max_threads)}
                for i in range(got.value)]

    def set_profiling(self, on: bool) -> None:
        """Switch per-dispatch profiling (the reference's creation option
        options.profiling, realizer.ts:899-914) on or off between calls."""
        self._check(self._lib.bg_set_profiling(self._ctx, 1 if on else 0))
        self.profiling = bool(on)

    # -- reference protocol methods outside this build's scope ---------------------------
    def run_user_kernel(self, *a: Any, **k: Any) -> Any:
        raise JitNotImplementedError("HIP bridge: run_user_kernel takes WGSL, which has no HIP meaning")


def inspect_tensor_plan(plan: Any, requests: Any = None) -> Dict[str, Any]:
    """Parse, validate and fuse a tensor plan without a device
    (bg_plan_inspect): the steps the executor would run, after its
    plan-level fusion, as {"steps": [{"value_id", "op", "inputs", ...}],
    "root_id"}.  Raises KernelError with the executor's own message for a
    plan it would refuse."""
    lib = N.load_library()
    pj = (plan if isinstance(plan, str) else json.dumps(plan, separators=(",", ":"))).encode()
    rj = None if requests is None else (requests if isinstance(requests, str)
                                         else json.dumps(requests, separators=(",", ":"))).encode()
    need = C.c_size_t(0)
    lib.bg_plan_inspect(pj, rj, None, 0, C.byref(need))
    buf = C.create_string_buffer(int(need.value))
    rc = lib.bg_plan_inspect(pj, rj, buf, len(buf), C.byref(need))
    text = buf.value.decode()
    if rc != N.BG_OK:
        raise KernelError(text, rc)
    return json.loads(text)
