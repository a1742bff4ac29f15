"""``LoadedModule``: the reference's operator API, backed by the gfx950 library.

The reference's kernels are methods of the ``LoadedModule`` generated by
``#[cuda_module] pub mod device`` (crates/inferrous-qwen3/src/kernels.rs:322-323),
created by ``device::load(&ctx)`` (src/gpu.rs:250) and called as
``module.op(&stream, LaunchConfig, args...)`` (src/gpu.rs:496-505,
src/conformance.rs:208-217).  This class keeps those names, argument order and
meanings so the parity tests read like src/conformance.rs:

* shapes come from buffer lengths exactly as in the reference:
  ``M = len(asc)``, ``N = len(ws)``, ``K = width``, ``len(out) == M * N``
  (src/kernels.rs:816-824);
* the ``LaunchConfig`` argument and the L2-prefetch hint arguments
  (``pf``, ``pf_from``, ``pf_to``, ``prefetch``, ``ck``, ``cv``, ``position``)
  are accepted and ignored -- outputs never depend on them
  (src/conformance.rs:108-128);
* the output buffer's dtype selects the epilogue: float32 = the reference's
  f32-holding-BF16 buffers, uint16 = BF16 bits, int32 = raw accumulators;
* errors raise ``W8A8Error`` (the reference returns ``Err``); there is no CPU
  fallback: every op runs the HIP library or raises.
"""
from __future__ import annotations

import ctypes

import numpy as np

from . import _lib
from ._lib import W8A8Error, check, lib
from .runtime import CudaContext, CudaStream, DeviceBuffer, is_capturing

_OUT = {np.dtype(np.float32): _lib.OUT_F32, np.dtype(np.uint16): _lib.OUT_BF16,
        np.dtype(np.int32): _lib.OUT_I32}


def _h(stream: CudaStream | None):
    return stream.handle if stream is not None else None


def _dtype_code(buf: DeviceBuffer) -> int:
    try:
        return _OUT[buf.dtype]
    except KeyError:
        raise TypeError(f"output dtype {buf.dtype} not supported (float32/uint16/int32)") from None


def _expect(buf: DeviceBuffer, dtype, what: str):
    if buf.dtype != np.dtype(dtype):
        raise TypeError(f"{what} must be {np.dtype(dtype)}, got {buf.dtype}")


def _shape(asc: DeviceBuffer, ws: DeviceBuffer, out: DeviceBuffer | None, width: int):
    m, n = len(asc), len(ws)
    if out is not None and len(out) != m * n:
        raise ValueError(f"out has {len(out)} elements, expected M*N = {m}*{n}")
    return m, n, int(width)


def _key(stream: CudaStream | None):
    return stream.handle if stream is not None else None


def _check_len(buf: DeviceBuffer, need: int, what: str):
    if len(buf) < need:
        raise ValueError(f"{what} has {len(buf)} elements, needs at least {need}")


class LoadedModule:
    """One instance per device context.  The split-K and selection
    workspaces are kept per stream (calls sharing one workspace must not
    overlap, and ops on different streams may), and an outgrown workspace is
    kept alive, not freed, because a graph captured earlier holds its
    address.  While a stream is being captured no workspace is allocated."""

    # lm_head of the Qwen3 family: selection workspace sized for it up front
    _SELECT_ROWS = 151936

    def __init__(self, ctx: CudaContext):
        self.ctx = ctx
        self._select_ws: dict = {}
        self._gemm_ws: dict = {}
        self._retired: list = []   # outgrown workspaces a captured graph may still use

    # ------------------------------------------------------------ quantizers
    def rounding_probe(self, stream, config, input: DeviceBuffer, out: DeviceBuffer) -> None:
        """src/kernels.rs:325-333."""
        _expect(input, np.float32, "input")
        _expect(out, np.int8, "out")
        if len(out) < len(input):
            raise ValueError("out shorter than input")
        check(lib().w8a8_rounding_probe(_h(stream), input.ptr, len(input), out.ptr), "rounding_probe")

    def quantize(self, stream, config, x: DeviceBuffer, width: int, q: DeviceBuffer,
                 scales: DeviceBuffer, pf=None, pf_from: int = 0, pf_to: int = 0,
                 maxima_reset: DeviceBuffer | None = None) -> None:
        """src/kernels.rs:414-452 (x float32 rows, or uint16 BF16 rows).
        ``maxima_reset`` reproduces the reset of src/kernels.rs:566."""
        rows = len(x) // width
        if rows * width != len(x) or len(q) != len(x) or len(scales) != rows:
            raise ValueError("quantize: x/q/scales lengths do not match width")
        _expect(q, np.int8, "q")
        _expect(scales, np.float32, "scales")
        mr = maxima_reset.ptr if maxima_reset is not None else None
        if x.dtype == np.float32:
            st = lib().w8a8_quantize(_h(stream), x.ptr, width, rows, q.ptr, scales.ptr, mr)
        elif x.dtype == np.uint16:
            st = lib().w8a8_quantize_bf16(_h(stream), x.ptr, width, rows, q.ptr, scales.ptr, mr)
        else:
            raise TypeError(f"x dtype {x.dtype} not supported")
        check(st, "quantize")

    def quantize_weights(self, stream, w_bf16: DeviceBuffer, k: int, q: DeviceBuffer,
                         scales: DeviceBuffer) -> None:
        """Offline per-output-channel weight quantization of tools/prepare.py:79-83
        on the device: for each BF16 row c of W[n, k], s_c = max(1e-8,
        max|W_c|) / 127 and q = clamp(round_half_even(W / s_c), -127, 127) --
        the same arithmetic as the activation quantizer, one row per channel."""
        self.quantize(stream, None, w_bf16, k, q, scales)

    def quantize_with_max(self, stream, config, x: DeviceBuffer, width: int, maxima: DeviceBuffer,
                          q: DeviceBuffer, scales: DeviceBuffer) -> None:
        """src/kernels.rs:453-475."""
        rows = len(x) // width
        if rows * width != len(x) or len(q) != len(x) or len(scales) < rows or len(maxima) < rows:
            raise ValueError("quantize_with_max: lengths do not match width")
        _expect(x, np.float32, "x")
        _expect(maxima, np.uint32, "maxima")
        check(lib().w8a8_quantize_with_max(_h(stream), x.ptr, width, rows, maxima.ptr, q.ptr,
                                           scales.ptr), "quantize_with_max")

    def norm_quantize(self, stream, config, x: DeviceBuffer, gain: DeviceBuffer, out: DeviceBuffer,
                      q: DeviceBuffer, scales: DeviceBuffer, maxima: DeviceBuffer) -> None:
        """src/kernels.rs:476-575 (host wrapper src/gpu.rs:340-363): RMSNorm of
        each 4096-wide row, the BF16-valued f32 output in ``out``, its
        quantization in ``q`` / ``scales``, and ``maxima`` reset to bits(1e-8).
        The rows come from ``scales`` (``rows(scale.len(), 1024)``)."""
        rows = len(scales)
        if len(gain) != 4096 or len(x) != rows * 4096 or len(out) != len(x) or len(q) != len(x) \
                or len(maxima) < rows:
            raise ValueError("norm_quantize: rows of 4096 with a 4096-wide gain expected")
        for b, dt, nm in ((x, np.float32, "x"), (gain, np.float32, "gain"), (out, np.float32, "out"),
                          (q, np.int8, "q"), (scales, np.float32, "scales"), (maxima, np.uint32, "maxima")):
            _expect(b, dt, nm)
        check(lib().w8a8_norm_quantize(_h(stream), x.ptr, gain.ptr, rows, 4096, out.ptr, q.ptr,
                                       scales.ptr, maxima.ptr), "norm_quantize")

    def head_packed(self, stream, config, x: DeviceBuffer, words: DeviceBuffer, offsets: DeviceBuffer,
                    exceptions: DeviceBuffer, out: DeviceBuffer, prefetch: int = 0) -> None:
        """src/kernels.rs:2258-2373 (call site src/gpu.rs:800-810): BF16 logits
        of the packed head against the last 4096 values of ``x``; one row per
        element of ``out``.  ``prefetch`` is the reference's L2 hint and does
        not change results."""
        rows = len(out)
        if len(words) < rows * 1536 or len(offsets) < rows * 16 or len(x) < 4096:
            raise ValueError("head_packed: packed rows of 4096 values and x of at least 4096 expected")
        _expect(x, np.float32, "x")
        _expect(words, np.uint32, "words")
        _expect(offsets, np.uint32, "offsets")
        _expect(exceptions, np.uint16, "exceptions")
        _expect(out, np.float32, "out")
        check(lib().w8a8_head_packed(_h(stream), x.ptr, len(x), words.ptr, offsets.ptr, exceptions.ptr,
                                     len(exceptions), rows, out.ptr), "head_packed")

    def unpack_head(self, stream, config, words: DeviceBuffer, offsets: DeviceBuffer,
                    exceptions: DeviceBuffer, out: DeviceBuffer) -> None:
        """src/kernels.rs:2376-2388: the packed values back as BF16 bits."""
        _expect(out, np.uint16, "out")
        check(lib().w8a8_unpack_bf16(_h(stream), words.ptr, offsets.ptr, exceptions.ptr, len(out), out.ptr),
              "unpack_head")

    # ------------------------------------------------------------ projections
    def reserve_workspace(self, nbytes: int, stream: CudaStream | None = None) -> None:
        """Make ``stream``'s split-K workspace at least nbytes (call before
        capturing a graph of large prefill projections)."""
        cur = self._gemm_ws.get(_key(stream))
        if cur is None or cur.nbytes < nbytes:
            if is_capturing(stream):
                raise W8A8Error(_lib.EWORKSPACE, "split-K workspace cannot grow while the stream is captured; "
                                "call reserve_workspace before capturing")
            if cur is not None:
                self._retired.append(cur)
            self._gemm_ws[_key(stream)] = DeviceBuffer((nbytes + 15) // 16 * 16, np.uint8)

    def _workspace_for(self, stream, m: int, n: int, k: int, path: int, split: bool = False):
        if path == _lib.PATH_MFMA and m > 4 and not split:
            path = _lib.PATH_AUTO   # the MFMA family too, split only where that is faster
        need = lib().w8a8_linear_workspace_bytes_path(m, n, k, path)
        if not need:
            return None, 0   # none used, or faster without
        if not is_capturing(stream):
            self.reserve_workspace(need, stream)
        # under capture a missing or small workspace selects the unsplit
        # kernels (identical results), so nothing is allocated
        ws = self._gemm_ws.get(_key(stream))
        return (ws.ptr, ws.nbytes) if ws is not None else (None, 0)

    def _linear(self, stream, q, asc, w, ws, width, out, path, residual=None, combined=None,
                split: bool = False) -> None:
        m, n, k = _shape(asc, ws, out, width)
        if len(q) < m * k or len(w) < n * k:
            raise ValueError("q or w shorter than M*K / N*K")
        wp, wb = self._workspace_for(stream, m, n, k, path, split)
        check(lib().w8a8_linear_ex(_h(stream), q.ptr, asc.ptr, m, w.ptr, ws.ptr, n, k,
                                   None if residual is None else residual.ptr, out.ptr,
                                   None if combined is None else combined.ptr, _dtype_code(out), path,
                                   wp, wb), "linear")

    def linear(self, stream, config, q, asc, w, ws, width, out) -> None:
        """src/kernels.rs:807-845 for any M (dispatched like src/gpu.rs:450-509)."""
        self._linear(stream, q, asc, w, ws, width, out, _lib.PATH_AUTO)

    def linear_dot4(self, stream, config, q, asc, w, ws, width, out) -> None:
        """Force the v_dot4 GEMV family at any M."""
        self._linear(stream, q, asc, w, ws, width, out, _lib.PATH_DOT4)

    def linear_mfma(self, stream, config, q, asc, w, ws, width, out) -> None:
        """Force the MFMA GEMM family at any M."""
        self._linear(stream, q, asc, w, ws, width, out, _lib.PATH_MFMA)

    # The reference's four M>1 tensor-core variants compute the same result
    # with different tilings (src/kernels.rs:846-1289).  Here one MFMA family
    # covers them; the names stay so reference call sites port unchanged.
    def linear_prefill(self, stream, config, q, asc, w, ws, width, out) -> None:
        self._linear(stream, q, asc, w, ws, width, out, _lib.PATH_MFMA)

    def linear_splitk(self, stream, config, q, asc, w, ws, width, out) -> None:
        """Split K wherever the shape's plan does, also where one launch is faster."""
        self._linear(stream, q, asc, w, ws, width, out, _lib.PATH_MFMA, split=True)

    def linear_tiled(self, stream, config, q, asc, w, ws, width, out) -> None:
        self._linear(stream, q, asc, w, ws, width, out, _lib.PATH_MFMA)

    def linear_large(self, stream, config, q, asc, w, ws, width, out) -> None:
        """src/kernels.rs:1142-1289; takes the activation and weight buffers
        where the reference takes their TMA descriptors (src/tensor.rs)."""
        self._linear(stream, q, asc, w, ws, width, out, _lib.PATH_MFMA)

    def linear_residual(self, stream, config, q, asc, w, ws, width, residual, out, combined,
                        prefetch: int = 0) -> None:
        """src/kernels.rs:577-618: out and combined = bf(residual + out)."""
        m, n, k = _shape(asc, ws, out, width)
        if len(residual) != m * n or len(combined) != m * n:
            raise ValueError("residual/combined must have M*N elements")
        if combined.dtype != out.dtype:
            raise TypeError("combined must have out's dtype")
        _expect(residual, np.float32, "residual")
        if _dtype_code(out) == _lib.OUT_I32:
            raise TypeError("linear_residual outputs f32 or BF16")
        self._linear(stream, q, asc, w, ws, width, out, _lib.PATH_AUTO, residual, combined)

    def linear_quantize_with_max(self, stream, config, x: DeviceBuffer, width: int,
                                 maxima: DeviceBuffer, q: DeviceBuffer, scales: DeviceBuffer, w, ws,
                                 out, residual=None, combined=None) -> None:
        """quantize_with_max (src/kernels.rs:453-475) then linear_residual /
        linear on the result, as GpuModel::linear_residual runs them at
        K = 12288 (src/gpu.rs:371-406)."""
        m = len(scales)
        n = len(ws)
        if len(x) != m * width or len(q) != m * width or len(out) != m * n:
            raise ValueError("linear_quantize_with_max: x/q/out sizes do not match")
        _expect(x, np.float32, "x")
        _expect(maxima, np.uint32, "maxima")
        _expect(q, np.int8, "q")
        _expect(scales, np.float32, "scales")
        _check_len(maxima, m, "maxima")
        _check_len(w, n * int(width), "w")
        if (residual is None) != (combined is None):
            raise ValueError("residual and combined go together")
        if residual is not None:
            _expect(residual, np.float32, "residual")
            if len(residual) != m * n or len(combined) != m * n or combined.dtype != out.dtype:
                raise ValueError("residual/combined must be M*N elements of out's dtype")
        check(lib().w8a8_linear_quantize_with_max(
            _h(stream), x.ptr, maxima.ptr, m, int(width), q.ptr, scales.ptr, w.ptr, ws.ptr, n,
            None if residual is None else residual.ptr, out.ptr,
            None if combined is None else combined.ptr, _dtype_code(out)), "linear_quantize_with_max")

    def linear_grouped(self, stream, q, asc, width, mats) -> None:
        """Sibling projections in one launch; ``mats`` = [(w, ws, out), ...]."""
        count = len(mats)
        m = len(asc)
        dt = {_dtype_code(o) for _, _, o in mats}
        if len(dt) != 1:
            raise TypeError("all outputs of a group must share one dtype")
        _check_len(q, m * int(width), "q")
        for i, (w, ws, o) in enumerate(mats):
            n = _shape(asc, ws, o, width)[1]
            _check_len(w, n * int(width), f"w[{i}]")
        W = (ctypes.c_void_p * count)(*[w.ptr for w, _, _ in mats])
        S = (ctypes.c_void_p * count)(*[s.ptr for _, s, _ in mats])
        N = (ctypes.c_size_t * count)(*[len(s) for _, s, _ in mats])
        O = (ctypes.c_void_p * count)(*[o.ptr for _, _, o in mats])
        check(lib().w8a8_linear_grouped(_h(stream), q.ptr, asc.ptr, m, int(width), count, W, S, N,
                                        O, dt.pop()), "linear_grouped")

    def linear_pair(self, stream, config, q, asc, width, w0, s0, out0, w1, s1, out1) -> None:
        """src/kernels.rs:696-735."""
        self.linear_grouped(stream, q, asc, width, [(w0, s0, out0), (w1, s1, out1)])

    def linear_triple(self, stream, config, q, asc, width, w0, s0, out0, w1, s1, out1, w2, s2,
                      out2, ck=None, cv=None, position=None, prefetch: int = 0) -> None:
        """src/kernels.rs:736-806 (KV-prefetch hint arguments ignored)."""
        self.linear_grouped(stream, q, asc, width, [(w0, s0, out0), (w1, s1, out1), (w2, s2, out2)])

    def linear_gate_up(self, stream, config, q, asc, width, w0, s0, gate, w1, s1, up) -> None:
        """The two projections of src/kernels.rs:619-695 (`linear_swiglu`)
        without the SiLU product: bit-exact gate/up outputs."""
        self.linear_grouped(stream, q, asc, width, [(w0, s0, gate), (w1, s1, up)])

    def linear_swiglu(self, stream, config, q, asc, width, w0, s0, gate, w1, s1, up, out,
                      maxima, prefetch: int = 0) -> None:
        """src/kernels.rs:619-695: gate, up (bit-exact), out = bf(silu(gate) * up)
        and the atomicMax of bits(|out|) per row into ``maxima`` (pass None to
        skip).  The prefetch hint is ignored."""
        m, n, k = _shape(asc, s0, gate, width)
        _shape(asc, s1, up, width)
        _check_len(q, m * k, "q")
        _check_len(w0, n * k, "w_gate")
        _check_len(w1, n * k, "w_up")
        if len(out) != m * n or up.dtype != gate.dtype or out.dtype != gate.dtype:
            raise ValueError("gate, up and out must be M*N elements of one dtype")
        if maxima is not None:
            _expect(maxima, np.uint32, "maxima")
            if len(maxima) < m:
                raise ValueError("maxima needs one word per row")
        check(lib().w8a8_linear_swiglu(_h(stream), q.ptr, asc.ptr, m, k, w0.ptr, s0.ptr, w1.ptr,
                                       s1.ptr, n, gate.ptr, up.ptr, out.ptr,
                                       None if maxima is None else maxima.ptr,
                                       _dtype_code(gate)), "linear_swiglu")

    def linear_swiglu_quantize(self, stream, config, q, asc, width, w0, s0, gate, w1, s1, up, out,
                               maxima, q_out, scales_out) -> None:
        """``linear_swiglu`` (src/kernels.rs:619-695) followed by
        ``quantize_with_max`` of its output (src/kernels.rs:453-475), the
        decode pair of src/gpu.rs:730 and :381, in one call: the same gate,
        up, out and maxima, plus ``q_out`` / ``scales_out`` for the next
        projection.  ``maxima`` is required."""
        m, n, k = _shape(asc, s0, gate, width)
        _shape(asc, s1, up, width)
        _check_len(q, m * k, "q")
        _check_len(w0, n * k, "w_gate")
        _check_len(w1, n * k, "w_up")
        if len(out) != m * n or up.dtype != gate.dtype or out.dtype != gate.dtype:
            raise ValueError("gate, up and out must be M*N elements of one dtype")
        _expect(maxima, np.uint32, "maxima")
        _expect(q_out, np.int8, "q_out")
        _expect(scales_out, np.float32, "scales_out")
        if len(maxima) < m or len(q_out) < m * n or len(scales_out) < m:
            raise ValueError("maxima / scales_out need one word per row, q_out M*N bytes")
        check(lib().w8a8_linear_swiglu_quantize(_h(stream), q.ptr, asc.ptr, m, k, w0.ptr, s0.ptr, w1.ptr,
                                                s1.ptr, n, gate.ptr, up.ptr, out.ptr, maxima.ptr, q_out.ptr,
                                                scales_out.ptr, _dtype_code(gate)), "linear_swiglu_quantize")

    def _produce_linear(self, stream, x, gain, normed, q, scales, maxima, w, ws, out, residual,
                        combined) -> None:
        n = len(ws)
        if len(x) != 4096 or (gain is not None and len(gain) != 4096):
            raise ValueError("one 4096-wide row (and a 4096-wide gain) expected")
        if n == 0 or len(out) != n:
            raise ValueError("out must hold the projection's N >= 1 outputs")
        _check_len(w, n * 4096, "w")
        _expect(x, np.float32, "x")
        _expect(q, np.int8, "q")
        _expect(scales, np.float32, "scales")
        _expect(ws, np.float32, "ws")
        if len(q) < 4096 or len(scales) < 1:
            raise ValueError("q needs 4096 codes, scales one word")
        if gain is not None:
            _expect(gain, np.float32, "gain")
        if normed is not None:
            _expect(normed, np.float32, "normed")
            if len(normed) < 4096:
                raise ValueError("normed needs 4096 values")
        if maxima is not None:
            _expect(maxima, np.uint32, "maxima")
        if (residual is None) != (combined is None):
            raise ValueError("residual and combined go together")
        if residual is not None:
            _expect(residual, np.float32, "residual")
            if len(residual) != n or len(combined) != n or combined.dtype != out.dtype:
                raise ValueError("residual/combined must be N elements, combined of out's dtype")
        ptr = lambda b: None if b is None else b.ptr  # noqa: E731
        if gain is not None:
            st = lib().w8a8_norm_quantize_linear(_h(stream), x.ptr, gain.ptr, ptr(normed), q.ptr, scales.ptr,
                                                 ptr(maxima), w.ptr, ws.ptr, n, ptr(residual), out.ptr,
                                                 ptr(combined), _dtype_code(out))
            check(st, "norm_quantize_linear")
        else:
            st = lib().w8a8_quantize_linear(_h(stream), x.ptr, 4096, q.ptr, scales.ptr, ptr(maxima), w.ptr,
                                            ws.ptr, n, ptr(residual), out.ptr, ptr(combined), _dtype_code(out))
            check(st, "quantize_linear")

    def norm_quantize_linear(self, stream, config, x, gain, normed, q, scales, maxima, w, ws, out,
                             residual=None, combined=None) -> None:
        """``norm_quantize`` (src/kernels.rs:476-575) of one 4096-wide row,
        then ``linear`` (or ``linear_residual`` with ``residual`` /
        ``combined``) of its codes at M = 1, in one launch.  Every output --
        ``normed`` (may be None), ``q``, ``scales``, the ``maxima`` reset (may
        be None), ``out``, ``combined`` -- equals the two calls' bit for bit."""
        self._produce_linear(stream, x, gain, normed, q, scales, maxima, w, ws, out, residual, combined)

    def quantize_linear(self, stream, config, x, q, scales, w, ws, out, residual=None, combined=None,
                        maxima_reset=None) -> None:
        """``quantize`` (src/kernels.rs:433-451) of one 4096-wide f32 row, then
        ``linear`` / ``linear_residual`` of its codes at M = 1, in one launch:
        the reference's decode ``linear_residual`` host step (src/gpu.rs:364-415)
        as one kernel, with the two calls' outputs bit for bit."""
        self._produce_linear(stream, x, None, None, q, scales, maxima_reset, w, ws, out, residual, combined)

    def norm_quantize_linear_swiglu(self, stream, config, x, gain, normed, q, scales, w0, s0, gate, w1, s1, up,
                                    out, maxima, q_out=None, scales_out=None) -> None:
        """``norm_quantize`` (src/kernels.rs:476-575) of one 4096-wide row,
        then ``linear_swiglu`` (src/kernels.rs:619-695) of its codes at M = 1
        -- and, with ``q_out`` / ``scales_out``, the ``quantize_with_max`` of
        ``out`` as ``linear_swiglu_quantize`` writes it: every output equals
        those calls' bit for bit.  ``maxima`` is required (reset by the norm,
        then the act maximum folded in); ``normed`` may be None."""
        n = len(s0)
        if len(x) != 4096 or len(gain) != 4096:
            raise ValueError("one 4096-wide row and a 4096-wide gain expected")
        if n == 0 or len(s1) != n or len(gate) != n or len(up) != n or len(out) != n:
            raise ValueError("gate, up, out and both scale vectors must hold N >= 1 values")
        if up.dtype != gate.dtype or out.dtype != gate.dtype:
            raise ValueError("gate, up and out must share one dtype")
        _check_len(w0, n * 4096, "w_gate")
        _check_len(w1, n * 4096, "w_up")
        for b, dt, nm in ((x, np.float32, "x"), (gain, np.float32, "gain"), (q, np.int8, "q"),
                          (scales, np.float32, "scales"), (maxima, np.uint32, "maxima")):
            _expect(b, dt, nm)
        if len(q) < 4096 or len(scales) < 1 or len(maxima) < 1:
            raise ValueError("q needs 4096 codes, scales and maxima one word")
        if normed is not None:
            _expect(normed, np.float32, "normed")
            if len(normed) < 4096:
                raise ValueError("normed needs 4096 values")
        if (q_out is None) != (scales_out is None):
            raise ValueError("q_out and scales_out go together")
        if q_out is not None:
            _expect(q_out, np.int8, "q_out")
            _expect(scales_out, np.float32, "scales_out")
            if len(q_out) < n or len(scales_out) < 1:
                raise ValueError("q_out needs N codes, scales_out one word")
        ptr = lambda b: None if b is None else b.ptr  # noqa: E731
        check(lib().w8a8_norm_quantize_linear_swiglu(_h(stream), x.ptr, gain.ptr, ptr(normed), q.ptr, scales.ptr,
                                                     w0.ptr, s0.ptr, w1.ptr, s1.ptr, n, gate.ptr, up.ptr, out.ptr,
                                                     maxima.ptr, ptr(q_out), ptr(scales_out), _dtype_code(gate)),
              "norm_quantize_linear_swiglu")

    def norm_quantize_mlp(self, stream, config, x, gain, normed, q, scales, w0, s0, gate, w1, s1, up, act, maxima,
                          wd, sd, out, residual=None, combined=None, q_act=None, scales_act=None) -> None:
        """The decode MLP block at M = 1 in two launches: ``norm_quantize``
        (src/kernels.rs:476-575) of one 4096-wide row, ``linear_swiglu``
        (src/kernels.rs:619-695) of its codes, then ``quantize_with_max``
        (src/kernels.rs:453-475) of ``act`` and ``linear_residual`` /
        ``linear`` (src/kernels.rs:577-618) through ``wd`` [N, 12288] -- the
        calls of src/gpu.rs:713-786.  Every output equals
        ``norm_quantize_linear_swiglu`` (with ``q_out``) followed by
        ``linear_residual`` / ``linear`` bit for bit.  ``gate``, ``up`` and
        ``act`` share one dtype (F32 or BF16), ``out`` and ``combined``
        another; ``normed``, ``q_act`` / ``scales_act`` and ``residual`` /
        ``combined`` are optional."""
        n_ff, n = len(s0), len(sd)
        if len(x) != 4096 or len(gain) != 4096:
            raise ValueError("one 4096-wide row and a 4096-wide gain expected")
        if n_ff != 12288:
            raise ValueError("the MLP width (len(s0)) must be 12288")
        if len(s1) != n_ff or len(gate) != n_ff or len(up) != n_ff or len(act) != n_ff:
            raise ValueError("gate, up, act and both scale vectors must hold 12288 values")
        if up.dtype != gate.dtype or act.dtype != gate.dtype:
            raise ValueError("gate, up and act must share one dtype")
        if n == 0 or len(out) != n:
            raise ValueError("out must hold N = len(sd) >= 1 values")
        _check_len(w0, n_ff * 4096, "w_gate")
        _check_len(w1, n_ff * 4096, "w_up")
        _check_len(wd, n * n_ff, "w_down")
        for b, dt, nm in ((x, np.float32, "x"), (gain, np.float32, "gain"), (q, np.int8, "q"),
                          (scales, np.float32, "scales"), (maxima, np.uint32, "maxima")):
            _expect(b, dt, nm)
        if len(q) < 4096 or len(scales) < 1 or len(maxima) < 1:
            raise ValueError("q needs 4096 codes, scales and maxima one word")
        if normed is not None:
            _expect(normed, np.float32, "normed")
            if len(normed) < 4096:
                raise ValueError("normed needs 4096 values")
        if (q_act is None) != (scales_act is None):
            raise ValueError("q_act and scales_act go together")
        if q_act is not None:
            _expect(q_act, np.int8, "q_act")
            _expect(scales_act, np.float32, "scales_act")
            if len(q_act) < n_ff or len(scales_act) < 1:
                raise ValueError("q_act needs 12288 codes, scales_act one word")
        if (residual is None) != (combined is None):
            raise ValueError("residual and combined go together")
        if residual is not None:
            _expect(residual, np.float32, "residual")
            if len(residual) != n or len(combined) != n or combined.dtype != out.dtype:
                raise ValueError("residual and combined must hold N values, combined in out's dtype")
        ptr = lambda b: None if b is None else b.ptr  # noqa: E731
        check(lib().w8a8_norm_quantize_mlp(_h(stream), x.ptr, gain.ptr, ptr(normed), q.ptr, scales.ptr,
                                           w0.ptr, s0.ptr, w1.ptr, s1.ptr, n_ff, gate.ptr, up.ptr, act.ptr,
                                           _dtype_code(gate), maxima.ptr, ptr(q_act), ptr(scales_act), wd.ptr,
                                           sd.ptr, n, ptr(residual), out.ptr, ptr(combined), _dtype_code(out)),
              "norm_quantize_mlp")

    def swiglu(self, stream, config, gate, up, out, maxima) -> None:
        """src/kernels.rs:2172-2190: out = bf(silu(gate) * up) elementwise;
        like the reference, the maximum is published into maxima[0] only when
        the input is one 12288-wide decode row."""
        n = len(gate)
        if len(up) != n or len(out) != n or up.dtype != gate.dtype or out.dtype != gate.dtype:
            raise ValueError("gate, up and out must have one length and dtype")
        publish = maxima is not None and n == 12288
        if publish:
            _expect(maxima, np.uint32, "maxima")
        check(lib().w8a8_swiglu(_h(stream), gate.ptr, up.ptr, 1, n, out.ptr,
                                maxima.ptr if publish else None, _dtype_code(gate)), "swiglu")

    # ------------------------------------------------------------ selection
    def _workspace(self, stream, nbytes: int) -> DeviceBuffer:
        """The stream's selection workspace, at least nbytes.  The first one
        already covers the Qwen3 lm_head, so decode never grows it; a buffer
        that does grow is retired, not freed (a captured graph may hold it),
        and growing under capture is refused instead of allocating."""
        cur = self._select_ws.get(_key(stream))
        if cur is None or cur.nbytes < nbytes:
            if is_capturing(stream):
                raise W8A8Error(_lib.EWORKSPACE, "selection workspace cannot grow while the stream is captured")
            if cur is not None:
                self._retired.append(cur)
            floor = max(lib().w8a8_linear_argmax_workspace_bytes(self._SELECT_ROWS),
                        lib().w8a8_select_workspace_bytes(self._SELECT_ROWS))
            cur = DeviceBuffer((max(nbytes, floor) + 7) // 8, np.uint64)
            self._select_ws[_key(stream)] = cur
        return cur

    def select_token(self, stream, config, x: DeviceBuffer, out: DeviceBuffer) -> None:
        """src/kernels.rs:2191-2231: lowest-index argmax, u32::MAX sentinel."""
        _expect(x, np.float32, "x")
        _expect(out, np.uint32, "out")
        need = lib().w8a8_select_workspace_bytes(len(x))
        ws = self._workspace(stream, need)
        check(lib().w8a8_select_token(_h(stream), x.ptr, len(x), out.ptr, ws.ptr, ws.nbytes),
              "select_token")

    def linear_argmax(self, stream, q, asc, w, ws, width, token: DeviceBuffer,
                      logits: DeviceBuffer | None = None) -> None:
        """W8A8 lm_head + fused greedy selection (src/gpu.rs:801-812 composition)."""
        if len(asc) != 1:
            raise ValueError("linear_argmax takes one activation row")
        _expect(token, np.uint32, "token")
        n = len(ws)
        if logits is not None and len(logits) != n:
            raise ValueError("logits must have N elements")
        _check_len(q, int(width), "q")
        _check_len(w, n * int(width), "w")
        need = lib().w8a8_linear_argmax_workspace_bytes(n)
        wsb = self._workspace(stream, need)
        check(lib().w8a8_linear_argmax(
            _h(stream), q.ptr, asc.ptr, w.ptr, ws.ptr, n, int(width), token.ptr,
            logits.ptr if logits is not None else None,
            _dtype_code(logits) if logits is not None else _lib.OUT_F32, wsb.ptr, wsb.nbytes),
            "linear_argmax")

    def linear_argmax_noalloc(self, stream, q, asc, w, ws, width, token: DeviceBuffer,
                              logits: DeviceBuffer | None = None) -> None:
        """linear_argmax with the selection keys in the library's own fixed
        device array (no workspace, no allocation): for callers that cannot
        allocate, e.g. while capturing a graph.  At most
        ``NOALLOC_MAX_ROWS`` vocabulary rows; concurrent calls on one GPU
        share that array and must not overlap."""
        if len(asc) != 1:
            raise ValueError("linear_argmax_noalloc takes one activation row")
        _expect(token, np.uint32, "token")
        n = len(ws)
        if n > _lib.NOALLOC_MAX_ROWS:
            raise ValueError(f"linear_argmax_noalloc: {n} rows exceed {_lib.NOALLOC_MAX_ROWS}")
        if logits is not None and len(logits) != n:
            raise ValueError("logits must have N elements")
        _check_len(q, int(width), "q")
        _check_len(w, n * int(width), "w")
        check(lib().w8a8_linear_argmax_noalloc(
            _h(stream), q.ptr, asc.ptr, w.ptr, ws.ptr, n, int(width), token.ptr,
            logits.ptr if logits is not None else None,
            _dtype_code(logits) if logits is not None else _lib.OUT_F32), "linear_argmax_noalloc")

    # ------------------------------------------------------------ decode sequence
    def prepare_sequence(self, entries) -> "SequencePlan":
        """Validate a dependent sequence of M = 1 projections and write its
        device table (w8a8_linear_sequence_prepare).  Each entry is a dict
        with ``q`` (int8 [k]), ``asc`` (float32 [1]), ``w`` (int8 [n*k]),
        ``ws`` (float32 [n]), ``out`` (float32 or uint16 [n]; None only for
        the selecting last entry), optional ``residual`` / ``combined``
        (linear_residual, src/kernels.rs:577-618) and ``select`` (the last
        entry only: the lm_head with select_token, src/kernels.rs:2191-2231).
        The plan keeps the buffers alive."""
        if not entries:
            raise ValueError("a sequence needs at least one entry")
        arr = (_lib.SeqEntry * len(entries))()
        keep = []
        for i, e in enumerate(entries):
            q, asc, w, ws, out = e["q"], e["asc"], e["w"], e["ws"], e.get("out")
            res, comb, sel = e.get("residual"), e.get("combined"), bool(e.get("select", False))
            _expect(q, np.int8, "q")
            _expect(asc, np.float32, "asc")
            _expect(w, np.int8, "w")
            _expect(ws, np.float32, "ws")
            k, n = len(q), len(ws)
            if len(asc) != 1:
                raise ValueError(f"entry {i}: one activation row (len(asc) == 1) expected")
            _check_len(w, n * k, f"entry {i}: w")
            if sel and i != len(entries) - 1:
                raise ValueError("only the last entry may select")
            if out is None and not sel:
                raise ValueError(f"entry {i}: out is required")
            dt = _dtype_code(out) if out is not None else _lib.OUT_F32
            if dt == _lib.OUT_I32:
                raise TypeError(f"entry {i}: out is float32 or uint16 (BF16)")
            if out is not None and len(out) != n:
                raise ValueError(f"entry {i}: out must hold N = len(ws) values")
            if (res is None) != (comb is None):
                raise ValueError(f"entry {i}: residual and combined go together")
            if res is not None:
                _expect(res, np.float32, "residual")
                if len(res) != n or len(comb) != n or comb.dtype != out.dtype:
                    raise ValueError(f"entry {i}: residual/combined must be N values, combined in out's dtype")
            ptr = lambda b: None if b is None else b.ptr  # noqa: E731
            arr[i] = _lib.SeqEntry(w.ptr, ws.ptr, q.ptr, asc.ptr, ptr(out), ptr(res), ptr(comb), n, k, dt,
                                   _lib.SEQ_SELECT if sel else 0)
            keep.append((q, asc, w, ws, out, res, comb))
        nbytes = lib().w8a8_linear_sequence_table_bytes(len(entries))
        table = DeviceBuffer((nbytes + 15) // 16 * 16, np.uint8)
        check(lib().w8a8_linear_sequence_prepare(arr, len(entries), table.ptr, table.nbytes),
              "linear_sequence_prepare")
        return SequencePlan(table, len(entries), bool(entries[-1].get("select", False)), keep)

    def linear_sequence(self, stream, plan: "SequencePlan", token: DeviceBuffer | None = None,
                        wait_us: int = 0) -> None:
        """Run a prepared sequence in one launch (w8a8_linear_sequence): every
        output equals the per-entry linear / linear_residual / linear_argmax
        call's.  ``token`` (uint32 [1]) receives the selection of a selecting
        last entry.  Not capturable; ``wait_us`` bounds every wait (0: the
        library's default)."""
        tok, wsp, wsb = None, None, 0
        if plan.select:
            if token is None:
                raise ValueError("the sequence selects: token (uint32 [1]) is required")
            _expect(token, np.uint32, "token")
            wb = self._workspace(stream, lib().w8a8_linear_sequence_workspace_bytes())
            tok, wsp, wsb = token.ptr, wb.ptr, wb.nbytes
        check(lib().w8a8_linear_sequence(_h(stream), plan.table.ptr, plan.count, tok, wsp, wsb, int(wait_us)),
              "linear_sequence")

    def sequence_status(self) -> int:
        """0, or 1 when a sequence wait ran out (synchronises the device)."""
        st = ctypes.c_uint32()
        check(lib().w8a8_linear_sequence_status(ctypes.byref(st)), "linear_sequence_status")
        return int(st.value)

    def sequence_reset(self) -> None:
        check(lib().w8a8_linear_sequence_reset(), "linear_sequence_reset")

    # ------------------------------------------------------------ synthetic
    def synth_i8(self, stream, out: DeviceBuffer, seed: int, stream_id: int) -> None:
        _expect(out, np.int8, "out")
        check(lib().w8a8_synth_i8(_h(stream), out.ptr, len(out), seed, stream_id), "synth_i8")

    def synth_f32(self, stream, out: DeviceBuffer, seed: int, stream_id: int, lo: float, hi: float) -> None:
        _expect(out, np.float32, "out")
        check(lib().w8a8_synth_f32(_h(stream), out.ptr, len(out), seed, stream_id, lo, hi),
              "synth_f32")


class SequencePlan:
    """A prepared decode sequence: its device table, entry count, whether the
    last entry selects, and references that keep its buffers alive."""

    def __init__(self, table: DeviceBuffer, count: int, select: bool, keep: list):
        self.table = table
        self.count = count
        self.select = select
        self._keep = keep


def load(ctx: CudaContext) -> LoadedModule:
    """``device::load(&ctx)`` (src/gpu.rs:250)."""
    return LoadedModule(ctx)
