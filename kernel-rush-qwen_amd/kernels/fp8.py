"""FP8 (OCP e4m3) decode matmuls on MI355X: quantizers, activation scales, the scaled cast, and
the dequant-fused skinny GEMM/GEMV that replaces torch._scaled_mm at decode sizes.

Drop-in for the reference's engine/kernels/fp8.py (signatures of quantize_weight, ActScale,
SharedScale, linear_fp8, pick_cast, FP8_MAX, HEADROOM kept as at fp8.py:13-106), plus the
per-channel / per-token family its experiments call (experiments/modal_fp8.py:59-85): quantize,
quant_rows, gemv_fp8, gemv_swiglu_fp8.

Numerics (every quantized byte is the OCP e4m3 round-to-nearest-even of the clamped value, as
torch's float8_e4m3fn cast gives):
  quantize_weight  scale = max(max|w|, 1e-12) / 448;  w8 = e4m3(clamp(w / scale, +-448))
  quantize         the same per output row (scale [N])
  ActScale         amax = max(max|x|, 1e-6) * headroom; inv = 448 / amax; scale = amax / 448
  quant_rows       ActScale per row, then x8 = e4m3(clamp(x * inv[m], +-448)); xs = scale [M, 1]
                   (quant_rows_tiled: the same bytes in the tiled activation layout)
  gemv_fp8 et al.  y = (sum_k x8 w8) * x_scale * w_scale with fp32 accumulation
Quantized weights carry, beside the reference's row-major [N, K] bytes, a copy in the GEMV
kernels' tiled layout (FP8Weight.tiled).
"""

import os

import torch

from . import _lib as L

FP8_MAX = 448.0
HEADROOM = float(os.environ.get("ENGINE_FP8_HEADROOM", "4"))
DECODE_MAX_ROWS = 32  # rows handled by one launch of the skinny kernels
# From this many rows linear_fp8 runs gemm_fp8. Per Qwen3-4B decoder layer (the four projections' products,
# weights cold in the caches) against hipBLASLt on MI355X, us: M = 33 44.6 / 46.1, M = 48 46.1 / 52.5,
# M = 77 52.1 / 53.1, M = 96 54.3 / 50.9, M = 127 58.4 / 60.4, M = 128 58.6 / 71.7, M = 160 64.8 / 62.3,
# M = 256 73.4 / 75.7, M = 512 97.6 / 95.4, M = 1024 157.6 / 152.3, M = 2048 231 / 230, M = 4096 380 / 358.
# The whole call is faster where it is short (_ring_pays, which also says on which weights it is taken
# below PER_CHANNEL_MIN_ROWS).
PREFILL_MIN_ROWS = DECODE_MAX_ROWS + 1
# The library takes one scale per weight; fewer rows than this keep refusing per-channel ones there.
PER_CHANNEL_MIN_ROWS = 128


class FP8Weight(tuple):
    """(w8, scale) as the reference returns it - w8 the row-major float8_e4m3fn [N, K] matrix,
    scale fp32 0-d (per tensor) or [N] (per output channel) - with the same bytes in the tiled
    layout of include/krq.h as .tiled (uint8 [N*K], or None when N % 16 or K % 64)."""

    def __new__(cls, w8, scale, tiled=None):
        self = super().__new__(cls, (w8, scale))
        self.tiled = tiled
        return self


def _check_weight(w):
    L.require_device(w)
    if w.dim() != 2 or w.dtype != torch.bfloat16:
        raise ValueError(f"expected a bf16 [N, K] weight, got {w.dtype} {tuple(w.shape)}")
    return w if w.stride(1) == 1 else w.contiguous()


def _weight_out(w, tiled):
    N, K = w.shape
    w8 = torch.empty((N, K), device=w.device, dtype=torch.float8_e4m3fn)
    t = None
    if tiled and N % 16 == 0 and K % 64 == 0:
        t = torch.empty((N * K,), device=w.device, dtype=torch.uint8)
    return w8, t


@torch.no_grad()
def quantize_weight(w, tiled=True):
    """w [N, K] bf16 -> (w8 [N, K] float8_e4m3fn, scale fp32 scalar), w ~= w8 * scale.
    Reference: engine/kernels/fp8.py:17-23."""
    w = _check_weight(w)
    N, K = w.shape
    w8, t = _weight_out(w, tiled)
    scale = torch.empty((), device=w.device, dtype=torch.float32)
    ws = torch.empty((N,), device=w.device, dtype=torch.float32)
    L.call("krq_quant_fp8_tensor", L.ptr(w), N, K, w.stride(0), L.ptr(ws), L.ptr(w8), L.ptr(t),
           L.ptr(scale), L.stream(w))
    return FP8Weight(w8, scale, t)


@torch.no_grad()
def quantize(w, tiled=True):
    """w [N, K] bf16 -> (w8 [N, K] float8_e4m3fn, scale fp32 [N]), w ~= w8 * scale[:, None].
    Per-output-channel form called by the reference's experiments/modal_fp8.py:59-60."""
    w = _check_weight(w)
    N, K = w.shape
    w8, t = _weight_out(w, tiled)
    scale = torch.empty((N,), device=w.device, dtype=torch.float32)
    L.call("krq_quant_fp8_rows", L.ptr(w), N, K, w.stride(0), L.ptr(w8), L.ptr(t), L.ptr(scale),
           L.stream(w))
    return FP8Weight(w8, scale, t)


def _rows(x):
    L.require_device(x)
    if x.dtype != torch.bfloat16:
        raise ValueError(f"expected bf16 activations, got {x.dtype}")
    x2 = x.reshape(-1, x.shape[-1]) if x.dim() != 2 else x
    return x2.contiguous()


class ActScale:
    """Activation scale for one call: x8 = clamp(x * inv), x ~= x8 * scale.
    Computed on device from this tensor's own range (no sync, graph-safe).
    Reference: engine/kernels/fp8.py:26-35."""

    def __init__(self, x, headroom=1.0):
        x2 = _rows(x)
        M, K = x2.shape
        dev = x2.device
        self.amax = torch.empty((), device=dev, dtype=torch.float32)
        self.inv = torch.empty((1,), device=dev, dtype=torch.float32)
        self.scale = torch.empty((), device=dev, dtype=torch.float32)
        ws = torch.empty((max(1, L.lib().krq_act_scale_ws_floats(M, K)),), device=dev,
                         dtype=torch.float32)
        L.call("krq_act_scale", L.ptr(x2), M, K, 0, float(headroom), L.ptr(self.amax),
               L.ptr(self.inv), L.ptr(self.scale), L.ptr(ws), L.stream(x2))


class SharedScale:
    """Scale slots living in caller-owned device tensors (read by decode graphs).
    Reference: engine/kernels/fp8.py:90-94."""

    def __init__(self, inv, scale):
        self.inv, self.scale = inv, scale


def quant_rows(x):
    """Per-token dynamic FP8: x [M, K] bf16 -> (x8 [M, K] float8_e4m3fn, xs fp32 [M, 1]) with
    x ~= x8 * xs, the operands of torch._scaled_mm(x8, w8.t(), scale_a=xs, ...) in the
    reference's experiments/modal_fp8.py:84-85."""
    x2 = _rows(x)
    M, K = x2.shape
    x8 = torch.empty((M, K), device=x2.device, dtype=torch.float8_e4m3fn)
    xs = torch.empty((M, 1), device=x2.device, dtype=torch.float32)
    L.call("krq_quant_rows", L.ptr(x2), M, K, L.ptr(x8), L.ptr(xs), L.stream(x2))
    return x8, xs


def quant_rows_tiled(x):
    """quant_rows with the e4m3 rows in the tiled activation layout the FP8 GEMV reads as
    X_FP8_TILED: the M rows padded with zero rows to MP = 16 * ceil(M / 16), in 16-row x 64-byte
    tiles (the tiling of FP8Weight.tiled), so each matrix-core operand load is one contiguous KiB.
    Returns (x8t uint8 [MP * K], xs fp32 [M, 1]); the bytes are quant_rows' bytes, permuted."""
    x2 = _rows(x)
    M, K = x2.shape
    mp = (M + 15) // 16 * 16
    x8t = torch.empty((mp * K,), device=x2.device, dtype=torch.uint8)
    xs = torch.empty((M, 1), device=x2.device, dtype=torch.float32)
    L.call("krq_quant_rows_tiled", L.ptr(x2), M, K, L.ptr(x8t), L.ptr(xs), L.stream(x2))
    return x8t, xs


def cast_tiled(x, a):
    """_cast(x, a) in the tiled activation layout of quant_rows_tiled (krq_cast_fp8_tiled): the
    static- or per-call-scale rows for the GEMV on X_FP8_TILED (up to 32 rows; from how many it pays:
    TILED_MIN_ROWS and the lines beside it).
    Returns uint8 [16 * ceil(M / 16) * K]; the bytes are _cast's, permuted, pad rows zero."""
    x2 = _rows(x)
    M, K = x2.shape
    L.require_device(a.inv)
    mp = (M + 15) // 16 * 16
    x8t = torch.empty((mp * K,), device=x2.device, dtype=torch.uint8)
    L.call("krq_cast_fp8_tiled", L.ptr(x2), M, K, L.ptr(_one(a.inv)), L.ptr(x8t), L.stream(x2))
    return x8t


def _cast_hip(x, a):
    x2 = _rows(x)
    M, K = x2.shape
    L.require_device(a.inv)
    y = torch.empty(x.shape, device=x.device, dtype=torch.float8_e4m3fn)
    L.call("krq_cast_fp8", L.ptr(x2), M, K, L.ptr(_one(a.inv)), 0, L.ptr(y), L.stream(x2))
    return y


def _act_scale_cast(x, headroom=1.0):
    """(ActScale(x, headroom), _cast_hip(x, a)) through krq_act_scale_cast_fp8: the same scale and
    bytes, one launch fewer (the fold of the partial maxima runs inside the cast)."""
    x2 = _rows(x)
    M, K = x2.shape
    dev = x2.device
    a = ActScale.__new__(ActScale)
    a.amax = torch.empty((), device=dev, dtype=torch.float32)
    a.inv = torch.empty((1,), device=dev, dtype=torch.float32)
    a.scale = torch.empty((), device=dev, dtype=torch.float32)
    ws = torch.empty((max(1, L.lib().krq_act_scale_ws_floats(M, K)),), device=dev, dtype=torch.float32)
    y = torch.empty(x.shape, device=x.device, dtype=torch.float8_e4m3fn)
    L.call("krq_act_scale_cast_fp8", L.ptr(x2), M, K, float(headroom), L.ptr(a.amax), L.ptr(a.inv),
           L.ptr(a.scale), L.ptr(ws), L.ptr(y), L.stream(x2))
    return a, y


def _cast_torch(x, a):
    return (x.float() * a.inv).clamp_(-FP8_MAX, FP8_MAX).to(torch.float8_e4m3fn)


_cast = _cast_hip


def pick_cast(log):
    """Validate the HIP cast against torch's cast on this GPU (bit-exact) and report both
    timings. Keeps the HIP cast when every byte matches; otherwise falls back to the torch cast
    and says so, as the reference does on a failed check (engine/kernels/fp8.py:62-87)."""
    global _cast
    _cast = _cast_hip
    try:
        x = torch.randn((4096, 2560), device="cuda", dtype=torch.bfloat16) * 3
        a = ActScale(x)
        ref = _cast_torch(x, a).view(torch.uint8)
        got = _cast_hip(x, a).view(torch.uint8)
        bad = int((ref != got).sum().item())
        ts = {}
        for name, fn in (("torch", _cast_torch), ("hip", _cast_hip)):
            fn(x, a)
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(5):
                fn(x, a)
            e1.record()
            e1.synchronize()
            ts[name] = e0.elapsed_time(e1) / 5
        if bad:
            _cast = _cast_torch
        log(f"fp8 cast: {ts} mismatched bytes={bad} -> {_cast.__name__}")
    except Exception as e:  # pragma: no cover - mirrors the reference's guarded check
        log(f"fp8 hip cast check failed: {e!r}")


# ---------------------------------------------------------------------------------------------
# skinny GEMM / GEMV
# ---------------------------------------------------------------------------------------------
def _check_weight_scale(ws, N):
    """The kernels read a weight's scale as one fp32 value or one per output row; 1 for the latter."""
    n = ws.numel()
    if ws.dtype != torch.float32 or (n != 1 and (n != N or not ws.is_contiguous())):
        raise ValueError(f"weight scale must be contiguous fp32 with 1 or {N} values, got {ws.dtype} {tuple(ws.shape)}")
    return 1 if n > 1 else 0


def _weight_operand(q):
    w8, ws = q[0], q[1]
    tiled = getattr(q, "tiled", None)
    L.require_device(w8, ws)
    shape = w8.shape
    _check_weight_scale(ws, shape[0])
    if tiled is not None:
        return tiled, L.W_TILED, ws, shape
    if w8.dtype != torch.float8_e4m3fn or w8.dim() != 2 or not w8.is_contiguous():
        raise ValueError("expected a contiguous float8_e4m3fn [N, K] weight")
    return w8, L.W_ROWMAJOR, ws, shape


FUSED_MAX_ELEMS = 8 * 64 * 64  # activation slice the GEMV can quantize in its prologue (static scale)
TILED_ROWS_MAX_K = 16384  # longest row krq_quant_rows_tiled takes (its vector kernel's register tile)
FUSED_MAX_ELEMS_DYN = 8 * 64 * 32  # row the GEMV can scale per token itself (M == 1)


def _gemv(xin, x_kind, x_scale, x_inv, M, q, split, mode, algo, out):
    w, layout, ws, (N, K) = _weight_operand(q)
    L.require_device(xin, x_scale, x_inv)
    xpr = 1 if (x_scale is not None and x_scale.numel() == M and M > 1) else 0
    wpr = 1 if ws.numel() > 1 else 0
    if out is None:
        if mode == L.OUT_PARTIAL:
            out = torch.empty((split, M, N), device=xin.device, dtype=torch.float32)
        else:
            out = torch.empty((M, N // 2 if mode == L.OUT_SWIGLU else N), device=xin.device,
                              dtype=torch.bfloat16)
    L.call("krq_gemv_fp8", L.ptr(xin), x_kind, L.ptr(x_scale), L.ptr(x_inv), xpr, L.ptr(w), layout,
           L.ptr(ws), wpr, M, N, K, split, mode, algo, L.ptr(out), L.stream(xin))
    return out


def gemv_fp8_launch(x8, xs, q, split=1, mode=L.OUT_BF16, algo=L.ALGO_AUTO, out=None):
    """One launch of the FP8 GEMV kernel on already-quantized activations.
    x8 float8_e4m3fn [M, K] (M <= 32); xs fp32 with 1 (per tensor) or M (per token) values;
    q = quantize(W) or quantize_weight(W). Returns out (allocated when None): bf16 [M, N],
    fp32 partials [split, M, N], or bf16 [M, N/2] for mode OUT_SWIGLU."""
    K = q[0].shape[1]
    M = x8.shape[0]
    if x8.dtype != torch.float8_e4m3fn or x8.dim() != 2 or x8.shape[1] != K or not x8.is_contiguous():
        raise ValueError(f"x8 must be a contiguous float8_e4m3fn [M, {K}] tensor")
    if xs.dtype != torch.float32 or xs.numel() not in (1, M):
        raise ValueError("xs must be fp32 with 1 or M values")
    return _gemv(x8, L.X_FP8, xs.reshape(-1), None, M, q, split, mode, algo, out)


def gemv_fp8_tiled_launch(x8t, xs, q, M, split=1, mode=L.OUT_BF16, out=None):
    """One launch of the FP8 GEMV (matrix-core kernel) on M rows of e4m3 activations in the tiled
    layout of quant_rows_tiled (x8t: 16 * ceil(M / 16) * K bytes) with their scales xs (1 or M
    values). Returns out as gemv_fp8_launch."""
    K = q[0].shape[1]
    mp = (M + 15) // 16 * 16
    if x8t.dtype != torch.uint8 or x8t.numel() != mp * K or not x8t.is_contiguous():
        raise ValueError(f"x8t must be a contiguous uint8 tensor of {mp * K} bytes (quant_rows_tiled)")
    if xs.dtype != torch.float32 or xs.numel() not in (1, M):
        raise ValueError("xs must be fp32 with 1 or M values")
    return _gemv(x8t, L.X_FP8_TILED, xs.reshape(-1), None, M, q, split, mode, L.ALGO_MFMA, out)


def gemv_fp8_bf16_launch(x, q, split=1, mode=L.OUT_BF16, a=None, algo=L.ALGO_AUTO, out=None):
    """One launch of the FP8 GEMV kernel on bf16 activations quantized inside the kernel:
    per token (M == 1, a is None) or with the inverse scale of an ActScale / SharedScale a."""
    x = _rows(x)
    M = x.shape[0]
    if a is None:
        return _gemv(x, L.X_BF16_DYN, None, None, M, q, split, mode, algo, out)
    return _gemv(x, L.X_BF16_STATIC, _one(a.scale), _one(a.inv), M, q, split, mode, algo, out)


def _one(scale):
    """A per-tensor scale (or its inverse) as the launches take it: one fp32 value (0-d or [1])."""
    if scale.dtype != torch.float32:
        raise ValueError(f"activation scales must be fp32, got {scale.dtype}")
    return scale if scale.numel() == 1 else scale.reshape(1)


def _fits_fused(x, M, K, split, a):
    """One row quantized in the GEMV's prologue (its activation wave). More rows with a given
    scale are cast first (row-major, or tiled from TILED_MIN_ROWS): quantizing them in the prologue
    measured slower on MI355X at every M > 1 (split 1, us, prologue / cast + GEMV): QKV M = 4
    9.19 / 6.92, M = 8 10.62 / 7.19; gate_up M = 4 15.78 / 11.33, M = 8 23.66 / 11.90."""
    if M != 1 or K % 64 or x.dtype != torch.bfloat16:
        return False
    if a is None:
        return K <= FUSED_MAX_ELEMS_DYN
    return K // split <= FUSED_MAX_ELEMS


def _activation_fp8(x, a, xs):
    """(x8, x_scale) for the GEMV when it does not quantize in its prologue: x8 given (fp8
    dtype) with xs; a static or per-call ActScale a (cast kernel); or per-token scales
    (quant_rows kernel)."""
    if x.dtype == torch.float8_e4m3fn:
        if xs is None:
            raise ValueError("float8 activations need their scale xs")
        if xs.dtype != torch.float32 or xs.numel() not in (1, x.shape[0]):
            raise ValueError("xs must be fp32 with 1 or M values")
        return x.contiguous(), xs.reshape(-1).contiguous()
    if a is not None:
        return _cast(x, a), _one(a.scale)
    x8, s = quant_rows(x)
    return x8, s.reshape(-1)


# From this many rows the GEMV reads tiled e4m3 rows (padded to 16-row tiles); below, row-major ones.
# Measured on MI355X (graph of 72 launches over 12 weight sets, per-token scales with the decode
# splits / a given scale at split 1), row-major against tiled, us: QKV M = 12 7.28 / 7.40, M = 16
# 7.52 / 7.40; gate_up M = 4 12.64 / 13.47, M = 16 14.19 / 13.70; down M = 4 9.70 / 10.35, M = 16
# 11.24 / 10.83; given scale M = 8 QKV 7.19 / 7.60, M = 16 8.25 / 7.68, M = 32 10.47 / 9.29.
TILED_MIN_ROWS = 13
# Split-K GEMVs take the tiled rows earlier where the launch whose workgroups share them in LDS
# (k_gemv_wide32; krq_gemv_fp8_shares_rows gives its workgroups) covers the chip. With a given scale,
# row-major / tiled, us, from three rows while they are one round on 256 compute units: eight layers'
# QKV (192 workgroups), O, down (160) and gate_up in one graph M = 2 273.8 / 279.7, M = 3 291.5 / 282.4,
# M = 7 303.7 / 288.2; 5,120 x 5,120 in two (160) M = 3 8.44 / 8.49, M = 8 9.21 / 8.54. On fewer a unit
# streams more (1,024 x 4,096 in four, 64, M = 5 5.02 / 5.64; 1,280 x 8,192 in two, 40, 7.23 / 9.58), on
# more the padding to sixteen rows costs (8,192 x 8,192 in four, 512, M = 5 15.4 / 17.7): there from
# eleven rows (11,008 x 4,096 in two, 344, M = 11 13.5 / 12.7, M = 5 12.2 / 12.6) and below 80
# workgroups not at all (1,280 x 8,192 in two M = 11 7.65 / 9.65). Scaled per token from eleven
# (the layers M = 9 284.8 / 287.1, M = 10 299.2 / 298.0, M = 12 305.2 / 298.7), by the same 80.
# Launches that do not share the rows lose by the padding: one K pass over a whole row (linear_fp8 over
# a layer's four projections at M = 5 36.4 us row-major, 43.0 tiled), weights without a tiled copy
# (down, given scale, M = 5 11.3 / 11.8), N = 16 mod 64 (2,576 x 9,728, M = 5 8.9 / 9.5), long splits
# (2,560 x 16,384 in two, M = 5 14.2 / 16.1). Split-K launches of those kinds take the tiled rows from
# TILED_MIN_ROWS (M = 12 per token 9.8 / 10.0 at 2,576 x 9,728), with a given scale from eleven (M = 11
# without a tiled copy: QKV 8.8 / 8.4, down 12.3 / 12.1).
TILED_MIN_ROWS_SPLIT = {"given": 3, "token": 11}
TILED_MIN_ROWS_SPLIT_APART = {"given": 11, "token": TILED_MIN_ROWS}
TILED_SPLIT_MANY_ROWS, TILED_SPLIT_LEAST_GROUPS, TILED_SPLIT_ONE_ROUND = 11, 80, (144, 240)


def _tiled_least(q, M, split, a):
    """The rows from which a split-K gemv_fp8 call of M < TILED_MIN_ROWS rows takes tiled rows."""
    kind = "token" if a is None else "given"
    if M < TILED_MIN_ROWS_SPLIT[kind]:
        return TILED_MIN_ROWS
    N, K = q[0].shape
    tiled = getattr(q, "tiled", None) is not None
    groups = L.lib().krq_gemv_fp8_shares_rows(M, N, K, split, L.W_TILED) if tiled else 0
    if groups == 0:
        return TILED_MIN_ROWS_SPLIT_APART[kind]
    least, most = TILED_SPLIT_ONE_ROUND
    if least <= groups <= most:
        return TILED_MIN_ROWS_SPLIT[kind]
    return TILED_SPLIT_MANY_ROWS if groups >= TILED_SPLIT_LEAST_GROUPS else TILED_MIN_ROWS


def _tiled_rows(x, M, K, a, xs, algo, least=TILED_MIN_ROWS):
    """bf16 rows at `least` <= M <= 32 go through quant_rows_tiled (scaled per token) or
    cast_tiled (a given scale) and the GEMV on tiled activations (the operands of quant_rows / _cast
    + the row-major e4m3 GEMV, with contiguous loads); fewer rows, rows longer than the tiled
    kernels take, and below TILED_MIN_ROWS rows that do not start on 16 bytes (the row-major
    quantizers take any address) use the row-major kernels, as do given-scale rows where pick_cast
    has put torch's cast in the place of the HIP one."""
    return (least <= M <= DECODE_MAX_ROWS and xs is None and x.dtype == torch.bfloat16 and K % 64 == 0
            and K <= TILED_ROWS_MAX_K and algo != L.ALGO_VALU and (a is None or _cast is _cast_hip)
            and (M >= TILED_MIN_ROWS or x.data_ptr() % 16 == 0))


def _tiled_operand(x, a):
    """(x8 tiled, x_scale) for _tiled_rows inputs: per token, or with the given scale."""
    if a is None:
        return quant_rows_tiled(x)
    return cast_tiled(x, a), _one(a.scale)


def _chunked(x8, xs, fn):
    M = x8.shape[0]
    if M <= DECODE_MAX_ROWS:
        return fn(x8, xs)
    outs = []
    for m0 in range(0, M, DECODE_MAX_ROWS):
        m1 = min(M, m0 + DECODE_MAX_ROWS)
        outs.append(fn(x8[m0:m1], xs[m0:m1] if xs.numel() == M else xs))
    return torch.cat(outs, dim=-2)


def gemv_fp8(x, q, split=1, a=None, xs=None, algo=L.ALGO_AUTO):
    """FP8 counterpart of kernels.gemv.gemv: x [M, K] bf16 (or float8_e4m3fn with xs), q from
    quantize / quantize_weight. split == 1: bf16 [M, N]; split > 1: fp32 partials [split, M, N]
    whose in-order sum is the product. Activations are scaled per token unless an ActScale /
    SharedScale `a` is given. Called as fp8.gemv_fp8(x, q, split) by the reference's
    experiments/modal_fp8.py:69."""
    M, K = x.shape
    assert K % split == 0
    mode = L.OUT_BF16 if split == 1 else L.OUT_PARTIAL
    if xs is None and _fits_fused(x, M, K, split, a):
        return gemv_fp8_bf16_launch(x, q, split, mode, a, algo)
    least = TILED_MIN_ROWS if split == 1 or M >= TILED_MIN_ROWS else _tiled_least(q, M, split, a)
    if _tiled_rows(x, M, K, a, xs, algo, least):
        x8t, s = _tiled_operand(x, a)
        return gemv_fp8_tiled_launch(x8t, s, q, M, split, mode)
    x8, s = _activation_fp8(x, a, xs)
    return _chunked(x8, s, lambda xc, sc: gemv_fp8_launch(xc, sc, q, split, mode, algo))


def gemv_swiglu_fp8(x, q, a=None, xs=None, algo=L.ALGO_AUTO):
    """FP8 counterpart of kernels.gemv.gemv_swiglu: q quantizes w_gu [2I, K] = [gate; up];
    returns bf16(bf16(silu(bf16 g)) * bf16 u) [M, I]. Called as fp8.gemv_swiglu_fp8(x, q) by the
    reference's experiments/modal_fp8.py:67."""
    M, K = x.shape
    if xs is None and _fits_fused(x, M, K, 1, a):
        return gemv_fp8_bf16_launch(x, q, 1, L.OUT_SWIGLU, a, algo)
    if _tiled_rows(x, M, K, a, xs, algo):
        x8t, s = _tiled_operand(x, a)
        return gemv_fp8_tiled_launch(x8t, s, q, M, 1, L.OUT_SWIGLU)
    x8, s = _activation_fp8(x, a, xs)
    return _chunked(x8, s, lambda xc, sc: gemv_fp8_launch(xc, sc, q, 1, L.OUT_SWIGLU, algo))


def swiglu_cast_fp8(x, q, out_a, a=None, xs=None):
    """gemv_swiglu_fp8(x, q, a, xs) cast for the next projection in the same launch
    (krq_gemv_swiglu_fp8_cast): the SwiGLU epilogue writes e4m3(clamp(act * out_a.inv, +-448)) of
    its bf16 act in the tiled activation layout of quant_rows_tiled, i.e. the bytes of
    _cast(act, out_a) permuted, with no bf16 act stored and no cast launch. out_a is the next
    projection's ActScale / SharedScale (device inv and scale), as the engine's static-scale decode
    MLP passes it to linear_fp8 (engine/engine.py:977-981). M <= 32. Returns (x8_tiled uint8
    [16 ceil(M / 16) * I], scale fp32 [1]) for gemv_fp8_tiled_launch."""
    w, layout, ws, (N, K) = _weight_operand(q)
    M = x.shape[0]
    if M > DECODE_MAX_ROWS or x.dim() != 2 or x.shape[1] != K:
        raise ValueError(f"swiglu_cast_fp8: x {tuple(x.shape)} against w [{N}, {K}] (M <= {DECODE_MAX_ROWS})")
    if N % 128:
        raise ValueError(f"swiglu_cast_fp8: the activation width {N // 2} must be a multiple of 64")
    if xs is None and _fits_fused(x, M, K, 1, a):
        xin = _rows(x)
        kind, x_scale, x_inv = (L.X_BF16_DYN, None, None) if a is None else \
            (L.X_BF16_STATIC, _one(a.scale), _one(a.inv))
    elif _tiled_rows(x, M, K, a, xs, L.ALGO_AUTO):
        xin, x_scale = _tiled_operand(x, a)
        kind, x_inv = L.X_FP8_TILED, None
    else:
        xin, x_scale = _activation_fp8(x, a, xs)
        kind, x_inv = L.X_FP8, None
    L.require_device(xin, x_scale, x_inv, out_a.inv)
    xpr = 1 if (x_scale is not None and x_scale.numel() == M and M > 1) else 0
    MP = 16 * ((M + 15) // 16)
    x8t = torch.empty((MP * (N // 2),), device=x.device, dtype=torch.uint8)
    L.call("krq_gemv_swiglu_fp8_cast", L.ptr(xin), kind, L.ptr(x_scale), L.ptr(x_inv), xpr, L.ptr(w), layout,
           L.ptr(ws), 1 if ws.numel() > 1 else 0, M, N, K, L.ptr(_one(out_a.inv)), L.ptr(x8t), L.stream(x))
    return x8t, _one(out_a.scale).reshape(1)


def gemm_fp8(x, q, a=None, xs=None):
    """Prefill FP8 GEMM (krq_gemm_fp8_ws): bf16 [M, N] = bf16(x8 . w8^T * x_scale[m] * w_scale[n]),
    the product torch._scaled_mm gives linear_fp8 (engine/kernels/fp8.py:105-106).
    x is bf16 [M, K] with an ActScale / SharedScale `a`, or float8_e4m3fn [M, K] with its scale xs
    (1 or M values); q from quantize_weight / quantize, N and K multiples of 128. bf16 rows are cast
    once (krq_cast_fp8) and multiplied by the e4m3 kernels where those run (K >= 256), else the
    cast is fused into the 128 x 128 kernel's A staging; both give the bytes of the reference's
    cast followed by the e4m3 product."""
    w8, ws = q[0], q[1]
    L.require_device(x, w8, ws)
    if w8.dtype != torch.float8_e4m3fn or w8.dim() != 2 or not w8.is_contiguous():
        raise ValueError("expected a contiguous float8_e4m3fn [N, K] weight")
    N, K = w8.shape
    _check_weight_scale(ws, N)
    if x.dim() != 2 or x.shape[1] != K:
        raise ValueError(f"x {tuple(x.shape)} does not match w8 {tuple(w8.shape)}")
    M = x.shape[0]
    if x.dtype == torch.float8_e4m3fn:
        if xs is None or xs.dtype != torch.float32 or xs.numel() not in (1, M):
            raise ValueError("float8 activations need their fp32 scale xs (1 or M values)")
        kind, xin, x_scale, x_inv = L.X_FP8, x.contiguous(), xs.reshape(-1).contiguous(), None
    else:
        if a is None:
            raise ValueError("bf16 activations need an ActScale / SharedScale a")
        if K % 128 == 0 and K >= 256:
            return gemm_fp8(_cast_hip(_rows(x), a), q, xs=_one(a.scale))
        kind, xin, x_scale, x_inv = L.X_BF16_STATIC, _rows(x), _one(a.scale), _one(a.inv)
    L.require_device(x_scale, x_inv)
    xpr = 1 if (x_scale.numel() == M and M > 1) else 0
    out = torch.empty((M, N), device=x.device, dtype=torch.bfloat16)
    nbytes = L.lib().krq_gemm_fp8_ws_bytes(kind, M, N, K)
    if nbytes < 0:
        raise RuntimeError("krq_gemm_fp8_ws_bytes: device query failed")
    work = torch.empty(nbytes, device=x.device, dtype=torch.uint8) if nbytes else None
    L.call("krq_gemm_fp8_ws", L.ptr(xin), kind, L.ptr(x_scale), L.ptr(x_inv), xpr, L.ptr(w8), L.ptr(ws),
           1 if ws.numel() > 1 else 0, M, N, K, L.ptr(work), nbytes, L.ptr(out), L.stream(xin))
    return out


def linear_fp8(x, q, a=None, amax_out=None):
    """bf16 [M, N] ~= x @ W^T with q = quantize_weight(W); a = given scale, or
    None to scale by this tensor's own range (running max kept in amax_out).
    Reference: engine/kernels/fp8.py:97-106. Decode sizes (M <= 32) run the HIP GEMV; more rows
    run this library's GEMM (gemm_fp8) where its e4m3 kernels take the weight (N and K multiples of
    128, K >= 256) and, below 128 rows, where it pays (_ring_pays); the rest keep the reference's
    library GEMM, torch._scaled_mm (hipBLASLt on ROCm)."""
    w8, ws = q[0], q[1]
    M, K = x.shape
    gemm = M > DECODE_MAX_ROWS and _takes_gemm(M, w8, ws)
    if gemm and _cast is _cast_hip:
        return _linear_gemm(x, q, a, amax_out)
    x8 = None
    if a is None:
        if M > DECODE_MAX_ROWS and _cast is _cast_hip:
            a, x8 = _act_scale_cast(x)
        else:
            a = ActScale(x)
        if amax_out is not None:
            amax_out.copy_(torch.maximum(amax_out, a.amax.reshape(1)))
    if x8 is None and _fits_fused(x, M, K, 1, a):
        return gemv_fp8_bf16_launch(x, q, 1, L.OUT_BF16, a)
    if x8 is None and _tiled_rows(x, M, K, a, None, L.ALGO_AUTO):
        return gemv_fp8_tiled_launch(cast_tiled(x, a), _one(a.scale), q, M, 1, L.OUT_BF16)
    if x8 is None:
        x8 = _cast(x, a)
    if M <= DECODE_MAX_ROWS:
        return gemv_fp8_launch(x8, _one(a.scale), q, 1, L.OUT_BF16)
    if gemm:
        return gemm_fp8(x8, q, xs=_one(a.scale))
    return torch._scaled_mm(x8, w8.t(), scale_a=a.scale, scale_b=ws, out_dtype=torch.bfloat16)


def _linear_gemm(x, q, a, amax_out):
    """linear_fp8 on the ring GEMM: the scale (without a given one), the cast and the product, their
    scale, e4m3 rows and partials in one allocation beside the output. A call on a short prompt is
    host work (the launches take 3 us each): 37 us with an allocation per piece and the launches
    through ActScale and gemm_fp8, 17 us this way."""
    w8, ws = q[0], q[1]
    N, K = w8.shape
    wpr = _check_weight_scale(ws, N)
    if a is not None:
        inv, given = _one(a.inv), _one(a.scale)
        L.require_device(inv, given)
    x2 = _rows(x)
    M, kx = x2.shape
    L.require_device(w8, ws)
    if kx != K:
        raise ValueError(f"x {tuple(x.shape)} does not match w8 {tuple(w8.shape)}")
    lib = L.lib()
    parts = 4 * lib.krq_act_scale_ws_floats(M, K) if a is None else 0
    split_bytes = lib.krq_gemm_fp8_ws_bytes(L.X_FP8, M, N, K)
    if split_bytes < 0:
        raise RuntimeError("krq_gemm_fp8_ws_bytes: device query failed")
    # amax, inv, scale and the maxima's partials | e4m3 rows | split-K partials
    at8 = (16 + parts + 255) & -256
    at_split = (at8 + M * K + 255) & -256
    work = torch.empty(at_split + split_bytes, device=x2.device, dtype=torch.uint8)
    out = torch.empty((M, N), device=x2.device, dtype=torch.bfloat16)
    p, st = work.data_ptr(), L.stream(x2)
    if a is None:
        scale = p + 8
        L.call("krq_act_scale_cast_fp8", L.ptr(x2), M, K, 1.0, p, p + 4, scale, p + 16, p + at8, st)
        if amax_out is not None:
            amax_out.copy_(torch.maximum(amax_out, work[:4].view(torch.float32)))
    else:
        scale = L.ptr(given)
        L.call("krq_cast_fp8", L.ptr(x2), M, K, L.ptr(inv), 0, p + at8, st)
    L.call("krq_gemm_fp8_ws", p + at8, L.X_FP8, scale, None, 0, L.ptr(w8), L.ptr(ws), wpr, M, N, K,
           p + at_split if split_bytes else None, split_bytes, L.ptr(out), st)
    return out


def _gemm_min_rows(w8, ws):
    """The rows from which linear_fp8 runs this library's GEMM on a weight. Below
    PER_CHANNEL_MIN_ROWS what the library's product refuses (per-channel scales, scales that are
    not fp32) or alone takes (a weight that does not start on 16 bytes) stays with it; see _ring_pays
    for the rest."""
    if not _ring_gemm_fits(w8):
        return float("inf")
    own = ws.numel() == 1 and ws.dtype == torch.float32 and w8.data_ptr() % 16 == 0
    return PREFILL_MIN_ROWS if own else PER_CHANNEL_MIN_ROWS


def _takes_gemm(M, w8, ws):
    """Whether linear_fp8 runs this library's GEMM on M > DECODE_MAX_ROWS rows of a weight."""
    return M >= _gemm_min_rows(w8, ws) and (M >= PER_CHANNEL_MIN_ROWS or _ring_pays(M, *w8.shape))


def _ring_pays(M, N, K):
    """Below PER_CHANNEL_MIN_ROWS rows: the weights on which a linear_fp8 call is no slower through this
    library's GEMM than through torch._scaled_mm. Such calls are made one by one (prefill), where the
    library's takes 39 us of host time and this one 16.5, so up to 64 MiB of weights it is the faster
    one, also where its product is not. Measured, us, called / captured in a graph with others:
      19,456 x 2,560  M = 77 24.7 against 40.6 / 25.2 against 25.5, M = 127 28.5 against 39.2 / 29.2, 26.5
      4,096 x 5,120   M = 64 21 against 42 / 21.7 against 16.7
      1,024 x 6,144   M = 64 18.7 against 42 / 17.0 against 12.5
      128 x 16,384    M = 64 33 against 42 / 33.2 against 15.1; 128 x 32,768 61 against 43
    (the last three: few tiles over a long K that the plan does not split, for which a captured call
    is slower; past K = 16,384 the called one is too). Larger weights keep the library (28,672 x 8,192
    M = 127 77 against 61, 32,000 x 4,096 51 against 40, 16,384 x 16,384 84 against 76) but for
    vocabularies over short rows (151,936 x 2,560 M = 77 92 against 114, 65,536 x 3,584 M = 64 50
    against 50; 80,000 x 4,096 M = 33 98 against 85) and long rows in split K (8,192 x 28,672 M = 77
    64 against 198, 2,560 x 32,768 42 against 108, 8,192 x 18,432 M = 64 46 against 60). From 2 GiB
    gemm_fp8 leaves the ring kernels all this was measured on."""
    if N * K > 1 << 26:
        return N * K < 0x7fffffff and ((N >= 65536 and K < 4096) or (2560 <= N <= 8192 and K >= 18432))
    return K <= 16384 or L.lib().krq_gemm_fp8_ws_bytes(L.X_FP8, M, N, K) != 0


def _ring_gemm_fits(w8):
    """The weight shapes gemm_fp8 multiplies with its ring kernels on e4m3 rows."""
    if w8.dtype != torch.float8_e4m3fn or w8.dim() != 2 or not w8.is_contiguous():
        return False
    N, K = w8.shape
    return N % 128 == 0 and K % 128 == 0 and K >= 256
