"""Host-side checks of the drop-in boundary that need no GPU: the C-ABI library loads and exports
every symbol include/krq.h declares, argument validation maps to the reference's exception
types, and nothing silently runs on the CPU."""

import ctypes
import os
import re

import pytest
import torch

from kernels import _lib as L
from kernels import fp8, gemv as G

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def header_symbols():
    text = open(os.path.join(ROOT, "include", "krq.h")).read()
    return set(re.findall(r"^\s*(?:int|int64_t|const char\*)\s+(krq_\w+)\s*\(", text, re.M))


def test_library_exports_every_header_symbol():
    lib = L.lib()
    declared = header_symbols()
    assert declared == set(L.EXPORTS), declared ^ set(L.EXPORTS)
    for name in declared:
        assert hasattr(lib, name)
    assert lib.krq_version().decode().startswith("krq")
    # the per-block stamps exist only in the timeline build (build_lib.py --timeline)
    assert not hasattr(lib, "krq_timeline_read")


def test_workspace_sizes_are_host_only():
    lib = L.lib()
    assert lib.krq_lmhead_ws_bytes(16, 151936) >= 256 + 16 * 8 * (151936 // 64)
    assert lib.krq_act_scale_ws_floats(16, 2560) >= 1


def _null():
    return ctypes.c_void_p(0)


def test_invalid_arguments_fail_before_any_launch():
    lib = L.lib()
    p = ctypes.c_void_p(4096)  # never dereferenced: validation rejects the call first
    # M out of range
    rc = lib.krq_gemv_fp8(p, 0, p, None, 0, p, 1, p, 1, 0, 64, 256, 1, 0, 0, p, _null())
    assert rc == L.KRQ_EINVAL and b"M=0" in lib.krq_last_error()
    # K/split not a multiple of 64
    rc = lib.krq_gemv_fp8(p, 0, p, None, 0, p, 1, p, 1, 1, 64, 200, 1, 0, 0, p, _null())
    assert rc == L.KRQ_EINVAL and b"K_SPLIT" in lib.krq_last_error()
    # in-kernel per-token scaling takes one row; static scaling needs x_inv
    rc = lib.krq_gemv_fp8(p, 1, None, None, 0, p, 1, p, 1, 2, 64, 256, 1, 0, 0, p, _null())
    assert rc == L.KRQ_EINVAL and b"M == 1" in lib.krq_last_error()
    rc = lib.krq_gemv_fp8(p, 2, p, None, 0, p, 1, p, 1, 2, 64, 256, 1, 0, 0, p, _null())
    assert rc == L.KRQ_EINVAL and b"x_inv" in lib.krq_last_error()
    # split > 1 without the partials output
    rc = lib.krq_gemv_bf16(p, p, 0, 1, 64, 256, 2, 0, p, _null())
    assert rc == L.KRQ_EINVAL
    # persistent BF16 GEMV: at least one program, whole 32-element K tiles
    rc = lib.krq_gemv_bf16_rows(p, p, 1, 64, 256, 0, 0, p, _null())
    assert rc == L.KRQ_EINVAL and b"programs=0" in lib.krq_last_error()
    rc = lib.krq_gemv_bf16_rows(p, p, 1, 64, 200, 4, 0, p, _null())
    assert rc == L.KRQ_EINVAL and b"multiple of 32" in lib.krq_last_error()
    # tiled activations take the matrix-core kernel; their quantizer needs K % 64 == 0
    rc = lib.krq_gemv_fp8(p, L.X_FP8_TILED, p, None, 0, p, 1, p, 1, 1, 64, 256, 1, 0, 2, p, _null())
    assert rc == L.KRQ_EINVAL and b"tiled activations" in lib.krq_last_error()
    # the activation scale with its cast: every pointer, a real shape
    rc = lib.krq_act_scale_cast_fp8(p, 16, 2560, 1.0, p, p, p, None, p, _null())
    assert rc == L.KRQ_EINVAL and b"null pointer" in lib.krq_last_error()
    rc = lib.krq_act_scale_cast_fp8(p, 0, 2560, 1.0, p, p, p, p, p, _null())
    assert rc == L.KRQ_EINVAL and b"bad shape" in lib.krq_last_error()
    rc = lib.krq_quant_rows_tiled(p, 16, 100, p, p, _null())
    assert rc == L.KRQ_EINVAL and b"K=100" in lib.krq_last_error()
    rc = lib.krq_quant_rows_tiled(p, 16, 16384 + 64, p, p, _null())
    assert rc == L.KRQ_EINVAL and b"K at most 16384" in lib.krq_last_error()
    rc = lib.krq_rmsnorm_quant_rows_tiled(p, p, p, 1e-6, 2, 2576, p, p, _null())
    assert rc == L.KRQ_EINVAL and b"multiple of 64" in lib.krq_last_error()
    # the tiled e4m3 lm_head rows need their per-row scales
    rc = lib.krq_lmhead_argmax(p, None, 1, p, L.LM_FP8_TILED_H, 1, p, 1, 16, 1024, 256, None, p, 1 << 20, p,
                               _null())
    assert rc == L.KRQ_EINVAL and b"h_scale" in lib.krq_last_error()
    # the allocation-free lm_head: its argument checks, then its scratch limit, before any HIP call
    rc = lib.krq_lmhead_argmax_noalloc(p, None, 1, p, L.LM_FP8_TILED_H, 1, p, 1, 16, 1024, 256, None, p,
                                       _null())
    assert rc == L.KRQ_EINVAL and b"h_scale" in lib.krq_last_error()
    assert lib.krq_lmhead_ws_bytes(32, 262144) == L.LMHEAD_SCRATCH_BYTES
    rc = lib.krq_lmhead_argmax_noalloc(p, p, 1, p, L.LM_FP8, 1, p, 1, 32, 262144 + 16, 2560, None, p, _null())
    assert rc == L.KRQ_EINVAL and b"scratch maximum of 4194304" in lib.krq_last_error()
    # null pointers
    rc = lib.krq_quant_fp8_rows(None, 16, 64, 64, p, None, p, _null())
    assert rc == L.KRQ_EINVAL
    # workspace too small
    rc = lib.krq_lmhead_argmax(p, None, 0, p, 0, 0, None, 0, 1, 1024, 256, None, p, 8, p, _null())
    assert rc == L.KRQ_EINVAL and b"workspace" in lib.krq_last_error()
    with pytest.raises(ValueError):
        L.call("krq_pack_fp8", p, 17, 64, p, _null())
    # fused MLP: one-row in-kernel scaling only; staging limit
    rc = lib.krq_mlp_fp8(p, 1, None, p, 1, p, 1, p, p, 1, 2, 2560, 9728, 4, p, p, 0, p, _null())
    assert rc == L.KRQ_EINVAL and b"M == 1" in lib.krq_last_error()
    rc = lib.krq_mlp_fp8(p, 0, p, p, 1, p, 1, p, p, 1, 32, 2560, 9728, 1, p, p, 0, p, _null())
    assert rc == L.KRQ_EINVAL and b"raise split" in lib.krq_last_error()
    # fused BF16 GEMV: residual epilogue needs its buffers; slices that do not fit are refused
    rc = lib.krq_gemv_bf16_fused(p, p, 0, 1, 2560, 4096, 4, L.OUT_RESIDUAL, None, None, 1e-6,
                                 None, None, None, None, p, _null())
    assert rc == L.KRQ_EINVAL and b"res_in" in lib.krq_last_error()
    rc = lib.krq_gemv_bf16_fused(p, p, 0, 16, 19456, 2560, 1, L.OUT_SWIGLU, p, p, 1e-6,
                                 None, None, None, None, p, _null())
    assert rc == L.KRQ_EINVAL and b"krq_rmsnorm_rows" in lib.krq_last_error()
    assert lib.krq_gemv_fused_fits(1, 6144, 2560, 2, L.OUT_PARTIAL, 1) == 1
    assert lib.krq_gemv_fused_fits(16, 19456, 2560, 1, L.OUT_SWIGLU, 1) == 0
    # fused FP8 GEMV: something to fuse; RMSNorm needs bf16 activations; per-token in-kernel
    # scaling takes one row; the residual epilogue needs its buffers
    args = (p, 1, None, None, 0, p, 1, p, 1)
    rc = lib.krq_gemv_fp8_fused(*args, 1, 6144, 2560, 2, L.OUT_PARTIAL, None, None, 1e-6, None, None, None,
                                None, p, _null())
    assert rc == L.KRQ_EINVAL and b"krq_gemv_fp8" in lib.krq_last_error()
    rc = lib.krq_gemv_fp8_fused(p, 0, p, None, 0, p, 1, p, 1, 1, 6144, 2560, 2, L.OUT_PARTIAL, p, p, 1e-6,
                                None, None, None, None, p, _null())
    assert rc == L.KRQ_EINVAL and b"bf16 activations" in lib.krq_last_error()
    rc = lib.krq_gemv_fp8_fused(*args, 2, 6144, 2560, 2, L.OUT_PARTIAL, p, p, 1e-6, None, None, None,
                                None, p, _null())
    assert rc == L.KRQ_EINVAL and b"M == 1" in lib.krq_last_error()
    # (split 2: at M = 1 the four-split residual runs folded and needs no counters)
    rc = lib.krq_gemv_fp8_fused(*args, 1, 2560, 4096, 2, L.OUT_RESIDUAL, None, None, 1e-6, p, p, p, None,
                                p, _null())
    assert rc == L.KRQ_EINVAL and b"cnt" in lib.krq_last_error()
    rc = lib.krq_gemv_fp8_fused(*args, 1, 2560, 4096, 4, L.OUT_RESIDUAL, p, p, 1e-6, p, p, p, p, p, _null())
    assert rc == L.KRQ_EINVAL and b"in one call" in lib.krq_last_error()
    assert lib.krq_gemv_fp8_fused_fits(1, 6144, 2560, 2, L.OUT_PARTIAL, L.X_BF16_DYN, 1) == 1
    assert lib.krq_gemv_fp8_fused_fits(16, 6144, 2560, 2, L.OUT_PARTIAL, L.X_BF16_DYN, 1) == 0
    assert lib.krq_gemv_fp8_fused_fits(4, 6144, 2560, 2, L.OUT_PARTIAL, L.X_BF16_STATIC, 1) == 1
    assert lib.krq_gemv_fp8_fused_fits(16, 6144, 2560, 2, L.OUT_PARTIAL, L.X_BF16_STATIC, 1) == 0
    assert lib.krq_gemv_fp8_fused_fits(32, 19456, 2560, 1, L.OUT_SWIGLU, L.X_BF16_STATIC, 1) == 0
    assert lib.krq_gemv_fp8_fused_fits(1, 2560, 9728, 4, L.OUT_RESIDUAL, L.X_FP8, 0) == 1
    rc = lib.krq_rmsnorm_quant_rows(p, p, p, 1e-6, 1, 16384 + 16, p, p, _null())
    assert rc == L.KRQ_EINVAL and b"at most 16384" in lib.krq_last_error()
    rc = lib.krq_rmsnorm_rows(p, p, p, 1e-6, 1, 20000, p, _null())
    assert rc == L.KRQ_EINVAL and b"at most 16384" in lib.krq_last_error()
    # prefill GEMM: N and K multiples of 128; bf16 activations need their inverse scale
    rc = lib.krq_gemm_fp8(p, L.X_FP8, p, None, 0, p, p, 1, 256, 200, 256, p, _null())
    assert rc == L.KRQ_EINVAL and b"multiples of 128" in lib.krq_last_error()
    rc = lib.krq_gemm_fp8(p, L.X_BF16_STATIC, p, None, 0, p, p, 1, 256, 256, 256, p, _null())
    assert rc == L.KRQ_EINVAL and b"x_inv" in lib.krq_last_error()
    rc = lib.krq_gemm_fp8(p, L.X_BF16_DYN, p, p, 0, p, p, 1, 256, 256, 256, p, _null())
    assert rc == L.KRQ_EINVAL and b"x_kind" in lib.krq_last_error()
    # the workspace form: the same checks, and a size that disagrees with its pointer is refused;
    # no split (0 bytes) where the ring kernels do not run (bf16 activations, K below 256)
    rc = lib.krq_gemm_fp8_ws(p, L.X_FP8, p, None, 0, p, p, 1, 256, 200, 256, p, 0, p, _null())
    assert rc == L.KRQ_EINVAL and b"multiples of 128" in lib.krq_last_error()
    rc = lib.krq_gemm_fp8_ws(p, L.X_FP8, p, None, 0, p, p, 1, 256, 256, 256, None, 1024, p, _null())
    assert rc == L.KRQ_EINVAL and b"workspace" in lib.krq_last_error()
    rc = lib.krq_gemm_fp8_ws(p, L.X_FP8, p, None, 0, p, p, 1, 256, 256, 256, p, -1, p, _null())
    assert rc == L.KRQ_EINVAL and b"workspace" in lib.krq_last_error()
    assert lib.krq_gemm_fp8_ws_bytes(L.X_BF16_STATIC, 256, 2560, 9728) == 0
    assert lib.krq_gemm_fp8_ws_bytes(L.X_FP8, 256, 2560, 128) == 0
    assert lib.krq_gemm_fp8_ws_bytes(L.X_FP8, 256, 200, 9728) == 0


def test_fused_buffers_and_mlp_contracts():
    from kernels.fused_gemv import FusedLayerBuffers
    from kernels.mlp import PersistentMLP
    b = FusedLayerBuffers(4, 2560, 151936, "cpu")
    assert b.res.shape == (2, 4, 2560) and b.res.dtype == torch.bfloat16
    assert b.ss.shape == (2, 4, 160) and b.cnt.shape == (151936 // 8,)
    pm = PersistentMLP(1, 2560, 9728, "cpu")
    assert pm.ctl.numel() == L.lib().krq_mlp_ctl_words() and int(pm.ctl.abs().sum()) == 0
    with pytest.raises(AssertionError):
        PersistentMLP(1, 2560, 9728 + 16, "cpu")          # the reference's chunk contract
    with pytest.raises(ValueError):
        pm(torch.zeros(1, 2560, dtype=torch.bfloat16), torch.zeros(1), torch.zeros(1))


def test_no_cpu_path():
    w = torch.zeros(16, 64, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="ROCm device"):
        fp8.quantize(w)
    with pytest.raises(RuntimeError, match="ROCm device"):
        G.gemv(torch.zeros(1, 64, dtype=torch.bfloat16), w)


def test_reference_helpers():
    assert G._bm(1) == 16 and G._bm(16) == 16 and G._bm(17) == 32 and G._bm(32) == 32
    with pytest.raises(ValueError):
        G._prune(G._CONFIGS, {"K_SPLIT": 48, "N": 64})
    assert G._prune(G._CONFIGS, {"K": 64, "N": 32})
    with pytest.raises(ValueError):
        G.gemv_tma(torch.zeros(1, 64), torch.zeros(64, 64))
    with pytest.raises(AssertionError):
        G.gemv_m1(torch.zeros(2, 64, dtype=torch.bfloat16), torch.zeros(16, 64, dtype=torch.bfloat16))
    assert fp8.FP8_MAX == 448.0
    q = fp8.FP8Weight(torch.zeros(1), torch.ones(()), None)
    w8, s = q
    assert isinstance(q, tuple) and q.tiled is None and s.item() == 1.0


def test_bench_refuses_more_than_one_gpu():
    """bench.py measures one GPU: --gpus N > 1 exits with a message before touching a device."""
    import subprocess
    import sys
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 2 and "one GPU" in r.stderr and r.stdout == ""


def test_fused_and_gemm_wrappers_refuse_cpu_tensors():
    from kernels import fused_gemv as FG
    x = torch.zeros(1, 256, dtype=torch.bfloat16)
    w = torch.zeros(32, 256, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="ROCm device"):
        FG.gemv_fused(x, w, 1)
    q = fp8.FP8Weight(torch.zeros(128, 256, dtype=torch.float8_e4m3fn), torch.ones(()), None)
    with pytest.raises(RuntimeError, match="ROCm device"):
        FG.gemv_fused(x, q, 1, ep=(x, x, x, x))
    with pytest.raises(RuntimeError, match="ROCm device"):
        fp8.gemm_fp8(torch.zeros(64, 256, dtype=torch.float8_e4m3fn), q, xs=torch.ones(1))


def test_linear_gemm_rows():
    """linear_fp8's line to this library's GEMM: one fp32 scale and an aligned weight from the first
    row past the decode sizes, other weights of its shapes from PER_CHANNEL_MIN_ROWS, the rest never."""
    w8 = torch.zeros(256 * 512 + 8, dtype=torch.uint8).view(torch.float8_e4m3fn)
    own, off = w8[:256 * 512].view(256, 512), w8[8:].view(256, 512)
    assert own.data_ptr() % 16 == 0
    one = torch.ones(())
    assert fp8._gemm_min_rows(own, one) == fp8._gemm_min_rows(own, one.reshape(1)) == fp8.PREFILL_MIN_ROWS
    for w, ws in ((off, one), (own, one.double()), (own, torch.ones(256))):
        assert fp8._gemm_min_rows(w, ws) == fp8.PER_CHANNEL_MIN_ROWS
    for w in (own[:, :128].contiguous(), own[:, :256], own[:200], own.view(torch.uint8)):
        assert fp8._gemm_min_rows(w, one) == float("inf")


def test_scales_are_fp32_of_the_right_count():
    """The kernels read scales through float pointers: another type, another number of values or
    strided ones are refused before any launch (and before the device is looked at)."""
    N, K = 256, 512
    w8 = torch.zeros(N, K, dtype=torch.uint8).view(torch.float8_e4m3fn)
    x = torch.zeros(128, K, dtype=torch.bfloat16)
    good = torch.ones(())
    for ws in (good.double(), torch.ones(N).bfloat16(), torch.ones(7), torch.ones(2 * N)[::2], good.expand(N)):
        with pytest.raises(ValueError, match="weight scale"):
            fp8._check_weight_scale(ws, N)
        with pytest.raises(ValueError, match="weight scale"):
            fp8.linear_fp8(x, (w8, ws))
    for ws in (good, good.reshape(1), torch.ones(N), torch.ones(N, 1)):
        fp8._check_weight_scale(ws, N)
    for a in (fp8.SharedScale(good, good.double()), fp8.SharedScale(good.bfloat16(), good)):
        with pytest.raises(ValueError, match="fp32"):
            fp8.linear_fp8(x, (w8, good), a)
    with pytest.raises(ValueError, match="fp32"):
        fp8._activation_fp8(x.to(torch.float8_e4m3fn), None, good.double())


def test_given_scale_rows_keep_the_picked_cast(monkeypatch):
    """Rows with a given scale take the tiled cast kernel only while pick_cast keeps the HIP cast."""
    a = fp8.SharedScale(torch.ones(1), torch.ones(()))
    x = {M: torch.zeros(M, 256, dtype=torch.bfloat16) for M in (3, 12, 13, 32)}
    assert all(fp8._tiled_rows(v, *v.shape, a, None, L.ALGO_AUTO, 3) for v in x.values())
    monkeypatch.setattr(fp8, "_cast", fp8._cast_torch)
    assert not any(fp8._tiled_rows(v, *v.shape, a, None, L.ALGO_AUTO, 3) for v in x.values())
    assert all(fp8._tiled_rows(v, *v.shape, None, None, L.ALGO_AUTO, 3) for v in x.values())


def test_tiled_rows_only_where_shared():
    """Below TILED_MIN_ROWS, tiled rows only for the launches that share them in LDS: tiled weights, N
    in whole groups of four row blocks, the split's tiles within LDS, one row block per wave; the
    head's persistent launch on a grid that fills the chip."""
    lib = L.lib()
    shares = lib.krq_gemv_fp8_shares_rows
    assert shares(5, 6144, 2560, 2, L.W_TILED) == 192 and shares(16, 2560, 9728, 4, L.W_TILED) == 160
    assert shares(3, 65536, 1024, 2, L.W_TILED) == 2048 and shares(5, 65536, 1024, 2, L.W_TILED) == 0  # (paired above 4)
    for bad in ((5, 6144, 2560, 2, L.W_ROWMAJOR), (5, 6160, 2560, 2, L.W_TILED), (5, 2560, 16384, 2, L.W_TILED),
                (5, 6144, 2560, 3, L.W_TILED), (5, 6144, 2592, 2, L.W_TILED), (1, 6144, 2560, 2, L.W_TILED),
                (17, 6144, 2560, 2, L.W_TILED), (5, 0, 2560, 2, L.W_TILED), (5, 6144, 2560, 0, L.W_TILED)):
        assert shares(*bad) == 0, bad
    head = lib.krq_lmhead_shares_rows
    assert head(5, 151936, 2560, L.W_TILED) == head(16, 32000, 4096, L.W_TILED) == 1
    for bad in ((5, 151936, 2560, L.W_ROWMAJOR), (5, 152064, 3584, L.W_TILED), (5, 16448, 2560, L.W_TILED),
                (5, 128256, 8192, L.W_TILED), (1, 151936, 2560, L.W_TILED), (17, 151936, 2560, L.W_TILED),
                (5, 0, 2560, L.W_TILED), (5, 151936, 0, L.W_TILED), (5, 151936, 2496, L.W_TILED)):
        assert head(*bad) == 0, bad

    a = fp8.SharedScale(torch.ones(1), torch.ones(()))
    t = torch.zeros(1)
    w8 = torch.empty(2560, 9728, device="meta")
    for scale, least, apart in ((a, 3, 11), (None, 11, 13)):
        for M in range(1, 13):
            for q, want in ((fp8.FP8Weight(w8, t, t), least), (fp8.FP8Weight(w8, t, None), apart), ((w8, t), apart),
                            (fp8.FP8Weight(w8[:2544], t, t), apart), (fp8.FP8Weight(w8[:1280], t, t), 11),
                            (fp8.FP8Weight(w8[:1216], t, t), 13), (fp8.FP8Weight(w8.expand(2, -1, -1).reshape(-1, 9728), t, t), 11)):
                assert (M >= fp8._tiled_least(q, M, 4, scale)) == (M >= want)


def test_linear_gemm_weights(monkeypatch):
    """linear_fp8 at 33 to 127 rows takes its own GEMM up to 64 MiB of weights (past K = 16,384 in split
    K), beyond that for long vocabularies over short rows and for long rows, never from 2 GiB; from
    128 rows always."""
    class Plan:
        def __init__(self, split):
            self.krq_gemm_fp8_ws_bytes = lambda kind, M, N, K: 1024 if split else 0

    for split in (False, True):
        monkeypatch.setattr(L, "lib", lambda: Plan(split))
        for M in (33, 64, 65, 127):
            for N, K in ((128, 256), (2560, 4096), (19456, 2560), (16384, 4096), (4096, 5120), (128, 16384),
                         (151936, 2560), (65536, 3584), (8192, 28672), (2560, 32768)):
                assert fp8._ring_pays(M, N, K), (M, N, K)
            for N, K in ((28672, 8192), (32000, 4096), (16384, 16384), (80000, 4096), (2048, 65536), (51200, 5120),
                         (1 << 20, 2048), (1 << 21, 1024)):
                assert not fp8._ring_pays(M, N, K), (M, N, K)
            assert fp8._ring_pays(M, 128, 32768) == fp8._ring_pays(M, 2048, 32768) == split
    w8 = torch.empty(1, 1, device="meta", dtype=torch.float8_e4m3fn).expand(28672, 8192)
    monkeypatch.setattr(fp8, "_gemm_min_rows", lambda w, ws: fp8.PREFILL_MIN_ROWS)
    assert not fp8._takes_gemm(127, w8, None) and fp8._takes_gemm(128, w8, None)


def test_linear_fp8_takes_two_dimensions():
    """linear_fp8 and swiglu_cast_fp8 refuse activations of other ranks before anything runs."""
    q = fp8.FP8Weight(torch.zeros(128, 256, dtype=torch.uint8).view(torch.float8_e4m3fn), torch.ones(()), None)
    for shape in ((256,), (1, 1, 256), (1, 40, 256)):
        with pytest.raises(ValueError):
            fp8.linear_fp8(torch.zeros(shape, dtype=torch.bfloat16), q)
