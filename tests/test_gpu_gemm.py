"""FP8 prefill GEMM (krq_gemm_fp8, kernels.fp8.gemm_fp8) against the exact oracle product of the
same e4m3 operands: max|y - ref| <= 1e-2 * max|ref| (the path's tolerance), for ragged M, per
tensor / per row scales, e4m3 activations and bf16 activations quantized in the kernel; the fused
cast is bit-identical to the reference's cast followed by the GEMM."""

import numpy as np
import pytest
import torch

from kernels import fp8 as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-2


def rel_err(y, ref):
    y = np.asarray(y, dtype=np.float64)
    ref = np.asarray(ref, dtype=np.float64)
    return float(np.abs(y - ref).max() / max(np.abs(ref).max(), 1e-30))


def codes(t):
    return t.cpu().view(torch.uint8).numpy()


def bf(shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16)


@pytest.mark.parametrize("M,N,K,per_row", [(33, 128, 128, True), (128, 256, 256, False), (300, 384, 640, True),
                                           (257, 6144, 2560, True), (256, 2560, 9728, False),
                                           (600, 512, 384, True), (1024, 2560, 9728, False), (777, 6144, 2560, True),
                                           # 256 x 256 ring tiles (>= 128 of them): ragged M, a tile count
                                           # that is not a multiple of the 8 XCDs, several tiles per CU
                                           (2000, 4096, 2560, True), (2100, 4352, 256, True),
                                           (4096, 8192, 384, False),
                                           # 192 x 256 tiles: ragged M (20 full row tiles + 160 rows)
                                           (4000, 2560, 512, True), (4096, 2560, 4096, False),
                                           # 64 x 64 tiles: small grids that do not split K
                                           (256, 2560, 4096, True), (100, 1024, 512, False),
                                           # a whole round of 256 x 256 tiles over the first 4096
                                           # columns, then 128 x 128 tiles over the last 2048 (two
                                           # launches into one output), also with ragged M
                                           (4096, 6144, 512, False), (3900, 6144, 384, True)])
def test_gemm_fp8_matches_oracle(dev, M, N, K, per_row):
    w = bf((N, K), 1, 0.02).to(dev)
    q = F.quantize(w) if per_row else F.quantize_weight(w)
    x = bf((M, K), 2).to(dev)
    x8, xs = F.quant_rows(x)                      # e4m3 activations, per-token scales
    y = F.gemm_fp8(x8, q, xs=xs)
    _, ref = O.fp8_matmul(codes(x8), xs.cpu().numpy().reshape(-1), codes(q[0]), q[1].cpu().numpy())
    e = rel_err(y.float().cpu().numpy(), ref)
    print(f"gemm M={M} N={N} K={K}: max-rel {e:.2e}")
    assert e <= TOL


@pytest.mark.parametrize("M,N,K,pad", [(4000, 19456, 2560, 4096),   # 256 x 256, ~5 tiles per block
                                       (3900, 19456, 2560, 4096),
                                       (2000, 19456, 2560, 2048),   # 256 x 256 rounds + 128 x 128 tail
                                       (3000, 6144, 2560, 3072)])   # 192 x 256, a second tile after a ragged one
def test_gemm_ragged_multi_tile(dev, M, N, K, pad):
    """More ring tiles than blocks with M not a multiple of the tile height (gate_up and QKV
    shapes), so blocks run tiles after one with rows past M: within the bar of the oracle on a
    sample of rows (the last 256, which hold the ragged row tile, and every 61st row), and bit for
    bit the rows of a run on M padded to a whole number of tiles (the same tile plan, no ragged
    tile; each output is the same sum of the same products in the same order)."""
    w = bf((N, K), 51, 0.02).to(dev)
    q = F.quantize(w)
    x = bf((pad, K), 52).to(dev)
    x8p, xsp = F.quant_rows(x)
    x8, xs = x8p[:M].contiguous(), xsp[:M].contiguous()
    y = F.gemm_fp8(x8, q, xs=xs)
    y_pad = F.gemm_fp8(x8p, q, xs=xsp)
    assert torch.equal(y, y_pad[:M])
    rows = np.unique(np.concatenate([np.arange(0, M, 61), np.arange(M - 256, M)]))
    _, ref = O.fp8_matmul(codes(x8)[rows], xs.cpu().numpy().reshape(-1)[rows], codes(q[0]), q[1].cpu().numpy())
    e = rel_err(y.float().cpu().numpy()[rows], ref)
    print(f"gemm ragged M={M} N={N} K={K}: max-rel {e:.2e} on {rows.size} rows")
    assert e <= TOL


@pytest.mark.parametrize("M,N,K,splits", [(256, 2560, 9728, 4), (200, 2560, 9728, 4), (300, 2560, 8192, 4),
                                          (130, 4096, 8192, 4), (1024, 2560, 9728, 2),
                                          # 64 x 64 tiles split (too few 128 x 128 ones to split)
                                          (64, 2560, 9728, 4), (100, 2560, 9728, 4)])
def test_gemm_split_k(dev, M, N, K, splits):
    """Split K (krq_gemm_fp8_ws with its workspace) and the unsplit kernel (krq_gemm_fp8, or the
    workspace form given too little workspace, which must then equal it bit for bit): both within
    the bar of the oracle."""
    from kernels import _lib as L
    lib = L.lib()
    assert lib.krq_gemm_fp8_ws_bytes(L.X_FP8, M, N, K) == splits * M * N * 4
    q = F.quantize(bf((N, K), 11, 0.02).to(dev))
    x8, xs = F.quant_rows(bf((M, K), 12).to(dev))
    _, ref = O.fp8_matmul(codes(x8), xs.cpu().numpy().reshape(-1), codes(q[0]), q[1].cpu().numpy())
    y_split = F.gemm_fp8(x8, q, xs=xs)
    args = (L.ptr(x8), L.X_FP8, L.ptr(xs), None, 1, L.ptr(q[0]), L.ptr(q[1]), 1, M, N, K)
    y_plain = torch.empty_like(y_split)
    L.call("krq_gemm_fp8", *args, L.ptr(y_plain), L.stream(x8))
    small = torch.empty(splits * M * N * 4 - 16, device=dev, dtype=torch.uint8)
    y_small = torch.empty_like(y_split)
    L.call("krq_gemm_fp8_ws", *args, L.ptr(small), small.numel(), L.ptr(y_small), L.stream(x8))
    assert torch.equal(y_small, y_plain)
    for y in (y_split, y_plain):
        e = rel_err(y.float().cpu().numpy(), ref)
        print(f"gemm M={M} N={N} K={K} splits={splits}: max-rel {e:.2e}")
        assert e <= TOL


@pytest.mark.parametrize("M,N,K", [(200, 256, 128), (200, 256, 384), (512, 2560, 4096)])
def test_gemm_fused_cast_is_cast_then_gemm(dev, M, N, K):
    """bf16 x with an ActScale: gemm_fp8 (the cast fused into the 128 x 128 kernel at K = 128,
    the HIP cast then the e4m3 kernels otherwise) equals fp8._cast + the e4m3 GEMM bit for bit; the
    C ABI's fused-cast kernel (krq_gemm_fp8 on bf16 rows) and linear_fp8 (prefill) are within the
    bar of the oracle."""
    from kernels import _lib as L
    w = bf((N, K), 3, 0.02).to(dev)
    q = F.quantize_weight(w)
    x = bf((M, K), 4).to(dev)
    a = F.ActScale(x)
    y = F.gemm_fp8(x, q, a)
    y2 = F.gemm_fp8(F._cast(x, a), q, xs=a.scale.reshape(1))
    assert torch.equal(y, y2)
    y3 = torch.empty_like(y)
    L.call("krq_gemm_fp8", L.ptr(x), L.X_BF16_STATIC, L.ptr(a.scale), L.ptr(a.inv), 0, L.ptr(q[0]), L.ptr(q[1]), 0,
           M, N, K, L.ptr(y3), L.stream(x))
    _, ref = O.fp8_matmul(codes(F._cast(x, a)), a.scale.cpu().numpy(), codes(q[0]), q[1].cpu().numpy())
    assert rel_err(F.linear_fp8(x, q).float().cpu().numpy(), ref) <= TOL
    assert rel_err(y.float().cpu().numpy(), ref) <= TOL
    assert rel_err(y3.float().cpu().numpy(), ref) <= TOL


@pytest.mark.parametrize("M,N,K", [(128, 2560, 4096), (300, 6144, 2560), (64, 2560, 4096), (200, 256, 128)])
def test_linear_fp8_prefill_route(dev, M, N, K):
    """linear_fp8 above the decode sizes (engine/kernels/fp8.py:105-106): from PREFILL_MIN_ROWS rows,
    on weights the ring kernels take, it is gemm_fp8 on the cast rows bit for bit; below that (or
    for K = 128) the library's torch._scaled_mm bit for bit. Both within the bar of the oracle."""
    q = F.quantize_weight(bf((N, K), 31, 0.02).to(dev))
    x = bf((M, K), 32).to(dev)
    a = F.ActScale(x)
    y = F.linear_fp8(x, q, a)
    # without a given scale linear_fp8 takes its own (ActScale and the cast in two launches),
    # the same bits, and records amax in amax_out
    amax_out = torch.zeros(1, device=dev)
    assert torch.equal(F.linear_fp8(x, q, amax_out=amax_out), y)
    assert torch.equal(amax_out, a.amax.reshape(1))
    x8 = F._cast(x, a)
    if M >= F.PREFILL_MIN_ROWS and K >= 256:
        assert torch.equal(y, F.gemm_fp8(x8, q, xs=a.scale.reshape(1)))
    else:
        assert torch.equal(y, torch._scaled_mm(x8, q[0].t(), scale_a=a.scale, scale_b=q[1], out_dtype=torch.bfloat16))
    _, ref = O.fp8_matmul(codes(x8), a.scale.cpu().numpy(), codes(q[0]), q[1].cpu().numpy())
    assert rel_err(y.float().cpu().numpy(), ref) <= TOL


# Short K (two pair buffers: fewer pairs of stages than four, as many, one more) and four pair buffers from
# K = 1,024 with 2 MiB of weights (one part on each side) or K = 2,048; rows from the first the GEMM
# takes, ragged and whole tiles; two 64 x 64 units per compute unit up to 1,024 rows and past them, one
# tile more (two buffers); 128 x 128 tiles, split K on either kind, one part per unit or past it.
@pytest.mark.parametrize("M,N,K", [(33, 2048, 1024), (100, 1920, 1024), (65, 128, 2048), (77, 1408, 1536),
                                   (100, 16384, 2048), (100, 16512, 2048), (1000, 2048, 2048), (2048, 1024, 4096),
                                   (33, 128, 256), (64, 128, 384), (77, 256, 512), (65, 384, 640), (127, 128, 1152),
                                   (100, 16384, 256), (100, 16512, 256), (33, 2560, 9728), (127, 2560, 9728),
                                   (129, 2560, 9728), (300, 2560, 8192), (200, 2560, 4096)])
def test_gemm_deep_ring(dev, M, N, K):
    q = F.quantize(bf((N, K), 51, 0.02).to(dev))
    for seed in (52, 53):  # (the second over the first's leftovers in LDS and the workspace)
        x8, xs = F.quant_rows(bf((M, K), seed).to(dev))
        y = F.gemm_fp8(x8, q, xs=xs)
        ref = (x8.double() @ q[0].double().t()) * xs.double() * q[1].double()
        assert rel_err(y.float().cpu().numpy(), ref.cpu().numpy()) <= TOL
        assert torch.equal(F.gemm_fp8(x8, q, xs=xs), y)


@pytest.mark.parametrize("M,takes", [(33, False), (127, False), (128, True)])
def test_linear_fp8_per_channel_rows(dev, M, takes):
    """Per-channel weights: refused below 128 rows (the library's scaled product takes one scale per
    weight), this library's GEMM from there."""
    q = F.quantize(bf((256, 512), 54, 0.02).to(dev))
    x = bf((M, 512), 55).to(dev)
    if takes:
        a = F.ActScale(x)
        assert torch.equal(F.linear_fp8(x, q), F.gemm_fp8(F._cast(x, a), q, xs=a.scale.reshape(1)))
    else:
        with pytest.raises((RuntimeError, ValueError)):
            F.linear_fp8(x, q)


@pytest.mark.parametrize("M,N,K", [(4096, 6144, 512), (256, 2560, 9728), (300, 6144, 2560)])
def test_gemm_graph_replays(dev, M, N, K):
    """gemm_fp8 captured in a graph (the two-launch tail plan, split K with its reduce and the
    workspace, a plain ring launch): every replay, with eager work between them, equals the eager
    result bit for bit."""
    q = F.quantize(bf((N, K), 41, 0.02).to(dev))
    x8, xs = F.quant_rows(bf((M, K), 42).to(dev))
    want = F.gemm_fp8(x8, q, xs=xs)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        F.gemm_fp8(x8, q, xs=xs)  # warm-up on a side stream, as before any capture
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = F.gemm_fp8(x8, q, xs=xs)
    for r in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), f"replay {r}"
        F.gemm_fp8(x8, q, xs=xs).sum().item()  # eager work between the replays
        y.zero_()
        torch.cuda.synchronize()


def test_gemm_matches_library_gemm(dev):
    """Against torch._scaled_mm (hipBLASLt) on the same operands: both within the bar of the oracle,
    and within a few bf16 ulps of each other."""
    M, N, K = 384, 2560, 2560
    q = F.quantize_weight(bf((N, K), 5, 0.02).to(dev))
    x = bf((M, K), 6).to(dev)
    a = F.ActScale(x)
    x8 = F._cast(x, a)
    ours = F.gemm_fp8(x8, q, xs=a.scale.reshape(1)).float()
    lib = torch._scaled_mm(x8, q[0].t(), scale_a=a.scale, scale_b=q[1], out_dtype=torch.bfloat16).float()
    assert rel_err(ours.cpu().numpy(), lib.cpu().numpy()) <= 2 * 2.0 ** -8


def test_gemm_rejects_bad_shapes(dev):
    q = F.quantize_weight(bf((200, 256), 7).to(dev))  # N not a multiple of 128
    x8, xs = F.quant_rows(bf((64, 256), 8).to(dev))
    with pytest.raises(ValueError):
        F.gemm_fp8(x8, q, xs=xs)


@pytest.mark.parametrize("M", [1, 5, 16, 33, 128])
def test_scales_refused(dev, M):
    """Scales of another type or count than the kernels read, from every row count's route."""
    q = F.quantize_weight(bf((256, 512), 56, 0.02).to(dev))
    x = bf((M, 512), 57).to(dev)
    a = F.ActScale(x)
    for ws in (q[1].double(), q[1].repeat(3)):
        bad = F.FP8Weight(q[0], ws, q.tiled)
        with pytest.raises((RuntimeError, ValueError)):
            F.linear_fp8(x, bad)
        with pytest.raises(ValueError):
            F.gemm_fp8(x, bad, a)
        if M <= 32:
            with pytest.raises(ValueError):
                F.gemv_fp8(x, bad, 2)
    for s in (F.SharedScale(a.inv.double(), a.scale), F.SharedScale(a.inv, a.scale.double())):
        with pytest.raises((RuntimeError, ValueError)):
            F.linear_fp8(x, q, s)


@pytest.mark.parametrize("given", [False, True])
@pytest.mark.parametrize("M,N,K", [(77, 384, 512), (40, 2560, 9728), (256, 2560, 9728)])
def test_linear_fp8_capture_and_streams(dev, M, N, K, given):
    """linear_fp8's one-allocation route (scale, e4m3 rows and split-K partials in one workspace freed at
    return) captured in a graph, with the running maximum: every replay on new inputs, eager calls on
    the same shapes in between, equals the eager result; and on two side streams whose calls overlap."""
    q = F.quantize_weight(bf((N, K), 61, 0.02).to(dev))
    xs = [bf((M, K), 62 + i, 1.0 + i).to(dev) for i in range(4)]
    a = F.ActScale(xs[3]) if given else None
    want = [F.linear_fp8(x, q, a) for x in xs]
    amax = [x.float().abs().amax().clamp_min(1e-6) for x in xs]
    torch.cuda.synchronize()

    buf, top = xs[0].clone(), torch.zeros(1, device=dev)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = F.linear_fp8(buf, q, a, amax_out=top)
    for i in (0, 2, 1, 3):
        buf.copy_(xs[i])
        top.zero_()
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want[i]), f"replay on input {i}"
        assert given or top.item() == amax[i].item()
        assert torch.equal(F.linear_fp8(xs[(i + 1) % 4], q, a), want[(i + 1) % 4])

    here = torch.cuda.current_stream()
    sides = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = [[], []]
    for s in sides:
        s.wait_stream(here)
    for r in range(8):  # (workspaces come and go on each stream while the other's are in use)
        for k, s in enumerate(sides):
            with torch.cuda.stream(s):
                got[k].append(F.linear_fp8(xs[(r + k) % 4], q, a))
    for s in sides:
        here.wait_stream(s)
    torch.cuda.synchronize()
    for k in range(2):
        for r in range(8):
            assert torch.equal(got[k][r], want[(r + k) % 4]), (k, r)
