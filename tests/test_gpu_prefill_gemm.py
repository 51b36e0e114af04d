"""GPU parity of the prefill (M > 16) linear: the MFMA GEMM on bf16 operands
with f32 accumulation, against ops::gemm restated in f32 (oracle) on the
decoded weights (compute.hpp:58-68, ops.hpp:254-305, convert_gguf.py:233-263).
Tolerance: the 1e-2 class of bf16 paths (max |diff| / max |ref|); measured
errors are ~3e-3."""
import numpy as np
import pytest

import vlrf_amd as V
from conftest import gemm_plan, rel_err
from vlrf_amd import _lib
from vlrf_amd import formats as F

pytestmark = pytest.mark.gpu
TOL = 1e-2


def _weight(ctx, seed, name, N, K, dtype):
    w = F.normal(seed, name, N * K, 0.02)
    blocks = F.quantize(w, dtype)
    dec = F.dequantize(blocks, dtype, N * K).reshape(N, K)
    return V.QuantWeight(ctx, blocks, dtype, N, K), dec


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
# Kernel selection: M <= 128 -> 128-row register-staged tiles; Q8_0 with M > 128 -> the
# direct-to-LDS kernel (256x128 tiles); Q4_0 with M > 128 -> the register-staged 256x128
# tiles (two per CU for 257..512 tiles, as 520 x 16600's 390).
# Wide 256x256 tiles (two 128-row halves of the one weight) where they give at
# least 192 workgroups: 520 x 16600 and 2048 x 6144 (the 8B layer's QKV at T = 2048).
@pytest.mark.parametrize("M,N,K", [(256, 6144, 4096), (128, 4096, 14336), (2048, 1024, 4096),
                                   (520, 16600, 64), (2048, 6144, 512)])
def test_prefill_gemm_config5_shapes(ctx, orc, dtype, M, N, K):
    """The 8B-layer projections (QKV 6144x4096, down 4096x14336) at prompt rows."""
    print(f"[case] qgemm dtype={dtype} M={M} N={N} K={K}", flush=True)
    w, dec = _weight(ctx, 21, f"P{N}x{K}", N, K, dtype)
    x = F.normal(21, f"px{M}x{K}", M * K).reshape(M, K)
    dx, dy = ctx.to_device(x), ctx.alloc(M * N * 4)
    ctx.qlinear(w, dx, dy, M)
    ref = x.astype(np.float64) @ dec.astype(np.float64).T
    assert rel_err(dy.download((M, N)), ref) <= TOL


@pytest.mark.parametrize("M,N,K", [(17, 37, 64), (200, 300, 128), (129, 130, 704), (300, 256, 2048),
                                   (1000, 8300, 192), (1500, 8300, 192), (300, 100, 256), (129, 37, 64)])
def test_prefill_gemm_ragged_with_norm_and_residual(ctx, orc, M, N, K):
    """Row/column counts off the 128x128 tile, with the fused RMSNorm prologue
    and the residual epilogue (in place on the residual)."""
    print(f"[case] qgemm ragged M={M} N={N} K={K}", flush=True)
    w, dec = _weight(ctx, 22, f"G{N}x{K}", N, K, V.DT_Q8_0)
    x = F.normal(22, f"gx{M}", M * K).reshape(M, K) * 3
    g = 1.0 + F.normal(22, f"gg{K}", K, 0.1)
    res = F.normal(22, f"gr{M}x{N}", M * N).reshape(M, N)
    dx, dg, dr = ctx.to_device(x), ctx.to_device(g), ctx.to_device(res)
    ctx.qlinear(w, dx, dr, M, norm_w=dg, eps=1e-5, residual=dr)
    ref = orc.linear(orc.rms_norm(x, g, 1e-5), dec) + res
    assert rel_err(dr.download((M, N)), ref) <= TOL


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
@pytest.mark.parametrize("M", [100, 192])
def test_prefill_swiglu(ctx, orc, dtype, M):
    """h = silu(x.Wg^T) * (x.Wu^T) at M rows (feedforward.hpp:54-62); M = 100 takes
    the 128-row tiles, M = 192 the 256-row ones."""
    Fd, K = 1408, 1024
    wg, gdec = _weight(ctx, 23, "PWg", Fd, K, dtype)
    wu, udec = _weight(ctx, 23, "PWu", Fd, K, dtype)
    x = F.normal(23, "psx", M * K).reshape(M, K)
    g = np.ones(K, np.float32)
    dx, dg, dh = ctx.to_device(x), ctx.to_device(g), ctx.alloc(M * Fd * 4)
    ctx.qlinear_swiglu(wg, wu, dx, dh, M, norm_w=dg, eps=1e-5)
    xn = orc.rms_norm(x, g, 1e-5)
    ref = orc.silu_mul(orc.linear(xn, udec), orc.linear(xn, gdec))
    assert rel_err(dh.download((M, Fd)), ref) <= TOL


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
@pytest.mark.parametrize("M,Fd,K", [(257, 1000, 192), (300, 100, 64)])
def test_prefill_swiglu_ragged(ctx, orc, dtype, M, Fd, K):
    """SwiGLU with the FFN width and the row count off the 256x128 tile (the
    gate and up tiles of the direct-to-LDS kernel share one workgroup)."""
    print(f"[case] swiglu ragged dtype={dtype} M={M} F={Fd} K={K}", flush=True)
    wg, gdec = _weight(ctx, 24, f"RWg{Fd}x{K}", Fd, K, dtype)
    wu, udec = _weight(ctx, 24, f"RWu{Fd}x{K}", Fd, K, dtype)
    x = F.normal(24, f"rsx{M}x{K}", M * K).reshape(M, K)
    g = 1.0 + F.normal(24, f"rsg{K}", K, 0.1)
    dx, dg, dh = ctx.to_device(x), ctx.to_device(g), ctx.alloc(M * Fd * 4)
    ctx.qlinear_swiglu(wg, wu, dx, dh, M, norm_w=dg, eps=1e-5)
    xn = orc.rms_norm(x, g, 1e-5)
    ref = orc.silu_mul(orc.linear(xn, udec), orc.linear(xn, gdec))
    assert rel_err(dh.download((M, Fd)), ref) <= TOL


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
# 17 <= M <= 128 over codes with K split into slices (64 x 256 tiles to M = 64,
# 128 x 128 above): the 1.1B up and down shapes, the 8B down shape (16 col
# tiles x 16 slices), ragged N, the residual form, and K = 128 (one slice).
@pytest.mark.parametrize("M,N,K,res", [(17, 5632, 2048, False), (64, 2048, 5632, True), (65, 300, 1024, False),
                                       (128, 4096, 14336, True), (100, 1000, 128, False), (33, 6144, 4096, False)])
def test_split_k_gemm_mid_m(ctx, orc, monkeypatch, dtype, M, N, K, res):
    """The K-split GEMM against the oracle, and against the unsplit
    register-staged kernel (VLRF_HIP_PREFILL_DQ=0): the same bf16 products,
    summed in another order (slices added last), so equal to f32 rounding."""
    print(f"[case] split-K qgemm dtype={dtype} M={M} N={N} K={K} res={res}", flush=True)
    w, dec = _weight(ctx, 26, f"S{N}x{K}", N, K, dtype)
    x = F.normal(26, f"sx{M}x{K}", M * K).reshape(M, K)
    r = F.normal(26, f"sr{M}x{N}", M * N).reshape(M, N)
    dx = ctx.to_device(x)

    def run():
        dy = ctx.to_device(r) if res else ctx.alloc(M * N * 4)
        ctx.qlinear(w, dx, dy, M, residual=dy if res else None)
        return dy.download((M, N))

    monkeypatch.delenv("VLRF_HIP_PREFILL_DQ", raising=False)
    got = run()
    monkeypatch.setenv("VLRF_HIP_PREFILL_DQ", "0")
    unsplit = run()
    monkeypatch.delenv("VLRF_HIP_PREFILL_DQ", raising=False)
    ref = x.astype(np.float64) @ dec.astype(np.float64).T + (r if res else 0)
    assert rel_err(got, ref) <= TOL
    assert rel_err(got, unsplit) <= 2e-5, rel_err(got, unsplit)


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
@pytest.mark.parametrize("M,Fd,K", [(17, 5632, 2048), (100, 1408, 1024), (128, 14336, 4096), (70, 200, 384)])
def test_split_k_swiglu_mid_m(ctx, orc, monkeypatch, dtype, M, Fd, K):
    """SwiGLU at 17 <= M <= 128 with K split: gate and up partial sums reduced
    before silu(g) * u, against the oracle and the unsplit kernel."""
    print(f"[case] split-K swiglu dtype={dtype} M={M} F={Fd} K={K}", flush=True)
    wg, gdec = _weight(ctx, 27, f"SG{Fd}x{K}", Fd, K, dtype)
    wu, udec = _weight(ctx, 27, f"SU{Fd}x{K}", Fd, K, dtype)
    x = F.normal(27, f"ssx{M}x{K}", M * K).reshape(M, K)
    dx = ctx.to_device(x)

    def run():
        dh = ctx.alloc(M * Fd * 4)
        ctx.qlinear_swiglu(wg, wu, dx, dh, M)
        return dh.download((M, Fd))

    monkeypatch.delenv("VLRF_HIP_PREFILL_DQ", raising=False)
    got = run()
    monkeypatch.setenv("VLRF_HIP_PREFILL_DQ", "0")
    unsplit = run()
    monkeypatch.delenv("VLRF_HIP_PREFILL_DQ", raising=False)
    ref = orc.silu_mul(orc.linear(x, udec), orc.linear(x, gdec))
    assert rel_err(got, ref) <= TOL
    assert rel_err(got, unsplit) <= 2e-5, rel_err(got, unsplit)


def _bf16(x):
    """x rounded to bf16 (nearest even)."""
    u = np.ascontiguousarray(x, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & np.uint32(0xFFFF0000)).view(np.float32)


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
@pytest.mark.parametrize("M,N,K,res", [(17, 300, 64, False), (64, 37, 576, True), (65, 700, 1216, False),
                                       (128, 520, 5504, True), (100, 129, 8128, False),       # 17..128 rows
                                       (129, 100, 64, True), (130, 300, 704, False), (300, 515, 5504, True),
                                       (257, 130, 8128, False), (600, 260, 1984, True)])      # more
def test_gemm_uneven_k_slices(ctx, monkeypatch, dtype, M, N, K, res):
    """K of any number of 64-column steps: odd step counts, slices that do not
    divide them (a shorter last one), one-step slices.  bf16 products summed
    over K in any order in f32 are within (K + slices) eps of their absolute sum of each other:
    the forms agree as _check_forms says, and with 64-bit sums of the same bf16 operands."""
    print(f"[case] uneven K slices dtype={dtype} M={M} N={N} K={K} res={res}", flush=True)
    x = F.normal(28, f"ux{M}x{K}", M * K).reshape(M, K)
    r = F.normal(28, f"ur{M}x{N}", M * N).reshape(M, N)
    dx = ctx.to_device(x)
    dec = []

    def run():
        w, d = _weight(ctx, 28, f"U{N}x{K}", N, K, dtype)
        dec.append(d)
        dy = ctx.to_device(r) if res else ctx.alloc(M * N * 4)
        ctx.qlinear(w, dx, dy, M, residual=dy if res else None)
        return dy.download((M, N))

    a, b, c = _all_forms(monkeypatch, run)
    _check_forms(a, b, c)
    xb, wb = (_bf16(t).astype(np.float64) for t in (x, dec[0]))
    ref = xb @ wb.T + (r if res else 0)
    bound = (K + 40) * 2.0 ** -24 * (np.abs(xb) @ np.abs(wb).T + (np.abs(r) if res else 0))
    assert (np.abs(a - ref) <= bound).all()


@pytest.mark.parametrize("M,Fd,K", [(33, 200, 704), (90, 515, 1984), (300, 130, 5504)])
def test_swiglu_uneven_k_slices(ctx, monkeypatch, M, Fd, K):
    print(f"[case] uneven K slices swiglu M={M} F={Fd} K={K}", flush=True)
    x = F.normal(29, f"vx{M}x{K}", M * K).reshape(M, K)
    dx = ctx.to_device(x)

    def run():
        wg, _ = _weight(ctx, 29, f"VG{Fd}x{K}", Fd, K, V.DT_Q4_0)
        wu, _ = _weight(ctx, 29, f"VU{Fd}x{K}", Fd, K, V.DT_Q4_0)
        dh = ctx.alloc(M * Fd * 4)
        ctx.qlinear_swiglu(wg, wu, dx, dh, M)
        return dh.download((M, Fd))

    a, b, c = _all_forms(monkeypatch, run)
    _check_forms(a, b, c)


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
# slices of 9 steps and a last one of 5 (128 x 128 tiles), 2 (64 x 256), 7, of 16 and 15 (256 rows)
@pytest.mark.parametrize("M,N,K,res", [(105, 2100, 5504, True), (50, 4500, 4160, False), (300, 2051, 2752, True),
                                       (700, 4120, 1984, False)])
def test_gemm_uneven_k_slices_on_whole_tiles(ctx, monkeypatch, dtype, M, N, K, res):
    """A shorter last slice on the plan's own tiles (the shapes above take the
    half-size ones): above 128 rows over the expansion and over the codes."""
    print(f"[case] uneven K slices, whole tiles dtype={dtype} M={M} N={N} K={K} res={res}", flush=True)
    S, kl, few, _ = gemm_plan(dtype, M, N, K)
    assert S > 1 and K % kl and not few
    x = F.normal(28, f"ux{M}x{K}", M * K).reshape(M, K)
    r = F.normal(28, f"ur{M}x{N}", M * N).reshape(M, N)
    dx, dec = ctx.to_device(x), []

    def run():
        w, d = _weight(ctx, 28, f"U{N}x{K}", N, K, dtype)
        dec.append(d)
        dy = ctx.to_device(r) if res else ctx.alloc(M * N * 4)
        ctx.qlinear(w, dx, dy, M, residual=dy if res else None)
        return dy.download((M, N))

    a, b, c = _all_forms(monkeypatch, run)
    _check_forms(a, b, c)
    xb, wb = (_bf16(t).astype(np.float64) for t in (x, dec[0]))
    ref = xb @ wb.T + (r if res else 0)
    bound = (K + 40) * 2.0 ** -24 * (np.abs(xb) @ np.abs(wb).T + (np.abs(r) if res else 0))
    assert (np.abs(a - ref) <= bound).all()


# last slices of 9, 1 and 7 steps
@pytest.mark.parametrize("M,Fd,K", [(128, 2048, 5504), (20, 773, 10432), (300, 2051, 2752)])
def test_swiglu_uneven_k_slices_on_whole_tiles(ctx, monkeypatch, M, Fd, K):
    print(f"[case] uneven K slices swiglu, whole tiles M={M} F={Fd} K={K}", flush=True)
    S, kl, few, _ = gemm_plan(V.DT_Q4_0, M, Fd, K, True)
    assert S > 1 and K % kl and not few
    dx = ctx.to_device(F.normal(29, f"vx{M}x{K}", M * K).reshape(M, K))

    def run():
        wg, _ = _weight(ctx, 29, f"VG{Fd}x{K}", Fd, K, V.DT_Q4_0)
        wu, _ = _weight(ctx, 29, f"VU{Fd}x{K}", Fd, K, V.DT_Q4_0)
        dh = ctx.alloc(M * Fd * 4)
        ctx.qlinear_swiglu(wg, wu, dx, dh, M)
        return dh.download((M, Fd))

    _check_forms(*_all_forms(monkeypatch, run))


def _check_forms(a, b, c):
    """The default and the in-LDS form identical bit for bit (at shapes on
    half-size tiles both are that one kernel: test_half_size_tiles_keep_the_bits
    compares it with the expansion); the in-register form identical too, except
    where the two others split K into slices, which it does not: there it
    differs by the f32 summation order only."""
    assert np.array_equal(a, b)
    assert np.array_equal(a, c) or rel_err(a, c) <= 2e-5, rel_err(a, c)


def _all_forms(monkeypatch, run):
    """run() as it comes (above 128 rows over the weights' bf16 expansion, but
    half-size tiles over the codes), with VLRF_HIP_PREFILL_BF16=0 (codes decoded
    into LDS tiles, once per workgroup) and with VLRF_HIP_PREFILL_DQ=0 as well
    (codes decoded in registers, K whole)."""
    monkeypatch.delenv("VLRF_HIP_PREFILL_BF16", raising=False)
    monkeypatch.delenv("VLRF_HIP_PREFILL_DQ", raising=False)
    a = run()
    monkeypatch.setenv("VLRF_HIP_PREFILL_BF16", "0")
    b = run()
    monkeypatch.setenv("VLRF_HIP_PREFILL_DQ", "0")
    c = run()
    monkeypatch.delenv("VLRF_HIP_PREFILL_BF16", raising=False)
    monkeypatch.delenv("VLRF_HIP_PREFILL_DQ", raising=False)
    return a, b, c


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
# 256x128 tiles (1000 x 1024), wide 256x256 tiles (2048 x 6144), a ragged
# wide edge (520 x 16600), the residual form (300 x 4096 x 2048), ragged rows
# and columns on the LDS-decode tiles (257 x 1000 x 256, 129 x 130 x 128, 300 x 100 x 384)
@pytest.mark.parametrize("M,N,K,res", [(1000, 1024, 512, False), (2048, 6144, 256, False),
                                       (520, 16600, 64, False), (300, 4096, 2048, True),
                                       (257, 1000, 256, False), (129, 130, 128, True),
                                       (300, 100, 384, True)])
def test_bf16_expansion_equals_in_register_decode(ctx, monkeypatch, dtype, M, N, K, res):
    """The GEMM over the weights' bf16 expansion multiplies the operands the
    in-register and in-LDS decodes form, in the same MFMA order: bit-identical
    outputs."""
    print(f"[case] bf16 expansion dtype={dtype} M={M} N={N} K={K} res={res}", flush=True)
    x = F.normal(24, f"bx{M}x{K}", M * K).reshape(M, K)
    r = F.normal(24, f"br{M}x{N}", M * N).reshape(M, N)
    dx = ctx.to_device(x)

    def run():
        w, _ = _weight(ctx, 24, f"B{N}x{K}", N, K, dtype)   # a fresh weight: no expansion yet
        dy = ctx.to_device(r) if res else ctx.alloc(M * N * 4)
        ctx.qlinear(w, dx, dy, M, residual=dy if res else None)
        return dy.download((M, N))

    a, b, c = _all_forms(monkeypatch, run)
    _check_forms(a, b, c)


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
# 2048 x 14336: 112 x 8 tiles of 256 x 128, the last round (128 columns x 8)
# as 128-row tiles over columns 12288..14335 (two launches)
@pytest.mark.parametrize("M,Fd,K", [(2048, 14336, 128), (257, 1000, 192), (257, 1000, 256), (600, 136, 512)])
def test_bf16_expansion_swiglu_equals_in_register_decode(ctx, monkeypatch, dtype, M, Fd, K):
    print(f"[case] bf16 expansion swiglu dtype={dtype} M={M} F={Fd} K={K}", flush=True)
    x = F.normal(25, f"sx{M}x{K}", M * K).reshape(M, K)
    dx = ctx.to_device(x)

    def run():
        wg, _ = _weight(ctx, 25, f"SG{Fd}x{K}", Fd, K, dtype)
        wu, _ = _weight(ctx, 25, f"SU{Fd}x{K}", Fd, K, dtype)
        dh = ctx.alloc(M * Fd * 4)
        ctx.qlinear_swiglu(wg, wu, dx, dh, M)
        return dh.download((M, Fd))

    a, b, c = _all_forms(monkeypatch, run)
    _check_forms(a, b, c)


@pytest.mark.parametrize("M,N,K,swiglu", [(233, 2560, 2048, False), (166, 2300, 1280, False), (300, 620, 4096, False),
                                          (317, 1100, 1536, True),                            # the plan's slices
                                          (1000, 1024, 512, False), (257, 1000, 256, False), (129, 130, 128, False),
                                          (300, 100, 384, False), (257, 1000, 192, True), (600, 136, 512, True)])   # K whole
def test_half_size_tiles_keep_the_bits(ctx, monkeypatch, M, N, K, swiglu):
    """Half-size tiles over the codes (the default at these shapes) add the same
    slices of K as the plan's own tiles over the bf16 expansion
    (VLRF_HIP_PREFILL_DQ=0): the same result to the bit."""
    print(f"[case] half-size tiles M={M} N={N} K={K} swiglu={swiglu}", flush=True)
    assert gemm_plan(V.DT_Q4_0, M, N, K, swiglu)[2]
    ws = [_weight(ctx, 30, f"H{i}.{N}x{K}", N, K, V.DT_Q4_0)[0] for i in range(1 + swiglu)]
    dx = ctx.to_device(F.normal(30, f"hx{M}x{K}", M * K).reshape(M, K))
    out = []
    for dq in (None, "0"):
        if dq is None:
            monkeypatch.delenv("VLRF_HIP_PREFILL_DQ", raising=False)
        else:
            monkeypatch.setenv("VLRF_HIP_PREFILL_DQ", dq)
        dy = ctx.alloc(M * N * 4)
        if swiglu:
            ctx.qlinear_swiglu(ws[0], ws[1], dx, dy, M)
        else:
            ctx.qlinear(ws[0], dx, dy, M)
        out.append(dy.download((M, N)))
    assert np.array_equal(*out)


def test_bf16_expansion_is_counted_in_the_weight_bytes(ctx):
    """vlrf_hip_weight_bytes: the packed codes and scales, plus 2 bytes per
    weight once a GEMM of more than 128 rows has made the bf16 expansion."""
    N, K, M = 384, 512, 200
    w, _ = _weight(ctx, 26, "WB", N, K, V.DT_Q8_0)
    packed = N * K + N * (K // 32) * 2
    assert w.device_bytes == packed
    x = ctx.to_device(F.normal(26, "wbx", M * K).reshape(M, K))
    y = ctx.alloc(M * N * 4)
    ctx.qlinear(w, x, y, 8)                      # M <= 128: no expansion
    assert w.device_bytes == packed
    ctx.qlinear(w, x, y, M)
    ctx.sync()
    assert w.device_bytes == packed + 2 * N * K


def _hip():
    import ctypes as C
    h = C.CDLL("libamdhip64.so")
    h.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    h.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    h.hipGraphInstantiate.argtypes = [C.POINTER(C.c_void_p), C.c_void_p, C.c_void_p, C.c_void_p, C.c_size_t]
    h.hipGraphLaunch.argtypes = [C.c_void_p, C.c_void_p]
    h.hipGraphExecDestroy.argtypes = [C.c_void_p]
    h.hipGraphDestroy.argtypes = [C.c_void_p]
    return h


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
@pytest.mark.parametrize("M,N,K,more", [(160, 512, 1024, 4), (64, 512, 1024, 4), (300, 2051, 2752, 10)])
def test_prefill_gemm_under_graph_capture(orc, dtype, M, N, K, more):
    """A stream under graph capture: the M > 128 GEMM records no allocation
    (the weight's bf16 expansion is not made, the tiles decode the blocks),
    the captured graph replays to the eager result (at 300 rows over the
    expansion, at the two others on half-size tiles over the codes) bit
    for bit, replay after replay with eager work between; a call whose rows
    alone would grow the context scratch while capturing is refused with an
    error instead of being recorded.  All three split K (partial sums in the
    context scratch after the bf16 rows) and launch the reduction."""
    import ctypes as C
    hip = _hip()
    ctx = V.Context(0)                  # its own scratch buffer, empty until the first call
    S, _, few, _ = gemm_plan(dtype, M, N, K)
    assert S > 1 and few == (M != 300)
    print(f"[case] qgemm under capture dtype={dtype} M={M} N={N} K={K}", flush=True)
    w1, dec = _weight(ctx, 31, "cap", N, K, dtype)
    w2, _ = _weight(ctx, 31, "cap", N, K, dtype)              # the same blocks, never expanded
    packed = w2.device_bytes
    x = F.normal(31, "capx", M * K).reshape(M, K)
    dx, y1, y2 = ctx.to_device(x), ctx.alloc(M * N * 4), ctx.alloc(M * N * 4)
    ctx.qlinear(w1, dx, y1, M)                                 # eager: grows the scratch, expands w1
    ctx.sync()
    eager = y1.download((M, N))
    ref = x.astype(np.float64) @ dec.astype(np.float64).T
    assert rel_err(eager, ref) <= TOL
    s = C.c_void_p(ctx.stream())
    assert hip.hipStreamBeginCapture(s, 2) == 0               # hipStreamCaptureModeRelaxed
    rc = V.lib().vlrf_hip_qlinear(ctx.h, w2.h, dx.ptr, y2.ptr, M, None, C.c_float(0.0), None)
    g = C.c_void_p()
    assert hip.hipStreamEndCapture(s, C.byref(g)) == 0
    assert rc == 0, V.lib().vlrf_hip_last_error()
    assert V.lib().vlrf_hip_weight_bytes(w2.h) == packed       # no expansion recorded
    ge = C.c_void_p()
    assert hip.hipGraphInstantiate(C.byref(ge), g, None, None, 0) == 0
    for i in range(3):
        y2.zero()
        ctx.qlinear(w1, dx, y1, M)                             # eager work between replays
        assert hip.hipGraphLaunch(ge, s) == 0
        ctx.sync()
        got = y2.download((M, N))
        assert rel_err(got, ref) <= TOL, i
        assert np.array_equal(got, eager), i
    hip.hipGraphExecDestroy(ge)
    hip.hipGraphDestroy(g)
    # Scratch growth while capturing: refused, the capture ends cleanly.
    M2 = more * M
    dx2, y3 = ctx.to_device(np.tile(x, (more, 1))), ctx.alloc(M2 * N * 4)
    assert hip.hipStreamBeginCapture(s, 2) == 0
    rc = V.lib().vlrf_hip_qlinear(ctx.h, w1.h, dx2.ptr, y3.ptr, M2, None, C.c_float(0.0), None)
    g = C.c_void_p()
    hip.hipStreamEndCapture(s, C.byref(g))
    if g.value:
        hip.hipGraphDestroy(g)
    assert rc == _lib.ERR_ARG and b"captured" in V.lib().vlrf_hip_last_error()
    ctx.qlinear(w1, dx2, y3, M2)                               # eagerly it runs
    ctx.sync()
    assert rel_err(y3.download((M2, N))[:M], ref) <= TOL


@pytest.mark.parametrize("M,N,K,swiglu", [(128, 2048, 5504, False), (300, 1024, 4096, False), (100, 600, 2048, True)])
def test_captured_gemm_with_scratch_for_its_rows_only(M, N, K, swiglu):
    """Captured when the context scratch holds the call's bf16 rows but not its
    partial sums: recorded with K whole, not refused; every replay is the eager
    result up to the order of the f32 sums."""
    import ctypes as C
    hip, ctx = _hip(), V.Context(0)
    print(f"[case] capture, scratch for the rows M={M} N={N} K={K} swiglu={swiglu}", flush=True)
    ws = [_weight(ctx, 32, f"c{i}", N, K, V.DT_Q8_0)[0] for i in range(1 + swiglu)]
    one, _ = _weight(ctx, 32, "one", 1, K, V.DT_Q8_0)
    dx, y, e = ctx.to_device(F.normal(32, "x", M * K).reshape(M, K)), ctx.alloc(M * N * 4), ctx.alloc(M * N * 4)
    S, _, _, part = gemm_plan(V.DT_Q8_0, M, N, K, swiglu)
    ctx.qlinear(one, dx, y, M)                                 # the same rows, one column
    held = (C.c_size_t * 2)()
    V.check(V.lib().vlrf_hip_scratch_bytes(ctx.h, held))
    assert S > 1 and 2 * M * K <= held[0] < 2 * M * K + part

    def call(out):
        if swiglu:
            return V.lib().vlrf_hip_qlinear_swiglu(ctx.h, ws[0].h, ws[1].h, dx.ptr, out.ptr, M, None, C.c_float(0.0))
        return V.lib().vlrf_hip_qlinear(ctx.h, ws[0].h, dx.ptr, out.ptr, M, None, C.c_float(0.0), None)

    s, g, ge = C.c_void_p(ctx.stream()), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(s, 2) == 0
    rc = call(y)
    assert hip.hipStreamEndCapture(s, C.byref(g)) == 0 and rc == 0, V.lib().vlrf_hip_last_error()
    assert hip.hipGraphInstantiate(C.byref(ge), g, None, None, 0) == 0
    for _ in range(3):
        y.zero()
        V.check(call(e))                                       # eager, split: grows the scratch the first time
        assert hip.hipGraphLaunch(ge, s) == 0
        ctx.sync()
        assert rel_err(y.download((M, N)), e.download((M, N))) <= 2e-5
    hip.hipGraphExecDestroy(ge)
    hip.hipGraphDestroy(g)
