"""GPU parity: dequant-fused quantized linear (compute::linear on weights
decoded from GGUF Q8_0/Q4_0 blocks, convert_gguf.py:233-263), benchmark
config 3 shapes, plus the fused RMSNorm prologue, residual epilogue and the
SwiGLU gate/up variant.  Oracle: ops::gemm restated (oracle/vlrf_oracle.c)
on the decoded f32 weights.  Tolerance: 1e-3 relative (fp32 path)."""
import numpy as np
import pytest

import vlrf_amd as V
from conftest import rel_err
from vlrf_amd import formats as F

pytestmark = pytest.mark.gpu


def _weight(ctx, seed, name, N, K, dtype):
    w = F.normal(seed, name, N * K, 0.02)
    blocks = F.quantize(w, dtype)
    dec = F.dequantize(blocks, dtype, N * K).reshape(N, K) if dtype != V.DT_F32 else w.reshape(N, K)
    return V.QuantWeight(ctx, blocks, dtype, N, K), dec


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
@pytest.mark.parametrize("N,K", [(5632, 2048), (2048, 5632)])
@pytest.mark.parametrize("M", [1, 4, 16])
def test_config3_qlinear(ctx, orc, dtype, N, K, M):
    print(f"[case] qlinear dtype={dtype} N={N} K={K} M={M}", flush=True)
    w, dec = _weight(ctx, 7, f"W{N}x{K}", N, K, dtype)
    x = F.normal(7, f"x{M}", M * K).reshape(M, K)
    dx, dy = ctx.to_device(x), ctx.alloc(M * N * 4)
    ctx.qlinear(w, dx, dy, M)
    y = dy.download((M, N))
    ref = orc.linear(x, dec)
    assert rel_err(y, ref) <= 1e-3
    np.testing.assert_allclose(y, ref, rtol=1e-3, atol=1e-5 * np.abs(ref).max())


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
@pytest.mark.parametrize("N,K", [(4096, 14336), (300, 14336), (37, 6176)])
def test_m1_wide_rows(ctx, orc, dtype, N, K):
    """M = 1 over rows wider than the general staging (K > 6144, up to the
    8B shape's d_ff 14336): plain and with the residual added."""
    print(f"[case] wide M=1 dtype={dtype} N={N} K={K}", flush=True)
    w, dec = _weight(ctx, 11, f"W{N}x{K}", N, K, dtype)
    x = F.normal(11, "xw", K).reshape(1, K)
    res = F.normal(11, "rw", N).reshape(1, N)
    dx, dy = ctx.to_device(x), ctx.alloc(N * 4)
    ctx.qlinear(w, dx, dy, 1)
    ref = orc.linear(x, dec)
    assert rel_err(dy.download((1, N)), ref) <= 1e-3
    dr = ctx.to_device(res)
    ctx.qlinear(w, dx, dr, 1, residual=dr)
    assert rel_err(dr.download((1, N)), ref + res) <= 1e-3


@pytest.mark.parametrize("M", [1, 3, 9])
@pytest.mark.parametrize("N,K", [(37, 64), (300, 96), (8, 1056)])
def test_qlinear_ragged_shapes(ctx, orc, M, N, K):
    """Row counts not divisible by the 8-row workgroup tile; K not a multiple of
    the 1024 staging tile; M between the 1/4/16 instantiations."""
    for dtype in (V.DT_Q8_0, V.DT_Q4_0, V.DT_F32):
        w, dec = _weight(ctx, 8, f"R{N}x{K}", N, K, dtype)
        x = F.normal(8, f"xr{M}", M * K).reshape(M, K)
        dx, dy = ctx.to_device(x), ctx.alloc(M * N * 4)
        ctx.qlinear(w, dx, dy, M)
        assert rel_err(dy.download((M, N)), orc.linear(x, dec)) <= 1e-3


def test_qlinear_fused_norm_and_residual(ctx, orc):
    """y = residual + W . rms_norm(x; g) (ops.hpp:478-499 then the residual add)."""
    N, K, M = 2560, 2048, 1
    w, dec = _weight(ctx, 9, "Wqkv", N, K, V.DT_Q8_0)
    x = F.normal(9, "xn", M * K).reshape(M, K) * 0.05
    g = 1.0 + F.normal(9, "g", K, 0.1)
    res = F.normal(9, "res", M * N).reshape(M, N)
    dx, dg, dr = ctx.to_device(x), ctx.to_device(g), ctx.to_device(res)
    dy = ctx.alloc(M * N * 4)
    ctx.qlinear(w, dx, dy, M, norm_w=dg, eps=1e-5)
    ref = orc.linear(orc.rms_norm(x, g, 1e-5), dec)
    assert rel_err(dy.download((M, N)), ref) <= 1e-3
    ctx.qlinear(w, dx, dr, M, norm_w=dg, eps=1e-5, residual=dr)      # in place on the residual
    assert rel_err(dr.download((M, N)), ref + res) <= 1e-3


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
@pytest.mark.parametrize("M", [1, 4])
def test_swiglu_gate_up(ctx, orc, dtype, M):
    """h = silu(x.Wg^T) * (x.Wu^T) (feedforward.hpp:54-62) with the fused norm."""
    Fd, K = 5632, 2048
    wg, gdec = _weight(ctx, 10, "Wg", Fd, K, dtype)
    wu, udec = _weight(ctx, 10, "Wu", Fd, K, dtype)
    x = F.normal(10, "xs", M * K).reshape(M, K)
    g = np.ones(K, np.float32)
    dx, dg, dh = ctx.to_device(x), ctx.to_device(g), ctx.alloc(M * Fd * 4)
    ctx.qlinear_swiglu(wg, wu, dx, dh, M, norm_w=dg, eps=1e-5)
    xn = orc.rms_norm(x, g, 1e-5)
    ref = orc.silu_mul(orc.linear(xn, udec), orc.linear(xn, gdec))
    assert rel_err(dh.download((M, Fd)), ref) <= 1e-3


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
@pytest.mark.parametrize("M,N,K", [(2, 37, 256), (7, 300, 2304), (16, 1000, 4352), (5, 16, 512)])
def test_small_m_matrix_core_path(ctx, orc, dtype, M, N, K):
    """2 <= M <= 16 with K % 256 == 0 runs on the matrix cores (codes exact in
    bf16, activations split into bf16 hi + lo): row counts off the 16-row tile,
    one 256-column slice, 9 slices over 16 waves (7 idle), 17 slices (one wave
    takes two).  Fused norm, then the residual added in place.  The split keeps
    the f32 class: 1e-4, ten times tighter than the path's stated 1e-3."""
    print(f"[case] qlinear small-M dtype={dtype} M={M} N={N} K={K}", flush=True)
    w, dec = _weight(ctx, 12, f"S{N}x{K}", N, K, dtype)
    x = F.normal(12, f"xs{M}x{K}", M * K).reshape(M, K)
    g = 1.0 + F.normal(12, f"gs{K}", K, 0.1)
    res = F.normal(12, f"rs{M}x{N}", M * N).reshape(M, N)
    dx, dg, dr, dy = ctx.to_device(x), ctx.to_device(g), ctx.to_device(res), ctx.alloc(M * N * 4)
    ctx.qlinear(w, dx, dy, M)
    assert rel_err(dy.download((M, N)), orc.linear(x, dec)) <= 1e-4
    ref = orc.linear(orc.rms_norm(x, g, 1e-5), dec)
    ctx.qlinear(w, dx, dr, M, norm_w=dg, eps=1e-5, residual=dr)
    assert rel_err(dr.download((M, N)), ref + res) <= 1e-4


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
def test_small_m_swiglu_ragged(ctx, orc, dtype):
    """SwiGLU on the small-M matrix-core path: M = 13, F = 1000 (not a multiple
    of 16), K = 4352 (17 slices)."""
    M, Fd, K = 13, 1000, 4352
    wg, gdec = _weight(ctx, 13, "SWg", Fd, K, dtype)
    wu, udec = _weight(ctx, 13, "SWu", Fd, K, dtype)
    x = F.normal(13, "sxs", M * K).reshape(M, K)
    g = 1.0 + F.normal(13, "sgs", K, 0.1)
    dx, dg, dh = ctx.to_device(x), ctx.to_device(g), ctx.alloc(M * Fd * 4)
    ctx.qlinear_swiglu(wg, wu, dx, dh, M, norm_w=dg, eps=1e-5)
    xn = orc.rms_norm(x, g, 1e-5)
    ref = orc.silu_mul(orc.linear(xn, udec), orc.linear(xn, gdec))
    assert rel_err(dh.download((M, Fd)), ref) <= 1e-4


def test_small_m_one_launch_calls_in_a_row(ctx, orc):
    """The small-M path reduces each row tile's slice partials in the tile's
    last workgroup, found by a per-tile counter that the reduction resets:
    calls in a row on one context with different tile and slice counts (a
    grid of fewer columns than slices, so workgroups take two slices, then
    one slice, then 22 slices) each match the oracle, twice over."""
    cases = [(4, 20000, 2048), (2, 300, 256), (16, 2048, 5632), (9, 5632, 2048)]
    for rep in range(2):
        for i, (M, N, K) in enumerate(cases):
            print(f"[case] small-M calls in a row: M={M} N={N} K={K} (pass {rep})", flush=True)
            w, dec = _weight(ctx, 40 + i, f"R{N}x{K}", N, K, V.DT_Q8_0)
            x = F.normal(40 + i, f"rx{M}x{K}", M * K).reshape(M, K)
            dx, dy = ctx.to_device(x), ctx.alloc(M * N * 4)
            ctx.qlinear(w, dx, dy, M)
            assert rel_err(dy.download((M, N)), orc.linear(x, dec)) <= 1e-4, (M, N, K)


def test_qlinear_rejects_bad_shapes(ctx):
    w, _ = _weight(ctx, 11, "Wbad", 64, 96, V.DT_Q8_0)
    x = ctx.alloc(96 * 4 * 17)
    with pytest.raises(V.HipError):
        ctx.qlinear(w, x, ctx.alloc(64 * 4 * 17), 17)      # M > 16 (MFMA path) needs K % 64 == 0
    wf, _ = _weight(ctx, 11, "Wbadf", 64, 64, V.DT_F32)
    with pytest.raises(V.HipError):
        ctx.qlinear(wf, x, ctx.alloc(64 * 4 * 17), 17)     # and a block-quantized weight
    with pytest.raises(V.HipError):
        ctx.qlinear(w, x, x, 1)                             # x aliasing y


@pytest.mark.parametrize("dtype,K", [(V.DT_Q8_0, 32), (V.DT_Q4_0, 32), (V.DT_Q8_0, 96), (V.DT_F32, 32), (V.DT_F32, 64)])
def test_qlinear_rejects_bad_k_above_128_rows(ctx, dtype, K):
    """K below a step of 64 (no step to split) or off it, and f32 weights: an
    argument error from both forms, and the context goes on."""
    M, N = 129, 64
    print(f"[case] refused K={K} dtype={dtype}", flush=True)
    wf = F.normal(11, f"Wk{K}", N * K, 0.02)
    w = V.QuantWeight(ctx, F.quantize(wf, dtype) if dtype != V.DT_F32 else wf, dtype, N, K)
    x, y = ctx.alloc(M * K * 4), ctx.alloc(M * N * 4)
    with pytest.raises(V.HipError):
        ctx.qlinear(w, x, y, M)
    with pytest.raises(V.HipError):
        ctx.qlinear_swiglu(w, w, x, y, M)
    ctx.qlinear(w, x, y, 16)
    ctx.sync()


def _small_bound(x, dec, nw, eps=1e-5):
    """(y, bound) in 64 bits: f32 sums of K products, exact in pieces, are off by
    at most (K + 60) eps of the absolute sum; a fused norm adds (K / 2 + 10) eps."""
    K = x.shape[1]
    x = x.astype(np.float64)
    if nw is not None:
        x = x / np.sqrt((x * x).mean(-1, keepdims=True) + eps) * nw.astype(np.float64)
    d = dec.astype(np.float64)
    return x @ d.T, (1.5 * K + 70 if nw is not None else K + 60) * 2.0 ** -24 * (np.abs(x) @ np.abs(d).T)


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
@pytest.mark.parametrize("M,N,K,norm,res", [
    (16, 64, 128, False, False), (16, 63, 224, True, False), (9, 65, 288, False, True), (2, 130, 1056, True, True),
    (5, 1, 480, False, False), (3, 700, 1824, True, False), (16, 300, 6176, False, True), (7, 257, 320, True, True),
    (2, 40, 320, True, False), (4, 64, 14304, False, False)])   # 320 x 2: stays on the vector kernel
def test_small_m_any_k(ctx, dtype, M, N, K, norm, res):
    """2..16 rows over K that is no multiple of 256: a last slice of 1..7 blocks,
    rows of an odd number of blocks, N off the row tile."""
    print(f"[case] small M any K dtype={dtype} M={M} N={N} K={K} norm={norm} res={res}", flush=True)
    wf = F.normal(33, f"W{N}x{K}", N * K, 0.02)
    blocks = F.quantize(wf, dtype)
    dec = F.dequantize(blocks, dtype, N * K).reshape(N, K)
    w = V.QuantWeight(ctx, blocks, dtype, N, K)
    x = F.normal(33, f"x{M}x{K}", M * K).reshape(M, K)
    nw = 1 + F.normal(33, f"n{K}", K, 0.1) if norm else None
    r = F.normal(33, f"r{M}x{N}", M * N).reshape(M, N)
    dy = ctx.to_device(r)
    ctx.qlinear(w, ctx.to_device(x), dy, M, norm_w=ctx.to_device(nw) if norm else None, residual=dy if res else None)
    ref, bound = _small_bound(x, dec, nw)
    if res:
        ref, bound = ref + r, bound + 2.0 ** -23 * (np.abs(ref) + np.abs(r))
    assert (np.abs(dy.download((M, N)) - ref) <= bound).all()


@pytest.mark.parametrize("M,N,K,norm", [(4, 60, 512 - 32, False), (4, 60, 544, False), (3, 60, 992, False), (3, 60, 1056, False),
                                        (2, 8193, 1056, False), (2, 8192, 1056, False), (3, 16385, 608, False),
                                        (2, 60, 992, True), (3, 60, 704, True)])
def test_small_m_any_k_lines_between_the_kernels(ctx, M, N, K, norm):
    """Either side of where such calls go over from the vector kernel: the same
    bound on both (it is theirs, not a kernel's)."""
    print(f"[case] small M lines M={M} N={N} K={K} norm={norm}", flush=True)
    w, dec = _weight(ctx, 38, f"W{N}x{K}", N, K, V.DT_Q4_0)
    x = F.normal(38, f"x{M}x{K}", M * K).reshape(M, K)
    nw = 1 + F.normal(38, f"n{K}", K, 0.1) if norm else None
    dy = ctx.alloc(M * N * 4)
    ctx.qlinear(w, ctx.to_device(x), dy, M, norm_w=ctx.to_device(nw) if norm else None)
    ref, bound = _small_bound(x, dec, nw)
    assert (np.abs(dy.download((M, N)) - ref) <= bound).all()


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
@pytest.mark.parametrize("M,K", [(16, 288), (5, 1056), (3, 4128)])
def test_small_m_any_k_every_piece_of_x_counts(ctx, dtype, M, K):
    """x = 1 + small parts that only the second, or only the third, bf16 piece
    holds, over weights c, -c, c, ..: the first piece (and the second) cancels in
    every block and the result is the small parts alone.  Of each block's 32
    products in three pieces, at most 100 additions round, each by eps of a
    partial sum, which is at most half of the absolute sum; a lost piece is five
    times that bound off, or more."""
    N, nb = 70, K // 32
    print(f"[case] small M pieces M={M} K={K} dtype={dtype}", flush=True)
    scale = np.frombuffer(np.float16(1 / 64).tobytes(), np.uint8)
    codes = np.tile(np.array([127, 129], np.uint8), 16) if dtype == V.DT_Q8_0 else np.full(16, 0x1F, np.uint8)
    blocks = np.tile(np.concatenate([scale, codes]), N * nb).reshape(N, -1)
    c = (127 if dtype == V.DT_Q8_0 else 7) / 64
    w = V.QuantWeight(ctx, blocks, dtype, N, K)
    k = 255 - np.arange(M)[:, None]
    for base, part in ((1.0, k * 2.0 ** -15), (1.0 + 2.0 ** -8, k * 2.0 ** -23)):
        x = np.full((M, K), base)
        x[:, ::2] += part
        assert (x.astype(np.float32) == x).all()
        dy = ctx.alloc(M * N * 4)
        ctx.qlinear(w, ctx.to_device(x.astype(np.float32)), dy, M)
        ref = c * (K // 2) * part                             # every column of the result alike
        bound = 100 * 2.0 ** -24 * (c * K * 1.01) / 2
        assert (ref > 4 * bound).all()
        assert (np.abs(dy.download((M, N)) - ref) <= bound).all()


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
def test_small_m_any_k_error_at_long_k(ctx, dtype):
    """56 slices added with their rounding errors: no further from 64 bits than the
    vector kernel at this shape (1.6e-7 of the 2-norm; 1.9e-7 without the errors)."""
    M, N, K = 16, 300, 14272
    print(f"[case] small M long K dtype={dtype}", flush=True)
    w, dec = _weight(ctx, 37, f"L{N}x{K}", N, K, dtype)
    x = F.normal(37, f"x{M}x{K}", M * K).reshape(M, K)
    dy = ctx.alloc(M * N * 4)
    ctx.qlinear(w, ctx.to_device(x), dy, M)
    ref = x.astype(np.float64) @ dec.astype(np.float64).T
    err = np.linalg.norm(dy.download((M, N)) - ref) / np.linalg.norm(ref)
    print(f"[error] {err:.3g}", flush=True)
    assert err <= 1.6e-7


@pytest.mark.parametrize("M,N,K,norm,res", [
    (2, 70, 256, True, False), (8, 64, 512, True, True), (9, 63, 2048, True, False), (16, 130, 2304, True, False),
    (7, 65, 2560, False, True), (16, 40, 4352, True, False), (3, 33, 2304, False, False)])
def test_small_m_slice_counts(ctx, M, N, K, norm, res):
    """1, 2, 8, 9, 10 and 17 slices of 256 columns, whose partial sums are added
    eight slices at a time or one; rows up to eight and more.  x in two bf16
    pieces is off by at most 2^-16 of itself; with a norm a rounding more."""
    print(f"[case] small M slices M={M} N={N} K={K} norm={norm} res={res}", flush=True)
    w, dec = _weight(ctx, 36, f"S{N}x{K}", N, K, V.DT_Q8_0)
    x = F.normal(36, f"x{M}x{K}", M * K).reshape(M, K)
    nw = 1 + F.normal(36, f"n{K}", K, 0.1) if norm else None
    r = F.normal(36, f"r{M}x{N}", M * N).reshape(M, N)
    dy = ctx.to_device(r)
    ctx.qlinear(w, ctx.to_device(x), dy, M, norm_w=ctx.to_device(nw) if norm else None, residual=dy if res else None)
    ref, bound = _small_bound(x, dec, nw)
    bound = bound * (1 + 2.0 ** 8 / K)   # + 2^-16 of the absolute sum, in units of K eps
    if res:
        ref, bound = ref + r, bound + 2.0 ** -23 * (np.abs(ref) + np.abs(r))
    assert (np.abs(dy.download((M, N)) - ref) <= bound).all()


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0])
@pytest.mark.parametrize("M,N,K", [(16, 70, 352), (3, 200, 1504)])
def test_small_m_any_k_swiglu_and_specials(ctx, orc, dtype, M, N, K):
    """SwiGLU over such K; and infinities and NaN in x stay in their rows with the
    vector kernel's meaning (they have no second and third piece), as does a
    value whose product with the largest code is still finite."""
    ws = []
    for n in "gu":
        b = F.quantize(F.normal(34, f"{n}{N}x{K}", N * K, 0.02), dtype)
        ws.append((V.QuantWeight(ctx, b, dtype, N, K), F.dequantize(b, dtype, N * K).reshape(N, K)))
    x = F.normal(34, f"x{M}x{K}", M * K).reshape(M, K)
    dh = ctx.alloc(M * N * 4)
    ctx.qlinear_swiglu(ws[0][0], ws[1][0], ctx.to_device(x), dh, M)
    ref = orc.silu_mul(orc.linear(x, ws[1][1]), orc.linear(x, ws[0][1]))
    assert rel_err(dh.download((M, N)), ref) <= 1e-5
    x[0, K - 1], x[1, 5], x[2] = np.inf, np.nan, 0.0
    x[2, 7] = 2e36
    dy = ctx.alloc(M * N * 4)
    ctx.qlinear(ws[0][0], ctx.to_device(x), dy, M)
    got, dec = dy.download((M, N)), ws[0][1]
    last, seven = dec[:, K - 1], dec[:, 7].astype(np.float64) * np.float64(x[2, 7])
    assert (np.sign(got[0][last != 0]) == np.sign(last[last != 0])).all() and np.isinf(got[0][last != 0]).all()
    assert np.isnan(got[0][last == 0]).all() and np.isnan(got[1]).all()
    assert np.allclose(got[2], seven, rtol=1e-6)
    if M > 3:
        ref3, bound3 = _small_bound(x[3:], dec, None)
        assert (np.abs(got[3:] - ref3) <= bound3).all()


def test_small_m_any_k_under_graph_capture(orc):
    """Under capture the call keeps no scratch address: it runs on the vector
    kernel, and replays to f32 rounding of the eager result, every time."""
    import ctypes as C
    from test_gpu_prefill_gemm import _hip
    hip, ctx = _hip(), V.Context(0)
    M, N, K = 8, 200, 1056
    b = F.quantize(F.normal(35, "w", N * K, 0.02), V.DT_Q8_0)
    w, dec = V.QuantWeight(ctx, b, V.DT_Q8_0, N, K), F.dequantize(b, V.DT_Q8_0, N * K).reshape(N, K)
    x = F.normal(35, "x", M * K).reshape(M, K)
    dx, dy, de = ctx.to_device(x), ctx.alloc(M * N * 4), ctx.alloc(M * N * 4)
    s, g, ge = C.c_void_p(ctx.stream()), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(s, 2) == 0
    rc = V.lib().vlrf_hip_qlinear(ctx.h, w.h, dx.ptr, dy.ptr, M, None, C.c_float(0.0), None)   # no call before it
    assert hip.hipStreamEndCapture(s, C.byref(g)) == 0 and rc == 0, V.lib().vlrf_hip_last_error()
    assert hip.hipGraphInstantiate(C.byref(ge), g, None, None, 0) == 0
    ref, bound = _small_bound(x, dec, None)
    for _ in range(3):
        dy.zero()
        ctx.qlinear(w, dx, de, M)
        assert hip.hipGraphLaunch(ge, s) == 0
        ctx.sync()
        for d in (dy, de):
            assert (np.abs(d.download((M, N)) - ref) <= bound).all()
    hip.hipGraphExecDestroy(ge)
    hip.hipGraphDestroy(g)
