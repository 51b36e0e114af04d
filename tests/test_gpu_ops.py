"""GPU parity of the engine's remaining per-op backend calls (IBackend::gemm,
layer_norm, softmax_inplace, gelu_inplace, add_inplace; ibackend.hpp:61-70)
against the oracle's restatements of ops.hpp (pinned against the reference
build in tests/test_oracle.py).  Tolerance 1e-3 relative (f32 paths); the
reductions run in a different order than the CPU's sequential loops."""
import numpy as np
import pytest

import vlrf_amd as V
from conftest import rel_err
from vlrf_amd import formats as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1, 300, 64), (37, 29, 64), (130, 257, 515), (64, 64, 16), (200, 768, 3072)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_gemm_f32(ctx, orc, M, N, K, ta, tb):
    print(f"[case] gemm_f32 {M}x{N}x{K} ta={ta} tb={tb}", flush=True)
    A = F.normal(60, f"A{M}x{K}", M * K).reshape(M, K)
    B = F.normal(60, f"B{K}x{N}", K * N).reshape(K, N)
    Ai = A.T.copy() if ta else A
    Bi = B.T.copy() if tb else B
    for alpha, beta in ((1.0, 0.0), (0.7, 1.0), (-1.25, 0.5)):
        C0 = F.normal(60, f"C{M}x{N}", M * N).reshape(M, N)
        if beta == 0.0:
            C0[:] = np.nan                        # beta == 0 must not read C (ops.hpp:186-188)
        dA, dB, dC = ctx.to_device(Ai), ctx.to_device(Bi), ctx.to_device(C0)
        ctx.gemm_f32(dA, dB, dC, M, N, K, alpha, beta, ta, tb)
        got = dC.download((M, N))
        ref = orc.gemm(Ai, Bi, np.nan_to_num(C0) if beta == 0.0 else C0, alpha, beta, ta, tb)
        assert np.isfinite(got).all()
        assert rel_err(got, ref) <= 1e-3, (alpha, beta)


def _gemm64(A, B):
    """(A.B, |A|.|B|) in 64 bits: f32 sums of K products in any order differ from
    the first by at most (K + slices + 2) eps of the second."""
    return A.astype(np.float64) @ B.astype(np.float64), np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)


@pytest.mark.parametrize("M,N,K,pad,off", [
    (32, 128, 64, 0, 0), (33, 129, 65, 0, 0), (31, 127, 63, 0, 0), (1, 1, 1, 0, 0),      # tile edges
    (64, 64, 128, 4, 0), (65, 63, 132, 4, 0), (4, 260, 4096, 8, 0),                       # padded rows, 16-byte loads
    (40, 72, 260, 3, 0), (40, 72, 260, 4, 1), (2, 130, 1000, 0, 3),                       # odd rows, odd addresses
    (100, 200, 6000, 0, 0), (1, 100, 8191, 0, 0), (700, 768, 1000, 0, 0),                 # split K, ragged slices
])
@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False), (True, True)])
def test_gemm_f32_tiles_and_splits(ctx, M, N, K, pad, off, ta, tb):
    """Edges of the tiles, of the K steps and of the slices; leading dimensions
    beyond the rows; addresses that forbid 16-byte loads."""
    print(f"[case] gemm_f32 {M}x{N}x{K} pad={pad} off={off} ta={ta} tb={tb}", flush=True)
    A, B = (F.normal(64, n, r * c).reshape(r, c) for n, r, c in ((f"a{M}.{K}", M, K), (f"b{K}.{N}", K, N)))

    def put(X, trans):
        X = X.T if trans else X
        rows, cols = X.shape
        host = np.full(off + rows * (cols + pad), np.nan, np.float32)   # the padding is not used
        host[off:].reshape(rows, cols + pad)[:, :cols] = X
        return ctx.to_device(host), cols + pad

    (dA, lda), (dB, ldb) = put(A, ta), put(B, tb)
    ldc = N + pad
    C0 = F.normal(64, f"c{M}.{N}", M * ldc).reshape(M, ldc)
    dC = ctx.to_device(C0)
    V.check(V.lib().vlrf_hip_gemm_f32(ctx.h, dA.ptr + 4 * off, dB.ptr + 4 * off, dC.ptr, M, N, K, lda, ldb, ldc,
                                      1.5, 0.5, int(ta), int(tb)))
    got = dC.download((M, ldc))
    ref, mag = _gemm64(A, B)
    bound = (K + 70) * 2.0 ** -24 * 1.5 * mag + 3 * 2.0 ** -24 * np.abs(0.5 * C0[:, :N].astype(np.float64)) + 1e-30
    assert (np.abs(got[:, :N] - (1.5 * ref + 0.5 * C0[:, :N])) <= bound).all()
    assert np.array_equal(got[:, N:], C0[:, N:])                        # between the rows of C


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (33, 3, 3), (64, 64, 4), (64, 65, 16), (17, 130, 15), (64, 64, 17),
                                   (2100, 1030, 32), (2100, 1030, 33), (70, 50001, 48), (70, 50001, 49),
                                   (65, 50000, 80), (65, 50000, 81)])
def test_gemm_f32_short_k(ctx, M, N, K, ta, tb):
    """Both sides of the lines between the two kernels: one step of 16, 512 and 1536
    tiles, K of 32, 48 and 80; alpha, beta and a gap between the rows of C."""
    print(f"[case] gemm short K M={M} N={N} K={K} ta={ta} tb={tb}", flush=True)
    A, B = F.normal(71, f"a{M}.{K}", M * K).reshape(M, K), F.normal(71, f"b{K}.{N}", K * N).reshape(K, N)
    ldc = N + 3
    C0 = F.normal(71, f"c{M}.{N}", M * ldc).reshape(M, ldc)
    dA, dB = (ctx.to_device(np.ascontiguousarray(t.T if x else t)) for t, x in ((A, ta), (B, tb)))
    dC = ctx.to_device(C0)
    V.check(V.lib().vlrf_hip_gemm_f32(ctx.h, dA.ptr, dB.ptr, dC.ptr, M, N, K, M if ta else K, K if tb else N, ldc,
                                      1.5, 0.5, int(ta), int(tb)))
    got = dC.download((M, ldc))
    ref, mag = _gemm64(A, B)
    bound = (K + 4) * 2.0 ** -24 * 1.5 * mag + 3 * 2.0 ** -24 * np.abs(0.5 * C0[:, :N].astype(np.float64)) + 1e-30
    assert (np.abs(got[:, :N] - (1.5 * ref + 0.5 * C0[:, :N])) <= bound).all()
    assert np.array_equal(got[:, N:], C0[:, N:])


@pytest.mark.parametrize("M,N,K", [(3, 40, 200), (70, 130, 1024)])
def test_gemm_f32_specials(ctx, M, N, K):
    """Infinities, NaN and denormals stay in their row of C and keep their meaning."""
    A, B = F.normal(65, f"sa{K}", M * K).reshape(M, K), F.normal(65, f"sb{K}", N * K).reshape(N, K)
    A[0, 1], A[1, K - 1], A[2] = np.inf, np.nan, 0.0
    A[2, 0], B[0] = 1e-39, 0.0                                          # a denormal times 2 is exact in f32
    B[0, 0] = 2.0
    dA, dB, dC = ctx.to_device(A), ctx.to_device(B), ctx.alloc(M * N * 4)
    ctx.gemm_f32(dA, dB, dC, M, N, K, trans_b=True)
    got = dC.download((M, N))
    ref, mag = _gemm64(A[2:], B.T)
    assert (np.isinf(got[0, 1:]).all() and (np.sign(got[0, 1:]) == np.sign(B[1:, 1])).all())
    assert np.isnan(got[0, 0]) and np.isnan(got[1]).all()               # inf * 0, NaN
    assert (np.abs(got[2:] - ref) <= (K + 70) * 2.0 ** -24 * mag + 1e-45).all()
    assert got[2, 0] == np.float32(1e-39) * np.float32(2.0)


def test_gemm_f32_under_graph_capture():
    """Under capture K stays whole (a captured launch keeps no scratch address
    that a later call may regrow); every replay gives the same result."""
    import ctypes as C
    from test_gpu_prefill_gemm import _hip
    hip, ctx = _hip(), V.Context(0)
    M, N, K = 60, 100, 4096
    A, B = F.normal(66, "ca", M * K).reshape(M, K), F.normal(66, "cb", N * K).reshape(N, K)
    dA, dB, dC, dE = ctx.to_device(A), ctx.to_device(B), ctx.alloc(M * N * 4), ctx.alloc(M * N * 4)
    ctx.gemm_f32(dA, dB, dE, M, N, K, trans_b=True)
    eager = dE.download((M, N))
    s, g, ge = C.c_void_p(ctx.stream()), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(s, 2) == 0
    rc = V.lib().vlrf_hip_gemm_f32(ctx.h, dA.ptr, dB.ptr, dC.ptr, M, N, K, K, K, N, 1.0, 0.0, 0, 1)
    assert hip.hipStreamEndCapture(s, C.byref(g)) == 0 and rc == 0
    assert hip.hipGraphInstantiate(C.byref(ge), g, None, None, 0) == 0
    ref, mag = _gemm64(A, B.T)
    big = ctx.alloc(4 * 64 * 8192)
    for _ in range(3):
        dC.zero()
        ctx.gemm_f32(dA, dB, big, M, 100, K, trans_b=True)              # eager work, with scratch, between
        assert hip.hipGraphLaunch(ge, s) == 0
        ctx.sync()
        got = dC.download((M, N))
        assert (np.abs(got - ref) <= (K + 70) * 2.0 ** -24 * mag).all()
        assert (np.abs(eager - ref) <= (K + 70) * 2.0 ** -24 * mag).all()
    hip.hipGraphExecDestroy(ge)
    hip.hipGraphDestroy(g)


def test_captured_calls_outlive_scratch_growth():
    """A captured K-split GEMM keeps the scratch address it recorded: eager calls
    that outgrow the buffer (an f32 GEMM, a small-M linear, twice) leave it in
    place, and every replay gives the eager result.  Replayed only once the
    context says that it kept the old buffer."""
    import ctypes as C
    from test_gpu_prefill_gemm import _hip
    hip, ctx = _hip(), V.Context(0)

    def held():
        out = (C.c_size_t * 2)()
        V.check(V.lib().vlrf_hip_scratch_bytes(ctx.h, out))
        return out[0], out[1]

    M, N, K = 64, 512, 1024
    w = V.QuantWeight(ctx, F.quantize(F.normal(69, "w", N * K, 0.02), V.DT_Q8_0), V.DT_Q8_0, N, K)
    dx, dy = ctx.to_device(F.normal(69, "x", M * K)), ctx.alloc(M * N * 4)
    ctx.qlinear(w, dx, dy, M)
    eager = dy.download((M, N))
    s, g, ge = C.c_void_p(ctx.stream()), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(s, 2) == 0
    rc = V.lib().vlrf_hip_qlinear(ctx.h, w.h, dx.ptr, dy.ptr, M, None, C.c_float(0.0), None)
    assert hip.hipStreamEndCapture(s, C.byref(g)) == 0 and rc == 0
    assert hip.hipGraphInstantiate(C.byref(ge), g, None, None, 0) == 0
    small, kept = held()
    assert small > 0 and kept == 0
    m, n, k = 64, 512, 16384                                            # splits K: m n 4 bytes a slice
    A, B, Cb = ctx.to_device(F.normal(69, "A", m * k)), ctx.to_device(F.normal(69, "B", n * k)), ctx.alloc(m * n * 4)
    n2, k2 = 9000, 4128                                                 # any-K small-M: more partials than that
    w2 = V.QuantWeight(ctx, F.quantize(F.normal(69, "w2", n2 * k2, 0.02), V.DT_Q8_0), V.DT_Q8_0, n2, k2)
    x2, y2 = ctx.to_device(F.normal(69, "x2", 16 * k2)), ctx.alloc(16 * n2 * 4)
    for grow in (lambda: ctx.gemm_f32(A, B, Cb, m, n, k, trans_b=True), lambda: ctx.qlinear(w2, x2, y2, 16)):
        before = held()[0]
        grow()
        ctx.sync()
        assert held()[0] > before and held()[1] == small                # the captured one, and no other
        for _ in range(3):
            dy.zero()
            grow()
            assert hip.hipGraphLaunch(ge, s) == 0
            ctx.sync()
            assert np.array_equal(dy.download((M, N)), eager)
    hip.hipGraphExecDestroy(ge)
    hip.hipGraphDestroy(g)


def test_gemm_f32_rejects_bad_shapes(ctx):
    a = ctx.alloc(64)
    with pytest.raises(V.HipError):
        ctx.gemm_f32(a, a, a, 0, 4, 4)
    with pytest.raises(V.HipError):
        ctx.gemm_f32(a, a, a, 4, 4, 4, lda=2)


@pytest.mark.parametrize("rows,D", [(1, 768), (7, 1000), (3, 5000), (2, 1)])
def test_layer_norm(ctx, orc, rows, D):
    x = F.normal(61, f"lx{D}", rows * D).reshape(rows, D) * 3 + 0.5
    w, b = 1 + F.normal(61, f"lw{D}", D, 0.1), F.normal(61, f"lb{D}", D, 0.1)
    dx, dw, db, do = ctx.to_device(x), ctx.to_device(w), ctx.to_device(b), ctx.alloc(x.nbytes)
    ctx.layer_norm(dx, dw, db, do, rows, D, 1e-5)
    assert rel_err(do.download(x.shape), orc.layer_norm(x, w, b, 1e-5)) <= 1e-3


@pytest.mark.parametrize("rows,D", [(1, 2048), (12, 77), (4, 5000), (3, 1)])
def test_softmax(ctx, orc, rows, D):
    x = F.normal(62, f"sx{D}", rows * D).reshape(rows, D) * 4
    if D > 2:
        x[0, 1] = -np.inf                         # a masked score: exp(-inf) = 0
    dx = ctx.to_device(x)
    ctx.softmax(dx, rows, D)
    got = dx.download(x.shape)
    ref = orc.softmax(x)        # the oracle sums sequentially for every D
    assert rel_err(got, ref) <= 1e-3
    assert np.allclose(got.sum(axis=1), 1.0, atol=1e-5)


@pytest.mark.parametrize("n", [1, 1000, 300001])
def test_gelu_and_add(ctx, orc, n):
    x = F.normal(63, f"gx{n}", n) * 5
    dx = ctx.to_device(x)
    ctx.gelu(dx, n)
    assert rel_err(dx.download(x.shape), orc.gelu(x)) <= 1e-5 * 10
    y = F.normal(63, f"gy{n}", n)
    a, b = ctx.to_device(x), ctx.to_device(y)
    ctx.add(a, b, n)
    assert np.array_equal(a.download(x.shape), x + y)       # one rounding per element, as the CPU


@pytest.mark.parametrize("n,off", [(3, 0), (4, 0), (5, 1), (1023, 0), (4099, 2), (70003, 0)])
def test_gelu_and_add_groups_of_four(ctx, orc, n, off):
    """Counts off the groups of four and addresses off 16 bytes: the same values as
    element by element, nothing beyond the end written."""
    x, y = F.normal(67, f"x{n}", n) * 3, F.normal(67, f"y{n}", n)
    pad = np.full(off, 9.0, np.float32)
    a, b = (ctx.to_device(np.concatenate([pad, t, pad, [9.0]]).astype(np.float32)) for t in (x, y))
    V.check(V.lib().vlrf_hip_gelu(ctx.h, a.ptr + 4 * off, n))
    g = a.download((n + 2 * off + 1,))
    assert rel_err(g[off:off + n], orc.gelu(x)) <= 1e-6
    V.check(V.lib().vlrf_hip_add(ctx.h, a.ptr + 4 * off, b.ptr + 4 * off, n))
    s = a.download((n + 2 * off + 1,))
    assert np.array_equal(s[off:off + n], g[off:off + n] + y)
    assert (np.delete(s, np.s_[off:off + n]) == 9.0).all() and (np.delete(g, np.s_[off:off + n]) == 9.0).all()


@pytest.mark.parametrize("rows,D,off", [(5, 4, 0), (3, 1020, 0), (2, 1028, 0), (2, 4096, 0), (2, 4100, 0), (3, 768, 1),
                                        (3, 1024, 0), (2, 2048, 0), (2, 2052, 0), (3000, 64, 0)])
def test_layer_norm_in_registers(ctx, rows, D, off):
    """Row lengths at the edges of the register form, and addresses that forbid it,
    against 64 bits: every step is an f32 sum of D terms."""
    x = F.normal(68, f"x{D}", rows * D).reshape(rows, D) * 2 + 1
    w, b = 1 + F.normal(68, f"w{D}", D, 0.1), F.normal(68, f"b{D}", D, 0.1)
    pad = np.zeros(off, np.float32)
    dx, dw, db = (ctx.to_device(np.concatenate([pad, t.ravel()]).astype(np.float32)) for t in (x, w, b))
    do = ctx.alloc(4 * (rows * D + off))
    V.check(V.lib().vlrf_hip_layer_norm(ctx.h, *[t.ptr + 4 * off for t in (dx, dw, db, do)], rows, D, 1e-5))
    got = do.download((rows * D + off,))[off:].reshape(rows, D)
    x64 = x.astype(np.float64)
    c = x64 - x64.mean(1, keepdims=True)
    inv = 1 / np.sqrt((c * c).mean(1, keepdims=True) + 1e-5)
    ref = c * inv * w + b
    bound = (D + 20) * 2.0 ** -24 * (np.abs(x64).max() * inv * np.abs(w) + np.abs(ref) + np.abs(b))
    assert (np.abs(got - ref) <= bound).all()
