"""GPU parity: f32 flash attention (IBackend::sdp_attention) and the Q8_0-KV
GQA decode attention, against the oracle's restatement of
AttentionBlock::flash_attn_head (attention.hpp:207-309).

Inputs are seeded N(0,1) from vlrf_amd.formats.normal (the reference test's
mt19937 stream is not reproducible outside libstdc++; shapes, masks and
tolerances follow tests/test_flash_attention.cpp:77-121)."""
import numpy as np
import pytest

from conftest import rel_err
from vlrf_amd import formats as F

pytestmark = pytest.mark.gpu

# (T, ctx, d_h, causal, seed): tests/test_flash_attention.cpp:96-121
REF_SHAPES = [(64, 64, 32, False, 1), (128, 128, 32, True, 2), (37, 37, 8, True, 5),
              (130, 130, 64, True, 6), (1, 1, 16, False, 3), (1, 200, 16, False, 4),
              (1, 1, 4, True, 8), (200, 500, 64, True, 7), (300, 300, 128, False, 9)]


def _qkv(seed, n_h, T, ctx_len, d):
    Q = F.normal(seed, "Q", n_h * T * d).reshape(n_h, T, d)
    K = F.normal(seed, "K", n_h * ctx_len * d).reshape(n_h, ctx_len, d)
    V = F.normal(seed, "V", n_h * ctx_len * d).reshape(n_h, ctx_len, d)
    return Q, K, V


def _run_gpu(ctx, Q, K, V, scale, causal):
    n_h, T, d = Q.shape
    ctx_len = K.shape[1]
    dq, dk, dv = ctx.to_device(Q), ctx.to_device(K), ctx.to_device(V)
    do = ctx.alloc(Q.nbytes)
    ctx.sdp_attention(dq, dk, dv, do, n_h, T, ctx_len, d, scale, causal)
    return do.download(Q.shape)


@pytest.mark.parametrize("T,ctx_len,d,causal,seed", REF_SHAPES)
def test_sdp_attention_reference_shapes(ctx, orc, T, ctx_len, d, causal, seed):
    print(f"[case] sdp T={T} ctx={ctx_len} d={d} causal={causal}", flush=True)
    n_h = 2
    Q, K, V = _qkv(seed, n_h, T, ctx_len, d)
    scale = np.float32(1.0) / np.sqrt(np.float32(d))
    out = _run_gpu(ctx, Q, K, V, scale, causal)
    ref = orc.sdp_attention(Q, K, V, scale, causal)
    assert np.max(np.abs(out - ref)) <= 1e-4          # the reference test's own bound
    assert rel_err(out, ref) <= 1e-3


def _sdp64(Q, K, V, scale, causal):
    """(attention in 64 bits, a bound on an f32 result's distance from it): every
    weight is off by at most eps ((d + 8) S + 40) relative, S the query's largest
    |scale| sum |q||k|; the sums over the keys add ctx eps each; both in the
    numerator and in the normaliser."""
    n_h, T, d = Q.shape
    n = K.shape[1]
    Q, K, V = (t.astype(np.float64) for t in (Q, K, V))
    keep = np.arange(n)[None, :] <= np.arange(T)[:, None] + (n - T) if causal else np.ones((T, n), bool)
    s = np.where(keep, Q @ K.transpose(0, 2, 1) * scale, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    S = np.where(keep, np.abs(Q) @ np.abs(K).transpose(0, 2, 1) * abs(scale), 0).max(-1, keepdims=True)
    return p @ V, 2 * 2.0 ** -24 * ((d + 8) * S + n + 40) * (p @ np.abs(V))


@pytest.mark.parametrize("T,ctx_len,d,causal,scale,off", [
    (1, 1, 1, True, 1.0, 0), (31, 31, 15, True, 0.5, 0), (32, 33, 16, True, 0.25, 0), (33, 64, 17, False, 0.3, 0),
    (64, 127, 48, True, 0.2, 0), (65, 65, 63, True, 0.125, 0), (40, 129, 64, True, 0.125, 1),   # odd addresses
    (1, 300, 64, True, 0.125, 0), (100, 100, 80, True, 0.11, 0), (7, 1000, 81, False, 0.11, 0),
    (50, 34, 96, False, 0.1, 0), (33, 200, 112, True, 0.1, 0), (70, 257, 127, True, 0.09, 0), (97, 97, 128, True, 0.09, 2),
    (40, 90, 64, True, -0.125, 0), (40, 90, 64, True, 0.0, 0), (5, 2050, 4, False, 0.5, 0)])
def test_sdp_attention_tiles(ctx, T, ctx_len, d, causal, scale, off):
    """Edges of the query blocks, key tiles and head-size steps; rows that forbid
    16-byte loads; negative and zero scales."""
    print(f"[case] sdp tiles T={T} ctx={ctx_len} d={d} causal={causal} scale={scale} off={off}", flush=True)
    n_h = 3
    Q, K, V = _qkv(T * 7 + d, n_h, T, ctx_len, d)
    bufs = [ctx.to_device(np.concatenate([np.full(off, np.nan, np.float32), t.ravel()])) for t in (Q, K, V)]
    do = ctx.to_device(np.full(Q.size + 8, 7.0, np.float32))
    import vlrf_amd as V_
    V_.check(V_.lib().vlrf_hip_attn_f32(ctx.h, *[b.ptr + 4 * off for b in bufs], do.ptr, n_h, T, ctx_len, d, scale,
                                        int(causal)))
    got = do.download((Q.size + 8,))
    ref, bound = _sdp64(Q, K, V, np.float32(scale), causal)
    assert (np.abs(got[:Q.size].reshape(Q.shape) - ref) <= bound).all()
    assert (got[Q.size:] == 7.0).all()


def test_sdp_attention_long_grid(ctx):
    """More blocks of queries than a grid takes along y: 2^20 queries a z step,
    past 65535 blocks, a ragged last one.  One key: the result is its value."""
    T, d = 65535 * 32 + 45, 4
    print(f"[case] sdp long grid T={T}", flush=True)
    Q = np.ones((1, T, d), np.float32)
    V1 = np.arange(1, d + 1, dtype=np.float32).reshape(1, 1, d)
    dq, dk, dv = ctx.to_device(Q), ctx.to_device(np.ones_like(V1)), ctx.to_device(V1)
    do = ctx.to_device(np.full(Q.size + 8, 7.0, np.float32))
    ctx.sdp_attention(dq, dk, dv, do, 1, T, 1, d, 0.5, False)
    got = do.download((Q.size + 8,))
    assert (got[:Q.size].reshape(T, d) == V1[0]).all()
    assert (got[Q.size:] == 7.0).all()


def test_sdp_attention_specials(ctx, orc):
    """-inf scores weigh nothing, a NaN query stays in its row, an infinite value
    in a key that every query of the block may see reaches all of them."""
    T, n, d = 40, 200, 64
    Q, K, V = _qkv(77, 2, T, n, d)
    Q[0], K[0, 3] = np.abs(Q[0]), -np.inf                     # head 0: key 3 scores -inf
    Q[1, 5] = np.nan
    V[1, 0, 2] = np.inf
    out = _run_gpu(ctx, Q, K, V, np.float32(0.125), True)
    K0, V0 = np.delete(K[:1], 3, 1), np.delete(V[:1], 3, 1)
    ref, bound = _sdp64(Q[:1], K0, V0, np.float32(0.125), True)
    assert (np.abs(out[0] - ref[0]) <= bound[0]).all()
    cpu = orc.sdp_attention(Q, K, V, np.float32(0.125), True)
    rows = np.arange(T) != 5
    assert np.isposinf(out[1][rows, 2]).all() and np.isposinf(cpu[1][rows, 2]).all()
    fine = np.ones(d, bool)
    fine[2] = False
    assert rel_err(out[1][rows][:, fine], cpu[1][rows][:, fine]) <= 1e-3


def test_config1_decode_f32(ctx, orc):
    """Benchmark config 1: 1 query, 8 heads, d 64, KV 512, non-causal, scale 1/8."""
    Q, K, V = _qkv(11, 8, 1, 512, 64)
    out = _run_gpu(ctx, Q, K, V, np.float32(0.125), False)
    ref = orc.sdp_attention(Q, K, V, np.float32(0.125), False)
    assert np.max(np.abs(out - ref)) <= 1e-4
    assert rel_err(out, ref) <= 1e-3


@pytest.mark.parametrize("ctx_len", [1, 255, 256, 257, 1000])
def test_decode_f32_split_boundaries(ctx, orc, ctx_len):
    """Split-K chunk boundaries (256 tokens) and a single-token context."""
    Q, K, V = _qkv(ctx_len, 4, 1, ctx_len, 128)
    s = np.float32(1.0) / np.sqrt(np.float32(128))
    out = _run_gpu(ctx, Q, K, V, s, False)
    ref = orc.sdp_attention(Q, K, V, s, False)
    assert rel_err(out, ref) <= 1e-3


def _gqa_reference(orc, q, kq, vq, ks, vs, n_heads, n_kv, d, ctx_len, scale):
    """Reference decode attention: dequant_into (kv_cache.hpp:259-286), GQA head
    h -> kv head h/(n_heads/n_kv) (attention.hpp:328-342), non-causal
    flash_attn_head per head."""
    row = n_kv * d
    Kd = kq[:ctx_len].astype(np.float32) * ks[:ctx_len, None]
    Vd = vq[:ctx_len].astype(np.float32) * vs[:ctx_len, None]
    out = np.zeros(n_heads * d, np.float32)
    rep = n_heads // n_kv
    for h in range(n_heads):
        g = h // rep
        out[h * d:(h + 1) * d] = orc.flash_attn_head(q[h * d:(h + 1) * d][None, :],
                                                     Kd[:, g * d:(g + 1) * d],
                                                     Vd[:, g * d:(g + 1) * d], scale, False)[0]
    assert Kd.shape[1] == row
    return out


@pytest.mark.parametrize("n_heads,n_kv,d,ctx_len", [(32, 4, 64, 4096), (32, 4, 64, 2048),
                                                    (8, 8, 64, 300), (16, 2, 128, 777),
                                                    (8, 1, 64, 1), (16, 8, 64, 509),
                                                    (32, 8, 64, 65), (32, 4, 64, 510),
                                                    (8, 2, 64, 4600)])
def test_q8_decode_attention(ctx, orc, n_heads, n_kv, d, ctx_len):
    """Benchmark config 2 (32q/4kv, d 64, ctx 4096) and other GQA groupings.
    d_head 64 takes the one-launch chunked kernel (64-row chunks up to 1024
    tokens; 509 + 3 rows fill a chunk's round), d_head 128 the split-K
    kernel and its combine."""
    import vlrf_amd as V_
    print(f"[case] q8 decode heads={n_heads}/{n_kv} d={d} ctx={ctx_len}", flush=True)
    row = n_kv * d
    kv = V_.KVCache(ctx, 1, ctx_len + 3, n_kv, d)
    K = F.normal(5, "Kc", ctx_len * row)
    Vv = F.normal(5, "Vc", ctx_len * row)
    kv.append(0, ctx.to_device(K), ctx.to_device(Vv), ctx_len)
    kq, vq, ks, vs = kv.read(0, 0, ctx_len)
    q = F.normal(5, "q", n_heads * d)
    dq = ctx.to_device(q)
    dout = ctx.alloc(q.nbytes)
    scale = np.float32(1.0) / np.sqrt(np.float32(d))
    kv.attention_decode(0, dq, dout, n_heads, ctx_len, scale)
    out = dout.download(q.shape)
    ref = _gqa_reference(orc, q, kq, vq, ks, vs, n_heads, n_kv, d, ctx_len, scale)
    assert rel_err(out, ref) <= 1e-3
    assert np.max(np.abs(out - ref)) <= 1e-4


def _dequant_rows(kv, ctx_len):
    import vlrf_amd as V_
    kq, vq, ks, vs = kv.read(0, 0, ctx_len)
    if kv.dtype == V_.KV_Q8_0:
        return kq.astype(np.float32) * ks[:, None], vq.astype(np.float32) * vs[:, None]
    if kv.dtype == V_.KV_F16:
        return kq.view(np.float16).astype(np.float32), vq.view(np.float16).astype(np.float32)
    return kq, vq


@pytest.mark.parametrize("kv_name", ["Q8_0", "F16", "F32"])
@pytest.mark.parametrize("n_heads,n_kv,ctx_len", [(32, 4, 1024), (32, 4, 1025), (8, 2, 2049),
                                                  (16, 16, 4097), (32, 4, 8192), (8, 8, 8193)])
def test_decode_attention_chunk_sizes(ctx, orc, kv_name, n_heads, n_kv, ctx_len):
    """d_head 64 decode attention in one launch: contexts at the chunk-size
    steps (64 rows up to 1024 tokens, then 128/256/512 so that at most 16
    chunks cover the context) and past 8192 (the split-K pair of launches).
    Two calls in a row, the second over a shorter context: the per-head
    counters left by the first must read zero again."""
    import vlrf_amd as V_
    dt = {"Q8_0": V_.KV_Q8_0, "F16": V_.KV_F16, "F32": V_.KV_F32}[kv_name]
    print(f"[case] decode chunks kv={kv_name} heads={n_heads}/{n_kv} ctx={ctx_len}", flush=True)
    d, row = 64, n_kv * 64
    kv = V_.KVCache(ctx, 1, ctx_len + 5, n_kv, d, dt)
    K = F.normal(9, "Kc", ctx_len * row)
    Vv = F.normal(9, "Vc", ctx_len * row)
    kv.append(0, ctx.to_device(K), ctx.to_device(Vv), ctx_len)
    Kd, Vd = _dequant_rows(kv, ctx_len)
    scale = np.float32(0.125)
    rep = n_heads // n_kv
    for call, n in enumerate((ctx_len, max(1, ctx_len // 3))):
        q = F.normal(call, "q", n_heads * d)
        dout = ctx.alloc(q.nbytes)
        kv.attention_decode(0, ctx.to_device(q), dout, n_heads, n, scale)
        out = dout.download(q.shape)
        ref = np.concatenate([orc.flash_attn_head(q[h * d:(h + 1) * d][None, :],
                                                  Kd[:n, (h // rep) * d:(h // rep + 1) * d],
                                                  Vd[:n, (h // rep) * d:(h // rep + 1) * d], scale, False)[0]
                              for h in range(n_heads)])
        assert rel_err(out, ref) <= 1e-3, (call, n)
        assert np.max(np.abs(out - ref)) <= 1e-4, (call, n)


@pytest.mark.parametrize("kv_name", ["Q8_0", "F16", "F32"])
@pytest.mark.parametrize("n_heads,n_kv,d,ctx_len,scale", [
    (4, 4, 128, 1, 0.1), (8, 8, 128, 63, 0.1), (8, 4, 128, 64, 0.1), (8, 2, 128, 65, 0.1), (16, 2, 128, 255, 0.1),
    (8, 8, 128, 256, 0.1), (32, 8, 128, 257, 0.1), (16, 4, 128, 1023, -0.1), (8, 1, 128, 4097, 0.1),
    (32, 8, 128, 6001, 0.1), (8, 8, 64, 8193, 0.125), (16, 8, 64, 8200, 0.0), (32, 4, 64, 8197, 0.125),
    (32, 8, 64, 4200, 0.125)])   # 8.6 MB of K/V at Q8_0 is past the one-launch form only in f16 and f32
def test_decode_attention_rows(ctx, kv_name, n_heads, n_kv, d, ctx_len, scale):
    """d_head 128, long contexts and large caches: edges of the rounds, of the
    chunks and of the single-chunk form; all GQA groups; rows past the context
    that hold infinities; the call that allocates nothing gives the same bits."""
    import vlrf_amd as V_
    dt = {"Q8_0": V_.KV_Q8_0, "F16": V_.KV_F16, "F32": V_.KV_F32}[kv_name]
    print(f"[case] decode rows kv={kv_name} heads={n_heads}/{n_kv} d={d} ctx={ctx_len} scale={scale}", flush=True)
    row, more = n_kv * d, 40
    K, V = (F.normal(21, f"{n}{ctx_len}", (ctx_len + more) * row).reshape(-1, row) for n in "kv")
    if dt != V_.KV_Q8_0:
        K[ctx_len:], V[ctx_len:] = np.nan, np.inf
    kv = V_.KVCache(ctx, 2, ctx_len + more, n_kv, d, dt)
    kv.append(1, ctx.to_device(K), ctx.to_device(V), ctx_len + more)
    Kd, Vd = (t[:ctx_len].reshape(ctx_len, n_kv, d).transpose(1, 0, 2).repeat(n_heads // n_kv, 0)
              for t in _dequant_rows_of(kv, 1, ctx_len + more))
    q = F.normal(22, f"q{ctx_len}", n_heads * d)
    dq, dout, dfix = ctx.to_device(q), ctx.alloc(q.nbytes), ctx.alloc(q.nbytes)
    kv.attention_decode(1, dq, dout, n_heads, ctx_len, scale)
    out = dout.download((n_heads, d))
    ref, bound = _sdp64(q.reshape(n_heads, 1, d), Kd, Vd, np.float32(scale), False)
    assert (np.abs(out - ref[:, 0]) <= bound[:, 0]).all()
    if n_heads * ((ctx_len + 63) // 64) * (d + 2) <= 1 << 19:
        V_.check(V_.lib().vlrf_hip_attn_decode_noalloc(kv.h, 1, dq.ptr, dfix.ptr, n_heads, ctx_len, float(scale)))
        assert np.array_equal(dfix.download((n_heads, d)), out)


def _dequant_rows_of(kv, layer, n):
    import vlrf_amd as V_
    kq, vq, ks, vs = kv.read(layer, 0, n)
    if kv.dtype == V_.KV_Q8_0:
        return kq.astype(np.float32) * ks[:, None], vq.astype(np.float32) * vs[:, None]
    if kv.dtype == V_.KV_F16:
        return kq.view(np.float16).astype(np.float32), vq.view(np.float16).astype(np.float32)
    return kq, vq
