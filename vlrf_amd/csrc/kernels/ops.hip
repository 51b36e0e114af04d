// ops.hip - the engine's remaining per-op backend calls on the device
// (IBackend::gemm / layer_norm / softmax_inplace / gelu_inplace / add_inplace,
// include/backend/ibackend.hpp:61-70), used by GPT-2-family models.
//
// Semantics follow the CPU ops (include/model/ops.hpp): gemm :170-310
// (C = beta*C first -- beta == 0 writes zeros -- then alpha*op(A)*op(B) added;
// op = transpose when transA / transB), layer_norm :443-476 (mean, variance of
// the deviations, (x - mean) * (1/sqrt(var + eps)) * w + b), softmax_inplace
// :501-540 (row max, exp(x - max), x * (1/(sum + 1e-9))), gelu_inplace
// :390-404 (tanh approximation 0.5 x (1 + tanh(sqrt(2/pi)(x + 0.044715 x^3)))),
// add_inplace :344-356.  f32 throughout; reductions are tree-ordered, so
// results agree with the sequential CPU loops to f32 rounding.
#include "../internal.hpp"

#include <cmath>

namespace vlrf_hip {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// f32 GEMM on the f32 matrix instructions.  A 256-lane workgroup owns a BM x BN
// tile of C (64x64, or 32x128 for M <= 32), each wave one 32x32 block of it in
// v_mfma_f32_32x32x2_f32: 4096 operations in 64 cycles, so a SIMD's one wave
// keeps its matrix core busy and two operand reads feed four instructions.  K
// advances in steps of 64 through two LDS buffers, the next step's operands in
// flight in registers while the current one is multiplied; a row's 64 values
// are contiguous in LDS (rows 68 floats apart: 16-byte reads of eight rows hit
// distinct banks), so lane half h takes k = 8s + 4h + 0..3 in one read (the
// order of k within a step is the same for both operands, and otherwise free).
// Products and sums are f32 FMAs as in the CPU loop; infinities and NaN pass
// through; rows and columns outside the matrices are copies of the last ones,
// whose products no stored element takes.
//
// Bound by the matrix rate (157 TFLOP/s f32) while the tiles fill the chip,
// else by the length of a workgroup's own K: the slices of a split K
// (gridDim.z, partial sums to P, added in slice order by gemm_f32_reduce_kernel)
// shorten it.  Measured against the vector-unit kernel before it (64x64 tiles, K
// steps of 16): 300x3072x768 144 -> 20.8 us, 300x768x3072 583 -> 23.0; the rate
// at 1024x1600x6400 is 108 TFLOP/s.  Steps of 64 with two register sets in
// flight; loads behind bounds branches ran 240 against 205 us at 1024x6400x1600.
constexpr int kGK = 64, kGS = kGK + 4;

// A step's loads are branch-free (a guarded load would be waited for where its
// branch ends): rows and k past the end read the last ones, and stage() zeroes
// what lies past kend.  KC: k runs contiguously in memory, else the row index
// does.  VEC: 16-byte loads, 32-bit offsets from the step's uniform base; the
// run's length is a multiple of 4, the base and the leading dimension (below
// 2^22) allow them.
template <int ROWS, bool KC, bool VEC>
__device__ __forceinline__ void gemm_f32_load(float4 (&st)[ROWS / 16], const float* __restrict__ X, int ld, int row0,
                                              int rows, int k0, int kend) {
    const float* base = KC ? X + (size_t)row0 * ld : X + (size_t)k0 * ld;
#pragma unroll
    for (int i = 0; i < ROWS / 16; ++i) {
        const int f = threadIdx.x + 256 * i;
        const int r = KC ? f / (kGK / 4) : 4 * (f % (ROWS / 4));   // within the tile
        const int k = KC ? 4 * (f % (kGK / 4)) : f / (ROWS / 4);
        if constexpr (VEC) {
            const uint32_t o = KC ? (uint32_t)(min(r, rows - 1 - row0) * ld) + min(k0 + k, kend - 4)
                                  : (uint32_t)(min(k, kend - 1 - k0) * ld) + min(row0 + r, rows - 4);
            st[i] = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(base) + 4u * o);
        } else {
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int rj = min(row0 + (KC ? r : r + j), rows - 1), kj = min(k0 + (KC ? k + j : k), kend - 1);
                v[j] = KC ? X[(size_t)rj * ld + kj] : X[(size_t)kj * ld + rj];
            }
            st[i] = make_float4(v[0], v[1], v[2], v[3]);
        }
    }
}

template <int ROWS, bool KC, bool TAIL>
__device__ __forceinline__ void gemm_f32_stage(const float4 (&st)[ROWS / 16], float* s, int left) {
#pragma unroll
    for (int i = 0; i < ROWS / 16; ++i) {
        const int f = threadIdx.x + 256 * i;
        const int k = KC ? 4 * (f % (kGK / 4)) : f / (ROWS / 4);
        float4 v = st[i];
        if constexpr (TAIL) {
            v.x = k < left ? v.x : 0.f;
            v.y = k + (KC ? 1 : 0) < left ? v.y : 0.f;
            v.z = k + (KC ? 2 : 0) < left ? v.z : 0.f;
            v.w = k + (KC ? 3 : 0) < left ? v.w : 0.f;
        }
        if constexpr (KC) {
            *reinterpret_cast<float4*>(s + (f / (kGK / 4)) * kGS + k) = v;
        } else {
            float* d = s + 4 * (f % (ROWS / 4)) * kGS + k;
            d[0] = v.x;
            d[kGS] = v.y;
            d[2 * kGS] = v.z;
            d[3 * kGS] = v.w;
        }
    }
}

template <int BM, int BN, bool TA, bool TB, bool VEC>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                       float* C, float* __restrict__ P, int M, int N, int K, int lda,
                                                       int ldb, int ldc, float alpha, float beta, int kslice) {
    constexpr int WN = BN / 32;                                   // waves across the tile's columns
    __shared__ __align__(16) float As[2][BM * kGS];
    __shared__ __align__(16) float Bs[2][BN * kGS];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int kbeg = blockIdx.z * kslice, kend = min(K, kbeg + kslice);
    const int ra = (w / WN) * 32 + (lane & 31), rb = (w % WN) * 32 + (lane & 31), h4 = 4 * (lane >> 5);
    struct Regs {
        float4 a[BM / 16], b[BN / 16];
    } r0, r1;
    auto load = [&](Regs& r, int k0) {
        gemm_f32_load<BM, !TA, VEC>(r.a, A, lda, m0, M, k0, kend);
        gemm_f32_load<BN, TB, VEC>(r.b, B, ldb, n0, N, k0, kend);
    };
    auto stage = [&](const Regs& r, int buf, int k0) {
        if (kend - k0 >= kGK) {
            gemm_f32_stage<BM, !TA, false>(r.a, As[buf], kGK);
            gemm_f32_stage<BN, TB, false>(r.b, Bs[buf], kGK);
        } else {
            gemm_f32_stage<BM, !TA, true>(r.a, As[buf], kend - k0);
            gemm_f32_stage<BN, TB, true>(r.b, Bs[buf], kend - k0);
        }
    };
    f32x16 acc = {};
    // Multiplies the step in buffer `buf`, with the step after the next one
    // requested into `fut` meanwhile, and moves the next (`nxt`) into LDS.
    auto step = [&](int buf, const Regs& nxt, Regs& fut, int k0) {
        if (k0 + 2 * kGK < kend) load(fut, k0 + 2 * kGK);
        const float* pa = As[buf] + ra * kGS + h4;
        const float* pb = Bs[buf] + rb * kGS + h4;
        float4 a[2], b[2];
        a[0] = *reinterpret_cast<const float4*>(pa);
        b[0] = *reinterpret_cast<const float4*>(pb);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
        for (int s = 0; s < kGK / 8; ++s) {   // the next eight k's operands are read under these four
            const int c = s & 1;
            if (s + 1 < kGK / 8) {
                a[c ^ 1] = *reinterpret_cast<const float4*>(pa + 8 * (s + 1));
                b[c ^ 1] = *reinterpret_cast<const float4*>(pb + 8 * (s + 1));
                __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            }
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[c].x, b[c].x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[c].y, b[c].y, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[c].z, b[c].z, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[c].w, b[c].w, acc, 0, 0, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
        }
        if (k0 + kGK < kend) stage(nxt, buf ^ 1, k0 + kGK);
        __syncthreads();
    };
    load(r0, kbeg);
    if (kbeg + kGK < kend) load(r1, kbeg + kGK);
    stage(r0, 0, kbeg);
    __syncthreads();
    for (int k0 = kbeg; k0 < kend; k0 += 2 * kGK) {
        step(0, r1, r0, k0);
        if (k0 + kGK < kend) step(1, r0, r1, k0 + kGK);
    }
    // Register r of lane l is row 8(r/4) + 4(l/32) + r%4, column l%32 of the block.
    const int n = n0 + rb;
    if (n >= N) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int m = m0 + (w / WN) * 32 + 8 * (r >> 2) + h4 + (r & 3);
        if (m >= M) continue;
        if (P) {
            P[((size_t)blockIdx.z * M + m) * N + n] = acc[r];
        } else {
            float* c = C + (size_t)m * ldc + n;
            const float prev = beta == 0.f ? 0.f : (beta == 1.f ? *c : *c * beta);
            *c = prev + alpha * acc[r];
        }
    }
}

// The same for short K on the vector units: a 256-lane workgroup owns a 64x64 tile
// of C, each lane a 4x4 block (rows ty + 16i, columns tx + 16j, so LDS reads of a
// wave are broadcast or conflict-free); K in steps of 16 staged through LDS.
// Bound by the stores of C and one trip to memory, where a step of 64 is mostly
// padding and its 68 KiB of LDS leave two workgroups a CU (us, that kernel / this
// one: 4096 x 4096 x 8 44.8 / 18.3, x 48 45.2 / 39.2, x 64 45.0 / 48.9; 100 x 50000 x 32
// 21.4 / 15.4; 1 x 4096 x 16 5.2 / 4.1).
constexpr int kShortT = 64, kShortK = 16;

__global__ __launch_bounds__(256) void gemm_f32_short_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                             float* C, int M, int N, int K, int lda, int ldb,
                                                             int ldc, float alpha, float beta, int transA, int transB) {
    __shared__ float As[kShortK][kShortT + 1];
    __shared__ float Bs[kShortK][kShortT + 1];
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    const int m0 = blockIdx.y * kShortT, n0 = blockIdx.x * kShortT;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += kShortK) {
        for (int i = tid; i < kShortT * kShortK; i += 256) {
            // A tile element (m, k): lanes walk k fastest when A is row-major in k
            const int r = transA ? i % kShortT : i / kShortK, c = transA ? i / kShortT : i % kShortK;
            const int m = m0 + r, k = k0 + c;
            float a = 0.f;
            if (m < M && k < K) a = transA ? A[(size_t)k * lda + m] : A[(size_t)m * lda + k];
            As[c][r] = a;
            const int rb = transB ? i / kShortK : i % kShortT, cb = transB ? i % kShortK : i / kShortT;   // (n, k)
            const int n = n0 + rb, kb = k0 + cb;
            float b = 0.f;
            if (n < N && kb < K) b = transB ? B[(size_t)n * ldb + kb] : B[(size_t)kb * ldb + n];
            Bs[cb][rb] = b;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < kShortK; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[kk][ty + 16 * i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx + 16 * j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] += a[i] * b[j];
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int m = m0 + ty + 16 * i, n = n0 + tx + 16 * j;
            if (m < M && n < N) {
                float* c = C + (size_t)m * ldc + n;
                const float prev = beta == 0.f ? 0.f : (beta == 1.f ? *c : *c * beta);
                *c = prev + alpha * acc[i][j];
            }
        }
}

// C = beta*C + alpha * (the S slices' partial sums, in slice order).
__global__ __launch_bounds__(256) void gemm_f32_reduce_kernel(const float* __restrict__ P, int S, float* C, int M,
                                                              int N, int ldc, float alpha, float beta) {
    const size_t mn = (size_t)M * N, i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= mn) return;
    float v = 0.f;
    for (int s = 0; s < S; s += 8) {   // eight loads in flight, added in slice order
        float p[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) p[j] = P[min(s + j, S - 1) * mn + i];
#pragma unroll
        for (int j = 0; j < 8; ++j) v += s + j < S ? p[j] : 0.f;
    }
    float* c = C + (i / N) * ldc + i % N;
    const float prev = beta == 0.f ? 0.f : (beta == 1.f ? *c : *c * beta);
    *c = prev + alpha * v;
}

__device__ __forceinline__ float block_sum(float v, float* red) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    v = wave_sum(v);
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

__device__ __forceinline__ float block_max(float v, float* red) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    v = wave_max(v);
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

__global__ __launch_bounds__(256) void layer_norm_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                         const float* __restrict__ b, float* out, int D,
                                                         float eps) {
    __shared__ float red[4];
    const float* r = x + (size_t)blockIdx.x * D;
    float s = 0.f;
    for (int j = threadIdx.x; j < D; j += 256) s += r[j];
    const float mean = block_sum(s, red) / (float)D;
    float v = 0.f;
    for (int j = threadIdx.x; j < D; j += 256) {
        const float d = r[j] - mean;
        v += d * d;
    }
    const float var = block_sum(v, red) / (float)D + eps;
    const float inv = 1.f / sqrtf(var);
    float* o = out + (size_t)blockIdx.x * D;
    for (int j = threadIdx.x; j < D; j += 256) o[j] = (r[j] - mean) * inv * w[j] + b[j];
}

// Rows of up to 4096 columns held in registers, NV float4 a thread (as many as the
// row has thousands of columns: with all four for every row, 20000 x 64 took 28.8 us):
// read once, and no load behind a reduction.  Against the kernel above, us: 1000 x
// 1600 5.1 -> 3.75, 4000 x 768 7.4 -> 5.5, 20000 x 1024 42.6 -> 24.4, 20000 x 64 10.8 -> 10.8.
template <int NV>
__global__ __launch_bounds__(256) void layer_norm_regs_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                              const float* __restrict__ b, float* out, int D,
                                                              float eps) {
    __shared__ float red[4];
    const float4* r = reinterpret_cast<const float4*>(x + (size_t)blockIdx.x * D);
    const int n4 = D / 4;
    float4 v[NV], wv[NV], bv[NV];
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int j = min((int)threadIdx.x + 256 * i, n4 - 1);
        v[i] = r[j];
        wv[i] = reinterpret_cast<const float4*>(w)[j];
        bv[i] = reinterpret_cast<const float4*>(b)[j];
    }
#pragma unroll
    for (int i = 0; i < NV; ++i)
        if ((int)threadIdx.x + 256 * i < n4) s += (v[i].x + v[i].y) + (v[i].z + v[i].w);
    const float mean = block_sum(s, red) / (float)D;
    float q = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        v[i] = make_float4(v[i].x - mean, v[i].y - mean, v[i].z - mean, v[i].w - mean);
        if ((int)threadIdx.x + 256 * i < n4)
            q += (v[i].x * v[i].x + v[i].y * v[i].y) + (v[i].z * v[i].z + v[i].w * v[i].w);
    }
    const float var = block_sum(q, red) / (float)D + eps;
    const float inv = 1.f / sqrtf(var);
    float4* o = reinterpret_cast<float4*>(out + (size_t)blockIdx.x * D);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int j = threadIdx.x + 256 * i;
        if (j < n4)
            o[j] = make_float4(v[i].x * inv * wv[i].x + bv[i].x, v[i].y * inv * wv[i].y + bv[i].y,
                               v[i].z * inv * wv[i].z + bv[i].z, v[i].w * inv * wv[i].w + bv[i].w);
    }
}

__global__ __launch_bounds__(256) void softmax_kernel(float* x, int D) {
    __shared__ float red[4];
    float* r = x + (size_t)blockIdx.x * D;
    float mx = -INFINITY;
    for (int j = threadIdx.x; j < D; j += 256) mx = fmaxf(mx, r[j]);
    mx = block_max(mx, red);
    float s = 0.f;
    for (int j = threadIdx.x; j < D; j += 256) {
        const float e = expf(r[j] - mx);
        r[j] = e;
        s += e;
    }
    const float inv = 1.f / (block_sum(s, red) + 1e-9f);
    for (int j = threadIdx.x; j < D; j += 256) r[j] *= inv;
}

__device__ __forceinline__ float gelu_tanh(float v) {
    constexpr float c1 = 0.7978845608028654f, c2 = 0.044715f;   // sqrt(2/pi), ops.hpp:393-394
    const float inner = c1 * (v + c2 * v * v * v);
    return 0.5f * v * (1.f + tanhf(inner));
}

// VEC: 16-byte accesses over whole groups of four (aligned bases), the rest singly
// (1000 x 6400: 7.9 -> 6.8 us; add of 1000 x 1600 3.9 -> 3.4).
template <bool VEC>
__global__ __launch_bounds__(256) void gelu_kernel(float* x, int64_t n) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256, n4 = VEC ? n / 4 : 0;
    for (int64_t i = t; i < n4; i += step) {
        const float4 v = reinterpret_cast<const float4*>(x)[i];
        reinterpret_cast<float4*>(x)[i] = make_float4(gelu_tanh(v.x), gelu_tanh(v.y), gelu_tanh(v.z), gelu_tanh(v.w));
    }
    for (int64_t i = 4 * n4 + t; i < n; i += step) x[i] = gelu_tanh(x[i]);
}

template <bool VEC>
__global__ __launch_bounds__(256) void add_kernel(float* dst, const float* __restrict__ src, int64_t n) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256, n4 = VEC ? n / 4 : 0;
    for (int64_t i = t; i < n4; i += step) {
        const float4 d = reinterpret_cast<const float4*>(dst)[i], s = reinterpret_cast<const float4*>(src)[i];
        reinterpret_cast<float4*>(dst)[i] = make_float4(d.x + s.x, d.y + s.y, d.z + s.z, d.w + s.w);
    }
    for (int64_t i = 4 * n4 + t; i < n; i += step) dst[i] += src[i];
}

bool aligned16(const void* a, const void* b = nullptr, const void* c = nullptr, const void* d = nullptr) {
    return (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c | (uintptr_t)d) & 15) == 0;
}

int grid_1d(int64_t n) {
    const int64_t g = (n + 255) / 256;
    return (int)(g < 4096 ? (g < 1 ? 1 : g) : 4096);
}

}  // namespace

namespace {

struct GemmF32Plan {
    bool wide;        // 32 x 128 tiles
    int S, kslice;    // slices of K, and the columns of one
};

// The split with the shortest estimated time, in K steps of one tile (about
// 1.1 us): rounds of 256 workgroups times the steps of a slice, plus, with more
// than one slice, the reduction: its launch (about 5 steps) and its partial
// sums at about 3.3 MB a step.  Slices keep at least two steps, and 512 tiles
// fill the chip twice without a split.  Measured (us, this split against one
// slice / the next candidates): 300x768x3072 (60 tiles) 23.0 with 4 slices, 38.2
// with 2, 22.7 with 8; 700x768x3072 (132) 42.6 with 3, 67.8 with 1; 300x3072x768
// (240) 20.8 with 1, 25.4 with 2; 1x768x3072 (6) 8.6 with 24, 10.6 with 12.
GemmF32Plan gemm_f32_plan(int M, int N, int K) {
    GemmF32Plan p;
    p.wide = M <= 32;
    const int bm = p.wide ? 32 : 64, bn = p.wide ? 128 : 64;
    const long tiles = (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
    const int steps = (K + kGK - 1) / kGK;
    int best = 1;
    if (tiles < 512) {
        float cost = (float)((tiles + 255) / 256) * steps;
        for (int S = 2; S <= 64 && S <= steps / 2; ++S) {
            const float c = (float)((tiles * S + 255) / 256) * ((steps + S - 1) / S) + 5.f +
                            8e-6f / 3.3f * S * (float)M * N;
            if (c < cost) {
                cost = c;
                best = S;
            }
        }
    }
    const int per = (steps + best - 1) / best;
    p.S = (steps + per - 1) / per;
    p.kslice = per * kGK;
    return p;
}

// Where K is short (it then stays whole) and the vector-unit kernel faster: one step
// of its 16, but for aligned operands of up to 256 tiles, and more of them as the
// tiles take more rounds of the other's two workgroups a CU.  us, steps of 64 / of
// 16: 1024 x 1024 x 16 5.5 / 6.2 (A transposed, x 4 6.6 / 6.0); 1024 x 2048 x 16 7.7 / 6.7,
// x 32 7.7 / 9.1; 1536 x 1536 x 32 10.5 / 9.2, x 48 10.5 / 11.7; 3072 x 3072 x 48 26.6 /
// 24.4, x 64 26.9 / 30.0, x 72 39.3 / 37.4 (B transposed 34.6 / 36.8); 16 x 200000 x 96
// 57.9 / 49.9.
bool gemm_f32_short(int M, int N, int K, bool transA, bool transB, bool vec) {
    const long tiles = (long)((M + kShortT - 1) / kShortT) * ((N + kShortT - 1) / kShortT);
    if (K <= 16) return !(vec && !transA && K >= 4 && M >= 64 && N >= 64 && tiles <= 256);
    if (K <= 32) return tiles > 512;
    return tiles >= 1536 && (K <= 48 || (K > 64 && K <= (M <= 32 ? 96 : 80) && !transB));
}

}  // namespace

size_t gemm_f32_part_bytes(int M, int N, int K) {
    if (M < 1 || N < 1 || K < 1) return 0;
    const GemmF32Plan p = gemm_f32_plan(M, N, K);
    return p.S > 1 ? (size_t)p.S * M * N * sizeof(float) : 0;
}

int launch_gemm_f32(hipStream_t s, const float* A, const float* B, float* C, int M, int N, int K, int lda,
                    int ldb, int ldc, float alpha, float beta, bool transA, bool transB, float* part) {
    VH_ARG(A && B && C, "gemm_f32: null operand");
    VH_ARG(M >= 1 && N >= 1 && K >= 1, "gemm_f32: empty shape %dx%dx%d", M, N, K);
    VH_ARG(lda >= (transA ? M : K) && ldb >= (transB ? K : N) && ldc >= N, "gemm_f32: leading dimension too small");
    GemmF32Plan p = gemm_f32_plan(M, N, K);
    if (!part) {
        p.S = 1;
        p.kslice = K;
    }
    float* P = p.S > 1 ? part : nullptr;
    const bool va = ((uintptr_t)A & 15) == 0 && lda % 4 == 0 && lda < (1 << 22) && (transA ? M : K) % 4 == 0;
    const bool vb = ((uintptr_t)B & 15) == 0 && ldb % 4 == 0 && ldb < (1 << 22) && (transB ? K : N) % 4 == 0;
    if (gemm_f32_short(M, N, K, transA, transB, va && vb)) {
        const dim3 grid((N + kShortT - 1) / kShortT, (M + kShortT - 1) / kShortT);
        hipLaunchKernelGGL(gemm_f32_short_kernel, grid, dim3(256), 0, s, A, B, C, M, N, K, lda, ldb, ldc, alpha, beta,
                           (int)transA, (int)transB);
        VH_LAUNCHED();
        return VLRF_HIP_OK;
    }
    const int bm = p.wide ? 32 : 64, bn = p.wide ? 128 : 64;
    const dim3 grid((N + bn - 1) / bn, (M + bm - 1) / bm, p.S);
#define VH_GF(BM, BN, TA, TB, VV)                                                                               \
    hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, TA, TB, VV>), grid, dim3(256), 0, s, A, B, C, P, M, N, K,    \
                       lda, ldb, ldc, alpha, beta, p.kslice)
#define VH_GF_T(BM, BN, VV)                                                                                      \
    if (transA) {                                                                                                \
        if (transB) VH_GF(BM, BN, true, true, VV);                                                               \
        else VH_GF(BM, BN, true, false, VV);                                                                     \
    } else {                                                                                                     \
        if (transB) VH_GF(BM, BN, false, true, VV);                                                              \
        else VH_GF(BM, BN, false, false, VV);                                                                    \
    }
    if (p.wide) {
        if (va && vb) { VH_GF_T(32, 128, true) } else { VH_GF_T(32, 128, false) }
    } else {
        if (va && vb) { VH_GF_T(64, 64, true) } else { VH_GF_T(64, 64, false) }
    }
#undef VH_GF_T
#undef VH_GF
    VH_LAUNCHED();
    if (P) {
        const size_t mn = (size_t)M * N;
        hipLaunchKernelGGL(gemm_f32_reduce_kernel, dim3((unsigned)((mn + 255) / 256)), dim3(256), 0, s, P, p.S, C, M,
                           N, ldc, alpha, beta);
        VH_LAUNCHED();
    }
    return VLRF_HIP_OK;
}

int launch_layer_norm(hipStream_t s, const float* x, const float* w, const float* b, float* out, int rows, int D,
                      float eps) {
    VH_ARG(x && w && b && out && rows >= 1 && D >= 1, "layer_norm: bad arguments");
    const bool regs = D % 4 == 0 && D <= 4096 && aligned16(x, w, b, out);
    if (regs && D <= 1024)
        hipLaunchKernelGGL(layer_norm_regs_kernel<1>, dim3(rows), dim3(256), 0, s, x, w, b, out, D, eps);
    else if (regs && D <= 2048)
        hipLaunchKernelGGL(layer_norm_regs_kernel<2>, dim3(rows), dim3(256), 0, s, x, w, b, out, D, eps);
    else if (regs)
        hipLaunchKernelGGL(layer_norm_regs_kernel<4>, dim3(rows), dim3(256), 0, s, x, w, b, out, D, eps);
    else
        hipLaunchKernelGGL(layer_norm_kernel, dim3(rows), dim3(256), 0, s, x, w, b, out, D, eps);
    VH_LAUNCHED();
    return VLRF_HIP_OK;
}

int launch_softmax(hipStream_t s, float* x, int rows, int D) {
    VH_ARG(x && rows >= 1 && D >= 1, "softmax: bad arguments");
    hipLaunchKernelGGL(softmax_kernel, dim3(rows), dim3(256), 0, s, x, D);
    VH_LAUNCHED();
    return VLRF_HIP_OK;
}

int launch_gelu(hipStream_t s, float* x, int64_t n) {
    VH_ARG(x && n >= 0, "gelu: bad arguments");
    if (n == 0) return VLRF_HIP_OK;
    if (aligned16(x)) hipLaunchKernelGGL((gelu_kernel<true>), dim3(grid_1d((n + 3) / 4)), dim3(256), 0, s, x, n);
    else hipLaunchKernelGGL((gelu_kernel<false>), dim3(grid_1d(n)), dim3(256), 0, s, x, n);
    VH_LAUNCHED();
    return VLRF_HIP_OK;
}

int launch_add(hipStream_t s, float* dst, const float* src, int64_t n) {
    VH_ARG(dst && src && n >= 0, "add: bad arguments");
    if (n == 0) return VLRF_HIP_OK;
    if (aligned16(dst, src)) hipLaunchKernelGGL((add_kernel<true>), dim3(grid_1d((n + 3) / 4)), dim3(256), 0, s, dst, src, n);
    else hipLaunchKernelGGL((add_kernel<false>), dim3(grid_1d(n)), dim3(256), 0, s, dst, src, n);
    VH_LAUNCHED();
    return VLRF_HIP_OK;
}

}  // namespace vlrf_hip
