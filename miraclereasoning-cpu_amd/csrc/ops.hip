// Op-level ABI: one entry point per reference kernel (kernels.cl), with the
// reference's argument lists.  These serve HIPBackend's op surface (the drop-in
// for OpenCLBackend); the fused decode step lives in engine.hip.
#include <algorithm>

#include "attention.h"
#include "gemm.h"
#include "linear.h"
#include "prefill.h"

namespace mr {
namespace {

constexpr int kThreads = 256;

inline int grid_for(int64_t n) { return (int)ceil_div64(n, kThreads); }

// Both pointers 16-byte aligned (null counts as aligned).
inline bool vec16(const void *a, const void *b = nullptr) { return (((uintptr_t)a | (uintptr_t)b) & 15) == 0; }

// Lanes that read `n` vectors of a row together: the power of two that covers
// them, at most a wave.
inline int lanes_for(int n) {
    int lpr = 1;
    while (lpr < n && lpr < kWave) lpr *= 2;
    return lpr;
}

// V consecutive floats from p (V = 4: p 16-byte aligned).
template <int V>
__device__ __forceinline__ void load_v(float (&o)[V], const float *p) {
    if constexpr (V == 4) {
        const float4 t = load_f4(p);
        o[0] = t.x; o[1] = t.y; o[2] = t.z; o[3] = t.w;
    } else {
        o[0] = gmem(p)[0];
    }
}
template <int V>
__device__ __forceinline__ void store_v(float *p, const float (&o)[V]) {
    if constexpr (V == 4) {
        typedef float f32x4 __attribute__((ext_vector_type(4)));
        *(MR_GLOBAL f32x4 *)gmem(p) = f32x4{o[0], o[1], o[2], o[3]};
    } else {
        gmem(p)[0] = o[0];
    }
}

// kernels.cl:19-28: a wave per row (BLOCK: a block per row), the row in
// registers (N x 4 floats a thread, every load in flight at once, one pass).
// A block of 256 threads that looped over its row twice took 31.3 us for
// 48,000 rows of 128 (49 MB) and 4.6 for one of 2048.
template <int N, bool BLOCK>
__global__ void __launch_bounds__(256) k_rms_reg(const float *x, const float *w, float *y, int rows, int width,
                                                 float eps) {
    __shared__ float red[kThreads / kWave];
    const int row = BLOCK ? blockIdx.x : blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int at = 4 * (BLOCK ? threadIdx.x : threadIdx.x & 63), step = 4 * (BLOCK ? kThreads : kWave);
    const float *xr = x + (int64_t)row * width;
    float v[N][4], g[N][4];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int c = at + i * step;
        if (c < width) {
            load_v<4>(v[i], xr + c);
            if (w) load_v<4>(g[i], w + c);
        }
        if (c >= width) v[i][0] = v[i][1] = v[i][2] = v[i][3] = 0.0f;
    }
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) ss = fmaf(v[i][e], v[i][e], ss);
    ss = BLOCK ? block_sum(ss, red) : wave_sum(ss);
    const float scale = 1.0f / sqrtf(ss / (float)width + eps);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int c = at + i * step;
        if (c >= width) break;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[i][e] = v[i][e] * scale * (w ? g[i][e] : 1.0f);
        store_v<4>(y + (int64_t)row * width + c, v[i]);
    }
}

// Rows past k_rms_reg's widths, or not of whole 16-byte vectors.
__global__ void __launch_bounds__(256) k_rms(const float *x, const float *w, float *y, int width, float eps) {
    __shared__ float red[kThreads / kWave];
    const float *xr = x + (int64_t)blockIdx.x * width;
    float ss = 0.0f;
    for (int j = threadIdx.x; j < width; j += blockDim.x) ss = fmaf(xr[j], xr[j], ss);
    ss = block_sum(ss, red);
    float scale = 1.0f / sqrtf(ss / (float)width + eps);
    for (int j = threadIdx.x; j < width; j += blockDim.x)
        y[(int64_t)blockIdx.x * width + j] = xr[j] * scale * (w ? w[j] : 1.0f);
}

// kernels.cl:30-44: a thread per (row, pair) and run of `per` heads: the FP32
// angle's cosine and sine (taken in double and rounded once, within half an
// ulp of the exact value at every angle the models reach) are the row's for
// every head (a thread per
// head's pair, 3 M of them for 3,000 rows of 16 x 128, took 21.4 us).
__global__ void __launch_bounds__(256) k_rope(const float *x, const float *freq, const float *pos, float *y, int rows,
                                              int heads, int dim, int split_half, int per) {
    const int half = dim / 2;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)rows * half) return;
    const int p = (int)(i % half), h0 = blockIdx.y * per, h1 = min(heads, h0 + per);
    const int64_t row = i / half;
    const double ad = (double)(pos[row] * freq[p]);
    const float c = (float)cos(ad), s = (float)sin(ad);
    const int64_t base = row * heads * dim;
    const int j = split_half ? p : 2 * p, k = split_half ? p + half : 2 * p + 1;
#pragma unroll 4
    for (int h = h0; h < h1; ++h) {
        float u = x[base + (int64_t)h * dim + j], v = x[base + (int64_t)h * dim + k];
        rope_rotate(u, v, c, s);
        y[base + (int64_t)h * dim + j] = u;
        y[base + (int64_t)h * dim + k] = v;
    }
}

__global__ void k_swiglu(const float *g, const float *u, float *y, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = (g[i] / (1.0f + expf(-g[i]))) * u[i];
}

__global__ void k_axpy(const float *x, const float *y, float *z, int n, float scale) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) z[i] = x[i] + scale * y[i];
}

__device__ __forceinline__ const float *row_of(const float *ring, const float *extra, int t, int kvw, int capacity,
                                               int start, int length, int kh, int dim) {
    if (t < length) return ring + (int64_t)((start + t) % capacity) * kvw + (int64_t)kh * dim;
    return extra + (int64_t)(t - length) * kvw + (int64_t)kh * dim;
}

// kernels.cl:58-73: `lpr` lanes (a power of two) read a key together, 64 / lpr
// keys a wave and round, for up to HN query heads of its KV head.  Block (run
// of keys, KV head, run of HN heads), flattened.  Bound by the keys' bytes: 16 heads over 3,000 keys of 16 x 128
// (24.6 MB) took 22.2 us with a thread per (key, head).
template <int V, int HN>
__global__ void __launch_bounds__(256) k_scores(const float *q, const float *k, const float *extra_k, float *s,
                                                int heads, int kv_heads, int dim, int capacity, int start, int length,
                                                int extra_length, int lpr, int runs) {
    constexpr int B = 4;   // keys of a lane group in flight
    const int lane = threadIdx.x & 63, sub = lane & (lpr - 1), total = length + extra_length;
    const int bx = blockIdx.x % runs, kh = (blockIdx.x / runs) % kv_heads, bz = blockIdx.x / runs / kv_heads;
    const int G = heads / kv_heads, g0 = bz * HN, ng = min(HN, G - g0), h0 = kh * G + g0;
    const int keys = kWave / lpr, per_block = 4 * keys * B;
    const int t0 = bx * per_block + (threadIdx.x >> 6) * keys * B + lane / lpr;
    const float *row[B];
#pragma unroll
    for (int b = 0; b < B; ++b)
        row[b] = row_of(k, extra_k, min(t0 + b * keys, total - 1), kv_heads * dim, capacity, start, length, kh, dim);
    float acc[B][HN] = {};
    for (int c = sub * V; c < dim; c += lpr * V) {
        float kv[B][V], qv[HN][V];
#pragma unroll
        for (int b = 0; b < B; ++b) load_v<V>(kv[b], row[b] + c);
#pragma unroll
        for (int g = 0; g < HN; ++g) load_v<V>(qv[g], q + (int64_t)(h0 + min(g, ng - 1)) * dim + c);
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
            for (int g = 0; g < HN; ++g)
#pragma unroll
                for (int e = 0; e < V; ++e) acc[b][g] = fmaf(qv[g][e], kv[b][e], acc[b][g]);
    }
#pragma unroll
    for (int b = 0; b < B; ++b)
#pragma unroll
        for (int g = 0; g < HN; ++g) {
            const float v = group_sum(acc[b][g], lpr);
            const int t = t0 + b * keys;
            if (sub == 0 && g < ng && t < total) s[(int64_t)(h0 + g) * total + t] = v / sqrtf((float)dim);
        }
}

// kernels.cl:75-84: one block of T threads per row, the row in registers (N
// values a thread; every exponential taken once).  256 threads walking the
// row three times took 9.4 us for 16 rows of 3,000.
template <int T, int N>
__global__ void __launch_bounds__(T) k_softmax_reg(const float *x, float *y, int width) {
    __shared__ float red[T / kWave];
    const float *xr = x + (int64_t)blockIdx.x * width;
    float v[N];
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int j = threadIdx.x + i * T;
        v[i] = j < width ? xr[j] : -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) m = fmaxf(m, v[i]);
    m = block_max(m, red);
    float den = 0.0f;
#pragma unroll
    for (int i = 0; i < N; ++i)
        if (threadIdx.x + i * T < width) {
            v[i] = expf(v[i] - m);
            den += v[i];
        }
    den = block_sum(den, red);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int j = threadIdx.x + i * T;
        if (j < width) y[(int64_t)blockIdx.x * width + j] = v[i] / den;
    }
}

// Rows wider than k_softmax_reg holds.
__global__ void __launch_bounds__(256) k_softmax(const float *x, float *y, int width) {
    __shared__ float red[kThreads / kWave];
    const float *xr = x + (int64_t)blockIdx.x * width;
    float *yr = y + (int64_t)blockIdx.x * width;
    float m = -INFINITY;
    for (int j = threadIdx.x; j < width; j += blockDim.x) m = fmaxf(m, xr[j]);
    m = block_max(m, red);
    float den = 0.0f;
    for (int j = threadIdx.x; j < width; j += blockDim.x) den += expf(xr[j] - m);
    den = block_sum(den, red);
    for (int j = threadIdx.x; j < width; j += blockDim.x) yr[j] = expf(xr[j] - m) / den;
}

__global__ void k_latent_mask(float *scores, const float *positions, int heads, int length, int memory,
                              int earliest) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)heads * length) return;
    int t = (int)(i % length);
    if (t >= memory && positions[t] < (float)earliest) scores[i] = -INFINITY;
}

// kernels.cl:93-107: block (key chunk, KV head, HN of its query heads, run of
// lpr V columns), flattened.  lpr lanes read a value row's columns together, the
// block's 256 / lpr lane groups take the chunk's rows in turn and add their
// sums in LDS; with several chunks `y` is chunk c's partial sum part[c][heads
// dim], which k_sum_chunks adds in order.  Bound by the values' bytes: one
// thread per output element walking 3,000 rows of 16 x 128 (24.6 MB) took 910
// us, 8 workgroups of dependent loads.
template <int V, int HN>
__global__ void __launch_bounds__(256) k_mix(const float *p, const float *v, const float *extra_v, float *y, int heads,
                                             int kv_heads, int dim, int capacity, int start, int length,
                                             int extra_length, int lpr, int chunk, int chunks) {
    constexpr int B = 4;   // rows of a lane group in flight
    __shared__ float red[HN][V][256];
    const int bx = blockIdx.x % chunks, kh = (blockIdx.x / chunks) % kv_heads, bz = blockIdx.x / chunks / kv_heads;
    const int total = length + extra_length, G = heads / kv_heads;
    const int hz = (G + HN - 1) / HN, g0 = (bz % hz) * HN;
    const int ng = min(HN, G - g0), h0 = kh * G + g0;
    const int sub = threadIdx.x & (lpr - 1), slot = threadIdx.x / lpr, slots = 256 / lpr;
    const int c = ((bz / hz) * lpr + sub) * V;
    const int t0 = bx * chunk, t1 = min(t0 + chunk, total);
    const bool live = c < dim;
    float acc[HN][V] = {};
    for (int t = t0 + slot; live && t < t1; t += slots * B) {
        float vv[B][V], w[B][HN];
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const int tb = min(t + b * slots, t1 - 1);
            load_v<V>(vv[b], row_of(v, extra_v, tb, kv_heads * dim, capacity, start, length, kh, dim) + c);
#pragma unroll
            for (int g = 0; g < HN; ++g) w[b][g] = p[(int64_t)(h0 + min(g, ng - 1)) * total + tb];
        }
#pragma unroll
        for (int b = 0; b < B; ++b) {
            if (t + b * slots >= t1) break;
#pragma unroll
            for (int g = 0; g < HN; ++g)
#pragma unroll
                for (int e = 0; e < V; ++e) acc[g][e] = fmaf(w[b][g], vv[b][e], acc[g][e]);
        }
    }
#pragma unroll
    for (int g = 0; g < HN; ++g)
#pragma unroll
        for (int e = 0; e < V; ++e) red[g][e][threadIdx.x] = acc[g][e];
    __syncthreads();
    float *out = y + (int64_t)bx * heads * dim;
    for (int i = threadIdx.x; i < ng * lpr * V; i += 256) {
        const int g = i / (lpr * V), r = i % (lpr * V), u = r / V, e = r % V;
        const int col = ((bz / hz) * lpr + u) * V + e;
        if (col >= dim) continue;
        float sum = 0.0f;
        for (int k = 0; k < slots; ++k) sum += red[g][e][k * lpr + u];
        out[(int64_t)(h0 + g) * dim + col] = sum;
    }
}

__global__ void __launch_bounds__(256) k_sum_chunks(const float *part, float *y, int n, int chunks) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float v = 0.0f;
#pragma unroll 8
    for (int c = 0; c < chunks; ++c) v += part[(int64_t)c * n + i];
    y[i] = v;
}

// kernels.cl:110-117: a wave per (slot, token) (a thread per dot, each walking
// its own rows, took 125 us for 64 tokens x 4 slots of 1024).
template <int V>
__global__ void __launch_bounds__(256) k_pool_scores(const float *u, const float *q, float *s, int tokens, int slots,
                                                     int width) {
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= tokens * slots) return;
    const int m = i / tokens, t = i % tokens;
    const float *ur = u + (int64_t)t * width, *qr = q + (int64_t)m * width;
    float v = 0.0f;
#pragma unroll 4
    for (int c = lane * V; c < width; c += kWave * V) {
        float a[V], b[V];
        load_v<V>(a, ur + c);
        load_v<V>(b, qr + c);
#pragma unroll
        for (int e = 0; e < V; ++e) v = fmaf(a[e], b[e], v);
    }
    v = wave_sum(v);
    if (lane == 0) s[(int64_t)m * tokens + t] = v / sqrtf((float)width);
}

// kernels.cl:119-130: block (64 columns, slot); its four waves take every
// fourth token each.  The first block of a slot also sums the anchor, in token
// order (it is rounded, so its last bits matter).
__global__ void __launch_bounds__(256) k_pool_mix(const float *u, const float *p, float *z, float *anchors, int tokens,
                                                  int slots, int width, int start_position, int runs) {
    __shared__ float red[4][kWave];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, m = blockIdx.x / runs;
    const int j = (blockIdx.x % runs) * kWave + lane;
    const float *pr = p + (int64_t)m * tokens;
    float v = 0.0f;
    if (j < width)
#pragma unroll 8
        for (int t = wave; t < tokens; t += 4) v = fmaf(pr[t], u[(int64_t)t * width + j], v);
    red[wave][lane] = v;
    if (blockIdx.x % runs == 0 && threadIdx.x == 0) {
        float pos = 0.0f;
#pragma unroll 8
        for (int t = 0; t < tokens; ++t) pos = fmaf(pr[t], (float)(start_position + t), pos);
        anchors[m] = rintf(pos);
    }
    __syncthreads();
    if (wave == 0 && j < width)
        z[(int64_t)m * width + j] = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
}

__global__ void k_merge_rows(const float *x, float *y, int width, float a, float b) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < width) y[j] = (a * x[j] + b * x[width + j]) / (a + b);
}

__global__ void k_block_means(const float *x, float *y, int length, int width, int block) {
    int blocks = (length + block - 1) / block;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)blocks * width) return;
    int b = (int)(i / width), j = (int)(i % width);
    int start = b * block, stop = min(start + block, length);
    float v = 0.0f;
    for (int t = start; t < stop; ++t) v += x[(int64_t)t * width + j];
    y[(int64_t)b * width + j] = v / (float)(stop - start);
}

}  // namespace
}  // namespace mr

using namespace mr;

#define OP_BEGIN(name)                                                      \
    MR_REQUIRE(ctx, name ": null context");                                \
    if (ctx->fail_next) {                                                   \
        ctx->fail_next = false;                                             \
        return fail(MR_ERR_INJECTED, name ": injected failure");            \
    }                                                                       \
    hipStream_t s = ctx->stream;

extern "C" {

int mr_linear(mr_ctx *ctx, const float *x, const void *w, int w_dtype, float *y, int rows, int out_dim, int in_dim) {
    OP_BEGIN("linear");
    MR_REQUIRE(x && w && y && rows > 0 && out_dim > 0 && in_dim > 0, "linear needs x[rows,in] and weight[out,in]");
    (void)s;
    return launch_linear(ctx, x, w, w_dtype, y, rows, out_dim, in_dim);
}

int mr_rms(mr_ctx *ctx, const float *x, const float *w, float *y, int rows, int width, float eps) {
    OP_BEGIN("rms");
    MR_REQUIRE(x && y && rows > 0 && width > 0, "RMSNorm shape mismatch");
    if (width % 4 == 0 && width <= 4096 && vec16(x, y) && vec16(w)) {
        // a wave per row where rows are short or enough to fill the device,
        // a block for a few long ones
        if (width <= 256) k_rms_reg<1, false><<<ceil_div(rows, 4), kThreads, 0, s>>>(x, w, y, rows, width, eps);
        else if (width <= 1024 && rows >= 256)
            k_rms_reg<4, false><<<ceil_div(rows, 4), kThreads, 0, s>>>(x, w, y, rows, width, eps);
        else if (width <= 1024) k_rms_reg<1, true><<<rows, kThreads, 0, s>>>(x, w, y, rows, width, eps);
        else if (width <= 2048) k_rms_reg<2, true><<<rows, kThreads, 0, s>>>(x, w, y, rows, width, eps);
        else k_rms_reg<4, true><<<rows, kThreads, 0, s>>>(x, w, y, rows, width, eps);
    } else {
        k_rms<<<rows, kThreads, 0, s>>>(x, w, y, width, eps);
    }
    MR_LAUNCHED("enqueue rms");
    return MR_OK;
}

int mr_rope(mr_ctx *ctx, const float *x, const float *freq, const float *pos, float *y, int rows, int heads, int dim,
            int split_half) {
    OP_BEGIN("rope");
    MR_REQUIRE(x && freq && pos && y && rows > 0 && heads > 0 && dim > 0 && dim % 2 == 0, "RoPE shape mismatch");
    // runs of heads a thread: all of them once the rows fill the device
    const int64_t pairs = (int64_t)rows * (dim / 2);
    const int per = (int)std::min<int64_t>(heads, std::max<int64_t>(ceil_div(heads, 65535), pairs * heads / 131072));
    const dim3 grid(grid_for(pairs), ceil_div(heads, per));
    k_rope<<<grid, kThreads, 0, s>>>(x, freq, pos, y, rows, heads, dim, split_half, per);
    MR_LAUNCHED("enqueue rope");
    return MR_OK;
}

int mr_swiglu(mr_ctx *ctx, const float *g, const float *u, float *y, int n) {
    OP_BEGIN("swiglu");
    MR_REQUIRE(g && u && y && n > 0, "SwiGLU shapes differ");
    k_swiglu<<<grid_for(n), kThreads, 0, s>>>(g, u, y, n);
    MR_LAUNCHED("enqueue swiglu");
    return MR_OK;
}

int mr_axpy(mr_ctx *ctx, const float *x, const float *y, float *z, int n, float scale) {
    OP_BEGIN("axpy");
    MR_REQUIRE(x && y && z && n > 0, "residual shapes differ");
    k_axpy<<<grid_for(n), kThreads, 0, s>>>(x, y, z, n, scale);
    MR_LAUNCHED("enqueue axpy");
    return MR_OK;
}

int mr_scores(mr_ctx *ctx, const float *q, const float *k, const float *extra_k, float *sc, int heads, int kv_heads,
              int dim, int capacity, int start, int length, int extra_length) {
    OP_BEGIN("scores");
    MR_REQUIRE(q && k && sc && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && capacity > 0 &&
                   length >= 0 && extra_length >= 0 && (extra_length == 0 || extra_k),
               "scores: bad arguments");
    int64_t n = (int64_t)(length + extra_length) * heads;
    if (n == 0) return MR_OK;
    const bool vec = dim % 4 == 0 && vec16(q, k) && vec16(extra_length ? extra_k : q);
    const int total = length + extra_length, lpr = lanes_for(vec ? dim / 4 : dim);
    const int hn = heads > kv_heads ? 4 : 1, runs = ceil_div(total, 16 * (kWave / lpr));
    const unsigned grid = (unsigned)runs * kv_heads * ceil_div(heads / kv_heads, hn);
#define MR_SCORES(V, HN)                                                                                          \
    k_scores<V, HN><<<grid, kThreads, 0, s>>>(q, k, extra_k, sc, heads, kv_heads, dim, capacity, start, length, \
                                              extra_length, lpr, runs)
    if (vec && hn == 4) MR_SCORES(4, 4);
    else if (vec) MR_SCORES(4, 1);
    else if (hn == 4) MR_SCORES(1, 4);
    else MR_SCORES(1, 1);
#undef MR_SCORES
    MR_LAUNCHED("enqueue scores");
    return MR_OK;
}

int mr_softmax(mr_ctx *ctx, const float *x, float *y, int rows, int width) {
    OP_BEGIN("softmax");
    MR_REQUIRE(x && y && rows > 0 && width > 0, "softmax: bad shape");
    if (width <= 1024) k_softmax_reg<256, 4><<<rows, 256, 0, s>>>(x, y, width);
    else if (width <= 8192) k_softmax_reg<1024, 8><<<rows, 1024, 0, s>>>(x, y, width);
    else k_softmax<<<rows, kThreads, 0, s>>>(x, y, width);
    MR_LAUNCHED("enqueue softmax");
    return MR_OK;
}

int mr_latent_mask(mr_ctx *ctx, float *scores, const float *positions, int heads, int length, int memory,
                   int earliest) {
    OP_BEGIN("latent_mask");
    MR_REQUIRE(scores && positions && heads > 0 && length > 0, "latent_mask: bad arguments");
    k_latent_mask<<<grid_for((int64_t)heads * length), kThreads, 0, s>>>(scores, positions, heads, length, memory,
                                                                         earliest);
    MR_LAUNCHED("enqueue latent_mask");
    return MR_OK;
}

int mr_mix(mr_ctx *ctx, const float *p, const float *v, const float *extra_v, float *y, int heads, int kv_heads,
           int dim, int capacity, int start, int length, int extra_length) {
    OP_BEGIN("mix");
    MR_REQUIRE(p && v && y && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && capacity > 0 &&
                   (extra_length == 0 || extra_v),
               "mix: bad arguments");
    const int total = std::max(length, 0) + std::max(extra_length, 0);
    const bool vec = dim % 4 == 0 && vec16(v, y) && vec16(extra_length > 0 ? extra_v : v);
    const int lpr = lanes_for(vec ? dim / 4 : dim);
    const int hn = heads > kv_heads ? 4 : 1;
    const int64_t units = (int64_t)kv_heads * ceil_div(heads / kv_heads, hn) * ceil_div(dim, lpr * (vec ? 4 : 1));
    // about two blocks per CU, each with a round of rows for its lane groups
    const int round = 4 * (256 / lpr);
    int chunks = (int)std::min<int64_t>(std::max<int64_t>(1, 512 / units), ceil_div(std::max(total, 1), round));
    void *part = nullptr;
    if (chunks > 1 && ctx_workspace(ctx, (size_t)chunks * heads * dim * sizeof(float), &part) != MR_OK) chunks = 1;
    const int chunk = ceil_div(std::max(total, 1), chunks);
    chunks = ceil_div(std::max(total, 1), chunk);
    float *out = chunks > 1 ? (float *)part : y;
    const unsigned grid = (unsigned)(chunks * units);
#define MR_MIX(V, HN)                                                                                             \
    k_mix<V, HN><<<grid, kThreads, 0, s>>>(p, v, extra_v, out, heads, kv_heads, dim, capacity, start,           \
                                           std::max(length, 0), std::max(extra_length, 0), lpr, chunk, chunks)
    if (vec && hn == 4) MR_MIX(4, 4);
    else if (vec) MR_MIX(4, 1);
    else if (hn == 4) MR_MIX(1, 4);
    else MR_MIX(1, 1);
#undef MR_MIX
    if (chunks > 1) k_sum_chunks<<<grid_for(heads * dim), kThreads, 0, s>>>(out, y, heads * dim, chunks);
    const hipError_t e = hipGetLastError();
    if (part) ctx_release(ctx, part);   // stream-ordered: later work on this stream reuses it safely
    MR_HIP(e, "enqueue mix");
    return MR_OK;
}

int mr_pool_scores(mr_ctx *ctx, const float *u, const float *q, float *sc, int tokens, int slots, int width) {
    OP_BEGIN("pool_scores");
    MR_REQUIRE(u && q && sc && tokens > 0 && slots > 0 && width > 0, "pool_scores: bad arguments");
    const int grid = (int)ceil_div64((int64_t)tokens * slots, 4);
    if (width % 4 == 0 && vec16(u, q)) k_pool_scores<4><<<grid, kThreads, 0, s>>>(u, q, sc, tokens, slots, width);
    else k_pool_scores<1><<<grid, kThreads, 0, s>>>(u, q, sc, tokens, slots, width);
    MR_LAUNCHED("enqueue pool_scores");
    return MR_OK;
}

int mr_pool_mix(mr_ctx *ctx, const float *u, const float *p, float *z, float *anchors, int tokens, int slots,
                int width, int start_position) {
    OP_BEGIN("pool_mix");
    MR_REQUIRE(u && p && z && anchors && tokens > 0 && slots > 0 && width > 0, "pool_mix: bad arguments");
    const int runs = ceil_div(width, kWave);
    k_pool_mix<<<(unsigned)runs * slots, kThreads, 0, s>>>(u, p, z, anchors, tokens, slots, width, start_position,
                                                           runs);
    MR_LAUNCHED("enqueue pool_mix");
    return MR_OK;
}

int mr_merge_rows(mr_ctx *ctx, const float *x, float *y, int width, float a, float b) {
    OP_BEGIN("merge_rows");
    MR_REQUIRE(x && y && width > 0, "merge_rows: bad arguments");
    k_merge_rows<<<grid_for(width), kThreads, 0, s>>>(x, y, width, a, b);
    MR_LAUNCHED("enqueue merge_rows");
    return MR_OK;
}

int mr_block_means(mr_ctx *ctx, const float *x, float *y, int length, int width, int block) {
    OP_BEGIN("block_means");
    MR_REQUIRE(x && y && length > 0 && width > 0 && block > 0, "block_means: bad arguments");
    int blocks = (length + block - 1) / block;
    k_block_means<<<grid_for((int64_t)blocks * width), kThreads, 0, s>>>(x, y, length, width, block);
    MR_LAUNCHED("enqueue block_means");
    return MR_OK;
}

int mr_attention(mr_ctx *ctx, const float *q, const float *k, const float *v, const float *extra_k,
                 const float *extra_v, float *y, int heads, int kv_heads, int dim, int capacity, int start,
                 int length, int extra_length) {
    OP_BEGIN("attention");
    (void)s;
    MR_REQUIRE(q && k && v && y && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && capacity > 0 &&
                   length >= 0 && extra_length >= 0 && length + extra_length > 0 &&
                   (extra_length == 0 || (extra_k && extra_v)),
               "attention: bad arguments");
    AttnProblem pr;
    pr.q = q; pr.ring_k = k; pr.ring_v = v; pr.extra_k = extra_k; pr.extra_v = extra_v;
    pr.heads = heads; pr.kv_heads = kv_heads; pr.dim = dim; pr.capacity = capacity;
    pr.start = start; pr.length = length; pr.extra_length = extra_length; pr.out = y;
    return launch_attention_op(ctx, pr);
}

int mr_attention_noalloc(mr_ctx *ctx, const float *q, const float *k, const float *v, const float *extra_k,
                         const float *extra_v, float *y, int heads, int kv_heads, int dim, int capacity, int start,
                         int length, int extra_length) {
    OP_BEGIN("attention_noalloc");
    (void)s;
    MR_REQUIRE(q && k && v && y && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && capacity > 0 &&
                   length >= 0 && extra_length >= 0 && length + extra_length > 0 &&
                   (extra_length == 0 || (extra_k && extra_v)),
               "attention_noalloc: bad arguments");
    AttnProblem pr;
    pr.q = q; pr.ring_k = k; pr.ring_v = v; pr.extra_k = extra_k; pr.extra_v = extra_v;
    pr.heads = heads; pr.kv_heads = kv_heads; pr.dim = dim; pr.capacity = capacity;
    pr.start = start; pr.length = length; pr.extra_length = extra_length; pr.out = y;
    return launch_attention_op_noalloc(ctx, pr);
}

int mr_debug_gemm(mr_ctx *ctx, const float *a, const void *w, float *c, float *ascale, int m, int n, int k,
                  int scheme) {
    OP_BEGIN("debug gemm");
    MR_REQUIRE(a && w && c && m > 0 && n > 0 && k > 0 && k % 8 == 0 && (scheme == 0 || (scheme == 1 && ascale)),
               "debug gemm: bad arguments");
    GemmArgs g;
    g.a = a; g.lda = k; g.w = w; g.dtype = MR_BF16; g.c = c; g.ldc = n; g.m = m; g.n = n; g.k = k;
    if (scheme == 1) {
        MR_TRY(gemm_f16_weight_scale(s, w, MR_BF16, (int64_t)n * k, &g.wscale));
        MR_REQUIRE(g.wscale > 0.0f, "debug gemm: weights not eligible for FP16 terms");
        g.ascale = ascale;
        MR_HIP(hipMalloc((void **)&g.ahl_ws, (size_t)2 * m * k * sizeof(_Float16)), "debug gemm workspace");
        void *wh = nullptr;
        const hipError_t ea = hipMalloc(&wh, (size_t)n * k * 2);
        if (ea != hipSuccess) {
            (void)hipFree(g.ahl_ws);
            MR_HIP(ea, "debug gemm workspace");
        }
        g.wh = wh;
        const int rc = gemm_f16_weight_copy(s, w, (int64_t)n * k, g.wscale, wh);
        if (rc != MR_OK) {
            (void)hipFree(g.ahl_ws);
            (void)hipFree(wh);
            return rc;
        }
        // the K slices' sums, as the batched prefill gives them (without, K stays whole)
        if (hipMalloc((void **)&g.part, kGemmPartFloats * sizeof(float)) != hipSuccess) g.part = nullptr;
    }
    int rc = launch_gemm(s, GEMM_STORE, g);
    const hipError_t e = hipStreamSynchronize(s);
    if (g.ahl_ws) (void)hipFree(g.ahl_ws);
    if (g.wh) (void)hipFree(const_cast<void *>(g.wh));
    if (g.part) (void)hipFree(g.part);
    MR_TRY(rc);
    MR_HIP(e, "debug gemm");
    return MR_OK;
}

int mr_debug_gemm_grouped(mr_ctx *ctx, const float *a, const void *w, const void *w2, float *c, const int *counts,
                          int groups, int n, int k, int swiglu, int tile_list) {
    OP_BEGIN("debug grouped gemm");
    MR_REQUIRE(a && w && c && counts && groups > 0 && groups <= 1024 && n > 0 && k > 0 && k % 8 == 0 &&
                   (!swiglu || w2),
               "debug grouped gemm: bad arguments");
    std::vector<int> offset(groups), start(groups + 1);
    int rows = 0, max_rows = 0;
    start[0] = 0;
    for (int z = 0; z < groups; ++z) {
        MR_REQUIRE(counts[z] >= 0, "debug grouped gemm: negative group size");
        offset[z] = rows;
        rows += counts[z];
        max_rows = std::max(max_rows, counts[z]);
        start[z + 1] = start[z] + ceil_div(counts[z], kGemmRowTile);
    }
    MR_REQUIRE(rows > 0, "debug grouped gemm: no rows");
    std::vector<void *> owned;   // freed on every return
    auto alloc = [&](size_t bytes, void **p) {
        const hipError_t e = hipMalloc(p, bytes);
        if (e == hipSuccess) owned.push_back(*p);
        return e;
    };
    struct Free {   // after the stream's work on them
        std::vector<void *> &v;
        hipStream_t s;
        ~Free() {
            (void)hipStreamSynchronize(s);
            for (void *p : v) (void)hipFree(p);
        }
    } release{owned, s};
    const int mats = swiglu ? 2 : 1;
    const int64_t nk = (int64_t)n * k;
    std::vector<void *> tab_w(mats * groups), tab_h(mats * groups);
    std::vector<float> scale(mats * groups);
    _Float16 *wh = nullptr;
    MR_HIP(alloc((size_t)mats * groups * nk * 2, (void **)&wh), "debug grouped gemm workspace");
    // a scale per matrix; a group's gate and up rows share the smaller, as
    // the model's expert copies do (the SwiGLU kernel unscales both by one)
    for (int t = 0; t < mats; ++t)
        for (int z = 0; z < groups; ++z) {
            const void *src = (const char *)(t ? w2 : w) + (size_t)z * nk * 2;
            float sc = 0.0f;
            MR_TRY(gemm_f16_weight_scale(s, src, MR_BF16, nk, &sc));
            MR_REQUIRE(sc > 0.0f, "debug grouped gemm: weights not eligible for FP16 terms");
            tab_w[t * groups + z] = const_cast<void *>(src);
            scale[t * groups + z] = sc;
        }
    for (int z = 0; z < groups && mats == 2; ++z)
        scale[z] = scale[groups + z] = std::min(scale[z], scale[groups + z]);
    for (int t = 0; t < mats; ++t)
        for (int z = 0; z < groups; ++z) {
            _Float16 *dst = wh + ((size_t)t * groups + z) * nk;
            MR_TRY(gemm_f16_weight_copy(s, tab_w[t * groups + z], nk, scale[t * groups + z], dst));
            tab_h[t * groups + z] = dst;
        }
    void **d_w = nullptr, **d_h = nullptr;
    float *d_scale = nullptr, *ascale = nullptr;
    int *d_off = nullptr, *d_cnt = nullptr, *d_start = nullptr;
    _Float16 *planes = nullptr;
    MR_HIP(alloc(tab_w.size() * sizeof(void *), (void **)&d_w), "debug grouped gemm workspace");
    MR_HIP(alloc(tab_h.size() * sizeof(void *), (void **)&d_h), "debug grouped gemm workspace");
    MR_HIP(alloc(scale.size() * sizeof(float), (void **)&d_scale), "debug grouped gemm workspace");
    MR_HIP(alloc((size_t)groups * sizeof(int), (void **)&d_off), "debug grouped gemm workspace");
    MR_HIP(alloc((size_t)groups * sizeof(int), (void **)&d_cnt), "debug grouped gemm workspace");
    MR_HIP(alloc((size_t)(groups + 1) * sizeof(int), (void **)&d_start), "debug grouped gemm workspace");
    MR_HIP(alloc((size_t)rows * sizeof(float), (void **)&ascale), "debug grouped gemm workspace");
    MR_HIP(alloc((size_t)2 * rows * k * sizeof(_Float16), (void **)&planes), "debug grouped gemm workspace");
    MR_HIP(hipMemcpy(d_w, tab_w.data(), tab_w.size() * sizeof(void *), hipMemcpyHostToDevice), "debug grouped gemm");
    MR_HIP(hipMemcpy(d_h, tab_h.data(), tab_h.size() * sizeof(void *), hipMemcpyHostToDevice), "debug grouped gemm");
    MR_HIP(hipMemcpy(d_scale, scale.data(), scale.size() * sizeof(float), hipMemcpyHostToDevice), "debug grouped gemm");
    MR_HIP(hipMemcpy(d_off, offset.data(), groups * sizeof(int), hipMemcpyHostToDevice), "debug grouped gemm");
    MR_HIP(hipMemcpy(d_cnt, counts, groups * sizeof(int), hipMemcpyHostToDevice), "debug grouped gemm");
    MR_HIP(hipMemcpy(d_start, start.data(), (groups + 1) * sizeof(int), hipMemcpyHostToDevice), "debug grouped gemm");
    GemmArgs g;
    g.a = a; g.lda = k; g.dtype = MR_BF16; g.c = c; g.ldc = n; g.m = rows; g.n = n; g.k = k;
    g.ascale = ascale; g.ahl_ws = planes;
    GemmGroups gg;
    gg.offset = d_off; gg.count = d_cnt; gg.groups = groups; gg.max_rows = max_rows;
    gg.w = d_w; gg.w2 = swiglu ? d_w + groups : nullptr;
    gg.wh = d_h; gg.wh2 = swiglu ? d_h + groups : nullptr; gg.wscale = d_scale;
    if (tile_list) {
        gg.row_tile_start = d_start;
        gg.row_tiles = start[groups];
    }
    MR_TRY(launch_gemm_grouped(s, swiglu ? GEMM_SWIGLU : GEMM_STORE, g, gg));
    MR_HIP(hipStreamSynchronize(s), "debug grouped gemm");
    return MR_OK;
}

int mr_debug_exp(mr_ctx *ctx, const float *x, float *y, int n, int which) {
    OP_BEGIN("debug exp");
    MR_TRY(launch_debug_exp(s, x, y, n, which));
    MR_HIP(hipStreamSynchronize(s), "debug exp");
    return MR_OK;
}

int mr_debug_prefill_attention(mr_ctx *ctx, const float *qkv, const float *ring_k, const float *ring_v, float *out,
                               int rows, int p0, int heads, int kv_heads, int d, int cap, int window, int presplit) {
    OP_BEGIN("debug prefill attention");
    MR_REQUIRE(qkv && ring_k && ring_v && out && rows > 0 && p0 >= 0 && heads > 0 && kv_heads > 0 && d > 0 &&
                   cap > 0 && window >= 0,
               "debug prefill attention: bad arguments");
    PrefillAttnArgs a;
    a.qkv = qkv; a.ld = (heads + 2 * kv_heads) * d; a.ring_k = ring_k; a.ring_v = ring_v; a.cap = cap;
    a.out = out; a.ldo = heads * d; a.p0 = p0; a.rows = rows; a.heads = heads; a.kv_heads = kv_heads; a.d = d;
    a.inv_root = 1.0f / sqrtf((float)d); a.window = window;
    void *ws = nullptr;
    if (presplit) {
        const int n = ceil_div(rows + std::min(p0, (window ? window : cap) - 1), 32) * 32;   // whole 32-row tiles
        const size_t planes = (size_t)4 * n * kv_heads * d * sizeof(_Float16);
        MR_HIP(hipMalloc(&ws, planes + 4 * kv_heads * sizeof(float)), "debug prefill attention workspace");
        a.kv16 = (_Float16 *)ws;
        a.kv16_rows = n;
        a.kv16_scale = (float *)((char *)ws + planes);
        a.kv16_max = (unsigned *)(a.kv16_scale + 2 * kv_heads);
    }
    const int rc = launch_prefill_attention(s, a);
    const hipError_t e = hipStreamSynchronize(s);
    if (ws) (void)hipFree(ws);
    MR_TRY(rc);
    MR_HIP(e, "debug prefill attention");
    return MR_OK;
}

}  // extern "C"
