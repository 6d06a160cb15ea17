// Companion elementwise kernels of the training step (reference: kernels.py:699-862,
// dataparallel.py:54-58).  One thread per element (or per row / column where the
// reference does that); they exist so a whole MLP train step can run on the
// device around the GEMMs, and are not tuned beyond coalesced access.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mi_gemm.h"

#include "act_math.h"
#include "ew_common.h"

namespace mg {

__device__ __forceinline__ float act_f(float x, int act) {
    return act == MG_ACT_GELU ? gelu_value(x) : (act == MG_ACT_RELU ? fmaxf(x, 0.f) : x);
}
__device__ __forceinline__ float dact_f(float x, int act) {
    return act == MG_ACT_GELU ? gelu_slope(x) : (act == MG_ACT_RELU ? (x > 0.f ? 1.f : 0.f) : 1.f);
}

__global__ void k_bias_act(const float *acc, const float *bias, float *z, uint16_t *y16, int64_t n,
                           int64_t ncol, int act, int dtype) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float v = !bias ? acc[i] : acc[i] + bias[(n | ncol) <= 0x7fffffff ? (uint32_t)i % (uint32_t)ncol : i % ncol];
    if (z) z[i] = v;
    if (y16) y16[i] = narrow16(act_f(v, act), dtype);
}

// The same four elements a thread (n and ncol multiples of 4, aligned): one 16-byte access per matrix, and one 32-bit
// remainder instead of a 64-bit one per element, which is what the kernel above spends its time on (2048 x 2048, GELU:
// 17.3 -> 9 us).  The arithmetic of an element is the same in both.
__device__ __forceinline__ uint2 narrow16x4(float a, float b, float c, float d, int dtype) {
    return make_uint2((uint32_t)narrow16(a, dtype) | ((uint32_t)narrow16(b, dtype) << 16),
                      (uint32_t)narrow16(c, dtype) | ((uint32_t)narrow16(d, dtype) << 16));
}
template <int ACT>
__global__ void __launch_bounds__(256) k_bias_act_v4(const float *acc, const float *bias, float *z, uint16_t *y16, uint32_t n4,
                                                     uint32_t ncol4, int dtype) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    float4 v = reinterpret_cast<const float4 *>(acc)[i];
    if (bias) {
        const float4 b = reinterpret_cast<const float4 *>(bias)[i % ncol4];
        v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w;
    }
    if (z) reinterpret_cast<float4 *>(z)[i] = v;
    if (y16) reinterpret_cast<uint2 *>(y16)[i] = narrow16x4(act_f(v.x, ACT), act_f(v.y, ACT), act_f(v.z, ACT), act_f(v.w, ACT), dtype);
}
template <int ACT, bool F32>
__global__ void __launch_bounds__(256) k_act_bwd_v4(const float *dy, const float *z, uint16_t *dz16, float *dz32, uint32_t n4, int dtype) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    float4 g = reinterpret_cast<const float4 *>(dy)[i];
    const float4 x = reinterpret_cast<const float4 *>(z)[i];
    g.x *= dact_f(x.x, ACT);
    g.y *= dact_f(x.y, ACT);
    g.z *= dact_f(x.z, ACT);
    g.w *= dact_f(x.w, ACT);
    if (dz16) reinterpret_cast<uint2 *>(dz16)[i] = narrow16x4(g.x, g.y, g.z, g.w, dtype);
    if (F32) reinterpret_cast<float4 *>(dz32)[i] = g;
}

__global__ void k_act_bwd(const float *dy, const float *z, uint16_t *dz16, float *dz32, int64_t n, int act,
                          int dtype) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float g = dy[i] * dact_f(z[i], act);
    if (dz16) dz16[i] = narrow16(g, dtype);
    if (dz32) dz32[i] = g;
}

// Column sums (the reference loops the rows in one thread per column, kernels.py:753-761:
// fine at batch 128 on 12 CUs, one long chain of dependent loads here).  A block takes 64
// columns and COL_SUM_ROWS rows: 8 threads per column stride through the rows (coalesced 256-byte
// row pieces), LDS adds the 8 partial sums.  One chunk of rows: the block writes (or adds to) the
// sum itself, in a fixed order.  More rows: the chunks add with atomics into sums, which the
// host has cleared unless accumulating.
// Up to COL_SUM_ONE rows one chunk with twice the threads per column takes them all: no clear in front, no atomics.
// 16 columns a workgroup: with 64, 2049 columns kept 33 CUs busy with 256 KB each (1000 rows 10.5 us, 8.1 so).  Rows beyond the
// end are clamped and not added: what an unrolled loop leaves over would be loaded one by one.
constexpr int COL_SUM_ONE_COLS = 16;
__global__ void __launch_bounds__(256) k_col_sum_one(const float *g, float *sums, int64_t ncol, int64_t nrow, int accumulate) {
    __shared__ float part[16][COL_SUM_ONE_COLS];
    const int tx = threadIdx.x % COL_SUM_ONE_COLS, ty = threadIdx.x / COL_SUM_ONE_COLS;
    const int64_t c = (int64_t)blockIdx.x * COL_SUM_ONE_COLS + tx;
    float s = 0.f;
    if (c < ncol) {
        for (int64_t r = ty; r < nrow; r += 16 * 16) {
            float v[16];
#pragma unroll
            for (int i = 0; i < 16; i++) v[i] = g[(r + 16 * i < nrow ? r + 16 * i : r) * ncol + c];
#pragma unroll
            for (int i = 0; i < 16; i++) s += r + 16 * i < nrow ? v[i] : 0.f;
        }
    }
    part[ty][tx] = s;
    __syncthreads();
    if (ty == 0 && c < ncol) {
#pragma unroll
        for (int i = 1; i < 16; i++) s += part[i][tx];
        sums[c] = accumulate ? sums[c] + s : s;
    }
}
__global__ void __launch_bounds__(512) k_col_sum(const float *g, float *sums, int64_t ncol, int64_t nrow,
                                                  int accumulate, int atomic) {
    __shared__ float part[8][64];
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int64_t c = (int64_t)blockIdx.x * 64 + tx;
    const int64_t r0 = (int64_t)blockIdx.y * COL_SUM_ROWS;
    const int64_t r1 = r0 + COL_SUM_ROWS < nrow ? r0 + COL_SUM_ROWS : nrow;
    float s = 0.f;
    if (c < ncol) {
#pragma unroll 8
        for (int64_t r = r0 + ty; r < r1; r += 8) s += g[r * ncol + c];
    }
    part[ty][tx] = s;
    __syncthreads();
    if (ty == 0 && c < ncol) {
        float t = part[0][tx];
#pragma unroll
        for (int i = 1; i < 8; i++) t += part[i][tx];
        if (atomic) atomicAdd(sums + c, t);
        else sums[c] = accumulate ? sums[c] + t : t;
    }
}

// Device-side copy of nbytes (a multiple of 4; 16-byte pieces when both ends are aligned).
__global__ void k_copy(const uint32_t *src, uint32_t *dst, int64_t nwords, int vec) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (vec) {
        if (i * 4 + 3 < nwords) reinterpret_cast<uint4 *>(dst)[i] = reinterpret_cast<const uint4 *>(src)[i];
        else for (int64_t j = i * 4; j < nwords; j++) dst[j] = src[j];
    } else if (i < nwords) {
        dst[i] = src[i];
    }
}

// A wavefront per row (the reference gives a row one thread, kernels.py:766-791, which walks it four times with every
// load behind the last: 28 us for 1000 rows of 37, 6 for 128 of 10; this form 5 and 3).
// Up to CE_IN_ORDER classes the sum has to be the one of that thread, to the last bit, so that a small model goes on
// training as it did: an add of a lane's value every few clocks, 0.4 us for 100 classes.  Beyond, where it would be the
// longest part of the kernel, the lanes' partial sums meet in a tree.
constexpr int CE_IN_ORDER = 128;
__global__ void __launch_bounds__(256) k_softmax_ce(const float *logits, const uint32_t *labels, uint16_t *dl16, float *dl32,
                                                    float *loss, int64_t nrows, int64_t stride, int64_t ncls, int dtype) {
    const int lane = threadIdx.x & 63;
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= nrows) return;
    const float *row = logits + i * stride;
    const float x0 = lane < ncls ? row[lane] : -1e30f;   // a row of up to 64 classes stays in registers
    float mx = x0;
    for (int64_t c = lane + 64; c < ncls; c += 64) mx = fmaxf(mx, row[c]);
    mx = wave_max(mx);
    float s = lane < ncls ? expf(x0 - mx) : 0.f;
    if (ncls <= CE_IN_ORDER) {
        // in the order of the classes, lane by lane: the sum of a serial loop to the last bit
        float t = 0.f;
        for (int c0 = 0; c0 < (int)ncls; c0 += 64) {
            if (c0) s = c0 + lane < ncls ? expf(row[c0 + lane] - mx) : 0.f;
            const int here = min(64, (int)ncls - c0);
            for (int j = 0; j < here; j++) t += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), j));
        }
        s = t;
    } else {
        for (int64_t c = lane + 64; c < ncls; c += 64) s += expf(row[c] - mx);
        s = wave_sum(s);
    }
    const float logZ = mx + logf(s);
    const int64_t y = labels[i];
    if (lane == 0) loss[i] = logZ - row[y];
    const float inv = 1.0f / (float)nrows;
    for (int64_t c = lane; c < stride; c += 64) {
        const float x = c < 64 ? x0 : c < ncls ? row[c] : 0.f;
        const float gv = c < ncls ? (expf(x - logZ) - (c == y ? 1.f : 0.f)) * inv : 0.f;
        if (dl16) dl16[i * stride + c] = narrow16(gv, dtype);
        if (dl32) dl32[i * stride + c] = gv;
    }
}

__global__ void k_adamw(float *w, const float *g, float *m, float *v, uint16_t *w16, const float *hp, int64_t n,
                        float wd, int dtype) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float lr = hp[0], b1 = hp[1], b2 = hp[2], bc1 = hp[3], bc2 = hp[4], eps = hp[5];
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float mh = mi / bc1;
    const float vh = vi / bc2;
    float wi = w[i];
    wi -= lr * (mh / (sqrtf(vh) + eps) + wd * wi);
    w[i] = wi;
    if (w16) w16[i] = narrow16(wi, dtype);
}

// AdamW over a list of parameters in one launch.  The table holds one entry per parameter and the
// number of its first workgroup; a workgroup finds its parameter by bisection and updates 1024
// consecutive elements of it, four per thread (same arithmetic as k_adamw, element by element).
__device__ __forceinline__ float adamw_one(float &w, float g, float &m, float &v, float lr, float b1, float b2,
                                           float bc1, float bc2, float eps, float wd) {
    m = b1 * m + (1.0f - b1) * g;
    v = b2 * v + (1.0f - b2) * g * g;
    w -= lr * ((m / bc1) / (sqrtf(v / bc2) + eps) + wd * w);
    return w;
}
__global__ void __launch_bounds__(256) k_adamw_multi(const mg_adamw_entry *table, int ntensors, const float *hp, int dtype) {
    int lo = 0, hi = ntensors - 1;
    while (lo < hi) {                      // last entry whose first_block <= blockIdx.x
        const int mid = (lo + hi + 1) >> 1;
        if (table[mid].first_block <= (int64_t)blockIdx.x) lo = mid;
        else hi = mid - 1;
    }
    const mg_adamw_entry e = table[lo];
    const float lr = hp[0], b1 = hp[1], b2 = hp[2], bc1 = hp[3], bc2 = hp[4], eps = hp[5];
    const int64_t i0 = (((int64_t)blockIdx.x - e.first_block) * 256 + threadIdx.x) * 4;
    if (i0 >= e.n) return;
    float *w = e.w + i0, *m = e.m + i0, *v = e.v + i0;
    const float *g = e.g + i0;
    uint16_t *w16 = e.w16 ? (uint16_t *)e.w16 + i0 : nullptr;
    if (i0 + 3 < e.n && e.vec) {
        float4 wv = *reinterpret_cast<float4 *>(w), mv = *reinterpret_cast<float4 *>(m), vv = *reinterpret_cast<float4 *>(v);
        const float4 gv = *reinterpret_cast<const float4 *>(g);
        adamw_one(wv.x, gv.x, mv.x, vv.x, lr, b1, b2, bc1, bc2, eps, e.wd);
        adamw_one(wv.y, gv.y, mv.y, vv.y, lr, b1, b2, bc1, bc2, eps, e.wd);
        adamw_one(wv.z, gv.z, mv.z, vv.z, lr, b1, b2, bc1, bc2, eps, e.wd);
        adamw_one(wv.w, gv.w, mv.w, vv.w, lr, b1, b2, bc1, bc2, eps, e.wd);
        *reinterpret_cast<float4 *>(w) = wv;
        *reinterpret_cast<float4 *>(m) = mv;
        *reinterpret_cast<float4 *>(v) = vv;
        if (w16)
            *reinterpret_cast<uint2 *>(w16) =
                make_uint2((uint32_t)narrow16(wv.x, dtype) | ((uint32_t)narrow16(wv.y, dtype) << 16),
                           (uint32_t)narrow16(wv.z, dtype) | ((uint32_t)narrow16(wv.w, dtype) << 16));
    } else {
        for (int k = 0; k < 4 && i0 + k < e.n; k++) {
            const float wi = adamw_one(w[k], g[k], m[k], v[k], lr, b1, b2, bc1, bc2, eps, e.wd);
            if (w16) w16[k] = narrow16(wi, dtype);
        }
    }
}

// Clears the gradient of every entry of an AdamW-style table in one launch (same block numbering).
__global__ void __launch_bounds__(256) k_zero_multi(const mg_adamw_entry *table, int ntensors) {
    int lo = 0, hi = ntensors - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (table[mid].first_block <= (int64_t)blockIdx.x) lo = mid;
        else hi = mid - 1;
    }
    const mg_adamw_entry e = table[lo];
    float *g = const_cast<float *>(e.g);
    const int64_t i0 = (((int64_t)blockIdx.x - e.first_block) * 256 + threadIdx.x) * 4;
    for (int k = 0; k < 4 && i0 + k < e.n; k++) g[i0 + k] = 0.f;
}

__global__ void k_zero(float *dst, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = 0.f;
}

__global__ void k_cast16(const float *src, uint16_t *dst, int64_t n, int dtype) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = narrow16(src[i], dtype);
}

// four elements per thread: one 16-byte load, one 8-byte store; the tail goes element by element
__global__ void k_cast16_v4(const float *src, uint16_t *dst, int64_t n, int dtype) {
    const int64_t i4 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i4 * 4 + 3 < n) {
        const float4 t = reinterpret_cast<const float4 *>(src)[i4];
        reinterpret_cast<uint2 *>(dst)[i4] =
            make_uint2((uint32_t)narrow16(t.x, dtype) | ((uint32_t)narrow16(t.y, dtype) << 16),
                       (uint32_t)narrow16(t.z, dtype) | ((uint32_t)narrow16(t.w, dtype) << 16));
    } else {
        for (int64_t i = i4 * 4; i < n; i++) dst[i] = narrow16(src[i], dtype);
    }
}

// Several copies in one launch (grid.y the copy): what a recorded step stages from CPU-written buffers.
struct CopyMulti {
    const uint32_t *src[MG_COPY_MAX];
    uint32_t *dst[MG_COPY_MAX];
    int64_t bytes[MG_COPY_MAX];
    int vec[MG_COPY_MAX], walk[MG_COPY_MAX];
};
// A thread takes 16 bytes, all of a copy on their way at once.  walk: COPY_WALK workgroups go through the buffer together, four
// loads a thread: over PCIe, requests in the order of their addresses are worth 54 GB/s from 16 workgroups, 50 from 64 and 41
// with a workgroup for every 4 KB.  Only for aligned host memory beyond COPY_WALK_BYTES (a workgroup for every 4 KB / walking, us,
// one copy and the wait for it: 128 KB 15.2 / 16.5, 256 KB 18.1 / 19.0, 384 KB 21.2 / 21.2, 512 KB 24.3 / 24.0, 1 MB 37.0 / 33.7, 3 MB
// 85 / 72; between others: 3 MB of host memory that is aligned to 4 bytes 64 / 241, 6 MB in HBM 5.5 / 18.7).
constexpr int COPY_WALK = 16;
constexpr int64_t COPY_WALK_BYTES = 384 << 10;
__global__ void __launch_bounds__(256) k_copy_multi(const CopyMulti a) {
    const int w = blockIdx.y;
    const int64_t n = a.bytes[w], i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const uint32_t *src = a.src[w];
    uint32_t *dst = a.dst[w];
    if (a.walk[w]) {
        if (blockIdx.x >= COPY_WALK) return;   // (the grid is that of the widest copy)
        constexpr int STEP = COPY_WALK * 256;
        const int64_t n16 = n / 16;
        for (int64_t at = i; at < n16; at += 4 * STEP) {
            uint4 v[4];
#pragma unroll
            for (int u = 0; u < 4; u++) v[u] = reinterpret_cast<const uint4 *>(src)[at + u * STEP < n16 ? at + u * STEP : at];
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (at + u * STEP < n16) reinterpret_cast<uint4 *>(dst)[at + u * STEP] = v[u];
        }
        if (i < n % 16) reinterpret_cast<uint8_t *>(dst)[n16 * 16 + i] = reinterpret_cast<const uint8_t *>(src)[n16 * 16 + i];
    } else if (a.vec[w] && i * 16 + 15 < n) {
        reinterpret_cast<uint4 *>(dst)[i] = reinterpret_cast<const uint4 *>(src)[i];
    } else {
        for (int64_t j = i * 4; j < i * 4 + 4 && j < n / 4; j++) dst[j] = src[j];
        if (i * 16 <= n && n < i * 16 + 16)   // the last piece: bytes behind the last whole word
            for (int64_t j = n / 4 * 4; j < n; j++) reinterpret_cast<uint8_t *>(dst)[j] = reinterpret_cast<const uint8_t *>(src)[j];
    }
}

// Gradients of a list of parameters into, or back out of, a flat accumulator in one launch (an AdamW-style table: g the
// gradient, w its place in the accumulator): the launches per parameter of dataparallel.py:47-73, most of them for a few
// hundred elements, cost 2 to 5 us each.
template <bool PULL>
__global__ void __launch_bounds__(256) k_arena_multi(const mg_adamw_entry *table, int ntensors, float scale) {
    int lo = 0, hi = ntensors - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (table[mid].first_block <= (int64_t)blockIdx.x) lo = mid;
        else hi = mid - 1;
    }
    const mg_adamw_entry e = table[lo];
    float *g = const_cast<float *>(e.g);
    const int64_t i0 = (((int64_t)blockIdx.x - e.first_block) * 256 + threadIdx.x) * 4;
    if (i0 + 3 < e.n && e.vec) {
        float4 w = *reinterpret_cast<float4 *>(e.w + i0);
        if (PULL) {
            *reinterpret_cast<float4 *>(g + i0) = make_float4(w.x * scale, w.y * scale, w.z * scale, w.w * scale);
        } else {
            const float4 x = *reinterpret_cast<const float4 *>(g + i0);
            w.x += x.x; w.y += x.y; w.z += x.z; w.w += x.w;
            *reinterpret_cast<float4 *>(e.w + i0) = w;
        }
    } else {
        for (int64_t i = i0; i < i0 + 4 && i < e.n; i++) {
            if (PULL) g[i] = e.w[i] * scale;
            else e.w[i] += g[i];
        }
    }
}

__global__ void k_scale_copy(float *dst, const float *src, int64_t n, float scale) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i] * scale;
}

__global__ void k_grad_add(float *dst, const float *src, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] += src[i];
}

// Pseudo-random 16-bit operands in [-1, 1) from a counter hash: timing a GEMM on
// zeros or on uninitialised memory misstates it (data toggling sets MFMA power,
// and with it the clock), so the tuner and warm-up fill their scratch with this.
__global__ void k_fill_uniform16(uint16_t *dst, int64_t n, uint32_t seed, int dtype) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t x = (uint32_t)i * 0x9E3779B1u + seed;
    x ^= x >> 16;
    x *= 0x85EBCA6Bu;
    x ^= x >> 13;
    x *= 0xC2B2AE35u;
    x ^= x >> 16;
    const float v = (float)(x >> 8) * (2.0f / 16777216.0f) - 1.0f;
    dst[i] = narrow16(v, dtype);
}

}  // namespace mg

using namespace mg;

static inline bool al16(const void *p) { return ((uintptr_t)p & 15) == 0; }
static inline bool act_ok(int a) { return a >= MG_ACT_NONE && a <= MG_ACT_RELU; }

extern "C" {

int mg_ew_bias_act(mg_ctx *ctx, const float *acc, const float *bias, float *z, void *y16, int64_t n, int64_t ncol,
                   int act, int dtype) {
    EW_PRECHECK("mg_ew_bias_act", acc && (z || y16) && count_ok(n) && ncol > 0 && act_ok(act) && dtype_ok(dtype));
    if (n % 4 == 0 && (!bias || ncol % 4 == 0) && (n | ncol) <= 0x7fffffff && al16(acc) && al16(bias) && al16(z) && ((uintptr_t)y16 & 7) == 0) {
        const auto kern = act == MG_ACT_GELU ? k_bias_act_v4<MG_ACT_GELU> : act == MG_ACT_RELU ? k_bias_act_v4<MG_ACT_RELU> : k_bias_act_v4<MG_ACT_NONE>;
        hipLaunchKernelGGL(kern, dim3(blocks_for(n / 4)), dim3(256), 0, ctx_stream(ctx), acc, bias, z, (uint16_t *)y16,
                           (uint32_t)(n / 4), bias ? (uint32_t)(ncol / 4) : 1u, dtype);
        EW_POSTCHECK("mg_ew_bias_act");
    }
    hipLaunchKernelGGL(k_bias_act, dim3(blocks_for(n)), dim3(256), 0, ctx_stream(ctx), acc, bias, z, (uint16_t *)y16, n,
                       ncol, act, dtype);
    EW_POSTCHECK("mg_ew_bias_act");
}

int mg_ew_act_bwd(mg_ctx *ctx, const float *dy, const float *z, void *dz16, float *dz32, int64_t n, int act,
                  int dtype) {
    EW_PRECHECK("mg_ew_act_bwd", dy && z && (dz16 || dz32) && count_ok(n) && act_ok(act) && dtype_ok(dtype));
    if (n % 4 == 0 && n <= 0x7fffffff && al16(dy) && al16(z) && al16(dz32) && ((uintptr_t)dz16 & 7) == 0) {
        const auto kern = dz32 ? (act == MG_ACT_GELU ? k_act_bwd_v4<MG_ACT_GELU, true> : act == MG_ACT_RELU ? k_act_bwd_v4<MG_ACT_RELU, true> : k_act_bwd_v4<MG_ACT_NONE, true>)
                               : (act == MG_ACT_GELU ? k_act_bwd_v4<MG_ACT_GELU, false> : act == MG_ACT_RELU ? k_act_bwd_v4<MG_ACT_RELU, false> : k_act_bwd_v4<MG_ACT_NONE, false>);
        hipLaunchKernelGGL(kern, dim3(blocks_for(n / 4)), dim3(256), 0, ctx_stream(ctx), dy, z, (uint16_t *)dz16, dz32, (uint32_t)(n / 4),
                           dtype);
        EW_POSTCHECK("mg_ew_act_bwd");
    }
    hipLaunchKernelGGL(k_act_bwd, dim3(blocks_for(n)), dim3(256), 0, ctx_stream(ctx), dy, z, (uint16_t *)dz16, dz32, n,
                       act, dtype);
    EW_POSTCHECK("mg_ew_act_bwd");
}

int mg_ew_col_sum(mg_ctx *ctx, const float *g, float *sums, int64_t ncol, int64_t nrow, int accumulate) {
    EW_PRECHECK("mg_ew_col_sum", g && sums && count_ok(ncol) && nrow > 0 && nrow <= (int64_t)65535 * COL_SUM_ROWS);
    const unsigned chunks = (unsigned)((nrow + COL_SUM_ROWS - 1) / COL_SUM_ROWS);
    if (chunks > 1 && nrow <= COL_SUM_ONE) {
        hipLaunchKernelGGL(k_col_sum_one, dim3((unsigned)((ncol + COL_SUM_ONE_COLS - 1) / COL_SUM_ONE_COLS)), dim3(256), 0, ctx_stream(ctx), g, sums, ncol, nrow,
                           accumulate);
        EW_POSTCHECK("mg_ew_col_sum");
    }
    if (chunks > 1 && !accumulate) hipLaunchKernelGGL(k_zero, dim3(blocks_for(ncol)), dim3(256), 0, ctx_stream(ctx), sums, ncol);
    hipLaunchKernelGGL(k_col_sum, dim3((unsigned)((ncol + 63) / 64), chunks), dim3(512), 0, ctx_stream(ctx), g, sums, ncol,
                       nrow, accumulate, chunks > 1 ? 1 : 0);
    EW_POSTCHECK("mg_ew_col_sum");
}

int mg_ew_copy(mg_ctx *ctx, void *dst, const void *src, int64_t nbytes) {
    EW_PRECHECK("mg_ew_copy", dst && src && count_ok(nbytes) && nbytes % 4 == 0 &&
                                  (((uintptr_t)dst | (uintptr_t)src) & 3) == 0);
    const int64_t nwords = nbytes / 4;
    const int vec = ((((uintptr_t)dst | (uintptr_t)src) & 15) == 0) ? 1 : 0;
    const int64_t threads = vec ? (nwords + 3) / 4 : nwords;
    hipLaunchKernelGGL(k_copy, dim3(blocks_for(threads)), dim3(256), 0, ctx_stream(ctx), (const uint32_t *)src,
                       (uint32_t *)dst, nwords, vec);
    EW_POSTCHECK("mg_ew_copy");
}

int mg_ew_copy_multi(mg_ctx *ctx, void *const *dst, const void *const *src, const int64_t *nbytes, int n) {
    EW_PRECHECK("mg_ew_copy_multi", dst && src && nbytes && n > 0 && n <= MG_COPY_MAX);
    CopyMulti a{};
    int64_t widest = 1;   // workgroups
    for (int i = 0; i < n; i++) {
        if (!dst[i] || !src[i] || !count_ok(nbytes[i]) || (((uintptr_t)dst[i] | (uintptr_t)src[i]) & 3))
            return mg::ctx_fail(MG_ERR_ARG, "mg_ew_copy_multi: bad argument");
        a.src[i] = (const uint32_t *)src[i];
        a.dst[i] = (uint32_t *)dst[i];
        a.bytes[i] = nbytes[i];
        a.vec[i] = (((uintptr_t)dst[i] | (uintptr_t)src[i]) & 15) == 0;
        if (a.vec[i] && nbytes[i] > COPY_WALK_BYTES) {   // (asking takes less than 0.2 us)
            hipPointerAttribute_t at{};
            const hipError_t e = hipPointerGetAttributes(&at, src[i]);
            if (e != hipSuccess) (void)hipGetLastError();
            a.walk[i] = e == hipSuccess && at.type == hipMemoryTypeHost;
        }
        const int64_t blocks = a.walk[i] ? COPY_WALK : blocks_for((nbytes[i] + 15) / 16);
        if (blocks > widest) widest = blocks;
    }
    hipLaunchKernelGGL(k_copy_multi, dim3((unsigned)widest, (unsigned)n), dim3(256), 0, ctx_stream(ctx), a);
    EW_POSTCHECK("mg_ew_copy_multi");
}

int mg_ew_arena_multi(mg_ctx *ctx, const mg_adamw_entry *table_dev, int ntensors, int64_t total_blocks, int pull, float scale) {
    EW_PRECHECK("mg_ew_arena_multi", table_dev && ntensors > 0 && total_blocks > 0 && total_blocks <= 0x7fffffff);
    if (pull) hipLaunchKernelGGL(k_arena_multi<true>, dim3((unsigned)total_blocks), dim3(256), 0, ctx_stream(ctx), table_dev, ntensors, scale);
    else hipLaunchKernelGGL(k_arena_multi<false>, dim3((unsigned)total_blocks), dim3(256), 0, ctx_stream(ctx), table_dev, ntensors, scale);
    EW_POSTCHECK("mg_ew_arena_multi");
}

int mg_ew_softmax_ce(mg_ctx *ctx, const float *logits, const uint32_t *labels, void *dl16, float *dl32, float *loss,
                     int64_t nrows, int64_t stride, int64_t ncls, int dtype) {
    EW_PRECHECK("mg_ew_softmax_ce", logits && labels && loss && count_ok(nrows) && ncls > 0 && stride >= ncls && dtype_ok(dtype) && nrows <= (int64_t)0x7fffffff * 4);
    hipLaunchKernelGGL(k_softmax_ce, dim3((unsigned)((nrows + 3) / 4)), dim3(256), 0, ctx_stream(ctx), logits, labels,
                       (uint16_t *)dl16, dl32, loss, nrows, stride, ncls, dtype);
    EW_POSTCHECK("mg_ew_softmax_ce");
}

int mg_ew_adamw(mg_ctx *ctx, float *w, const float *g, float *m, float *v, void *w16, const float *hp, int64_t n,
                float wd, int dtype) {
    EW_PRECHECK("mg_ew_adamw", w && g && m && v && hp && count_ok(n) && dtype_ok(dtype));
    hipLaunchKernelGGL(k_adamw, dim3(blocks_for(n)), dim3(256), 0, ctx_stream(ctx), w, g, m, v, (uint16_t *)w16, hp, n,
                       wd, dtype);
    EW_POSTCHECK("mg_ew_adamw");
}

int mg_ew_adamw_multi(mg_ctx *ctx, const mg_adamw_entry *table_dev, int ntensors, int64_t total_blocks, const float *hp,
                      int dtype) {
    EW_PRECHECK("mg_ew_adamw_multi", table_dev && ntensors > 0 && total_blocks > 0 && total_blocks <= 0x7fffffff && hp &&
                                         dtype_ok(dtype));
    hipLaunchKernelGGL(k_adamw_multi, dim3((unsigned)total_blocks), dim3(256), 0, ctx_stream(ctx), table_dev, ntensors, hp,
                       dtype);
    EW_POSTCHECK("mg_ew_adamw_multi");
}

int mg_ew_zero_multi(mg_ctx *ctx, const mg_adamw_entry *table_dev, int ntensors, int64_t total_blocks) {
    EW_PRECHECK("mg_ew_zero_multi", table_dev && ntensors > 0 && total_blocks > 0 && total_blocks <= 0x7fffffff);
    hipLaunchKernelGGL(k_zero_multi, dim3((unsigned)total_blocks), dim3(256), 0, ctx_stream(ctx), table_dev, ntensors);
    EW_POSTCHECK("mg_ew_zero_multi");
}

int mg_ew_zero(mg_ctx *ctx, float *dst, int64_t n) {
    EW_PRECHECK("mg_ew_zero", dst && count_ok(n));
    hipLaunchKernelGGL(k_zero, dim3(blocks_for(n)), dim3(256), 0, ctx_stream(ctx), dst, n);
    EW_POSTCHECK("mg_ew_zero");
}

int mg_ew_cast16(mg_ctx *ctx, const float *src, void *dst, int64_t n, int dtype) {
    EW_PRECHECK("mg_ew_cast16", src && dst && count_ok(n) && dtype_ok(dtype));
    if ((((uintptr_t)src & 15) | ((uintptr_t)dst & 7)) == 0)
        hipLaunchKernelGGL(k_cast16_v4, dim3(blocks_for((n + 3) / 4)), dim3(256), 0, ctx_stream(ctx), src, (uint16_t *)dst, n,
                           dtype);
    else
        hipLaunchKernelGGL(k_cast16, dim3(blocks_for(n)), dim3(256), 0, ctx_stream(ctx), src, (uint16_t *)dst, n, dtype);
    EW_POSTCHECK("mg_ew_cast16");
}

int mg_ew_fill_uniform16(mg_ctx *ctx, void *dst, int64_t n, uint32_t seed, int dtype) {
    EW_PRECHECK("mg_ew_fill_uniform16", dst && count_ok(n) && dtype_ok(dtype));
    hipLaunchKernelGGL(k_fill_uniform16, dim3(blocks_for(n)), dim3(256), 0, ctx_stream(ctx), (uint16_t *)dst, n, seed,
                       dtype);
    EW_POSTCHECK("mg_ew_fill_uniform16");
}

int mg_ew_scale_copy(mg_ctx *ctx, float *dst, const float *src, int64_t n, float scale) {
    EW_PRECHECK("mg_ew_scale_copy", dst && src && count_ok(n));
    hipLaunchKernelGGL(k_scale_copy, dim3(blocks_for(n)), dim3(256), 0, ctx_stream(ctx), dst, src, n, scale);
    EW_POSTCHECK("mg_ew_scale_copy");
}

int mg_ew_grad_add(mg_ctx *ctx, float *dst, const float *src, int64_t n) {
    EW_PRECHECK("mg_ew_grad_add", dst && src && count_ok(n));
    hipLaunchKernelGGL(k_grad_add, dim3(blocks_for(n)), dim3(256), 0, ctx_stream(ctx), dst, src, n);
    EW_POSTCHECK("mg_ew_grad_add");
}

}  // extern "C"
