// What the attention kernels of flash_kernels.hip and flash_small_kernels.hip share: operand types, the
// layout of a tile in LDS, products with it, reductions over a lane's 16 values and between the half-waves.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mi_gemm.h"

#include "ew_common.h"

namespace mg {

typedef _Float16 fk_half8 __attribute__((ext_vector_type(8)));
typedef __bf16 fk_bf8 __attribute__((ext_vector_type(8)));
typedef float fk_f32x16 __attribute__((ext_vector_type(16)));
typedef float fk_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t fk_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t fk_u32x2 __attribute__((ext_vector_type(2)));
typedef short fk_short4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) fk_short4 fk_lds_short4;

template <int DT>
__device__ __forceinline__ fk_f32x16 fk_mfma(fk_u32x4 a, fk_u32x4 b, fk_f32x16 c) {
    if constexpr (DT == MG_F16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(fk_half8, a), __builtin_bit_cast(fk_half8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(fk_bf8, a), __builtin_bit_cast(fk_bf8, b), c, 0, 0, 0);
}
template <int DT>
__device__ __forceinline__ float fk_widen(uint32_t b) {
    if constexpr (DT == MG_F16) return (float)__builtin_bit_cast(_Float16, (uint16_t)b);
    else return __builtin_bit_cast(float, b << 16);
}

// A masked score is -inf (its exponential is 0 against any finite reference), a row that has seen nothing yet refers to a
// finite number far below every score.
#define FK_MASKED (-__builtin_inff())
constexpr float FK_NOTHING = -1e30f;
// Keeps a uniform condition a branch: turned into selects, a mask costs every tile what only the diagonal ones need.
#define FK_BRANCH asm volatile("")
// Values narrowed to pairs, and as they survive that.
template <int DT>
__device__ __forceinline__ void fk_round(float (&e)[16], uint32_t (&w)[8]) {
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
        const uint32_t u = pack16<DT>(e[r], e[r + 1]);
        w[r / 2] = u;
        e[r] = fk_widen<DT>(u & 0xffffu);
        e[r + 1] = fk_widen<DT>(u >> 16);
    }
}
template <int DT>
__device__ __forceinline__ void fk_narrow(const float (&e)[16], uint32_t (&w)[8]) {
#pragma unroll
    for (int r = 0; r < 16; r += 2) w[r / 2] = pack16<DT>(e[r], e[r + 1]);
}

constexpr int FK_BN = 64;   // rows of a staged tile

// Shapes of one instantiation: KK steps of 16 along the head width (zero-filled beyond it).
template <int KK>
struct FkShape {
    static constexpr int MB = (KK + 1) / 2;           // 32-row blocks of an output with the head width along the rows
    static constexpr int W = MB * 32;                 // columns of a staged row
    static constexpr int PITCH = W * 2 + 16;          // its bytes: 16 of padding spread both kinds of reads over the banks
    static constexpr int CPR = W / 8;                 // 16-byte chunks of a row
    static constexpr int NCH = CPR / 4;               // chunks per thread (256) and tile of 64 rows
    static constexpr int TILE = FK_BN * PITCH;
    static constexpr int NBUF = 4 * TILE <= 65536 ? 2 : 1;   // two tensors, double-buffered where a static array allows it
};

// One tile of 64 rows of a (rows, pitch) matrix, on its way to LDS through registers.
template <int KK>
struct FkStage {
    using S = FkShape<KK>;
    fk_u32x4 reg[S::NCH];
    __device__ __forceinline__ void load(const uint16_t *base, int64_t pitch, int row0, int nrows, int hd, int tid) {
#pragma unroll
        for (int i = 0; i < S::NCH; i++) {
            const int c = tid + 256 * i, r = c / S::CPR, ch = c % S::CPR;
            const fk_u32x4 zero = {0u, 0u, 0u, 0u};
            // rows beyond the matrix repeat the last one: what they produce is masked
            reg[i] = ch * 8 < hd ? *reinterpret_cast<const fk_u32x4 *>(base + (int64_t)min(row0 + r, nrows - 1) * pitch + ch * 8) : zero;
        }
    }
    __device__ __forceinline__ void store(char *lds, int tid) const {
#pragma unroll
        for (int i = 0; i < S::NCH; i++) {
            const int c = tid + 256 * i, r = c / S::CPR, ch = c % S::CPR;
            *reinterpret_cast<fk_u32x4 *>(lds + r * S::PITCH + ch * 16) = reg[i];
        }
    }
};

// This lane's row as B operands: k = 16 kk + 8 half .. + 7.
template <int KK>
__device__ __forceinline__ void fk_load_row(fk_u32x4 (&f)[KK], const uint16_t *row, int half, int hd) {
#pragma unroll
    for (int kk = 0; kk < KK; kk++) {
        const fk_u32x4 zero = {0u, 0u, 0u, 0u};
        const int d = kk * 16 + half * 8;
        f[kk] = d < hd ? *reinterpret_cast<const fk_u32x4 *>(row + d) : zero;
    }
}

// 32 rows of a tile (block b) times the rows in registers.
template <int DT, int KK>
__device__ __forceinline__ fk_f32x16 fk_product(const char *lds_rows, const fk_u32x4 (&bf)[KK]) {
    fk_f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.f;
#pragma unroll
    for (int kk = 0; kk < KK; kk++)
        acc = fk_mfma<DT>(*reinterpret_cast<const fk_u32x4 *>(lds_rows + kk * 32), bf[kk], acc);
    return acc;
}

// out += (32 rows of the tile)^T * p; p: this lane's 16 neighbouring rows of its column, narrowed, in pairs.
template <int DT, int KK>
__device__ __forceinline__ void fk_accumulate(fk_f32x16 (&out)[FkShape<KK>::MB], const char *lds_tr, const uint32_t (&p)[8]) {
    using S = FkShape<KK>;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const fk_u32x4 o = {p[4 * u], p[4 * u + 1], p[4 * u + 2], p[4 * u + 3]};
#pragma unroll
        for (int i = 0; i < S::MB; i++) {
            // transposing read (ds_read_b64_tr_b16): 16 lanes supply 4 rows x 16 columns and receive a column each
            const char *a = lds_tr + 8 * u * S::PITCH + i * 64;
            const fk_u32x2 lo = __builtin_bit_cast(fk_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((fk_lds_short4 *)a));
            const fk_u32x2 hi = __builtin_bit_cast(fk_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((fk_lds_short4 *)(a + 4 * S::PITCH)));
            out[i] = fk_mfma<DT>(fk_u32x4{lo[0], lo[1], hi[0], hi[1]}, o, out[i]);
        }
    }
}

// Columns of `o` (head width along the rows, this lane's column) times f, as a row of 16-bit values.
template <int DT, int MB>
__device__ __forceinline__ void fk_store_row16(uint16_t *row, const fk_f32x16 (&o)[MB], float f, int half, int hd) {
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int d = 32 * i + 8 * g + 4 * half;
            if (d < hd)
                *reinterpret_cast<fk_u32x2 *>(row + d) = fk_u32x2{pack16<DT>(o[i][4 * g] * f, o[i][4 * g + 1] * f),
                                                                  pack16<DT>(o[i][4 * g + 2] * f, o[i][4 * g + 3] * f)};
        }
}

// What the two half-waves hold for a column, combined (in both).
template <class F>
__device__ __forceinline__ float fk_both(float x, F f) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return f(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
}
__device__ __forceinline__ float fk_max16(const fk_f32x16 &v) {
    float m[4];
#pragma unroll
    for (int i = 0; i < 4; i++) m[i] = fmaxf(fmaxf(v[i], v[4 + i]), fmaxf(v[8 + i], v[12 + i]));
    return fmaxf(fmaxf(m[0], m[1]), fmaxf(m[2], m[3]));
}
__device__ __forceinline__ float fk_sum16(const float (&v)[16]) {
    float t[4];
#pragma unroll
    for (int i = 0; i < 4; i++) t[i] = (v[i] + v[4 + i]) + (v[8 + i] + v[12 + i]);
    return (t[0] + t[1]) + (t[2] + t[3]);
}

// sum over d of g16[d] out32[d] for this lane's row, its half of the columns; both halves hold the sum
template <int DT, int KK>
__device__ __forceinline__ float fk_row_term(const fk_u32x4 (&g)[KK], const float *row, int half, int hd) {
    float t = 0.f;
#pragma unroll
    for (int kk = 0; kk < KK; kk++) {
        const int d = kk * 16 + half * 8;
        if (d < hd) {
            const fk_f32x4 x = *reinterpret_cast<const fk_f32x4 *>(row + d), y = *reinterpret_cast<const fk_f32x4 *>(row + d + 4);
#pragma unroll
            for (int w = 0; w < 4; w++) {
                const float lo = fk_widen<DT>(g[kk][w] & 0xffffu), hi = fk_widen<DT>(g[kk][w] >> 16);
                t += w < 2 ? lo * x[2 * w] + hi * x[2 * w + 1] : lo * y[2 * w - 4] + hi * y[2 * w - 3];
            }
        }
    }
    return fk_both(t, [](float a, float b) { return a + b; });
}

// Where the lanes of a wavefront read a tile: block b's rows as A operands, and transposed.
struct FkLane {
    int lane, wave, n, half, arow, trow, tcol;
    __device__ __forceinline__ FkLane() {
        lane = threadIdx.x & 63;
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        n = lane & 31;
        half = lane >> 5;
        arow = 16 * ((n >> 2) & 1) + 4 * (n >> 3) + (n & 3);
        const int j = lane & 15, g4 = lane >> 4;
        trow = (g4 >> 1) * 16 + (j >> 2);
        tcol = (g4 & 1) * 16 + (j & 3) * 4;
    }
};

struct FkArgs {
    const uint16_t *qkv;        // (B*T, 3D)
    const uint32_t *seg;        // (B*T) or NULL
    uint16_t *out16;            // (B*T, D)                      forward
    float *out32;               // (B*T, D)                      forward writes, backward reads
    float *lse;                 // (B*H, T)
    const uint16_t *dout;       // (B*T, D)                      backward
    float *dsum;                // (B*H, T): row term            dQ writes, dK / dV reads
    uint16_t *dqkv;             // (B*T, 3D)
    int T, H, hd;
    float scale;
};

// Steps of 16 along the head width that an instantiation exists for.
static inline int fk_steps(int64_t hd) { return hd <= 16 ? 1 : hd <= 32 ? 2 : hd <= 64 ? 4 : hd <= 96 ? 6 : 8; }

// flash_small_kernels.hip: a workgroup a block of 32 rows, where that many workgroups are no more than the chip holds.
bool fk_small_forward(const FkArgs &a, int64_t nbh);
bool fk_small_backward(const FkArgs &a, int64_t nbh);
void fk_small_launch(hipStream_t s, const FkArgs &a, int64_t nbh, int dtype, bool backward);

}  // namespace mg
