// Shared by the companion kernel files: context access, 16-bit narrowing and widening,
// argument checks of the C entry points.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mi_gemm.h"

struct mg_ctx;
namespace mg {
hipStream_t ctx_stream(mg_ctx *ctx);
int ctx_fail(int code, const char *msg);
int ctx_hip_fail(hipError_t e, const char *what);

__device__ __forceinline__ uint16_t narrow16(float x, int dtype) {
    if (dtype == MG_F16) {
        _Float16 h = (_Float16)x;   // round to nearest even
        return __builtin_bit_cast(uint16_t, h);
    }
    uint32_t u = __builtin_bit_cast(uint32_t, x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;   // NaN
    u += 0x7fffu + ((u >> 16) & 1u);                        // round to nearest even
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float widen16(uint16_t h, int dtype) {
    if (dtype == MG_F16) return (float)__builtin_bit_cast(_Float16, h);
    return __builtin_bit_cast(float, (uint32_t)h << 16);
}

// Two values to 16 bits, round to nearest even, the first in the low half.
template <int DT>
__device__ __forceinline__ uint32_t pack16(float a, float b) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    if constexpr (DT == MG_F16) return __builtin_bit_cast(uint32_t, h2{(_Float16)a, (_Float16)b});
    else return __builtin_bit_cast(uint32_t, b2{(__bf16)a, (__bf16)b});
}

// What all 64 lanes of a wavefront hold, combined by a commutative f (in all of them): with the value 32, 16, 8, 4, 2 and 1
// lanes away in turn, the order - and so the bits - of a butterfly of __shfl_xor, but in VALU moves (v_permlane32_swap, v_permlane16_swap, DPP
// rotations within 16 lanes) instead of six LDS round trips of 100 clocks and more, one behind the other.
template <int CTRL>
__device__ __forceinline__ float wave_dpp(float v) {
    const int i = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, CTRL, 0xf, 0xf, false));
}
template <class F>
__device__ __forceinline__ float wave_all(float v, F f) {
    const auto pair = [&](auto r) { return f(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1])); };
    uint32_t u = __builtin_bit_cast(uint32_t, v);
    v = pair(__builtin_amdgcn_permlane32_swap(u, u, false, false));
    u = __builtin_bit_cast(uint32_t, v);
    v = pair(__builtin_amdgcn_permlane16_swap(u, u, false, false));
    v = f(v, wave_dpp<0x128>(v));   // row_ror:8
    v = f(v, wave_dpp<0x124>(v));   // row_ror:4, of values that repeat every 8 lanes
    v = f(v, wave_dpp<0x4e>(v));    // quad_perm 2 3 0 1
    return f(v, wave_dpp<0xb1>(v)); // quad_perm 1 0 3 2
}
__device__ __forceinline__ float wave_sum(float v) {
    return wave_all(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float wave_max(float v) {
    return wave_all(v, [](float a, float b) { return fmaxf(a, b); });
}

// Column sums: rows of a chunk - several chunks add with atomics -, and how many rows of an f32 matrix one chunk of
// twice the threads takes at the most.  The sums that share a launch with products (gemm_backward_kernel.h) have the same chunks, and so
// the same bits.
constexpr int COL_SUM_ROWS = 512;
constexpr int COL_SUM_ONE = 1024;

static inline unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }
static inline bool dtype_ok(int d) { return d == MG_F16 || d == MG_BF16; }
static inline bool count_ok(int64_t n) { return n > 0 && n <= (int64_t)0x7fffffff * 256; }

}  // namespace mg

#define EW_PRECHECK(name, cond)                                            \
    if (!ctx) return mg::ctx_fail(MG_ERR_ARG, name ": ctx is NULL");       \
    if (!(cond)) return mg::ctx_fail(MG_ERR_ARG, name ": bad argument");
#define EW_POSTCHECK(name)                                                 \
    do {                                                                   \
        hipError_t e_ = hipGetLastError();                                 \
        if (e_ != hipSuccess) return mg::ctx_hip_fail(e_, name);           \
        return MG_OK;                                                      \
    } while (0)
