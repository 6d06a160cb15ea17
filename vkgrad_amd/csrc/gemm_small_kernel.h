// Products that take microseconds: the plan of the 64 x 64 tile - its K slices, and the order in which each adds up - run with
// a wavefront a slice instead of a workgroup a slice.
//
// A workgroup owns 32 x 32 outputs; wavefront s takes K slice s, asks for the operands of four K-blocks of 64 at once (two where B comes
// element by element; the rule that takes a product keeps most slices to that) and multiplies them without meeting anybody:
// K-contiguous operands go from memory straight into MFMA fragments, the N-contiguous B of layout NN through a few kilobytes of LDS of the wavefront's own, read back transposed.
// The partial sums meet in LDS, added in slice order, and one wavefront runs the usual epilogue: the bits are those of the
// slices that meet in the workspace, without its round trip through memory, its counter and its waiting.
//
// Bound by latency: one load, a chain of MFMAs, one meeting, one store.
// Measured (f16, in a recorded step, us, a workgroup a slice / this): 128 x 512 x 784 in five slices 9.0 / 7.0, 33 rows 8.2 / 7.1, 128 x
// 10 x 512 in four, B in rows of 20 bytes, 9.0 / 6.5; the MNIST MLP step 88.9 / 83.7, its prediction of 33 rows 43.3 / 38.6.
// The quarter tiles read every operand twice as often as 64 x 64 ones: only where the chip is nearly empty.
#pragma once
#include "gemm_kernel.h"

namespace mg {

constexpr int SMALL_MAX_SPLIT = 8;
constexpr int SMALL_PITCH = 80;                       // bytes of a row of 32 columns of B in LDS
constexpr int SMALL_WAVE_LDS = 64 * SMALL_PITCH;      // a K-block of B, then 32 x 32 partial sums
static_assert(SMALL_WAVE_LDS >= 32 * 32 * 4, "partial sums take the place of the staged block");

// One 64-wide K-block on its way: the fragments of K-contiguous operands, or pieces of rows of B.
// ANY: a B of any alignment, element by element (A is in 16-byte pieces all the same).
template <int LAYOUT, bool ANY>
struct SmallBlock {
    u32x4 a[4], b[4];
    // eight consecutive elements, all or none of them there
    static __device__ __forceinline__ u32x4 piece(const uint16_t *p, bool there) {
        const u32x4 zero = {0u, 0u, 0u, 0u};
        return there ? *reinterpret_cast<const u32x4 *>(p) : zero;
    }
    // eight elements `stride` apart, those from `valid` on zero; without branches, so that all loads of a block are on their
    // way together (what is beyond the last repeats it)
    static __device__ __forceinline__ u32x4 elements(const uint16_t *p, int64_t stride, int valid) {
        uint32_t x[8];
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = p[(valid > e ? e : valid - 1) * stride];
        u32x4 v = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int e = 0; e < 8; e++) v[e >> 1] |= (valid > e ? x[e] : 0u) << (16 * (e & 1));
        return v;
    }
    // arow: this lane's row of A; b: NT this lane's row of B, NN B itself (ANY: from this lane's column)
    __device__ __forceinline__ void load(const GemmParams &p, const uint16_t *arow, const uint16_t *bsrc, int k0, int len, int n0,
                                         int lane) {
        const int half = lane >> 5;
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            const int k = 16 * kk + 8 * half;
            a[kk] = piece(arow + k0 + k, k < len);
            if constexpr (ANY) b[kk] = elements(bsrc + (int64_t)(k0 + k) * (LAYOUT == L_NT ? 1 : p.ldb), LAYOUT == L_NT ? 1 : p.ldb, len - k);
            else if constexpr (LAYOUT == L_NT) b[kk] = piece(bsrc + k0 + k, k < len);
            else {
                const int c = lane + 64 * kk, r = c >> 2;
                const u32x4 zero = {0u, 0u, 0u, 0u};
                // (columns beyond the matrix repeat the last piece: they are not stored)
                b[kk] = r < len ? *reinterpret_cast<const u32x4 *>(bsrc + (int64_t)(k0 + r) * p.ldb + min(n0 + 8 * (c & 3), p.N - 8)) : zero;
            }
        }
    }
    template <int DT>
    __device__ __forceinline__ void multiply(f32x16 &acc, char *lds, int lane) const {
        if constexpr (LAYOUT == L_NT || ANY) {
#pragma unroll
            for (int kk = 0; kk < 4; kk++) acc = mfma32<DT>(a[kk], b[kk], acc);
        } else {
            // (LDS accesses of one wavefront complete in order)
            asm volatile("" ::: "memory");
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                const int c = lane + 64 * kk;
                *reinterpret_cast<u32x4 *>(lds + (c >> 2) * SMALL_PITCH + (c & 3) * 16) = b[kk];
            }
            asm volatile("" ::: "memory");
            // 16 lanes supply 4 rows x 16 columns and receive a column each
            const int g = lane >> 4, j = lane & 15;
            const char *at = lds + (8 * (g >> 1) + (j >> 2)) * SMALL_PITCH + ((g & 1) * 16 + (j & 3) * 4) * 2;
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                const u32x2 lo = lds_read_tr((const uint16_t *)(at + 16 * kk * SMALL_PITCH));
                const u32x2 hi = lds_read_tr((const uint16_t *)(at + (16 * kk + 4) * SMALL_PITCH));
                acc = mfma32<DT>(a[kk], u32x4{lo[0], lo[1], hi[0], hi[1]}, acc);
            }
            asm volatile("" ::: "memory");
        }
    }
};

template <int LAYOUT, int DT, bool ANY, bool ACT>
__global__ void __launch_bounds__(64 * SMALL_MAX_SPLIT)
gemm_small_kernel(const GemmParams p) {
    static_assert(LAYOUT != L_TN, "A is K-contiguous");
    extern __shared__ __attribute__((aligned(16))) char dsm[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nbn = (p.N + 31) / 32, m0 = (int)(blockIdx.x / nbn) * 32, n0 = (int)(blockIdx.x % nbn) * 32;
    const int kbeg = wave * p.k_per_split, kend = min(p.K, kbeg + p.k_per_split);
    const uint16_t *arow = p.A + (int64_t)min(m0 + (lane & 31), p.M - 1) * p.lda;
    const int col = min(n0 + (lane & 31), p.N - 1);
    const uint16_t *bsrc = LAYOUT == L_NT ? p.B + (int64_t)col * p.ldb : ANY ? p.B + col : p.B;
    char *lds = dsm + wave * SMALL_WAVE_LDS;
    // the blocks in the order of the kernels with direct loads (what is left of K first) or of the register-staged ones (last)
    const int rem = ANY ? 0 : (kend - kbeg) & 63, first = rem ? 1 : 0, nblk = first + (kend - kbeg - rem + 63) / 64;
    constexpr int CH = ANY ? 2 : 4;
    f32x16 acc[1][1];
#pragma unroll
    for (int r = 0; r < 16; r++) acc[0][0][r] = 0.f;
    for (int c = 0; c < nblk; c += CH) {
        SmallBlock<LAYOUT, ANY> blk[CH];
#pragma unroll
        for (int i = 0; i < CH; i++)
            if (c + i < nblk) {
                const bool is_rem = c + i < first;
                const int k0 = is_rem ? kbeg : kbeg + rem + (c + i - first) * 64;
                blk[i].load(p, arow, bsrc, k0, is_rem ? rem : min(64, kend - k0), n0, lane);
            }
#pragma unroll
        for (int i = 0; i < CH; i++)
            if (c + i < nblk) blk[i].template multiply<DT>(acc[0][0], lds, lane);
    }
    {
        f32x4 *mine = reinterpret_cast<f32x4 *>(lds) + lane;
#pragma unroll
        for (int g = 0; g < 4; g++) mine[64 * g] = f32x4{acc[0][0][4 * g], acc[0][0][4 * g + 1], acc[0][0][4 * g + 2], acc[0][0][4 * g + 3]};
        __syncthreads();
        if (wave > 0) return;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[0][0][r] = 0.f;
        for (int s = 0; s < p.split_k; s++) {
            const f32x4 *part = reinterpret_cast<const f32x4 *>(dsm + s * SMALL_WAVE_LDS) + lane;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const f32x4 t = part[64 * g];
#pragma unroll
                for (int e = 0; e < 4; e++) acc[0][0][4 * g + e] += t[e];
            }
        }
    }
    store_tile<DT, 1, 1, 32, 32, ACT>(p, p.C, acc, m0, n0, 0, 0, lane, p.bias != nullptr, p.beta ? 1 : 0,
                                      m0 + 32 <= p.M && n0 + 32 <= p.N);
}

template <int LAYOUT, int DT, bool ANY, bool ACT>
hipError_t launch_gemm_small(const GemmParams &p, hipStream_t stream, KernelQuery *query) {
    auto kern = gemm_small_kernel<LAYOUT, DT, ANY, ACT>;
    const int lds = p.split_k * SMALL_WAVE_LDS;
    if (query) return query_kernel((const void *)kern, 64 * p.split_k, lds, query);
    const unsigned grid = (unsigned)(((p.M + 31) / 32) * ((p.N + 31) / 32));
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * p.split_k), lds, stream, p);
    return hipGetLastError();
}
static_assert(SMALL_MAX_SPLIT * SMALL_WAVE_LDS <= 65536, "dynamic LDS needs no attribute");

typedef hipError_t (*small_launch_fn)(const GemmParams &, hipStream_t, KernelQuery *);
// [layout NN, NT][dtype][any alignment][fused 16-bit output]
extern small_launch_fn small_table[2][2][2][2];

}  // namespace mg
