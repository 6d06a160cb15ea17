// Causal attention without the (T, T) matrices (flash_kernels.hip) for calls that leave the chip idle there: a workgroup owns
// 32 rows of one side instead of 128, and its four wavefronts share out the other side, every fourth block of 32 rows each.
// They meet twice: forward with the maximum and sum of their keys, and in both directions with their part of the output,
// added in wavefront order.  No tile is shared, so there is no barrier in the walk: a wavefront passes its blocks through LDS
// of its own, the next one on its way in registers.
//
// Forward, the scores of a row stay in registers between the sum and P V (16 registers a block; up to NB blocks a
// wavefront, T <= 128 NB): one walk over the keys, and P is exp2(score - lse), narrowed, as in flash_kernels.hip and as the backward pass rebuilds it.
// Backward, dQ and dK / dV are one launch; the row term, which the dQ kernel of flash_kernels.hip leaves for
// the dK / dV kernel behind it, is formed by both.
//
// Bound by the chain from one block to the next, an eighth as long as with 128 rows a workgroup and all blocks in turn, against
// four times the operand traffic from L2.
// Measured (us, between others of its kind, this / flash_kernels.hip): 2 heads x 1024 x 64 forward 12.3 / 28.8, backward 21.4 / 52.4; 5 x
// 333, 6 of 64 9.1 / 15.0 and 17.1 / 26.7; 2 x 64, 4 of 16 4.3 / 5.3 and 5.4 / 8.2; 4 x 512, 8 of 32, packed, 8.7 / 20.9 and 16.5 / 39.9.
#include "flash_common.h"

namespace mg {

// LDS accesses of one wavefront complete in order; this keeps the compiler from moving them across.
#define FK_WAVE_FENCE asm volatile("" ::: "memory")

// One block of 32 rows on its way to a wavefront's own LDS.
template <int KK>
struct FkBlock {
    using S = FkShape<KK>;
    static constexpr int N = S::CPR / 2;
    fk_u32x4 reg[N];
    __device__ __forceinline__ void load(const uint16_t *base, int64_t pitch, int row0, int nrows, int hd, int lane) {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int c = lane + 64 * i, r = c / S::CPR, ch = c % S::CPR;
            const fk_u32x4 zero = {0u, 0u, 0u, 0u};
            // rows beyond the matrix repeat the last one: what they produce is masked
            reg[i] = ch * 8 < hd ? *reinterpret_cast<const fk_u32x4 *>(base + (int64_t)min(row0 + r, nrows - 1) * pitch + ch * 8) : zero;
        }
    }
    __device__ __forceinline__ void store(char *lds, int lane) const {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int c = lane + 64 * i, r = c / S::CPR, ch = c % S::CPR;
            *reinterpret_cast<fk_u32x4 *>(lds + r * S::PITCH + ch * 16) = reg[i];
        }
    }
};

template <int KK>
constexpr int fk_block_bytes() { return 32 * FkShape<KK>::PITCH; }
constexpr int FK_MEET = 4 * 8 * 64 * 16;   // four wavefronts, eight groups of four values a lane

// The four wavefronts' parts of an output (head width along the rows, this lane's column), added up in wavefront order; every
// wavefront passes its share of the sums to put(d, values).  lds: FK_MEET bytes, free for everybody on entry.
template <int MB, class F>
__device__ __forceinline__ void fk_meet(const fk_f32x16 (&o)[MB], char *lds, const FkLane &L, F put) {
    fk_f32x4 *m = reinterpret_cast<fk_f32x4 *>(lds);
#pragma unroll
    for (int i0 = 0; i0 < MB; i0 += 2) {
        const int nb = MB - i0 < 2 ? 1 : 2;
        if (i0) __syncthreads();
#pragma unroll
        for (int k = 0; k < 4 * nb; k++) {
            const fk_f32x16 &v = o[i0 + k / 4];
            const int g = k % 4;
            m[(L.wave * 8 + k) * 64 + L.lane] = fk_f32x4{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < nb; j++) {
            const int k = L.wave * nb + j;
            fk_f32x4 t = m[k * 64 + L.lane];
#pragma unroll
            for (int w = 1; w < 4; w++) {
                const fk_f32x4 u = m[(w * 8 + k) * 64 + L.lane];
#pragma unroll
                for (int e = 0; e < 4; e++) t[e] += u[e];
            }
            put(32 * (i0 + k / 4) + 8 * (k % 4) + 4 * L.half, t);
        }
    }
}
template <int DT>
__device__ __forceinline__ void fk_put16(uint16_t *row, int d, const fk_f32x4 &v, int hd) {
    if (d < hd) *reinterpret_cast<fk_u32x2 *>(row + d) = fk_u32x2{pack16<DT>(v[0], v[1]), pack16<DT>(v[2], v[3])};
}
__device__ __forceinline__ int fk_first_block(int first) {
    int f = first;
#pragma unroll
    for (int m = 16; m >= 1; m >>= 1) f = min(f, __shfl_xor(f, m, 64));
    return __builtin_amdgcn_readfirstlane(f) / 32;
}

// ---- forward -------------------------------------------------------------------------
template <int DT, int KK, int NB>
__global__ void __launch_bounds__(256, 2)
k_flash_fwd_row(const FkArgs p) {
    using S = FkShape<KK>;
    constexpr int VB = 4 * fk_block_bytes<KK>();
    __shared__ __attribute__((aligned(16))) char smem[VB > FK_MEET ? VB : FK_MEET];
    __shared__ float st_m[4][32], st_l[4][32];
    const FkLane L;
    const int T = p.T, hd = p.hd, D = p.H * hd;
    const int b = blockIdx.x / p.H, h = blockIdx.x % p.H;
    const int yb = gridDim.y - 1 - blockIdx.y, i0 = yb * 32;   // the long rows first
    const int q = i0 + L.n, qc = min(q, T - 1);
    const int64_t pitch = 3 * (int64_t)D;
    const uint16_t *qb = p.qkv + (int64_t)b * T * pitch + h * hd, *kb = qb + D, *vb = kb + D;
    const int first = p.seg ? (int)p.seg[(int64_t)b * T + qc] : 0;
    const int b0 = (p.seg ? fk_first_block(first) : 0) + L.wave;   // this wavefront: blocks b0, b0 + 4, ... up to yb
    fk_u32x4 qf[KK], kf[2][KK];
    fk_load_row<KK>(qf, qb + qc * pitch, L.half, hd);
    auto load_k = [&](fk_u32x4 (&f)[KK], int blk) {
        fk_load_row<KK>(f, kb + (int64_t)min(blk * 32 + L.arow, T - 1) * pitch, L.half, hd);
    };
    if (b0 <= yb) load_k(kf[0], b0);
    fk_f32x16 s[NB];
    float mt = FK_MASKED;
#pragma unroll
    for (int t = 0; t < NB; t++) {
        const int blk = b0 + 4 * t;
        if (blk <= yb) {
            if (t + 1 < NB && blk + 4 <= yb) load_k(kf[(t + 1) & 1], blk + 4);
            fk_f32x16 acc;
#pragma unroll
            for (int r = 0; r < 16; r++) acc[r] = 0.f;
#pragma unroll
            for (int kk = 0; kk < KK; kk++) acc = fk_mfma<DT>(kf[t & 1][kk], qf[kk], acc);
            if (p.seg || blk == yb) {
                FK_BRANCH;
                const int lo = first - blk * 32 - 16 * L.half, hi = q - blk * 32 - 16 * L.half;
#pragma unroll
                for (int r = 0; r < 16; r++) acc[r] = (r <= hi && r >= lo) ? acc[r] : FK_MASKED;
            }
            mt = fmaxf(mt, fk_max16(acc));
            s[t] = acc;
        }
    }
    FkBlock<KK> vs;
    if (b0 <= yb) vs.load(vb, pitch, b0 * 32, T, hd, L.lane);
    const float c2 = p.scale * 1.4426950408889634f;   // base 2: an exponential is one v_exp_f32
    mt = fk_both(mt, [](float x, float y) { return fmaxf(x, y); });
    const float mw = fmaxf(mt * c2, FK_NOTHING);
    float l = 0.f;
#pragma unroll
    for (int t = 0; t < NB; t++)
        if (b0 + 4 * t <= yb) {
            float e[16];
#pragma unroll
            for (int r = 0; r < 16; r++) e[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][r], c2, -mw));
            l += fk_sum16(e);
        }
    l = fk_both(l, [](float x, float y) { return x + y; });
    st_m[L.wave][L.n] = mw;
    st_l[L.wave][L.n] = l;
    __syncthreads();
    float m = mw;
#pragma unroll
    for (int w = 0; w < 4; w++) m = fmaxf(m, st_m[w][L.n]);
    l = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) l += st_l[w][L.n] * __builtin_amdgcn_exp2f(st_m[w][L.n] - m);
    const float lse = m + __builtin_amdgcn_logf(l);
    fk_f32x16 o[S::MB];
#pragma unroll
    for (int i = 0; i < S::MB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[i][r] = 0.f;
    char *vt = smem + L.wave * fk_block_bytes<KK>();
#pragma unroll
    for (int t = 0; t < NB; t++) {
        const int blk = b0 + 4 * t;
        if (blk <= yb) {
            FK_WAVE_FENCE;
            vs.store(vt, L.lane);
            FK_WAVE_FENCE;
            if (t + 1 < NB && blk + 4 <= yb) vs.load(vb, pitch, (blk + 4) * 32, T, hd, L.lane);
            float e[16];   // the very P that the backward pass rebuilds
#pragma unroll
            for (int r = 0; r < 16; r++) e[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][r], c2, -lse));
            uint32_t w[8];
            fk_narrow<DT>(e, w);
            fk_accumulate<DT, KK>(o, vt + L.trow * S::PITCH + L.tcol * 2, w);
        }
    }
    if (L.wave == 0 && L.half == 0 && q < T) p.lse[(int64_t)blockIdx.x * T + q] = lse;
    __syncthreads();
    const int64_t row = ((int64_t)b * T + q) * D + h * hd;
    fk_meet<S::MB>(o, smem, L, [&](int d, const fk_f32x4 &v) {
        if (q >= T || d >= hd) return;
        fk_put16<DT>(p.out16 + row, d, v, hd);
        if (p.out32) *reinterpret_cast<fk_f32x4 *>(p.out32 + row + d) = v;
    });
}

// ---- backward ------------------------------------------------------------------------
template <int DT, int KK>
__device__ __forceinline__ void fk_dq_row(const FkArgs &p, char *smem, int yb) {
    using S = FkShape<KK>;
    const FkLane L;
    const int T = p.T, hd = p.hd, D = p.H * hd;
    const int b = blockIdx.x / p.H, h = blockIdx.x % p.H;
    const int i0 = yb * 32, q = i0 + L.n, qc = min(q, T - 1);
    const int64_t pitch = 3 * (int64_t)D;
    const uint16_t *qb = p.qkv + (int64_t)b * T * pitch + h * hd, *kb = qb + D, *vb = kb + D;
    const int64_t orow = ((int64_t)b * T + qc) * D + h * hd;
    const int first = p.seg ? (int)p.seg[(int64_t)b * T + qc] : 0;
    int blk = (p.seg ? fk_first_block(first) : 0) + L.wave;
    FkBlock<KK> ks, vs;
    if (blk <= yb) {
        ks.load(kb, pitch, blk * 32, T, hd, L.lane);
        vs.load(vb, pitch, blk * 32, T, hd, L.lane);
    }
    fk_u32x4 qf[KK], gf[KK];
    fk_load_row<KK>(qf, qb + qc * pitch, L.half, hd);
    fk_load_row<KK>(gf, p.dout + orow, L.half, hd);
    const int64_t stat = (int64_t)blockIdx.x * T + qc;
    const float lse = p.lse[stat], dsum = fk_row_term<DT, KK>(gf, p.out32 + orow, L.half, hd);
    const float dscaled = dsum * p.scale;
    if (L.wave == 0 && L.half == 0 && q < T) p.dsum[stat] = dsum;
    const float c2 = p.scale * 1.4426950408889634f;
    fk_f32x16 o[S::MB];
#pragma unroll
    for (int i = 0; i < S::MB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[i][r] = 0.f;
    char *kt = smem + L.wave * 2 * fk_block_bytes<KK>(), *vt = kt + fk_block_bytes<KK>();
    for (; blk <= yb; blk += 4) {
        FK_WAVE_FENCE;
        ks.store(kt, L.lane);
        vs.store(vt, L.lane);
        FK_WAVE_FENCE;
        if (blk + 4 <= yb) {
            ks.load(kb, pitch, (blk + 4) * 32, T, hd, L.lane);
            vs.load(vb, pitch, (blk + 4) * 32, T, hd, L.lane);
        }
        const fk_f32x16 s = fk_product<DT, KK>(kt + L.arow * S::PITCH + L.half * 16, qf);
        const fk_f32x16 dp = fk_product<DT, KK>(vt + L.arow * S::PITCH + L.half * 16, gf);
        float e[16];
#pragma unroll
        for (int r = 0; r < 16; r++) e[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c2, -lse));
        uint32_t w[8];
        fk_round<DT>(e, w);   // P as the forward pass multiplied it
#pragma unroll
        for (int r = 0; r < 16; r++) e[r] *= __builtin_fmaf(dp[r], p.scale, -dscaled);
        if (p.seg || blk == yb) {
            FK_BRANCH;
            const int hi = q - blk * 32 - 16 * L.half, lo = first - blk * 32 - 16 * L.half;
#pragma unroll
            for (int r = 0; r < 16; r++) e[r] = (r <= hi && r >= lo) ? e[r] : 0.f;
        }
        fk_narrow<DT>(e, w);
        fk_accumulate<DT, KK>(o, kt + L.trow * S::PITCH + L.tcol * 2, w);
    }
    __syncthreads();
    uint16_t *row = p.dqkv + ((int64_t)b * T + qc) * pitch + h * hd;
    fk_meet<S::MB>(o, smem, L, [&](int d, const fk_f32x4 &v) {
        if (q < T) fk_put16<DT>(row, d, v, hd);
    });
}

template <int DT, int KK>
__device__ __forceinline__ void fk_dkv_row(const FkArgs &p, char *smem, float (&st)[4][3][32], int jb, int nblk) {
    using S = FkShape<KK>;
    const FkLane L;
    const int T = p.T, hd = p.hd, D = p.H * hd;
    const int b = blockIdx.x / p.H, h = blockIdx.x % p.H;
    const int j0 = jb * 32, key = j0 + L.n, kc = min(key, T - 1);
    const int64_t pitch = 3 * (int64_t)D;
    const uint16_t *qb = p.qkv + (int64_t)b * T * pitch + h * hd, *kb = qb + D, *vb = kb + D;
    const uint16_t *gb = p.dout + (int64_t)b * T * D + h * hd;
    int blk = jb + L.wave;
    FkBlock<KK> qs, gs;
    if (blk < nblk) {
        qs.load(qb, pitch, blk * 32, T, hd, L.lane);
        gs.load(gb, D, blk * 32, T, hd, L.lane);
    }
    fk_u32x4 kf[KK], vf[KK];
    fk_load_row<KK>(kf, kb + kc * pitch, L.half, hd);
    fk_load_row<KK>(vf, vb + kc * pitch, L.half, hd);
    const float c2 = p.scale * 1.4426950408889634f;
    fk_f32x16 dk[S::MB], dv[S::MB];
#pragma unroll
    for (int i = 0; i < S::MB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) dk[i][r] = dv[i][r] = 0.f;
    char *qt = smem + L.wave * 2 * fk_block_bytes<KK>(), *gt = qt + fk_block_bytes<KK>();
    float *lse = st[L.wave][0], *dsum = st[L.wave][1], *seg = st[L.wave][2];
    for (; blk < nblk; blk += 4) {
        const int i0 = blk * 32, rq = min(i0 + L.n, T - 1);
        // (this block's, while the next one's rows are on their way)
        fk_u32x4 gr[KK];
        fk_load_row<KK>(gr, gb + (int64_t)rq * D, L.half, hd);
        const float r_lse = p.lse[(int64_t)blockIdx.x * T + rq];
        const int r_first = p.seg ? (int)p.seg[(int64_t)b * T + rq] : 0;
        FK_WAVE_FENCE;
        qs.store(qt, L.lane);
        gs.store(gt, L.lane);
        FK_WAVE_FENCE;
        if (blk + 4 < nblk) {
            qs.load(qb, pitch, (blk + 4) * 32, T, hd, L.lane);
            gs.load(gb, D, (blk + 4) * 32, T, hd, L.lane);
        }
        const float r_d = fk_row_term<DT, KK>(gr, p.out32 + ((int64_t)b * T + rq) * D + h * hd, L.half, hd);
        lse[L.n] = r_lse;
        dsum[L.n] = r_d * p.scale;
        seg[L.n] = __builtin_bit_cast(float, r_first);
        FK_WAVE_FENCE;
        const fk_f32x16 s = fk_product<DT, KK>(qt + L.arow * S::PITCH + L.half * 16, kf);
        const fk_f32x16 dp = fk_product<DT, KK>(gt + L.arow * S::PITCH + L.half * 16, vf);
        float e[16], ds[16];
#pragma unroll
        for (int r = 0; r < 16; r++) e[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c2, -lse[16 * L.half + r]));
        if (p.seg || blk == jb || i0 + 31 >= T) {
            FK_BRANCH;
            const int lo = key - i0 - 16 * L.half, hi = T - 1 - i0 - 16 * L.half;
#pragma unroll
            for (int r = 0; r < 16; r++)
                e[r] = (r >= lo && r <= hi && key >= __builtin_bit_cast(int, seg[16 * L.half + r])) ? e[r] : 0.f;
        }
        uint32_t we[8], wd[8];
        fk_round<DT>(e, we);
#pragma unroll
        for (int r = 0; r < 16; r++) ds[r] = e[r] * __builtin_fmaf(dp[r], p.scale, -dsum[16 * L.half + r]);
        fk_narrow<DT>(ds, wd);
        fk_accumulate<DT, KK>(dv, gt + L.trow * S::PITCH + L.tcol * 2, we);
        fk_accumulate<DT, KK>(dk, qt + L.trow * S::PITCH + L.tcol * 2, wd);
    }
    uint16_t *row = p.dqkv + ((int64_t)b * T + kc) * pitch + h * hd;
    __syncthreads();
    fk_meet<S::MB>(dk, smem, L, [&](int d, const fk_f32x4 &v) {
        if (key < T) fk_put16<DT>(row + D, d, v, hd);
    });
    __syncthreads();
    fk_meet<S::MB>(dv, smem, L, [&](int d, const fk_f32x4 &v) {
        if (key < T) fk_put16<DT>(row + 2 * D, d, v, hd);
    });
}

template <int DT, int KK>
__global__ void __launch_bounds__(256, (KK <= 4 ? 2 : 1))
k_flash_bwd_row(const FkArgs p) {
    constexpr int TB = 8 * fk_block_bytes<KK>();
    __shared__ __attribute__((aligned(16))) char smem[TB > FK_MEET ? TB : FK_MEET];
    __shared__ __attribute__((aligned(16))) float st[4][3][32];
    // the longest first: the keys that most queries see, the queries that see most keys
    const int nblk = gridDim.y / 2, y = blockIdx.y / 2;
    if (blockIdx.y % 2 == 0) fk_dkv_row<DT, KK>(p, smem, st, y, nblk);
    else fk_dq_row<DT, KK>(p, smem, nblk - 1 - y);
}

// The line is where four times the operand traffic costs more than idle CUs, in blocks of 32 rows.  Forward (us, here / 128 rows a
// workgroup): 512 blocks (16 x 128, 8 of 64) 7.4 / 10.2, 696 (3 x 900, 8 of 80) 24 / 36, 1024 (8 x 512, 8 of 64) 16.6 / 20.2.  2048
// (64 x 256, 4 of 64) 20.5 / 18.9, 2048 (4 x 1024, 16 of 64) 43 / 35.  Scores of more than 1024 keys do not fit a row's registers.
bool fk_small_forward(const FkArgs &a, int64_t nbh) { return a.T <= 1024 && nbh * ((a.T + 31) / 32) <= 1024; }
// Backward a block is two workgroups, of which a CU holds two with heads of up to 64 and one with wider ones (324 registers): the
// rounds are 256 and 128 blocks, and more of them are worth it the longer a row is, whose chain they shorten, and in packed rows, where
// 128 rows walk the tiles of the earliest of them.  Where 128 rows a workgroup overtake (their time over this one's; 32 to 1024 rows,
// 128 to 512 blocks, bf16): heads of 32 nowhere (512 blocks of 64 rows 0.95, of 256 1.28); of 64, 64 rows 256 blocks 1.19, 320 0.90, 96 rows
// 312 1.09, 384 0.96 (packed 504 1.02), 128 rows 512 0.99; of 80, 64 rows 128 blocks 1.39, 192 0.89, 128 rows 256 1.18, 320 0.92 (packed
// 1.03), 256 rows 320 1.08, 384 0.99, 448 0.84 (packed 1.04), 512 rows 384 1.17, 448 0.97, packed 512 1.14.  The tiles of four wavefronts for heads
// wider than 96 do not fit static LDS.
static int fk_small_backward_most(int steps, int T, bool packed) {
    if (steps <= 2) return 512;
    if (steps == 4) return T <= 64 ? 256 : T < 128 && !packed ? 320 : 512;
    if (steps > 6) return 0;
    if (T < 96) return 128;
    if (T < 256) return packed && T >= 128 ? 320 : 256;
    return T < 384 ? (packed ? 448 : 320) : packed ? 512 : 384;
}
bool fk_small_backward(const FkArgs &a, int64_t nbh) {
    return nbh * ((a.T + 31) / 32) <= fk_small_backward_most(fk_steps(a.hd), a.T, a.seg != nullptr);
}

template <int DT, int KK>
static void fk_small_forward_launch(hipStream_t s, const FkArgs &a, dim3 grid) {
    if (a.T <= 128) hipLaunchKernelGGL((k_flash_fwd_row<DT, KK, 1>), grid, dim3(256), 0, s, a);
    else if (a.T <= 256) hipLaunchKernelGGL((k_flash_fwd_row<DT, KK, 2>), grid, dim3(256), 0, s, a);
    else if (a.T <= 512) hipLaunchKernelGGL((k_flash_fwd_row<DT, KK, 4>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((k_flash_fwd_row<DT, KK, 8>), grid, dim3(256), 0, s, a);
}
template <int DT, int KK>
static void fk_small_launch_as(hipStream_t s, const FkArgs &a, int64_t nbh, bool backward) {
    const unsigned nblk = (unsigned)((a.T + 31) / 32);
    if (!backward) fk_small_forward_launch<DT, KK>(s, a, dim3((unsigned)nbh, nblk));
    else if constexpr (KK <= 6) hipLaunchKernelGGL((k_flash_bwd_row<DT, KK>), dim3((unsigned)nbh, 2 * nblk), dim3(256), 0, s, a);
}
template <int DT>
static void fk_small_launch_width(hipStream_t s, const FkArgs &a, int64_t nbh, bool backward) {
    switch (fk_steps(a.hd)) {
    case 1: return fk_small_launch_as<DT, 1>(s, a, nbh, backward);
    case 2: return fk_small_launch_as<DT, 2>(s, a, nbh, backward);
    case 4: return fk_small_launch_as<DT, 4>(s, a, nbh, backward);
    case 6: return fk_small_launch_as<DT, 6>(s, a, nbh, backward);
    default: return fk_small_launch_as<DT, 8>(s, a, nbh, backward);
    }
}
void fk_small_launch(hipStream_t s, const FkArgs &a, int64_t nbh, int dtype, bool backward) {
    if (dtype == MG_F16) fk_small_launch_width<MG_F16>(s, a, nbh, backward);
    else fk_small_launch_width<MG_BF16>(s, a, nbh, backward);
}

}  // namespace mg
