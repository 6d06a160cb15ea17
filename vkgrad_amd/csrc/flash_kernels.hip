// Causal attention without the (T, T) matrices: forward, and backward from the row statistics.
//
//   out[q] = sum_j P[q][j] v[j],  P = softmax over the keys first(q) <= j <= q of scale * q . k
//
// (reference call sites transformer.py:144-182; attn_softmax / attn_softmax_doc / attn_softmax_bwd,
// tkernels.py:105-187, and the head permutes around them, tkernels.py:195-301.)  The operands
// are the merged (B*T, 3D) 16-bit output of the QKV projection and the merged (B*T, D)
// gradient of the output, the results the merged (B*T, D) output and (B*T, 3D) gradient: no head
// permutes, and of P only the two numbers per row that rebuild it leave the forward kernel -
// lse = log2 of the sum of exponentials, base 2.
//
// All three kernels share one scheme.  A wavefront owns 32 rows of one side (queries, or keys in
// the dK / dV kernel), one per lane along the accumulator columns of v_mfma_f32_32x32x16; their
// 16-bit rows stay in registers as B operands.  The other side passes through LDS in tiles of 64
// rows shared by the four wavefronts, loaded one tile ahead through registers.  Row n = 8g + 4h +
// e of an A operand is given row 16h + 4g + e of its block of 32, so a lane of half-wave h ends
// up with 16 neighbouring rows of its column: narrowed, they are the B operand of the second product
// (k = rows of the tile), whose A operand is read transposed from the same LDS rows.  What a row
// needs - maximum, sum, lse, row term - is one number per lane, so there are no lane exchanges but
// one between the half-waves.
//
// The forward kernel walks the keys twice - once for the row's sum, once for P V - so that P is narrowed to 16 bits after
// it is normalised, which is what multiplying a stored P does, and the backward kernels round the P they rebuild the same
// way: the row term then cancels against the very P that made the output.  (One walk with P relative to a running
// reference point, and dS from P in 32 bits, is 34 + 83 us where this is 46 + 89, and its errors against 64 bits are no
// larger; but in rows that are nearly one-hot the terms no longer cancel, and single gradients of a packed batch moved by
// as much as the root mean square of all.)
//
// What bounds them: the exponentials and the arithmetic around them (a transcendental takes 16
// clocks a wavefront, 256 a block of 32 x 32, as much as its MFMAs) and the latency from one to the next, not memory:
// 96 heads x 1024 x 64 read and write 60 MB forward.  Masks are branches over whole tiles (FK_BRANCH), maxima
// trees; the sum of a row goes key by key.  Measured there (bf16, kernel by kernel): forward 41.8 us (40.5 with sums as trees and
// no maximum of a tile until a sum reaches 2^100, which costs lse up to six bits; 48 with a serial maximum and a branch a block),
// backward 39.5 + 49.8 (44.8 + 62 with P narrowed twice and a mask test an element in the dK / dV kernel, which the
// compiler made a branch an element).
// P is rebuilt twice in the backward pass, once per kernel: that costs 7 products instead of 5, but dQ needs no
// atomics, no clear and no narrowing pass.  Three wavefronts a SIMD forward, two in the dK / dV kernel.
#include "flash_common.h"

namespace mg {

// Which head and which rows (longest first) a workgroup takes.  Consecutive workgroups fill the CUs round by round; every
// second round is dealt out backwards, eight at a time so that a head stays on its XCD, and a CU's
// share evens out: in order, one CU gets the longest of every round (96 heads x 1024 x 64: 45.3 + 88.3
// us in order, 43.1 + 85.5 so).
struct FkWork {
    int bh, y;
    __device__ __forceinline__ FkWork() {
        const int n = gridDim.x * gridDim.y, w = blockIdx.y * gridDim.x + blockIdx.x, round = w >> 8;
        int v = w;
        if ((round & 1) && (round + 1) * 256 <= n) v = (round << 8) + ((31 - ((w & 255) >> 3)) << 3) + (w & 7);
        bh = v % (int)gridDim.x;
        y = v / (int)gridDim.x;
    }
};

// ---- forward -------------------------------------------------------------------------
template <int DT, int KK>
__global__ void __launch_bounds__(256, (KK <= 4 ? 3 : 2))
k_flash_fwd(const FkArgs p) {
    using S = FkShape<KK>;
    __shared__ __attribute__((aligned(16))) char smem[2 * S::NBUF * S::TILE];
    const FkLane L;
    const int tid = threadIdx.x, T = p.T, hd = p.hd, D = p.H * hd;
    const FkWork wk;
    const int b = wk.bh / p.H, h = wk.bh % p.H;
    const int iw = (gridDim.y - 1 - wk.y) * 128;   // the long rows first
    const int i0 = iw + L.wave * 32, q = i0 + L.n, qc = min(q, T - 1);
    const int64_t pitch = 3 * (int64_t)D;
    const uint16_t *qb = p.qkv + (int64_t)b * T * pitch + h * hd, *kb = qb + D, *vb = kb + D;
    fk_u32x4 qf[KK];
    fk_load_row<KK>(qf, qb + qc * pitch, L.half, hd);
    const int first = p.seg ? (int)p.seg[(int64_t)b * T + qc] : 0;
    // tiles that hold a key some query of the workgroup sees
    int t0 = 0;
    if (p.seg) {
        int f = first;
#pragma unroll
        for (int m = 16; m >= 1; m >>= 1) f = min(f, __shfl_xor(f, m, 64));
        int *fmin = reinterpret_cast<int *>(smem);
        if (L.lane == 0) fmin[L.wave] = f;
        __syncthreads();
        t0 = min(min(fmin[0], fmin[1]), min(fmin[2], fmin[3])) / FK_BN;
        __syncthreads();
    }
    const int t1 = min(iw + 127, T - 1) / FK_BN + 1;
    const float c2 = p.scale * 1.4426950408889634f;   // base 2: an exponential is one v_exp_f32
    float m = FK_NOTHING, l = 0.f;
    // scores of a tile, masked where the diagonal or a sample's start crosses it
    auto scores = [&](const char *kt, int j0, fk_f32x16 (&s)[2]) {
#pragma unroll
        for (int bl = 0; bl < 2; bl++) s[bl] = fk_product<DT, KK>(kt + (bl * 32 + L.arow) * S::PITCH + L.half * 16, qf);
        if (p.seg || j0 + FK_BN - 1 > i0) {
            FK_BRANCH;
            const int lo = first - j0 - 16 * L.half, hi = q - j0 - 16 * L.half;
#pragma unroll
            for (int bl = 0; bl < 2; bl++)
#pragma unroll
                for (int r = 0; r < 16; r++) s[bl][r] = (32 * bl + r <= hi && 32 * bl + r >= lo) ? s[bl][r] : FK_MASKED;
        }
    };
    FkStage<KK> ks, vs;
    // First walk over the keys: the row's reference point and its sum of exponentials.
    ks.load(kb, pitch, t0 * FK_BN, T, hd, tid);
    for (int t = t0; t < t1; t++) {
        const int j0 = t * FK_BN;
        char *kt = smem + (t & 1) * S::TILE;
        ks.store(kt, tid);
        if (t + 1 < t1) ks.load(kb, pitch, j0 + FK_BN, T, hd, tid);
        __syncthreads();
        if (j0 > i0 + 31) continue;          // every key beyond every query of this wavefront
        fk_f32x16 s[2];
        scores(kt, j0, s);
        // The reference point need not be the maximum, but stays within 8 of it: further off, the exponents that matter would be
        // held with fewer bits (a first tile 60 below the rest, a sum up to 2^100: an error of lse of 3.9e-6 for 0.8e-6).
        float mt = fmaxf(fk_max16(s[0]), fk_max16(s[1]));
        mt = fk_both(mt, [](float x, float y) { return fmaxf(x, y); }) * c2;
        if (__any(mt > m + 8.f)) {
            const float mn = fmaxf(m, mt);
            l *= __builtin_amdgcn_exp2f(m - mn);
            m = mn;
        }
#pragma unroll
        for (int bl = 0; bl < 2; bl++)
#pragma unroll
            for (int r = 0; r < 16; r++) l += __builtin_amdgcn_exp2f(__builtin_fmaf(s[bl][r], c2, -m));
    }
    ks.load(kb, pitch, t0 * FK_BN, T, hd, tid);
    vs.load(vb, pitch, t0 * FK_BN, T, hd, tid);
    l = fk_both(l, [](float x, float y) { return x + y; });
    const float lse = m + __builtin_amdgcn_logf(l);
    __syncthreads();
    // Second walk: P, normalised before it is narrowed, times V.
    fk_f32x16 o[S::MB];
#pragma unroll
    for (int i = 0; i < S::MB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[i][r] = 0.f;
    for (int t = t0; t < t1; t++) {
        const int j0 = t * FK_BN;
        char *kt = smem + (S::NBUF == 2 ? (t & 1) * 2 * S::TILE : 0), *vt = kt + S::TILE;
        if (S::NBUF == 1) __syncthreads();   // everybody is done with the tile before
        ks.store(kt, tid);
        vs.store(vt, tid);
        if (t + 1 < t1) {
            ks.load(kb, pitch, j0 + FK_BN, T, hd, tid);
            vs.load(vb, pitch, j0 + FK_BN, T, hd, tid);
        }
        __syncthreads();
        if (j0 > i0 + 31) continue;
        fk_f32x16 s[2];
        scores(kt, j0, s);
#pragma unroll
        for (int bl = 0; bl < 2; bl++) {
            float e[16];
#pragma unroll
            for (int r = 0; r < 16; r++) e[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[bl][r], c2, -lse));
            uint32_t w[8];
            fk_narrow<DT>(e, w);
            fk_accumulate<DT, KK>(o, vt + (bl * 32 + L.trow) * S::PITCH + L.tcol * 2, w);
        }
    }
    if (q >= T) return;
    if (L.half == 0) p.lse[(int64_t)wk.bh * T + q] = lse;
    const int64_t row = ((int64_t)b * T + q) * D + h * hd;
    fk_store_row16<DT, S::MB>(p.out16 + row, o, 1.f, L.half, hd);
    if (p.out32) {
#pragma unroll
        for (int i = 0; i < S::MB; i++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int d = 32 * i + 8 * g + 4 * L.half;
                if (d < hd)
                    *reinterpret_cast<fk_f32x4 *>(p.out32 + row + d) = fk_f32x4{o[i][4 * g], o[i][4 * g + 1], o[i][4 * g + 2], o[i][4 * g + 3]};
            }
    }
}

// ---- backward: dQ, and the row term sum_d dOut[q][d] Out[q][d] ------------------------
template <int DT, int KK>
__global__ void __launch_bounds__(256, 2)
k_flash_dq(const FkArgs p) {
    using S = FkShape<KK>;
    __shared__ __attribute__((aligned(16))) char smem[2 * S::NBUF * S::TILE];
    const FkLane L;
    const int tid = threadIdx.x, T = p.T, hd = p.hd, D = p.H * hd;
    const FkWork wk;
    const int b = wk.bh / p.H, h = wk.bh % p.H;
    const int iw = (gridDim.y - 1 - wk.y) * 128;
    const int i0 = iw + L.wave * 32, q = i0 + L.n, qc = min(q, T - 1);
    const int64_t pitch = 3 * (int64_t)D;
    const uint16_t *qb = p.qkv + (int64_t)b * T * pitch + h * hd, *kb = qb + D, *vb = kb + D;
    const int64_t orow = ((int64_t)b * T + qc) * D + h * hd;
    fk_u32x4 qf[KK], gf[KK];
    fk_load_row<KK>(qf, qb + qc * pitch, L.half, hd);
    fk_load_row<KK>(gf, p.dout + orow, L.half, hd);
    const float dsum = fk_row_term<DT, KK>(gf, p.out32 + orow, L.half, hd);
    const int64_t stat = (int64_t)wk.bh * T + qc;
    if (L.half == 0 && q < T) p.dsum[stat] = dsum;
    const float lse = p.lse[stat], dscaled = dsum * p.scale;
    const int first = p.seg ? (int)p.seg[(int64_t)b * T + qc] : 0;
    int t0 = 0;
    if (p.seg) {
        int f = first;
#pragma unroll
        for (int m = 16; m >= 1; m >>= 1) f = min(f, __shfl_xor(f, m, 64));
        int *fmin = reinterpret_cast<int *>(smem);
        if (L.lane == 0) fmin[L.wave] = f;
        __syncthreads();
        t0 = min(min(fmin[0], fmin[1]), min(fmin[2], fmin[3])) / FK_BN;
        __syncthreads();
    }
    const int t1 = min(iw + 127, T - 1) / FK_BN + 1;
    const float c2 = p.scale * 1.4426950408889634f;
    fk_f32x16 o[S::MB];
#pragma unroll
    for (int i = 0; i < S::MB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[i][r] = 0.f;
    FkStage<KK> ks, vs;
    ks.load(kb, pitch, t0 * FK_BN, T, hd, tid);
    vs.load(vb, pitch, t0 * FK_BN, T, hd, tid);
    for (int t = t0; t < t1; t++) {
        const int j0 = t * FK_BN;
        char *kt = smem + (S::NBUF == 2 ? (t & 1) * 2 * S::TILE : 0), *vt = kt + S::TILE;
        if (S::NBUF == 1) __syncthreads();
        ks.store(kt, tid);
        vs.store(vt, tid);
        if (t + 1 < t1) {
            ks.load(kb, pitch, j0 + FK_BN, T, hd, tid);
            vs.load(vb, pitch, j0 + FK_BN, T, hd, tid);
        }
        __syncthreads();
#pragma unroll
        for (int bl = 0; bl < 2; bl++) {
            const int jb = j0 + 32 * bl;
            if (jb > i0 + 31) continue;
            const fk_f32x16 s = fk_product<DT, KK>(kt + (bl * 32 + L.arow) * S::PITCH + L.half * 16, qf);
            const fk_f32x16 dp = fk_product<DT, KK>(vt + (bl * 32 + L.arow) * S::PITCH + L.half * 16, gf);
            float e[16];
#pragma unroll
            for (int r = 0; r < 16; r++) e[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c2, -lse));
            uint32_t w[8];
            fk_round<DT>(e, w);   // P as the forward pass multiplied it
#pragma unroll
            for (int r = 0; r < 16; r++) e[r] *= __builtin_fmaf(dp[r], p.scale, -dscaled);
            if (p.seg || jb + 31 > i0) {
                FK_BRANCH;
                const int hi = q - jb - 16 * L.half, lo = first - jb - 16 * L.half;
#pragma unroll
                for (int r = 0; r < 16; r++) e[r] = (r <= hi && r >= lo) ? e[r] : 0.f;
            }
            fk_narrow<DT>(e, w);
            fk_accumulate<DT, KK>(o, kt + (bl * 32 + L.trow) * S::PITCH + L.tcol * 2, w);
        }
    }
    if (q < T) fk_store_row16<DT, S::MB>(p.dqkv + ((int64_t)b * T + q) * pitch + h * hd, o, 1.f, L.half, hd);
}

// ---- backward: dK and dV; a wavefront owns 32 keys, the queries that see them pass through LDS ----
template <int DT, int KK>
__global__ void __launch_bounds__(256, (KK <= 4 ? 2 : 1))
k_flash_dkv(const FkArgs p) {
    using S = FkShape<KK>;
    __shared__ __attribute__((aligned(16))) char smem[2 * S::NBUF * S::TILE];
    __shared__ __attribute__((aligned(16))) float st_lse[2][FK_BN], st_d[2][FK_BN];
    __shared__ int st_first[2][FK_BN];
    const FkLane L;
    const int tid = threadIdx.x, T = p.T, hd = p.hd, D = p.H * hd;
    const FkWork wk;
    const int b = wk.bh / p.H, h = wk.bh % p.H;
    const int jw = wk.y * 128;                     // the keys that most queries see first
    const int j0 = jw + L.wave * 32, key = j0 + L.n, kc = min(key, T - 1);
    const int64_t pitch = 3 * (int64_t)D;
    const uint16_t *qb = p.qkv + (int64_t)b * T * pitch + h * hd, *kb = qb + D, *vb = kb + D;
    const uint16_t *gb = p.dout + (int64_t)b * T * D + h * hd;
    fk_u32x4 kf[KK], vf[KK];
    fk_load_row<KK>(kf, kb + kc * pitch, L.half, hd);
    fk_load_row<KK>(vf, vb + kc * pitch, L.half, hd);
    const float c2 = p.scale * 1.4426950408889634f;
    fk_f32x16 dk[S::MB], dv[S::MB];
#pragma unroll
    for (int i = 0; i < S::MB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) dk[i][r] = dv[i][r] = 0.f;
    const int t0 = jw / FK_BN, t1 = (T - 1) / FK_BN + 1;
    FkStage<KK> qs, gs;
    float r_lse = 0.f, r_d = 0.f;
    int r_first = 0;
    auto load = [&](int t) {
        qs.load(qb, pitch, t * FK_BN, T, hd, tid);
        gs.load(gb, D, t * FK_BN, T, hd, tid);
        if (tid < FK_BN) {
            const int qq = min(t * FK_BN + tid, T - 1);
            r_lse = p.lse[(int64_t)wk.bh * T + qq];
            r_d = p.dsum[(int64_t)wk.bh * T + qq];
            if (p.seg) r_first = (int)p.seg[(int64_t)b * T + qq];
        }
    };
    load(t0);
    for (int t = t0; t < t1; t++) {
        const int i0 = t * FK_BN, buf = S::NBUF == 2 ? t & 1 : 0;
        char *qt = smem + buf * 2 * S::TILE, *gt = qt + S::TILE;
        if (S::NBUF == 1) __syncthreads();
        qs.store(qt, tid);
        gs.store(gt, tid);
        if (tid < FK_BN) {
            st_lse[buf][tid] = r_lse;
            st_d[buf][tid] = r_d * p.scale;
            st_first[buf][tid] = r_first;
        }
        if (t + 1 < t1) load(t + 1);
        __syncthreads();
#pragma unroll
        for (int bl = 0; bl < 2; bl++) {
            const int ib = i0 + 32 * bl;
            if (ib + 31 < j0 || ib >= T) continue;       // no query of the block sees a key of this wavefront
            const int r0 = 32 * bl + 16 * L.half;        // this lane's queries: ib + 16 half + r
            float e[16], ds[16], d[16];
            const fk_f32x16 s = fk_product<DT, KK>(qt + (bl * 32 + L.arow) * S::PITCH + L.half * 16, kf);
            const fk_f32x16 dp = fk_product<DT, KK>(gt + (bl * 32 + L.arow) * S::PITCH + L.half * 16, vf);
#pragma unroll
            for (int r = 0; r < 16; r++) {
                e[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c2, -st_lse[buf][r0 + r]));
                d[r] = st_d[buf][r0 + r];
            }
            if (p.seg || ib < j0 + 31 || ib + 31 >= T) {
                FK_BRANCH;
                const int lo = key - i0 - r0, hi = T - 1 - i0 - r0;
#pragma unroll
                for (int r = 0; r < 16; r++) e[r] = (r >= lo && r <= hi && key >= st_first[buf][r0 + r]) ? e[r] : 0.f;
            }
            uint32_t we[8], wd[8];
            fk_round<DT>(e, we);
#pragma unroll
            for (int r = 0; r < 16; r++) ds[r] = e[r] * __builtin_fmaf(dp[r], p.scale, -d[r]);
            fk_narrow<DT>(ds, wd);
            fk_accumulate<DT, KK>(dv, gt + (bl * 32 + L.trow) * S::PITCH + L.tcol * 2, we);
            fk_accumulate<DT, KK>(dk, qt + (bl * 32 + L.trow) * S::PITCH + L.tcol * 2, wd);
        }
    }
    if (key >= T) return;
    uint16_t *row = p.dqkv + ((int64_t)b * T + key) * pitch + h * hd;
    fk_store_row16<DT, S::MB>(row + D, dk, 1.f, L.half, hd);
    fk_store_row16<DT, S::MB>(row + 2 * D, dv, 1.f, L.half, hd);
}

template <int DT, int KK>
static void fk_launch(hipStream_t s, const FkArgs &a, int64_t nbh, bool backward) {
    // heads fastest: the blocks of a head, which share its K and V, land on one XCD when the head count is a
    // multiple of 8
    const dim3 grid((unsigned)nbh, (unsigned)((a.T + 127) / 128));
    if (!backward) {
        hipLaunchKernelGGL((k_flash_fwd<DT, KK>), grid, dim3(256), 0, s, a);
    } else {
        hipLaunchKernelGGL((k_flash_dq<DT, KK>), grid, dim3(256), 0, s, a);
        hipLaunchKernelGGL((k_flash_dkv<DT, KK>), grid, dim3(256), 0, s, a);
    }
}

static void fk_dispatch(hipStream_t s, const FkArgs &a, int64_t nbh, int dtype, bool backward) {
    if (backward ? fk_small_backward(a, nbh) : fk_small_forward(a, nbh)) return fk_small_launch(s, a, nbh, dtype, backward);
    const int kk = fk_steps(a.hd);
    if (dtype == MG_F16) {
        if (kk == 1) fk_launch<MG_F16, 1>(s, a, nbh, backward);
        else if (kk == 2) fk_launch<MG_F16, 2>(s, a, nbh, backward);
        else if (kk == 4) fk_launch<MG_F16, 4>(s, a, nbh, backward);
        else if (kk == 6) fk_launch<MG_F16, 6>(s, a, nbh, backward);
        else fk_launch<MG_F16, 8>(s, a, nbh, backward);
    } else {
        if (kk == 1) fk_launch<MG_BF16, 1>(s, a, nbh, backward);
        else if (kk == 2) fk_launch<MG_BF16, 2>(s, a, nbh, backward);
        else if (kk == 4) fk_launch<MG_BF16, 4>(s, a, nbh, backward);
        else if (kk == 6) fk_launch<MG_BF16, 6>(s, a, nbh, backward);
        else fk_launch<MG_BF16, 8>(s, a, nbh, backward);
    }
}

static bool fk_shape_ok(int64_t B, int64_t T, int64_t H, int64_t hd) {
    return B > 0 && H > 0 && B <= 0x7fffffff / H && T > 0 && T <= 65535 * 128 && mg_tk_flash_supported(hd) &&
           B * T <= 0x7fffffff && H * hd <= 0x7fffffff / 3;
}

}  // namespace mg

using namespace mg;

extern "C" {

// 16-byte pieces of a head's row: the width is a multiple of 8
int mg_tk_flash_supported(int64_t hd) { return hd > 0 && hd <= 128 && hd % 8 == 0; }

int mg_tk_flash_fwd(mg_ctx *ctx, const void *qkv16, const uint32_t *seg, void *out16, float *out32, float *lse, int64_t B,
                    int64_t T, int64_t H, int64_t hd, float scale, int dtype) {
    EW_PRECHECK("mg_tk_flash_fwd", qkv16 && out16 && lse && fk_shape_ok(B, T, H, hd) && dtype_ok(dtype) && scale > 0.f &&
                                       (((uintptr_t)qkv16 | (uintptr_t)out32) & 15) == 0 && ((uintptr_t)out16 & 7) == 0 &&
                                       (((uintptr_t)lse | (uintptr_t)seg) & 3) == 0);
    FkArgs a{};
    a.qkv = (const uint16_t *)qkv16;
    a.seg = seg;
    a.out16 = (uint16_t *)out16;
    a.out32 = out32;
    a.lse = lse;
    a.T = (int)T;
    a.H = (int)H;
    a.hd = (int)hd;
    a.scale = scale;
    fk_dispatch(ctx_stream(ctx), a, B * H, dtype, false);
    EW_POSTCHECK("mg_tk_flash_fwd");
}

int mg_tk_flash_bwd(mg_ctx *ctx, const void *qkv16, const uint32_t *seg, const void *dout16, const float *out32,
                    const float *lse, float *dsum, void *dqkv16, int64_t B, int64_t T, int64_t H, int64_t hd, float scale,
                    int dtype) {
    EW_PRECHECK("mg_tk_flash_bwd", qkv16 && dout16 && out32 && lse && dsum && dqkv16 && fk_shape_ok(B, T, H, hd) &&
                                       dtype_ok(dtype) && scale > 0.f &&
                                       (((uintptr_t)qkv16 | (uintptr_t)dout16 | (uintptr_t)out32) & 15) == 0 &&
                                       ((uintptr_t)dqkv16 & 7) == 0 &&
                                       (((uintptr_t)lse | (uintptr_t)dsum | (uintptr_t)seg) & 3) == 0);
    FkArgs a{};
    a.qkv = (const uint16_t *)qkv16;
    a.seg = seg;
    a.dout = (const uint16_t *)dout16;
    a.out32 = const_cast<float *>(out32);
    a.lse = const_cast<float *>(lse);
    a.dsum = dsum;
    a.dqkv = (uint16_t *)dqkv16;
    a.T = (int)T;
    a.H = (int)H;
    a.hd = (int)hd;
    a.scale = scale;
    fk_dispatch(ctx_stream(ctx), a, B * H, dtype, true);
    EW_POSTCHECK("mg_tk_flash_bwd");
}

}  // extern "C"
