// gemm_impl.h — the prompt (prefill) GEMM: Y[n][rows] = X[n][K] . W^T for
// many activation vectors (n = prompt tokens), instantiated per weight
// format by gemm_q4.hip / gemm_q5.hip / gemm_q8.hip / gemm_q4k.hip /
// gemm_q6k.hip.
//
// One work-group of four waves computes a 32-vector x 128-row output tile:
// its vectors are two groups of 16, each with a 16-row high and a 16-row low
// operand block in LDS, and wave w owns output rows 32w .. 32w+31 (two 16-row
// "virtual tiles").  The k loop walks block quads through a two-stage
// pipeline: the activation operand of quad kk+1 is copied into LDS with
// direct-to-LDS loads and each wave loads the weight codes of its two
// virtual tiles for it into registers while quad kk is contracted.  32 KiB
// of LDS (40 or 48 where a range is summed in two halves, see launch_gemm_dt)
// and 128 VGPRs keep four work-groups on a CU (three at 48), each with its own
// barrier.  Eight-wave 64 x 128 tiles (two work-groups per CU, half the weight
// decoding per product) took, Q4_0 11008 inputs x 2048 rows / 2048 x 22016:
// 2048 vectors 211 / 417 us against 216 / 406, 1500 vectors 192 / 321 against
// 170 / 315, 512 vectors 67 / 126 (k split) against 66 / 119, and at 128
// vectors or fewer up to 40 % longer.
// Weights of any fold are read in place: virtual tile V of part p gathers,
// for column c', the codes of row 16V + c' from tile (16V + c') / R,
// column p*R + c' % R.
//
// Arithmetic follows the decode matvec's (gemv_impl.h): codes decoded to
// exact f16 integers, v_mfma_f32_16x16x32_f16 against the exact hi/lo
// operand, fp32 per-block scaling, and the same fused epilogues.  Unlike the
// matvec, each block's low-part products join the high-part MFMA sum (codes
// times 2^-11 against the low part times 2^11), so one scale FMA per output
// and block serves both.
#pragma once
#include "gemm_slices.h"
#include "gemv_impl.h"

#include <algorithm>

// Adds the ks k ranges' partial sums of a prompt GEMM in order, applies the
// RMSNorm factor and runs the epilogue (gemv.hip).
int launch_gemm_finish(const GemvArgs &a, int epi, int ks, hipStream_t s);

#define GEMM_NT 256   // threads per work-group
#define GEMM_BM 32    // vectors per work-group
#define GEMM_BN 128   // output rows per work-group (8 virtual tiles)
#define GEMM_STAGES 2 // quads in flight

struct GemmShape {
    int epi;
    int mt;          // vector tiles (GEMM_BM vectors each)
    int nt;          // 128-row tiles
    int ga;          // XCD slices along the vector tiles (1, 2, 4, 8)
    int mts, nts;    // vector / row tiles per slice (gemm_slices.h)
    int ks, kq;      // k ranges (grid.y) of kq block quads each; ks > 1: fp32 partial sums to a.part
    int fq;          // > 0: after fq quads (even) of its range a work-group sets its sums aside
};

// acc += the block's contribution for 16 vectors: xh holds their high
// operand parts, xl their low parts (scaled by LO_SCALE), wv the decoded
// codes and wl the codes times LO_INV_SCALE (exact: a power of two).  The
// low products go into the same fp32 sum as the high ones, so one scale FMA
// per output and block applies the block's factor to both.
template <int DT>
__device__ __forceinline__ void mfma_block_hl(f32x4 &acc, const f16x8 &xh, const f16x8 &xl, const f16x8 &wv,
                                              const f16x8 &wl, const BlockScale &s)
{
    const f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (DT == DT_Q4_K) {
        const _Float16 o = (_Float16)1, ol = (_Float16)LO_INV_SCALE;
        const f16x8 ones = {o, o, o, o, o, o, o, o};
        const f16x8 onesl = {ol, ol, ol, ol, ol, ol, ol, ol};
        f32x4 cc = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, wv, z, 0, 0, 0);
        cc = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, wl, cc, 0, 0, 0);
        f32x4 cs = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, ones, z, 0, 0, 0);
        cs = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, onesl, cs, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i] = fmaf(s.s1, cs[i], fmaf(s.s0, cc[i], acc[i]));
    } else if constexpr (DT == DT_Q6_K) {
        const _Float16 o = (_Float16)0;
        const f16x8 w0 = {wv[0], wv[1], wv[2], wv[3], o, o, o, o};
        const f16x8 w1 = {o, o, o, o, wv[4], wv[5], wv[6], wv[7]};
        const f16x8 l0 = {wl[0], wl[1], wl[2], wl[3], o, o, o, o};
        const f16x8 l1 = {o, o, o, o, wl[4], wl[5], wl[6], wl[7]};
        f32x4 c0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, w0, z, 0, 0, 0);
        c0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, l0, c0, 0, 0, 0);
        f32x4 c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, w1, z, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, l1, c1, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i] = fmaf(s.s1, c1[i], fmaf(s.s0, c0[i], acc[i]));
    } else {
        f32x4 cc = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, wv, z, 0, 0, 0);
        cc = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, wl, cc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i] = fmaf(s.s0, cc[i], acc[i]);
    }
}

// q_load with precomputed element offsets: e = cell * 64 + lane (codes,
// Q5_0 fifth bits, Q6_K high bits) and ds = the scale record's index
// (cell * 64 + col * 4 halves, or cell * 16 + col K-quant records).
template <int DT>
__device__ __forceinline__ void gemm_wload(const QTensor &w, uint32_t e, uint32_t ds, u32x4 &c0, u32x4 &c1,
                                           typename QScale<DT>::T &sv, uint32_t &h)
{
    constexpr uint32_t LB = QFmt<DT>::LANE_BYTES;
    const u32x4 *p = (const u32x4 *)(w.qs + e * LB);
    c0 = p[0];
    if constexpr (DT == DT_Q8_0) c1 = p[1];
    else if constexpr (DT == DT_Q6_K) {
        const u32x2 hb = *(const u32x2 *)((const uint8_t *)w.qh + e * 8u);
        c1 = u32x4{hb[0], hb[1], 0u, 0u};
    } else c1 = u32x4{0, 0, 0, 0};
    if constexpr (is_kquant(DT)) sv = *(const u32x4 *)((const uint8_t *)w.d + ds * 16u);
    else sv = *(const u32x2 *)((const uint8_t *)w.d + ds * 2u);
    if constexpr (DT == DT_Q5_0) h = *(const uint32_t *)((const uint8_t *)w.qh + e * 4u);
    else h = 0u;
}

// RMSNorm factors of vectors m0 .. m0 + BM - 1 (past the last: its own) from
// the producer's partial sums of squares, by NT threads into LDS: NT / BM
// lanes per vector, eight partials in flight per lane.
template <int BM, int NT>
__device__ __forceinline__ void gemm_norms(const GemvArgs &a, int m0, float *s_nrm, int tid)
{
    constexpr int LPV = NT / BM;
    static_assert(LPV >= 1 && LPV <= 64 && (LPV & (LPV - 1)) == 0, "lanes per vector");
    const int vi = tid / LPV, sub = tid % LPV;
    const float *p = a.in.ss + (size_t)min(m0 + vi, a.n - 1) * a.in.ss_stride;
    float s = 0.0f;
    for (int i0 = sub; i0 < a.in.ss_count; i0 += 8 * LPV) {
        float q[8];
#pragma unroll
        for (int k = 0; k < 8; k++) q[k] = i0 + k * LPV < a.in.ss_count ? p[i0 + k * LPV] : 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k++) s += q[k];
    }
    for (int o = LPV >> 1; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (sub == 0) s_nrm[vi] = 1.0f / sqrtf(s / (float)a.w.cols + a.in.eps);
}

// Epilogues of a tile of BM vectors x BR output rows (vectors m0 .., rows
// r0 .., r0 a multiple of BR) by NT threads; src(vi, rl) gives the products of
// vector m0 + vi and rows r0 + rl .. +3, scaled.  EPI_RESID and EPI_SWIGLU:
// a thread per operand piece of the consumer (eight inputs, 32 contiguous
// bytes for a vector's high and low rows), a wave over 16 vectors and the
// block's four k-groups, so a k-group's stores are 512 contiguous bytes and
// residual lines are used whole.  EPI_QKV: a thread per four rows (two RoPE
// pairs), 16 lanes along a vector's rows.  The stores bound these epilogues:
// one lane per row and 2-byte operand stores took 571 us for the gate/up
// projection of 2048 tokens (22016 x 2048 Q4_0) where the same product with
// plain stores took 431; 470-479 (400) with 16-byte ones and gemm_norms.
// Rows come in whole operand blocks (RESID, SWIGLU: the consumer's inputs)
// or whole 16-row heads (QKV).
template <int EPI, int BM, int BR, int NT, typename Src>
__device__ __forceinline__ void epi_runs(const GemvArgs &a, Src src, int m0, int r0, int tid)
{
#pragma clang fp contract(off)
    static_assert(BM % 16 == 0, "vectors per tile");
    if constexpr (EPI == EPI_RESID || EPI == EPI_SWIGLU) {
        constexpr int RPK = EPI == EPI_SWIGLU ? 2 : 1;   // rows per consumer input
        constexpr int PV = BR / (8 * RPK);               // pieces per vector
        static_assert(BR % (32 * RPK) == 0 && (BM * PV) % NT == 0, "whole blocks");
        const bool q8 = a.next.dt == DT_Q8_0;
#pragma unroll
        for (int it = 0; it < BM * PV / NT; it++) {
            const int i = tid + it * NT;
            const int g = i & 3, vi = (i >> 2) % BM, bl = (i >> 2) / BM, v = m0 + vi;
            const int b = r0 / RPK / 32 + bl;
            const int o0 = q8 ? 8 * g : 4 * g, o1 = q8 ? o0 + 4 : o0 + 16;   // the piece's inputs in its block
            const bool act = v < a.n && 32 * b * RPK < a.w.rows;
            if constexpr (EPI == EPI_RESID) {
                f32x4 x0 = {}, x1 = {};
                if (act) {
                    const size_t base = (size_t)v * a.out_stride + 32 * b;
                    const float *res = (a.res ? a.res : a.out) + base;
                    x0 = *(const f32x4 *)(res + o0) + src(vi, 32 * bl + o0);
                    x1 = *(const f32x4 *)(res + o1) + src(vi, 32 * bl + o1);
                    *(f32x4 *)(a.out + base + o0) = x0;
                    *(f32x4 *)(a.out + base + o1) = x1;
                    if (a.next.q) act_put8(a.next, v, b, g, 32 * b + o0, 32 * b + o1, x0, x1);
                }
                if (a.next.ss) {
                    // sums of squares per 16 rows: Q8_0 lanes 0, 1 hold the
                    // block's first 16 and lanes 2, 3 its second; otherwise
                    // x0 belongs to the first and x1 to the second
                    float s0 = x0[0] * x0[0] + x0[1] * x0[1] + x0[2] * x0[2] + x0[3] * x0[3];
                    float s1 = x1[0] * x1[0] + x1[1] * x1[1] + x1[2] * x1[2] + x1[3] * x1[3];
                    float *ss = a.next.ss + (size_t)v * a.next.ss_stride + 2 * b;
                    if (q8) {
                        s0 += s1;
                        s0 += __shfl_xor(s0, 1, 64);
                        if (act && !(g & 1)) ss[g >> 1] = s0;
                    } else {
                        s0 += __shfl_xor(s0, 1, 64);
                        s0 += __shfl_xor(s0, 2, 64);
                        s1 += __shfl_xor(s1, 1, 64);
                        s1 += __shfl_xor(s1, 2, 64);
                        if (act && g == 0) {
                            ss[0] = s0;
                            ss[1] = s1;
                        }
                    }
                }
            } else if (act) {
                f32x4 hv[2];
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    const int rl = 2 * (32 * bl + (p ? o1 : o0));
                    const f32x4 ya = src(vi, rl), yb = src(vi, rl + 4);   // gate, up alternating
                    hv[p][0] = (ya[0] / (1.0f + expf(-ya[0]))) * ya[1];
                    hv[p][1] = (ya[2] / (1.0f + expf(-ya[2]))) * ya[3];
                    hv[p][2] = (yb[0] / (1.0f + expf(-yb[0]))) * yb[1];
                    hv[p][3] = (yb[2] / (1.0f + expf(-yb[2]))) * yb[3];
                    if (a.out) *(f32x4 *)(a.out + (size_t)v * a.out_stride + 32 * b + (p ? o1 : o0)) = hv[p];
                }
                if (a.next.q) act_put8(a.next, v, b, g, 32 * b + o0, 32 * b + o1, hv[0], hv[1]);
            }
        }
    } else {
        static_assert(EPI == EPI_QKV && BR % 64 == 0 && (BM * BR / 4) % NT == 0, "whole rows");
#pragma unroll
        for (int it = 0; it < BM * BR / 4 / NT; it++) {
            const int i = tid + it * NT;
            const int vi = (i >> 4) % BM, rl = 64 * ((i >> 4) / BM) + 4 * (i & 15), v = m0 + vi;
            if (v >= a.n || r0 + rl >= a.w.rows) continue;
            const f32x4 y = src(vi, rl);
            const int pos = epi_pos(a, v), row = r0 + rl + a.row_base;
            const bool isq = row < a.nq, isk = !isq && row < a.nq + a.nkv;
            const int rr = isq ? row : isk ? row - a.nq : row - a.nq - a.nkv;
            const int h = rr / a.d_head, d = rr % a.d_head;
            f32x4 x = y;
            if (a.rope_on && (isq || isk)) {
                const f32x4 cs = *(const f32x4 *)(a.rope + ((size_t)pos * (a.d_head / 2) + (d >> 1)) * 2);
                x[0] = y[0] * cs[0] - y[1] * cs[1];
                x[1] = y[0] * cs[1] + y[1] * cs[0];
                x[2] = y[2] * cs[2] - y[3] * cs[3];
                x[3] = y[2] * cs[3] + y[3] * cs[2];
            }
            if (isq) {
                *(f32x4 *)(a.out + (size_t)v * a.out_stride + row) = x;
                continue;
            }
            void *base = isk ? a.kv.k_base : a.kv.v_base;
            const size_t o = kv_offset(a.kv, v) + ((size_t)h * a.max_ctx + pos) * a.d_head + d;
            if (a.kv_f16)
                *(f16x4 *)((_Float16 *)base + o) =
                    f16x4{(_Float16)x[0], (_Float16)x[1], (_Float16)x[2], (_Float16)x[3]};
            else *(f32x4 *)((float *)base + o) = x;
        }
    }
}

// Held to four waves per SIMD (128 VGPRs).  Unheld, the Q8_0 and K-quant
// instances took 129-160 and ran half the work-groups: 22016 x 2048 at 2048
// vectors, Q8_0 590 -> 462 us, Q4_K 822 -> 612 (4 VGPRs spilled), Q6_K 1031
// -> 791 (18 spilled).
template <int DT, bool SLIM>
__global__ __launch_bounds__(GEMM_NT) __attribute__((amdgpu_waves_per_eu(4))) void k_gemm(GemvArgs a, GemmShape sh)
{
    constexpr int HG = 2, NJ = 2;                 // vector groups and virtual tiles per wave
    constexpr int PW = 16 / (GEMM_NT / 64);       // 64-row operand copies per wave and stage
    constexpr int ASTAGE = 4 * 4 * 2 * GEMM_BM * 16;   // [block][k-group][2 GEMM_BM rows][16 B]
    constexpr int BN = GEMM_BN;
    static_assert(GEMM_BM == 16 * HG && GEMM_BN == 16 * NJ * (GEMM_NT / 64), "tile");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint8_t *s_a = smem;                                 // GEMM_STAGES x ASTAGE
    static_assert(GEMM_BM * (BN + 4) * 4 <= GEMM_STAGES * ASTAGE, "epilogue tile");

    // XCD-aware tile order: work-groups b, b+8, b+16, ... share an XCD.  The
    // (vector tile, row tile) grid is cut into ga x (8 / ga) slices, one per
    // XCD; an XCD walks its slice vector tile fastest, so the operand tiles
    // of its slice stay in its L2 while the weights stream past
    const int b = blockIdx.x, xcd = b & 7, i = b >> 3;
    const int mt_ = (xcd % sh.ga) * sh.mts + i % sh.mts;
    const int nt_ = (xcd / sh.ga) * sh.nts + i / sh.mts;
    if (mt_ >= sh.mt || nt_ >= sh.nt) return;
    const int m0 = mt_ * GEMM_BM;

    const int tid = threadIdx.x, l = tid & 63, g = l >> 4, cl = l & 15;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = a.n, nrows = 2 * n;
    const int BQ = a.w.block_quads, F = a.w.fold, R = 16 / F;
    const int nblk = a.w.cols >> 5;
    const int KQ = F * BQ;
    // this work-group's k range (split-K over grid.y): quads kb .. ke - 1
    const int kb = (int)blockIdx.y * sh.kq, ke = min(KQ, kb + sh.kq);

    // RMSNorm scales of the tile's vectors from the producer's partials,
    // passed through the last stage's LDS (untouched until the k loop's
    // first copy into it, which follows a wait and a barrier) to the lanes
    // that apply them: lane l's vectors 16h + 4(l>>4) + e
    float nrm[HG][4] = {};
    if (a.in.ss) {
        float *s_nrm = (float *)(smem + (GEMM_STAGES - 1) * ASTAGE);
        gemm_norms<GEMM_BM, GEMM_NT>(a, m0, s_nrm, tid);
        __syncthreads();
#pragma unroll
        for (int h = 0; h < HG; h++)
#pragma unroll
            for (int e = 0; e < 4; e++) nrm[h][e] = s_nrm[16 * h + 4 * (l >> 4) + e];
    }

    // weight gather for this lane: virtual tile V -> (tile, column).  The
    // lane's element offsets within the tensor (32-bit: the host checks the
    // size) are fixed here; each quad adds a uniform part
    uint32_t wq[NJ], wd[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int V = (nt_ * 4 + wid) * NJ + j;
        const int row = V * 16 + cl;
        const uint32_t wt = (uint32_t)min(row / R, a.w.row_tiles - 1), wc = (uint32_t)(row % R);
        wq[j] = wt * (uint32_t)BQ * 64u + wc + 16u * (uint32_t)g;   // cell * 64 + lane
        wd[j] = is_kquant(DT) ? wt * (uint32_t)BQ * 16u + wc : wt * (uint32_t)BQ * 64u + 4u * wc;
    }
    // operand row of this lane's copies (LDS rows of each 32-row group: the 16
    // high parts, then the 16 low parts of its 16 vectors, operand rows 2v and
    // 2v+1)
    const int l5 = l & 31;
    const uint32_t arow = 16u * (uint32_t)min(2 * m0 + (l & 32) + 2 * (l5 & 15) + (l5 >> 4), nrows - 1);

    u32x4 c0[GEMM_STAGES][NJ], c1[GEMM_STAGES][NJ];
    typename QScale<DT>::T dv[GEMM_STAGES][NJ];
    uint32_t hv[GEMM_STAGES][NJ];
    // loads of quad kk into stage st: 4 operand copies (of the tile's 32
    // 1 KiB pieces) and the codes/scales of the wave's two virtual tiles;
    // every load is issued unconditionally (padding blocks re-read a valid
    // block) so the per-stage load count is fixed
    auto load_stage = [&](int st, int kk) {
        kk = min(kk, ke - 1);
        const int p = kk / BQ, q = kk - p * BQ;
        const int b0 = p * 4 * BQ + 4 * q;
#pragma unroll
        for (int i = 0; i < PW; i++) {
            const int s = wid * PW + i, bi = s >> 2, gg = s & 3;   // (block, k-group)
            const int blk = min(b0 + bi, nblk - 1);
            const uint8_t *src = (const uint8_t *)a.in.q + ((size_t)blk * 4 + gg) * nrows * 16 + arow;
            uint8_t *dst = s_a + st * ASTAGE + s * 2 * GEMM_BM * 16;
            __builtin_amdgcn_global_load_lds((const gvoid_t *)src, (lvoid_t *)dst, 16, 0, 0);
        }
        const uint32_t uq = (uint32_t)(q * 64 + p * R);
        const uint32_t ud = is_kquant(DT) ? (uint32_t)(q * 16 + p * R) : (uint32_t)(q * 64 + 4 * p * R);
#pragma unroll
        for (int j = 0; j < NJ; j++) gemm_wload<DT>(a.w, wq[j] + uq, wd[j] + ud, c0[st][j], c1[st][j], dv[st][j], hv[st][j]);
    };

    const f32x4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 acc[HG][NJ];
#pragma unroll
    for (int h = 0; h < HG; h++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[h][j] = zero4;

    auto compute = [&](int st, int kk) {
        const int p = kk / BQ, q = kk - p * BQ;
        // blocks of this quad: padding blocks of the last part and the steps
        // past the end of the k range contribute nothing
        const int nb = kk < ke ? min(4, nblk - (p * 4 * BQ + 4 * q)) : 0;
        const uint8_t *sa = s_a + st * ASTAGE;
        auto block = [&](int bi) {
            f16x8 wv[NJ], wl[NJ];
            BlockScale bs[NJ];
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                wv[j] = deq_block<DT>(c0[st][j], c1[st][j], hv[st][j], bi);
                wl[j] = wv[j] * (_Float16)LO_INV_SCALE;
                bs[j] = block_scale<DT>(dv[st][j], bi);
            }
#pragma unroll
            for (int h = 0; h < HG; h++) {
                const uint8_t *row = &sa[((bi * 4 + g) * 2 * GEMM_BM + 32 * h + cl) * 16];
                const f16x8 xh = *(const f16x8 *)row;
                const f16x8 xl = *(const f16x8 *)(row + 16 * 16);
#pragma unroll
                for (int j = 0; j < NJ; j++) mfma_block_hl<DT>(acc[h][j], xh, xl, wv[j], wl[j], bs[j]);
            }
        };
        // a whole quad is one straight run (the four blocks' loads, MFMA
        // chains and scale FMAs interleave); the uniform test keeps branches
        // between blocks to the rare partial quads
        if (nb == 4) {
#pragma unroll
            for (int bi = 0; bi < 4; bi++) block(bi);
        } else {
#pragma unroll
            for (int bi = 0; bi < 4; bi++) {
                if (bi >= nb) break;
                block(bi);
            }
        }
    };

    // two-stage k loop: at the top of step kk only the loads of kk are
    // outstanding; the wait and the barrier publish every wave's copy of kk
    // (and every wave is done with kk-1), then kk+1 is issued into the stage
    // kk-1 freed
    load_stage(0, kb);
    __builtin_amdgcn_sched_barrier(0);
    // the body is unconditional (steps past the end compute nothing and
    // re-read the last quad) so every wait count is the same on each pass
    const bool halves = sh.fq && kb + sh.fq < ke;
    // the first half's sums: [HG NJ][threads] in LDS, each thread its own;
    // SLIM: those of the last vector group in registers
    constexpr int HL = SLIM ? HG - 1 : HG;
    f32x4 *aside = (f32x4 *)(smem + GEMM_STAGES * ASTAGE) + tid;
    f32x4 keep[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) keep[j] = zero4;
    for (int k0 = kb; k0 < ke; k0 += GEMM_STAGES) {
        if (halves && k0 == kb + sh.fq) {
#pragma unroll
            for (int h = 0; h < HG; h++)
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    if (h < HL) aside[(h * NJ + j) * GEMM_NT] = acc[h][j];
                    else keep[j] = acc[h][j];
                    acc[h][j] = zero4;
                }
        }
#pragma unroll
        for (int u = 0; u < GEMM_STAGES; u++) {
            const int kk = k0 + u;
            __builtin_amdgcn_s_waitcnt(WAITCNT_VM_LGKM0(0));
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            load_stage((u + 1) % GEMM_STAGES, kk + 1);
            __builtin_amdgcn_sched_barrier(0);
            compute(u, kk);
        }
    }
    // drain the trailing re-reads before the LDS can be released
    __builtin_amdgcn_s_waitcnt(WAITCNT_VM_LGKM0(0));
    __syncthreads();

    // lane l holds, per vector group h and tile j, output row 16V + cl for
    // vectors m0 + 16h + 4(l>>4) + {0, 1, 2, 3}.  Plain and partial
    // sums leave from here (64-byte runs of a vector's rows); the other
    // epilogues take the tile through LDS, 16 bytes at a time
    const bool logits = sh.epi == EPI_LOGITS;
    const bool direct = sh.ks > 1 || sh.epi == EPI_STORE || logits;
    float *tile = (float *)smem;
#pragma unroll
    for (int h = 0; h < HG; h++) {
        unsigned long long key[4] = {};   // EPI_LOGITS: the lane's best row per vector
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            if (halves) acc[h][j] += h < HL ? aside[(h * NJ + j) * GEMM_NT] : keep[j];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int rl = (wid * NJ + j) * 16 + cl, row = nt_ * BN + rl;
                const int vi = 16 * h + 4 * (l >> 4) + e, v = m0 + vi;
                float y = acc[h][j][e] * ACT_INV_SCALE;
                // partial sums of a k range: the finish kernel adds the
                // ranges in order, then scales and runs the epilogue
                if (a.in.ss && sh.ks == 1) y *= nrm[h][e];
                if (!direct) tile[vi * (BN + 4) + rl] = y;
                else if (v < n && row < a.w.rows) {
                    if (sh.ks > 1) a.part[((size_t)blockIdx.y * n + v) * a.w.rows + row] = y;
                    else a.out[(size_t)v * a.out_stride + row] = y;
                    if (logits) {
                        const unsigned long long k = argmax_key(y, (uint32_t)row);
                        key[e] = k > key[e] ? k : key[e];
                    }
                }
            }
        }
        if (!logits) continue;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            for (int o = 8; o > 0; o >>= 1) {
                const unsigned long long other = __shfl_xor(key[e], o, 64);
                key[e] = other > key[e] ? other : key[e];
            }
            const int v = m0 + 16 * h + 4 * (l >> 4) + e;
            if (cl == 0 && v < n)
                atomicMax(a.argmax + (size_t)v * ARGMAX_SLOTS + ((nt_ * 4 + wid) & (ARGMAX_SLOTS - 1)), key[e]);
        }
    }
    if (direct) return;
    __syncthreads();
    auto src = [&](int vi, int rl) { return *(const f32x4 *)&tile[vi * (BN + 4) + rl]; };
    switch (sh.epi) {
    case EPI_RESID: epi_runs<EPI_RESID, GEMM_BM, BN, GEMM_NT>(a, src, m0, nt_ * BN, tid); break;
    case EPI_SWIGLU: epi_runs<EPI_SWIGLU, GEMM_BM, BN, GEMM_NT>(a, src, m0, nt_ * BN, tid); break;
    default: epi_runs<EPI_QKV, GEMM_BM, BN, GEMM_NT>(a, src, m0, nt_ * BN, tid); break;
    }
}

// k ranges of the prompt GEMM.  The tiles of a narrow matrix or a short
// prompt leave CUs idle, and every work-group walks its k range at the
// latency of a step (about 1.2 us per block quad), so the ranges are doubled
// while the grid still fits one work-group per CU (two block quads or more
// each), and further, up to four per CU, while they keep ten quads.  Each range
// costs a write and a read of its partial sums in the finish kernel, which
// is why short ranges stop at one per CU: Q4_0, with finish, 64 vectors:
// 2048 x 2048 18.2 us in one range, 11.6 / 11.4 in 4 / 8 (taken), 14.6 in 16;
// 2048 x 11008 76, 26.8 in 4, 19.5 in 8 (taken), 19.7 in 16; 22016 x 2048 28.1
// in one (taken), 27.5 in 2, 30.1 in 4.  At 512 vectors 2048 x 2048 20.2 in
// one (taken), 23.9 in 2; 2048 x 11008 82.9, 72.6 in 2, 66.1 in 4 (taken).
// Within the partial-sum buffer (part_cap floats).  CMOL_GEMM_KSPLIT=0 turns
// it off (measurements).
static inline int gemm_ks(const QTensor &w, int n, size_t part_cap)
{
    static const bool on = [] {
        const char *e = getenv("CMOL_GEMM_KSPLIT");
        return !(e && e[0] == '0');
    }();
    if (!on) return 1;
    const long tiles = (long)((n + GEMM_BM - 1) / GEMM_BM) * ((w.rows + GEMM_BN - 1) / GEMM_BN);
    const int KQ = w.fold * w.block_quads;
    int ks = 1;
    while (ks < GEMM_KS_MAX && (size_t)(2 * ks) * n * w.rows <= part_cap &&
           ((tiles * 2 * ks <= gemv_cus() && KQ / (2 * ks) >= 2) ||
            (tiles * 2 * ks <= 4L * gemv_cus() && KQ / (2 * ks) >= 10)))
        ks *= 2;
    return ks;
}

template <int DT>
int launch_gemm_dt(const GemvArgs &a, int epi, hipStream_t s)
{
    if (epi < EPI_STORE || epi > EPI_LOGITS) return -6;
    // the kernel's per-lane weight offsets are 32-bit
    if ((size_t)a.w.row_tiles * a.w.block_quads * 64 * QFmt<DT>::LANE_BYTES > 0xffffffffUL) return -6;
    GemmShape sh;
    sh.epi = epi;
    const int KQ = a.w.fold * a.w.block_quads;
    const int ks = a.part && epi != EPI_LOGITS ? gemm_ks(a.w, a.n, a.part_cap) : 1;   // (the finish has no argmax)
    sh.ks = ks;
    sh.kq = (KQ + ks - 1) / ks;
    sh.mt = (a.n + GEMM_BM - 1) / GEMM_BM;
    sh.nt = (a.w.rows + GEMM_BN - 1) / GEMM_BN;
    const GemmSlices sl = gemm_slices(sh.mt, sh.nt, ks, sh.kq, std::max(1, gemv_cus() / 8));
    sh.ga = sl.ga;
    sh.mts = sl.mts;
    sh.nts = sl.nts;
    const long wgs = 8L * sh.mts * sh.nts;
    if (wgs > 0x7fffffffL) return -6;
    // fewer than four work-groups per CU (the grids that two ranges of twice
    // the work would also serve): each range is summed in two halves, so a
    // range costs no precision against two of half its length (2048 inputs:
    // 1.39e-7 of the result in 2-norm, 1.69e-7 in one chain; 20.2 us against
    // 19.7 at 2048 x 2048 x 512 vectors).  Fuller grids run in one chain: the
    // first half's sums, 16 KiB of LDS, would leave a CU three work-groups of
    // four.
    sh.fq = (long)sh.mt * sh.nt * ks < 4L * gemv_cus() ? 2 * ((sh.kq + 3) / 4) : 0;
    // where that already makes a second round, with more than three work-groups
    // per CU on the fullest XCD, half of those sums stay in registers instead.
    // us, all in LDS / half: Q4_0 22016 x 2048 x 160 47.4 / 45.1, 5120 x 2048 x
    // 700 49.4 / 46.0; Q4_K 2048 x 2048 x 1600 68.0 / 61.1; Q6_K (24 VGPRs
    // spilled) 4096 x 4096 x 800 161 / 150.  Grids of one vector tile, bound by
    // their weights, and several k ranges gain only in the formats that it makes
    // spill nothing (128256 x 2048 x 17: Q4_0 49.4 / 46.8, Q5_0 63.2 / 61.7, Q8_0
    // 55.5 / 56.8, Q6_K 93.9 / 96.2; 2048 x 11008 x 224, eight ranges: Q4_0 42.1
    // / 39.6, Q4_K 52.7-53.7 / 54.0-54.5).
    constexpr bool spills = DT != DT_Q4_0 && DT != DT_Q5_0;
    const bool slim = sh.fq && (long)sh.mts * sh.nts * ks > 3L * (gemv_cus() / 8) && (!spills || (sh.mt > 1 && ks == 1));
    const size_t lds = (size_t)GEMM_STAGES * 4 * 4 * 2 * GEMM_BM * 16 + (sh.fq ? (size_t)GEMM_NT * (slim ? 32 : 64) : 0);
    const dim3 grid((unsigned)wgs, (unsigned)ks), block(GEMM_NT);
    auto go = [&](auto kern) {
        if (a.ev_start) hipExtLaunchKernelGGL(kern, grid, block, lds, s, a.ev_start, ks > 1 ? nullptr : a.ev_stop, 0, a, sh);
        else hipLaunchKernelGGL(kern, grid, block, lds, s, a, sh);
    };
    if (slim) go(k_gemm<DT, true>);
    else go(k_gemm<DT, false>);
    return ks > 1 ? launch_gemm_finish(a, epi, ks, s) : 0;
}
