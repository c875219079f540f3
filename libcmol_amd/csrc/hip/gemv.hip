// gemv.hip — quantised matvec / small-batch GEMM for gfx950.
//
// y[n] = W . x[n] for a Q4_0/Q5_0/Q8_0/Q4_K/Q6_K weight in the quad-tile layout and up
// to 32 activation vectors (kernel template in gemv_impl.h).  One work-group
// owns one 16-row tile and its NW wavefronts split the k range.  The
// activation operand of the whole k range is copied into LDS once with
// direct-to-LDS loads (in chunks only when it exceeds the LDS budget); each
// wave streams its weight quads through a ring of U in-flight loads (one
// coalesced 16/32-byte load per lane per quad), decodes the codes to exact
// small integers in f16 (common.h) and contracts them with
// v_mfma_f32_16x16x32_f16 against the operand (kernels.h: f16 high part and
// scaled f16 remainder in two MFMA rows per vector, eight vectors per MFMA),
// so every product is exact and the sum is carried in fp32.  The per-block
// fp16 scale multiplies each block's 16x16 result tile.  Partial sums of the
// waves meet in LDS in a fixed order.
//
// Fused around the product (reference arithmetic in brackets):
//   RMSNorm: 1/sqrt(mean(x^2)+eps) from the producer's sum-of-squares
//            partials, applied to the result [src/model.c:90-97];
//   epilogues: store; residual add + next operand [src/model.c:232,259];
//            SwiGLU over interleaved gate/up rows [src/model.c:117-123];
//            RoPE on q/k rows + KV-cache write at pos [src/attn.c:83-101];
//            logits + first-index argmax [src/sampler.c:199-204].
#include "gemm_impl.h"

int launch_gemv_q4(const GemvArgs &a, int epi, hipStream_t s);
int launch_gemv_q5(const GemvArgs &a, int epi, hipStream_t s);
int launch_gemv_q8(const GemvArgs &a, int epi, hipStream_t s);
int launch_gemm_q4(const GemvArgs &a, int epi, hipStream_t s);
int launch_gemm_q5(const GemvArgs &a, int epi, hipStream_t s);
int launch_gemm_q8(const GemvArgs &a, int epi, hipStream_t s);
int launch_gemv_q4k(const GemvArgs &a, int epi, hipStream_t s);
int launch_gemv_q6k(const GemvArgs &a, int epi, hipStream_t s);
int launch_gemm_q4k(const GemvArgs &a, int epi, hipStream_t s);
int launch_gemm_q6k(const GemvArgs &a, int epi, hipStream_t s);

// four floats at any float address
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

size_t act_bytes(int K, int n)
{
    const size_t blocks = (size_t)((K / 32 + 3) / 4) * 4;
    return blocks * 4 * (size_t)(2 * n) * 8 * sizeof(_Float16);
}


// Whether 9 .. 32 vectors over w run the prompt GEMM, which decodes each
// weight once for all of them, rather than the batched matvec, which decodes
// it once per 8 or 16 vectors but has more and shorter work-groups.  us,
// matvec / GEMM: above 16 vectors the GEMM wins once its 128-row tiles cover
// the CUs (32 vectors Q4_0: 22016 x 2048 16.1 / 19.9, 32768 x 2048 28.8 /
// 20.6; Q8_0 128256 x 2048 91.8 / 62.1), for 2^26 weights or more (17 vectors
// Q8_0 8192 x 8192 26.2 / 24.5), and for the K-quants, whose decoding costs
// more, from 2^25 (Q4_K, 20 vectors: 22016 x 2048 30.1 / 27.3; 11008 x 2048
// 20.1 / 18.9 with the weights in the caches, but 22.0 / 22.5 with the
// preparation and weights from HBM) or above 2^24 (Q6_K: 11008 x 2048 29.8 /
// 23.8, 2048 x 5632 15.8 / 16.1); up to 16 vectors from two tiles per CU on (16
// vectors Q8_0 49152 x 2048 27.9 / 29.6, 65536 x 2048 32.4 / 30.9).  Narrow
// heads above 16 vectors (17): Q8_0 49152 x 576 17.5 / 13.8, Q5_0 49152 x 960
// 28.4 / 19.9.  Inside lock-step steps of four 3B blocks (fp16 caches), with
// the SwiGLU and residual epilogues, the same order: all matrices Q4_K, 17
// sessions 410 / 397, 24 427 / 412, 32 474 / 442; Q6_K 550 / 491, 568 / 513,
// 612 / 527.
static bool batch_by_gemm(const QTensor &w, int n)
{
    // (folded tensors serve one session; the GEMM's weight offsets are 32-bit)
    if (n <= 8 || w.fold != 1 || (size_t)w.row_tiles * w.block_quads * 64 * lane_bytes_of(w.dtype) > 0xffffffffUL)
        return false;
    const long tiles = (w.rows + GEMM_BN - 1) / GEMM_BN, weights = (long)w.rows * w.cols;
    if (n <= 16) return tiles >= 2L * gemv_cus();
    return tiles >= gemv_cus() || weights >= 1L << 26 || (w.dtype == DT_Q4_K && weights >= 1L << 25) ||
           (w.dtype == DT_Q6_K && weights > 1L << 24);
}

int launch_gemv(const GemvArgs &a, int epi, hipStream_t s)
{
    if (a.n < 1 || a.n > 32 || a.in.nrows != 2 * a.n || !a.in.q) return -6;
    if (batch_by_gemm(a.w, a.n)) return launch_gemm(a, epi, s);
    int rc;
    switch (a.w.dtype) {
    case DT_Q4_0: rc = launch_gemv_q4(a, epi, s); break;
    case DT_Q5_0: rc = launch_gemv_q5(a, epi, s); break;
    case DT_Q8_0: rc = launch_gemv_q8(a, epi, s); break;
    case DT_Q4_K: rc = launch_gemv_q4k(a, epi, s); break;
    case DT_Q6_K: rc = launch_gemv_q6k(a, epi, s); break;
    default: return -4;
    }
    if (rc) return rc;
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

int launch_gemm(const GemvArgs &a, int epi, hipStream_t s)
{
    if (a.n < 1 || a.in.nrows != 2 * a.n || !a.in.q) return -6;
    int rc;
    switch (a.w.dtype) {
    case DT_Q4_0: rc = launch_gemm_q4(a, epi, s); break;
    case DT_Q5_0: rc = launch_gemm_q5(a, epi, s); break;
    case DT_Q8_0: rc = launch_gemm_q8(a, epi, s); break;
    case DT_Q4_K: rc = launch_gemm_q4k(a, epi, s); break;
    case DT_Q6_K: rc = launch_gemm_q6k(a, epi, s); break;
    default: return -4;
    }
    if (rc) return rc;
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

size_t gemm_part_floats(const QTensor &w, int n)
{
    const int ks = gemm_ks(w, n, (size_t)-1);
    return ks > 1 ? (size_t)ks * n * w.rows : 0;
}

size_t gemm_part_least(const QTensor &w, int n)
{
    const long tiles = (long)((n + 63) / 64) * ((w.rows + 127) / 128);
    int ks = 1;
    while (ks < 4 && tiles * ks < 2L * gemv_cus() && w.fold * w.block_quads / (2 * ks) >= 8) ks *= 2;
    return ks > 1 ? (size_t)ks * n * w.rows : 0;
}

size_t gemv_part_floats(const QTensor &w, int n)
{
    return batch_by_gemm(w, n) ? gemm_part_floats(w, n) : gemv_part_least(w, n);
}

size_t gemv_part_least(const QTensor &w, int n)
{
    if (!gemv_batched(w, n)) return 0;
    GbShape sh;
    gb_plan(w, n, sh);
    size_t f = sh.splits > 1 ? (size_t)sh.splits * n * w.rows : 0;
    Gb16Shape p;
    if (gb16_plan(w, n, p) && p.splits > 1) f = std::max(f, (size_t)p.splits * n * w.rows);
    return f;
}

// k-split finish of the batched matvec: a wave per 64 rows of one vector; the
// lanes of a 16-row tile are a 16-lane group, as the epilogues need.  The
// epilogue's own inputs and the first FS slices' partial sums are loaded
// together, unconditionally (rows past the matrix re-read the last one), so
// the kernel waits for one round trip before the epilogues.
template <int EPI>
__global__ __launch_bounds__(256) void k_gemv_b_finish(GemvArgs a, int splits, int ss_count)
{
#pragma clang fp contract(off)
    constexpr int FS = 16;
    // the arguments of the partial-sum and epilogue-input loads, fetched in
    // one round trip
    sgpr_pin(a.w.rows);
    sgpr_pin(a.n);
    sgpr_pin(a.part);
    sgpr_pin(splits);
    sgpr_pin(ss_count);
    sgpr_pin(a.in.ss);
    sgpr_pin(a.in.ss_stride);
    sgpr_pin(a.in.q);
    sgpr_pin(a.in.tail);
    sgpr_pin(a.out);
    sgpr_pin(a.out_stride);
    if constexpr (EPI == EPI_RESID) sgpr_pin(a.res);
    if constexpr (EPI == EPI_QKV) {
        sgpr_pin(a.kv.layer_off);
        sgpr_pin(a.kv.slot_ids);
        sgpr_pin(a.pos);
        sgpr_pin(a.pos_stride);
        sgpr_pin(a.pos0);
    }
    const int v = blockIdx.y, l = threadIdx.x & 63;
    const int r0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 64;   // the wave's first row
    if (r0 >= a.w.rows) return;   // whole waves past the matrix
    const size_t kstride = (size_t)a.n * a.w.rows;
    const int row = r0 + l;
    const bool act = row < a.w.rows;
    EpiPre pre;
    epi_pre_load(a, EPI, v, row, act, pre);
    float pv[FS];
    const float *pp = a.part + (size_t)v * a.w.rows + min(row, a.w.rows - 1);
#pragma unroll
    for (int k = 0; k < FS; k++) pv[k] = pp[(size_t)min(k, splits - 1) * kstride];
    float nrm = 1.0f;
    if (ss_count) {
        float s = 0.0f;
        for (int i = l; i < ss_count; i += 64) s += a.in.ss[(size_t)v * a.in.ss_stride + i];
        s = wave_sum(s);
        nrm = 1.0f / sqrtf(s / (float)a.w.cols + a.in.eps);
    }
    epi_pre_cs(a, EPI, v, row, act, pre);
    // slices added in ascending order
    float y = 0.0f;
#pragma unroll
    for (int k = 0; k < FS; k++)
        if (k < splits) y += pv[k];
    for (int k = FS; k < splits; k++) y += pp[(size_t)k * kstride];
    y *= nrm;
    epilogue<EPI>(a, row >> 4, row & 15, 16, v, act, y, true, pre);
}

int launch_gemv_b_finish(const GemvArgs &a, int epi, int splits, int ss_count, hipStream_t s)
{
    const dim3 grid((a.w.rows + 255) / 256, a.n), block(256);
    auto go = [&](auto kern) {
        if (a.ev_stop) hipExtLaunchKernelGGL(kern, grid, block, 0, s, nullptr, a.ev_stop, 0, a, splits, ss_count);
        else hipLaunchKernelGGL(kern, grid, block, 0, s, a, splits, ss_count);
    };
    switch (epi) {
    case EPI_STORE: go(k_gemv_b_finish<EPI_STORE>); break;
    case EPI_RESID: go(k_gemv_b_finish<EPI_RESID>); break;
    case EPI_SWIGLU: go(k_gemv_b_finish<EPI_SWIGLU>); break;
    case EPI_QKV: go(k_gemv_b_finish<EPI_QKV>); break;
    default: go(k_gemv_b_finish<EPI_LOGITS>); break;
    }
    return 0;
}

// k-split finish of the prompt GEMM: a work-group per 16 vectors and BR rows
// (a piece of eight inputs or four rows per thread, see epi_runs), the
// partial sums read 16 bytes at a time, up to four ranges in flight.
template <int EPI> constexpr int gfin_rows() { return EPI == EPI_SWIGLU ? 256 : EPI == EPI_RESID ? 128 : 64; }

template <int EPI>
__global__ __launch_bounds__(256) void k_gemm_finish(GemvArgs a, int ks)
{
#pragma clang fp contract(off)
    constexpr int BR = gfin_rows<EPI>();
    __shared__ float s_nrm[16];
    const int m0 = blockIdx.y * 16, r0 = blockIdx.x * BR, tid = threadIdx.x;
    const size_t kstride = (size_t)a.n * a.w.rows;
    if (a.in.ss) {
        gemm_norms<16, 256>(a, m0, s_nrm, tid);
        __syncthreads();
    }
    // rows r0 + rl .. +3 of vector m0 + vi (callers ask for real ones only;
    // the last of an odd row count re-read its own row)
    auto src = [&](int vi, int rl) {
        const int left = a.w.rows - (r0 + rl);
        const float *p = a.part + (size_t)(m0 + vi) * a.w.rows + r0 + rl;
        f32x4 y = {};
        for (int k = 0; k < ks; k += 4) {
            f32x4 q[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const float *pk = p + (size_t)min(k + u, ks - 1) * kstride;
                if (left >= 4) {
                    const f4u t = *(const f4u *)pk;
                    q[u] = f32x4{t[0], t[1], t[2], t[3]};
                } else {
                    q[u] = f32x4{pk[0], pk[min(1, left - 1)], pk[min(2, left - 1)], 0.0f};
                }
            }
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (k + u < ks) y += q[u];
        }
        if (a.in.ss) y *= s_nrm[vi];
        return y;
    };
    if constexpr (EPI == EPI_STORE) {
        const int vi = tid >> 4, rl = 4 * (tid & 15), left = a.w.rows - (r0 + rl);
        if (m0 + vi >= a.n || left <= 0) return;
        const f32x4 y = src(vi, rl);
        float *o = a.out + (size_t)(m0 + vi) * a.out_stride + r0 + rl;
        if (left >= 4) *(f4u *)o = f4u{y[0], y[1], y[2], y[3]};
        else
            for (int i = 0; i < left; i++) o[i] = y[i];
    } else {
        epi_runs<EPI, 16, BR, 256>(a, src, m0, r0, tid);
    }
}

template <int EPI>
static void launch_gfin(const GemvArgs &a, int ks, hipStream_t s)
{
    constexpr int BR = gfin_rows<EPI>();
    const dim3 grid((a.w.rows + BR - 1) / BR, (a.n + 15) / 16), block(256);
    if (a.ev_stop) hipExtLaunchKernelGGL(k_gemm_finish<EPI>, grid, block, 0, s, nullptr, a.ev_stop, 0, a, ks);
    else hipLaunchKernelGGL(k_gemm_finish<EPI>, grid, block, 0, s, a, ks);
}

int launch_gemm_finish(const GemvArgs &a, int epi, int ks, hipStream_t s)
{
    switch (epi) {
    case EPI_STORE: launch_gfin<EPI_STORE>(a, ks, s); break;
    case EPI_RESID: launch_gfin<EPI_RESID>(a, ks, s); break;
    case EPI_SWIGLU: launch_gfin<EPI_SWIGLU>(a, ks, s); break;
    default: launch_gfin<EPI_QKV>(a, ks, s); break;
    }
    return 0;
}

// Standalone operand preparation: one thread per (vector, block of 32,
// k-group), i.e. per 16-byte piece of the operand's high and low rows: two
// 4-float loads, two 16-byte stores; the block's sum of squares meets over
// the four k-group lanes.  Bound by its launch and one load-to-store round
// trip (a 2048-input vector is 256 threads), then by the operand's bytes.
// The earlier thread per 32-value block stored each half separately, 64
// dependent 2-byte stores per thread: 13.2 us at 1 x 2048, now 2.0; 14.4 at
// 32 x 2048, now 3.8.
// VS: log2 of the vectors a wave covers.  The operand interleaves the
// vectors per (block, k-group), so with 16 or more of them a wave takes 16
// vectors of one block (512 contiguous bytes stored per k-group, whole
// 128-byte lines read); with fewer, one vector of 16 blocks.
// x and norm_w carry no alignment beyond a float's.
template <int VS>
__global__ __launch_bounds__(256) void k_act_prep(const float *__restrict__ x, int x_stride, int K, int n, ActOut o)
{
#pragma clang fp contract(off)
    const int l = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int g = l & 3;
    const int v = blockIdx.y * (1 << VS) + ((l >> 2) & ((1 << VS) - 1));
    const int b = ((blockIdx.x * 4 + wid) << (4 - VS)) + (l >> (2 + VS));
    const bool act = v < n && b < K / 32;   // the four lanes of a block alike
    // the k-group's inputs in operand order (the inverse of act_put's map):
    // Q8_0 eight consecutive ones, the nibble formats 4g .. +3 and 16+4g ..
    // +3, each four in the order 0, 2, 1, 3
    const bool q8 = o.dt == DT_Q8_0;
    const int k0 = 32 * b + (q8 ? 8 * g : 4 * g), k1 = k0 + (q8 ? 4 : 16);
    float xv[8] = {}, wv[8];
    if (act) {
        const f4u a0 = *(const f4u *)(x + (size_t)v * x_stride + k0), a1 = *(const f4u *)(x + (size_t)v * x_stride + k1);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            xv[e] = a0[e];
            xv[4 + e] = a1[e];
        }
    }
    if (o.norm_w && act) {
        const f4u w0 = *(const f4u *)(o.norm_w + k0), w1 = *(const f4u *)(o.norm_w + k1);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            wv[e] = w0[e];
            wv[4 + e] = w1[e];
        }
    }
    float ss = 0.0f;
    f16x8 hi, lo;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        ss += xv[e] * xv[e];
        const float t = (o.norm_w ? wv[e] * xv[e] : xv[e]) * ACT_SCALE;
        const _Float16 h = (_Float16)t;
        hi[e] = h;
        lo[e] = (_Float16)((t - (float)h) * LO_SCALE);
    }
    if (!q8) {
        hi = __builtin_shufflevector(hi, hi, 0, 2, 1, 3, 4, 6, 5, 7);
        lo = __builtin_shufflevector(lo, lo, 0, 2, 1, 3, 4, 6, 5, 7);
    }
    ss += __shfl_xor(ss, 1, 64);
    ss += __shfl_xor(ss, 2, 64);
    if (!act) return;
    f16x8 *dst = (f16x8 *)(o.q + (((size_t)b * 4 + g) * o.nrows + 2 * v) * 8);
    dst[0] = hi;
    dst[1] = lo;
    if (o.ss && g == 0) o.ss[(size_t)v * o.ss_stride + b] = ss;
}

int launch_act_prep(const float *x, int x_stride, int K, int n, const ActOut &o, hipStream_t s)
{
    const int nb = K / 32;
    if (n >= 16)
        hipLaunchKernelGGL(k_act_prep<4>, dim3((nb + 3) / 4, (n + 15) / 16), dim3(256), 0, s, x, x_stride, K, n, o);
    else
        hipLaunchKernelGGL(k_act_prep<0>, dim3((nb + 63) / 64, n), dim3(256), 0, s, x, x_stride, K, n, o);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}
