// attn.hip — the decode attention kernels over the work-group functions of
// attn_impl.h: one work-group of ATT_THREADS per (kv head, split, vector),
// then one per (query head, vector) to merge the splits.
#include "attn_impl.h"

#define ATT_THREADS 256
// Positions per chunk of a 256-thread work-group (a split is a multiple).
#define ATT_CHUNK (ATT_THREADS / 4)

template <int DH, typename KT>
__global__ __launch_bounds__(ATT_THREADS) void k_attn(AttnArgs a)
{
    if constexpr (sizeof(KT) == 2 && DH >= 64 && ATT_THREADS == 256)
        attn_split_mf<DH, StPlain>(a, blockIdx.x, blockIdx.y, blockIdx.z);
    else
        attn_split<DH, KT, ATT_THREADS, StPlain>(a, blockIdx.x, blockIdx.y, blockIdx.z);
}

template <int DH>
__global__ __launch_bounds__(ATT_THREADS) void k_attn_merge(AttnArgs a)
{
    attn_merge_head<DH, ATT_THREADS, StPlain>(a, blockIdx.x, blockIdx.y);
}

// Head-per-wave decode attention for d_head 64 and 128: one work-group of
// four waves per (kv head, split, vector); wave w serves query heads w and
// w + 4 of the group.  The split is walked in chunks of CH (32 or 64) positions whose
// K and V rows are staged in LDS by all 256 threads (coalesced 16-byte
// loads of the next chunk are in flight while the current one is used):
//   * scores: four lanes per position, each holding a quarter of the head's
//     query in registers (interleaved 16-byte pieces) against the same pieces
//     of the K row; K rows are padded to an odd multiple of 64 bytes so the
//     four rows a 16-lane pass reads fall in alternate LDS bank halves;
//   * online softmax over the 64 scores with wave reductions;
//   * weighted sum with lanes over the dimensions: each position's weight is
//     broadcast with readlane and its V row read once per wave.
// With NWV = 8 waves and at most four query heads per kv head, two waves
// serve each head, each on one half of every chunk's positions (their
// online softmaxes meet at the end of the split), so each wave's dependent
// chains are half as long and two waves share a SIMD; with more heads wave
// w serves head w alone.
// Same partial format as attn_split, merged by k_attn_merge.
#define ATH_CH 64
template <int DH, typename KT, int CH, int NWV>
__global__ __launch_bounds__(NWV * 64) void k_attn_h(AttnArgs a)
{
#pragma clang fp contract(off)
    constexpr int RB = DH * (int)sizeof(KT);        // row bytes
    constexpr int KS = RB + 64;                      // padded K row stride (bytes)
    constexpr int PE = 16 / (int)sizeof(KT);         // elements per 16-byte piece
    constexpr int NPL = RB / 16 / 4;                 // pieces per lane (a quarter of the row)
    constexpr int DL = DH / 64;                      // output dims per lane
    constexpr int NT = NWV * 64;
    constexpr int UNITS = CH * RB / 16;              // 16-byte units of a chunk's K (and of V)
    constexpr int UPT = UNITS / NT;                  // per thread
    constexpr int PS = CH / 16;                      // 16-position passes per chunk
    static_assert(UNITS % NT == 0 && CH % 16 == 0, "chunk size");
    static_assert(NWV == 4 || (NWV == 8 && PS % 2 == 0), "waves");
    __shared__ __attribute__((aligned(16))) uint8_t ks[2][CH * KS];
    __shared__ __attribute__((aligned(16))) uint8_t vs[2][CH * RB];
    __shared__ float xm[4], xl[4], xo[4][DH];        // NWV = 8: the second halves' results

    const int kvh = blockIdx.x, sp = blockIdx.y, n = blockIdx.z;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the prologue's launch arguments in one batch of loads, then the
    // vector's length and cache slot together (the slot read from a valid
    // address either way): two round trips before the K/V loads, not four
    sgpr_pin(a.seqlen);
    sgpr_pin(a.seqlen_stride);
    sgpr_pin(a.max_ctx);
    sgpr_pin(a.split);
    sgpr_pin(a.kv.k_base);
    sgpr_pin(a.kv.v_base);
    sgpr_pin(a.kv.slot_ids);
    sgpr_pin(a.kv.slot_stride);
    sgpr_pin(a.kv.layer_off);
    sgpr_pin(a.q);
    sgpr_pin(a.q_stride);
    const int32_t *lenp = a.seqlen + (size_t)n * a.seqlen_stride;
    const int32_t *slotp = a.kv.slot_ids ? a.kv.slot_ids + n : lenp;
    const int len = *lenp, slot = *slotp;
    sgpr_pin(len);
    sgpr_pin(slot);
    const int G = a.n_heads / a.n_kv;
    const int L = min(len, a.max_ctx);
    const int t0 = sp * a.split;
    if (t0 >= L) return;
    const int cnt = min(L, t0 + a.split) - t0;
    const int nch = (cnt + CH - 1) / CH;
    const int nact = (L + a.split - 1) / a.split;
    const size_t kvo = kv_offset_of(a.kv, n, slot);
    const size_t off = kvo + (size_t)kvh * a.max_ctx * DH + (size_t)t0 * DH;
    const uint8_t *kb = (const uint8_t *)((const KT *)a.kv.k_base + off);
    const uint8_t *vb = (const uint8_t *)((const KT *)a.kv.v_base + off);

    // staging: thread tid moves units tid + NT u of K and V (rows past the
    // split re-read its last row; their weights are zero)
    u32x4 kr[UPT], vr[UPT];
    auto fetch = [&](int c) {
#pragma unroll
        for (int u = 0; u < UPT; u++) {
            const int unit = tid + NT * u, row = unit / (RB / 16), col = unit % (RB / 16);
            const size_t src = (size_t)min(c * CH + row, cnt - 1) * RB + col * 16;
            kr[u] = ldg((const u32x4 *)(kb + src));
            vr[u] = ldg((const u32x4 *)(vb + src));
        }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int u = 0; u < UPT; u++) {
            const int unit = tid + NT * u, row = unit / (RB / 16), col = unit % (RB / 16);
            *(u32x4 *)&ks[buf][row * KS + col * 16] = kr[u];
            *(u32x4 *)&vs[buf][row * RB + col * 16] = vr[u];
        }
    };

    // queries of this wave's heads: lane quarter j holds pieces j, j+4, ...
    // (NWV = 8: head hw, passes ps0 .. ps0 + PSW - 1 of each chunk)
    const int j = lane & 3;
    constexpr bool PAIRS = NWV == 8;
    constexpr int PSW = PAIRS ? PS / 2 : PS;
    const int hw = PAIRS ? (wid & 3) : wid, half = PAIRS ? (wid >> 2) : 0;
    const int ps0 = half * PSW;
    const int nh = PAIRS ? (hw < G ? 1 : 0) : (wid < G ? (wid + 4 < G ? 2 : 1) : 0);
    float q[2][NPL * PE];
    float m[2], l[2], o[2][DL];
#pragma unroll
    for (int hh = 0; hh < 2; hh++) {
        m[hh] = -INFINITY;
        l[hh] = 0.0f;
#pragma unroll
        for (int d = 0; d < DL; d++) o[hh][d] = 0.0f;
        const int g = min(PAIRS ? hw : wid + 4 * hh, G - 1);
        const float *qh = a.q + (size_t)n * a.q_stride + (size_t)(kvh * G + g) * DH;
#pragma unroll
        for (int i = 0; i < NPL; i++)
#pragma unroll
            for (int e = 0; e < PE; e++) q[hh][i * PE + e] = ldg(qh + (j + 4 * i) * PE + e);
    }
    // scores and m stay raw dot products; a weight is 2^((t - m) c) with
    // c = log2(e)/sqrt(d_head) on the hardware exponential (exp2(-inf) = 0)
    const float scale = 1.0f / sqrtf((float)DH), c2 = scale * 1.44269504088896341f;

    fetch(0);
    put(0);
    __syncthreads();
    for (int c = 0; c < nch; c++) {
        const int buf = c & 1;
        if (c + 1 < nch) fetch(c + 1);
        const int np = min(CH, cnt - c * CH);
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
            if (hh >= nh) break;
            // scores: pass ps covers positions 16 ps + lane/4
            float sc[PSW];
#pragma unroll
            for (int pw = 0; pw < PSW; pw++) {
                const int ps = ps0 + pw;
                const uint8_t *kr0 = &ks[buf][(16 * ps + (lane >> 2)) * KS];
                float dot = 0.0f;
#pragma unroll
                for (int i = 0; i < NPL; i++) {
                    const u32x4 w = *(const u32x4 *)(kr0 + (j + 4 * i) * 16);
                    float kv[PE];
                    if constexpr (sizeof(KT) == 4) {
                        const f32x4 wf = __builtin_bit_cast(f32x4, w);
#pragma unroll
                        for (int e = 0; e < 4; e++) kv[e] = wf[e];
                    } else {
                        const f16x8 h8 = __builtin_bit_cast(f16x8, w);
#pragma unroll
                        for (int e = 0; e < 8; e++) kv[e] = (float)h8[e];
                    }
#pragma unroll
                    for (int e = 0; e < PE; e++) dot = fmaf(q[hh][i * PE + e], kv[e], dot);
                }
                dot += __shfl_xor(dot, 1, 64);
                dot += __shfl_xor(dot, 2, 64);
                sc[pw] = (16 * ps + (lane >> 2)) < np ? dot : -INFINITY;   // raw score
            }
            float mc = sc[0];
#pragma unroll
            for (int pw = 1; pw < PSW; pw++) mc = fmaxf(mc, sc[pw]);
            mc = wave_max(mc);
            const float mn = fmaxf(m[hh], mc);
            // a half-chunk wave may not have met a valid position yet
            // (uniform over the wave)
            if (PAIRS && mn == -INFINITY) continue;
            float ev[PSW], ls = 0.0f;
#pragma unroll
            for (int pw = 0; pw < PSW; pw++) {
                ev[pw] = __builtin_amdgcn_exp2f((sc[pw] - mn) * c2);
                if (j == 0) ls += ev[pw];
            }
            ls = wave_sum(ls);
            const float al = __builtin_amdgcn_exp2f((m[hh] - mn) * c2);
            l[hh] = l[hh] * al + ls;
            m[hh] = mn;
#pragma unroll
            for (int d = 0; d < DL; d++) o[hh][d] *= al;
            // weighted sum: lane covers dims DL*lane ..
#pragma unroll
            for (int pw = 0; pw < PSW; pw++) {
                const int ps = ps0 + pw;
#pragma unroll 4
                for (int r = 0; r < 16; r++) {
                    const float ep = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ev[pw]), 4 * r));
                    const uint8_t *vrow = &vs[buf][(16 * ps + r) * RB];
                    if constexpr (sizeof(KT) == 4) {
                        if constexpr (DL == 2) {
                            const float2 v = *(const float2 *)(vrow + lane * 8);
                            o[hh][0] = fmaf(ep, v.x, o[hh][0]);
                            o[hh][1] = fmaf(ep, v.y, o[hh][1]);
                        } else {
                            o[hh][0] = fmaf(ep, *(const float *)(vrow + lane * 4), o[hh][0]);
                        }
                    } else {
                        if constexpr (DL == 2) {
                            const f16x2 v = *(const f16x2 *)(vrow + lane * 4);
                            o[hh][0] = fmaf(ep, (float)v[0], o[hh][0]);
                            o[hh][1] = fmaf(ep, (float)v[1], o[hh][1]);
                        } else {
                            o[hh][0] = fmaf(ep, (float)*(const _Float16 *)(vrow + lane * 2), o[hh][0]);
                        }
                    }
                }
            }
        }
        if (c + 1 < nch) {
            __syncthreads();   // every wave is done with the other buffer
            put(buf ^ 1);
            __syncthreads();
        }
    }

    // NWV = 8: the second halves hand their (m, l, o) to the first, which
    // combine them with the log-sum-exp rule
    if constexpr (PAIRS) {
        if (half == 1 && nh) {
#pragma unroll
            for (int d = 0; d < DL; d++) xo[hw][DL * lane + d] = o[0][d];
            if (lane == 0) {
                xm[hw] = m[0];
                xl[hw] = l[0];
            }
        }
        __syncthreads();
        if (half == 1) return;
        if (nh) {
            const float m1 = xm[hw], M = fmaxf(m[0], m1);
            const float a0 = m[0] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m[0] - M) * c2);
            const float a1 = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m1 - M) * c2);
            l[0] = l[0] * a0 + xl[hw] * a1;
            m[0] = M;
#pragma unroll
            for (int d = 0; d < DL; d++) o[0][d] = o[0][d] * a0 + xo[hw][DL * lane + d] * a1;
        }
    }
    // partials (or the finished output when the session fits one split)
    const bool single = nact == 1;
    const size_t sbase = (((size_t)n * a.n_kv + kvh) * a.max_splits + sp) * G;
#pragma unroll
    for (int hh = 0; hh < 2; hh++) {
        if (hh >= nh) break;
        const int g = PAIRS ? hw : wid + 4 * hh;
#pragma unroll
        for (int d = 0; d < DL; d++) {
            const int dim = DL * lane + d;
            if (single) {
                const float ov = o[hh][d] / l[hh];
                const int k = (kvh * G + g) * DH + dim;
                if (a.out) a.out[(size_t)n * a.out_stride + k] = ov;
                if (a.next.q) act_put(a.next, n, k, ov);
            } else {
                a.po[(sbase + g) * DH + dim] = o[hh][d];
            }
        }
        if (!single && lane == 0) {
            a.pm[sbase + g] = m[hh] * scale;   // natural units, as the merge reads them
            a.pl[sbase + g] = l[hh];
        }
    }
}

// One wave per (head of q|k|v, vector): lane l holds dims DL*l .. DL*l+DL-1
// (DL = d_head/64; d_head 16/32 use the first d_head lanes).  q and k heads:
// RMSNorm s = 1/sqrtf(sum x^2 / d_head + eps), y = w * (x * s) (the
// reference's cmol_rms_norm order, wave-order sum), then RoPE on the pairs
// (2i, 2i+1) with the QKV epilogue's arithmetic; then q -> a.q, k and v ->
// the cache at the vector's position.
template <int DL>
__global__ __launch_bounds__(64) void k_qk_rope(QkArgs a)
{
#pragma clang fp contract(off)
    const int hh = blockIdx.x, v = blockIdx.y, lane = threadIdx.x;
    const int dh = a.d_head;
    const bool isq = hh < a.n_heads, isk = !isq && hh < a.n_heads + a.n_kv;
    const int row0 = hh * dh;   // q rows, then k rows, then v rows
    const bool act = lane * DL < dh;
    const float *src = a.raw + (size_t)v * a.raw_stride + row0;
    float x[DL];
#pragma unroll
    for (int j = 0; j < DL; j++) x[j] = act ? src[lane * DL + j] : 0.0f;
    const float *w = isq ? a.qn_w : isk ? a.kn_w : nullptr;
    if (w) {
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < DL; j++) ss += x[j] * x[j];
        ss = wave_sum(ss);
        const float sc = 1.0f / sqrtf(ss / (float)dh + a.eps);
#pragma unroll
        for (int j = 0; j < DL; j++) x[j] = act ? w[lane * DL + j] * (x[j] * sc) : 0.0f;
    }
    const int pos = min(max(a.pos[(size_t)v * a.pos_stride], 0), a.max_ctx - 1);
    if ((isq || isk) && a.rope_on) {
        float partner[DL];
        if constexpr (DL >= 2) {
#pragma unroll
            for (int j = 0; j < DL; j++) partner[j] = x[j ^ 1];
        } else {
            partner[0] = __shfl_xor(x[0], 1, 64);
        }
        float y[DL];
#pragma unroll
        for (int j = 0; j < DL; j++) {
            const int i = lane * DL + j;
            const float *cs = a.rope + ((size_t)pos * (dh / 2) + (i >> 1)) * 2;
            const float c = act ? cs[0] : 1.0f, sn = act ? cs[1] : 0.0f;
            y[j] = !(i & 1) ? x[j] * c - partner[j] * sn : partner[j] * sn + x[j] * c;
        }
#pragma unroll
        for (int j = 0; j < DL; j++) x[j] = y[j];
    }
    if (!act) return;
    if (isq) {
#pragma unroll
        for (int j = 0; j < DL; j++) a.q[(size_t)v * a.q_stride + row0 + lane * DL + j] = x[j];
        return;
    }
    const int kvh = isk ? hh - a.n_heads : hh - a.n_heads - a.n_kv;
    const size_t o = kv_offset(a.kv, v) + ((size_t)kvh * a.max_ctx + pos) * dh + lane * DL;
    void *base = isk ? a.kv.k_base : a.kv.v_base;
#pragma unroll
    for (int j = 0; j < DL; j++) {
        if (a.kv_f16) ((_Float16 *)base)[o + j] = (_Float16)x[j];
        else ((float *)base)[o + j] = x[j];
    }
}

int launch_qk_rope(const QkArgs &a, hipStream_t s)
{
    if (a.n < 1 || a.d_head < 16 || a.d_head > 256 || (a.d_head & (a.d_head - 1))) return -4;
    const dim3 grid(a.n_heads + 2 * a.n_kv, a.n), block(64);
    switch (a.d_head) {
    case 256: hipLaunchKernelGGL(k_qk_rope<4>, grid, block, 0, s, a); break;
    case 128: hipLaunchKernelGGL(k_qk_rope<2>, grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL(k_qk_rope<1>, grid, block, 0, s, a); break;
    }
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

int attn_max_splits(int max_ctx, int split) { return (max_ctx + split - 1) / split; }

int launch_attn(const AttnArgs &a, hipStream_t s)
{
    const int G = a.n_heads / a.n_kv;
    // splits of whole 64-position chunks, or (head-per-wave kernel, d_head
    // 64 / 128) of whole 32-position chunks
    const bool half_chunks = a.split % ATT_CHUNK != 0;
    if (G < 1 || G > ATT_MAX_G || a.n_heads % a.n_kv || a.split < 1 || a.split % (ATT_CHUNK / 2) ||
        (half_chunks && a.d_head != 64 && a.d_head != 128))
        return -4;
    if (a.max_splits > ATT_MAX_MERGE) return -4;
    dim3 grid(a.n_kv, a.max_splits, a.n), block(ATT_THREADS), mgrid(a.n_heads, a.n);
    if (a.bal > 0) return launch_attn_bal(a, s);
#define ATT(DHV)                                                                          \
    if (a.kv_f16) hipLaunchKernelGGL((k_attn<DHV, _Float16>), grid, block, 0, s, a);      \
    else hipLaunchKernelGGL((k_attn<DHV, float>), grid, block, 0, s, a);
#define ATH(DHV)                                                                                      \
    if (half_chunks) {                                                                                \
        if (a.kv_f16) hipLaunchKernelGGL((k_attn_h<DHV, _Float16, 32, 4>), grid, block, 0, s, a);     \
        else hipLaunchKernelGGL((k_attn_h<DHV, float, 32, 4>), grid, block, 0, s, a);                \
    } else if (h8) {                                                                                  \
        if (a.kv_f16) hipLaunchKernelGGL((k_attn_h<DHV, _Float16, ATH_CH, 8>), grid, block8, 0, s, a); \
        else hipLaunchKernelGGL((k_attn_h<DHV, float, ATH_CH, 8>), grid, block8, 0, s, a);           \
    } else {                                                                                          \
        if (a.kv_f16) hipLaunchKernelGGL((k_attn_h<DHV, _Float16, ATH_CH, 4>), grid, block, 0, s, a); \
        else hipLaunchKernelGGL((k_attn_h<DHV, float, ATH_CH, 4>), grid, block, 0, s, a);            \
    }
    // head-per-wave kernel for short splits (one or two chunks); the
    // thread-per-dimension kernel streams long splits better
    const char *e = getenv("CMOL_ATTN_H");
    const bool head_waves = half_chunks || (e ? e[0] == '1' : a.split <= 2 * ATH_CH);
    // eight waves (two per query head) when the kv head has at most four
    // query heads (CMOL_ATTN_H8=0: four waves, measurements)
    static const bool h8_on = [] {
        const char *v = getenv("CMOL_ATTN_H8");
        return !(v && v[0] == '0');
    }();
    const bool h8 = h8_on && G <= 4;
    const dim3 block8(512);
    switch (a.d_head) {
    case 16: ATT(16); break;
    case 32: ATT(32); break;
    case 64: if (head_waves) { ATH(64); } else { ATT(64); } break;
    case 128: if (head_waves) { ATH(128); } else { ATT(128); } break;
    case 256: ATT(256); break;
    default: return -4;
    }
    if (a.max_splits > 1) {
        switch (a.d_head) {
        case 16: hipLaunchKernelGGL((k_attn_merge<16>), mgrid, block, 0, s, a); break;
        case 32: hipLaunchKernelGGL((k_attn_merge<32>), mgrid, block, 0, s, a); break;
        case 64: hipLaunchKernelGGL((k_attn_merge<64>), mgrid, block, 0, s, a); break;
        case 128: hipLaunchKernelGGL((k_attn_merge<128>), mgrid, block, 0, s, a); break;
        default: hipLaunchKernelGGL((k_attn_merge<256>), mgrid, block, 0, s, a); break;
        }
    }
#undef ATT
#undef ATH
    return hipGetLastError() == hipSuccess ? 0 : -4;
}
