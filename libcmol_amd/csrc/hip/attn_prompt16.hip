// attn_prompt16.hip — prompt-pass attention over an fp16 cache, flash style
// on MFMA: the counterpart of k_attn_prompt (attn.hip) for caches that need
// no high/low split.  A translation unit of its own, beside the decode
// attention kernels' code object.
//
// One work-group of four waves per (kv head, block of QT = 64 / G prompt
// tokens, split of `split` positions), its 64 query rows (row r = token
// r / G, head r % G) sharing every K/V tile.  Wave w owns rows
// 16w .. 16w+15, lane (col, g) row 16w + col.
// The split's positions (up to its last token's) are walked in tiles of 64,
// double-buffered in LDS by direct-to-LDS loads straight from the cache:
//   K: for 16 positions c and k-step s a 1 KiB piece whose lane (col, g) holds
//      dimensions 32s + 8g .. +7 of position 16c + col, gathered by the
//      loads' per-lane addresses: the MFMA operand order, no conversion pass;
//   V: the rows as cached, their 32-byte units (16 dimensions) XOR-swizzled
//      by the row so the transposing reads of four rows fall in different
//      banks.
//   * transposed scores S^T = K Q^T (16x16x32 f16): the query split once into
//      exact f16 high and low parts (q = hi + lo/2048), two products per step;
//   * lazy online softmax as in attn_piece_mfw: a row's reference moves only
//      when a score exceeds it by more than PA_LAZY (in log2 units; a wave
//      vote), so most tiles need no cross-lane step and no rescale; lanes sum
//      their own weights and meet at the end;
//   * weights times 2^13 as f16 high + low parts (at most 2^15; the low part
//      needs no scale of its own, so both products go into one accumulator)
//      are the B operand of O^T = V^T P^T; the A operand comes from V through
//      ds_read_b64_tr_b16 (see attn_piece_mfw).
// Products are exact and sums fp32.  Same partial format as attn_split; a
// token whose positions fit one split is finished here.
//
// Bound: per tile and wave 64 MFMAs (1024 cycles of the matrix pipe), about
// 640 cycles of softmax VALU and 32 KiB of LDS reads (256 cycles of a pipe the
// CU's waves share); 64 KiB of LDS keep two work-groups on a CU.  Before,
// these passes ran the decode split kernel, one work-group per (kv head,
// split, token), each re-reading the token's whole prefix.  At 16/4 heads of
// 128, per layer: 512 tokens behind 1300 positions 314 + 17 us (merge) -> 27 +
// 8, 188 tokens behind 1812 120 + 8 -> 18 + 5.5; 2048 tokens in one pass 68.
// Work-groups of 128 rows (each K/V fragment read once per two row groups,
// 251 VGPRs) took 28.8, 18.7 and 70: the LDS reads do not bound it, and
// the grid halves.
#include "attn_impl.h"

constexpr int PA_TP = 64;            // positions per tile
constexpr float PA_LAZY = 2.0f;      // log2: weights stay below 4
constexpr float PA_WS = 8192.0f;     // weight scale: 4 * 8192 < 65504

template <int DH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_attn_prompt16(AttnArgs a)
{
#pragma clang fp contract(off)
    constexpr int KS = DH / 32, DT = DH / 16, TP = PA_TP, CT = TP / 16;
    constexpr int KB = TP * DH * 2, STAGE = 2 * KB;   // K, then V (bytes)
    constexpr int RPP = 1024 / (2 * DH);              // V rows per 1 KiB piece
    constexpr int VPW = TP / RPP / 4;                 // V pieces per wave
    extern __shared__ __attribute__((aligned(256))) uint8_t smem_p[];

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, col = lane & 15;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = a.n_heads / a.n_kv, QT = 64 / G;
    // the longest prefixes first
    const int kvh = blockIdx.x, vb = (int)(gridDim.y - 1 - blockIdx.y) * QT, sp = blockIdx.z;
    const int nt = min(QT, a.n - vb);
    if (nt <= 0) return;
    const int last = min(a.seqlen[(size_t)(vb + nt - 1) * a.seqlen_stride], a.max_ctx);
    const int pa = sp * a.split, pb = min(pa + a.split, last);
    if (pa >= last) return;
    const int whole = min(min(a.seqlen[(size_t)vb * a.seqlen_stride], a.max_ctx), pb);   // visible to every row
    const float scale = 1.0f / sqrtf((float)DH), c2 = scale * 1.44269504088896341f;
    const float lazy = PA_LAZY / c2;

    const size_t off = kv_offset(a.kv, 0) + (size_t)kvh * a.max_ctx * DH;
    const uint8_t *kb = (const uint8_t *)uniform_ptr((const _Float16 *)a.kv.k_base + off);
    const uint8_t *vbp = (const uint8_t *)uniform_ptr((const _Float16 *)a.kv.v_base + off);
    // this lane's piece of a V row: row lane / (DH / 8) of the piece, LDS
    // unit u holding dimensions 16 (u ^ f(row)) .. +15
    const int vrow = lane / (DH / 8), vch = lane % (DH / 8);
    auto issue = [&](int st, int p0) {
        uint8_t *dst = smem_p + st * STAGE;
        const uint32_t kp = (uint32_t)min(p0 + 16 * wid + col, last - 1) * (2 * DH) + 16 * g;
#pragma unroll
        for (int s = 0; s < KS; s++)
            __builtin_amdgcn_global_load_lds((const gvoid_t *)(kb + kp + 64 * s),
                                             (lvoid_t *)(dst + (wid * KS + s) * 1024), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < VPW; i++) {
            const int r = (wid * VPW + i) * RPP + vrow;   // row of the tile
            const int f = DH == 128 ? r & 7 : (r >> 1) & 3;
            const uint32_t vp = (uint32_t)min(p0 + r, last - 1) * (2 * DH) +
                                32 * ((vch >> 1) ^ f) + 16 * (vch & 1);
            __builtin_amdgcn_global_load_lds((const gvoid_t *)(vbp + vp),
                                             (lvoid_t *)(dst + KB + (wid * VPW + i) * 1024), 16, 0, 0);
        }
    };
    issue(0, pa);

    // query operands of this lane's row 16w + col = (token at, head ah)
    const int ar = 16 * wid + col, at = ar / G, ah = ar - at * G;
    const bool arow = at < nt;
    f16x8 qh[KS], ql[KS];
    const float *qp = a.q + (size_t)(vb + (arow ? at : 0)) * a.q_stride + (size_t)(kvh * G + ah) * DH;
#pragma unroll
    for (int s = 0; s < KS; s++) {
        const float4 q0 = *(const float4 *)(qp + 32 * s + 8 * g), q1 = *(const float4 *)(qp + 32 * s + 8 * g + 4);
        const float qv[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float x = arow ? qv[e] : 0.0f;
            const _Float16 hi = (_Float16)x;
            qh[s][e] = hi;
            ql[s][e] = (_Float16)((x - (float)hi) * 2048.0f);
        }
    }
    const int L = arow ? min(a.seqlen[(size_t)(vb + at) * a.seqlen_stride], a.max_ctx) : 0;
    const int lim = min(L, pb);   // visible positions of this split: pa .. lim-1
    const f32x4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 o[DT];
#pragma unroll
    for (int t = 0; t < DT; t++) o[t] = zero4;
    // mk = -m c2; a row with no visible position yet (m = -inf) has weights 0
    float m = -INFINITY, mk = 0.0f, lsum = 0.0f;
    // transposing reads: this lane's bytes of row 4g + col/4 (+ 16 per c) of
    // dimension tile t at vaddr ^ 32t
    const int vr = 4 * g + (col >> 2);
    const uint32_t vaddr = (uint32_t)(vr * (2 * DH) + 32 * (DH == 128 ? vr & 7 : (vr >> 1) & 3) + 8 * (col & 3));

    int st = 0;
    for (int p0 = pa; p0 < pb; p0 += TP, st ^= 1) {
        // the tile has landed and every wave is done with the other stage
        __builtin_amdgcn_s_waitcnt(WAITCNT_VM_LGKM0(0));
        __syncthreads();
        if (p0 + TP < pb) issue(st ^ 1, p0 + TP);
        const uint8_t *ks_ = smem_p + st * STAGE, *vs_ = ks_ + KB;
        // ---- scores: sc[c][i] = position p0 + 16c + 4g + i of this lane's row
        float sc[CT][4];
#pragma unroll
        for (int c = 0; c < CT; c++) {
            f32x4 s1 = zero4, s2 = zero4;
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const f16x8 kf = *(const f16x8 *)(ks_ + (c * KS + s) * 1024 + lane * 16);
                s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qh[s], s1, 0, 0, 0);
                s2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, ql[s], s2, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) sc[c][i] = fmaf(s2[i], 1.0f / 2048.0f, s1[i]);
        }
        if (p0 + TP > whole) {   // uniform: the causal edge and the split's end
#pragma unroll
            for (int c = 0; c < CT; c++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (p0 + 16 * c + 4 * g + i >= lim) sc[c][i] = -INFINITY;
        }
        // ---- online softmax of the row (its scores: lanes col + 16 g) ----
        float mx = sc[0][0];
#pragma unroll
        for (int c = 0; c < CT; c++)
#pragma unroll
            for (int i = 0; i < 4; i++) mx = fmaxf(mx, sc[c][i]);
        if (__ballot(mx > m + lazy)) {
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float mn = fmaxf(m, mx);
            const float mref = mn == -INFINITY ? 0.0f : mn;
            const float al = mn == m ? 1.0f : __builtin_amdgcn_exp2f((m - mref) * c2);
            m = mn;
            mk = -mref * c2;
            lsum *= al;
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) o[t][i] *= al;
        }
        f16x8 ph[CT / 2], pl[CT / 2];
#pragma unroll
        for (int c = 0; c < CT; c++) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float e = __builtin_amdgcn_exp2f(fmaf(sc[c][i], c2, mk));
                lsum += e;
                const _Float16 hi = (_Float16)fmaf(e, PA_WS, 0.0f);
                ph[c >> 1][4 * (c & 1) + i] = hi;
                pl[c >> 1][4 * (c & 1) + i] = (_Float16)fmaf(e, PA_WS, -(float)hi);
            }
        }
        // ---- O^T += V^T P^T: k-step k covers positions 32k + 4g .. +3 and 32k + 16 + 4g .. +3
#pragma unroll
        for (int k = 0; k < CT / 2; k++) {
#pragma unroll
            for (int t = 0; t < DT; t++) {
                typedef short s16x4 __attribute__((ext_vector_type(4)));
                typedef __attribute__((address_space(3))) s16x4 ls16x4;
                const uint8_t *src = vs_ + 32 * k * (2 * DH) + (vaddr ^ (32u * t));
                const s16x4 lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls16x4 *)src);
                const s16x4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls16x4 *)(src + 16 * (2 * DH)));
                const f16x8 vf = __builtin_bit_cast(f16x8, __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
                o[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, ph[k], o[t], 0, 0, 0);
                o[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pl[k], o[t], 0, 0, 0);
            }
        }
    }

    // ---- outputs: lane (col, g) holds dimensions 16t + 4g + i of its row ----
    lsum += __shfl_xor(lsum, 16, 64);
    lsum += __shfl_xor(lsum, 32, 64);
    const int nact = (L + a.split - 1) / a.split;
    if (!arow || sp >= nact) return;   // no positions of this token here
    const int v = vb + at;
    if (nact == 1) {
        const float inv = 1.0f / lsum;
#pragma unroll
        for (int t = 0; t < DT; t++) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float ov = o[t][i] * (1.0f / PA_WS) * inv;
                const int k = (kvh * G + ah) * DH + 16 * t + 4 * g + i;
                if (a.out) a.out[(size_t)v * a.out_stride + k] = ov;
                if (a.next.q) act_put(a.next, v, k, ov);
            }
        }
    } else {
        const size_t sb = (((size_t)v * a.n_kv + kvh) * a.max_splits + sp) * G + ah;
#pragma unroll
        for (int t = 0; t < DT; t++) {
            float4 ov;
            ov.x = o[t][0] * (1.0f / PA_WS);
            ov.y = o[t][1] * (1.0f / PA_WS);
            ov.z = o[t][2] * (1.0f / PA_WS);
            ov.w = o[t][3] * (1.0f / PA_WS);
            *(float4 *)&a.po[sb * DH + 16 * t + 4 * g] = ov;
        }
        if (g == 0) {
            a.pm[sb] = m * scale;   // natural units, as the merge reads them
            a.pl[sb] = lsum;
        }
    }
}

template <int DH>
static int go(const AttnArgs &a, hipStream_t s)
{
    constexpr int LDS = 2 * 2 * PA_TP * DH * 2;
    static const bool lds_ok =
        hipFuncSetAttribute((const void *)k_attn_prompt16<DH>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) ==
        hipSuccess;
    if (!lds_ok) return -4;
    const int QT = 64 / (a.n_heads / a.n_kv);
    const dim3 grid(a.n_kv, (a.n + QT - 1) / QT, a.max_splits), block(256);
    hipLaunchKernelGGL(k_attn_prompt16<DH>, grid, block, LDS, s, a);
    return a.max_splits > 1 ? launch_attn_merge_wave(a, s) : 0;
}

int launch_attn_prompt16(const AttnArgs &a, hipStream_t s)
{
    return a.d_head == 128 ? go<128>(a, s) : go<64>(a, s);
}
