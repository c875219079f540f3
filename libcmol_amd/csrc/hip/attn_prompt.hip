// attn_prompt.hip — prompt-pass attention, flash style on MFMA: the n vectors
// are consecutive prompt tokens of one session (vector v at position
// seqlen[v] - 1).  A translation unit of its own, beside the decode attention
// kernels' code object.
//
// One work-group of eight waves per (kv head, block of QT = 64 / G prompt
// tokens, split of `split` positions): its 64 query rows (row r = token
// r / G, head r % G) share every K/V tile.  The split's positions (up to its
// last token's) are walked in pairs of tiles of TP positions, one tile per
// half of the work-group, each copied into LDS with direct-to-LDS loads
// while the previous one is used.  Wave w4 of a half owns query rows
// 16 w4 .. +15, lane (col, g) row 16 w4 + col, over the half's tiles; the
// halves' softmaxes and outputs meet at the end.
//
// fp16 cache (TP = 64), tiles straight from the cache:
//   K: for 16 positions c and k-step s a 1 KiB piece whose lane (col, g) holds
//      dimensions 32s + 8g .. +7 of position 16c + col, gathered by the
//      loads' per-lane addresses: the MFMA operand order;
//   V: the rows as cached, their 32-byte units (16 dimensions) XOR-swizzled
//      by the row so the transposing reads of four rows fall in different
//      banks.
// fp32 cache (TP = 32), from the exact f16 high and low parts (x = hi +
// lo / 2048) that k_kv_hilo lays out once per pass and layer, per (kv head,
// 32-position tile):
//   K: the same pieces, a high and a low one each;
//   V: for dimension tile t a high and a low piece whose lane (col, g) holds
//      dimension 16t + col of positions 4g .. 4g+3 and 16+4g .. 16+4g+3 (the
//      positions whose scores that lane holds after the score products).
// Positions past `last` repeat position last-1, so every value is finite.
//   * transposed scores S^T = K Q^T (16x16x32 f16), the query split once into
//      exact f16 high and low parts: lane (col, g) holds positions
//      16c + 4g + i of its row, those past the row's token masked (causal).
//      Two products per step over fp16, three over fp32 (the dropped
//      low.low term is below 2^-22 of each product);
//   * lazy online softmax as in attn_piece_mfw: a row's reference moves only
//      when a score exceeds it by more than PA_LAZY (in log2 units; a wave
//      vote), so most tiles need no cross-lane step and no rescale; lanes sum
//      their own weights and meet at the end;
//   * the weights, as exact f16 high and low parts, are the B operand of
//      O^T = V^T P^T; products with a low part (of the weights, of V) have an
//      accumulator of their own, so the output takes one rounding per tile.
//      Over fp16 the A operand comes from V through ds_read_b64_tr_b16 (see
//      attn_piece_mfw).
// Products are exact and sums fp32.  A masked position's weight is 0, so a
// cached V row that is not finite would make the earlier tokens that share its
// tile NaN (0 * inf); a work-group whose outputs are not all finite walks its
// split again with such rows taken apart, and only the rows that attend to one
// are NaN, as in a decode of the tokens one by one.  A token whose positions
// fit one split is finished here; otherwise each split leaves (max, sum of
// exp, unnormalised output) in the partial format of attn_split and
// k_attn_merge_wave combines them.
//
// Bound: latency and the causal imbalance.  Per tile a wave has 1024 (fp16)
// or 768 (fp32) cycles of the matrix pipe and about 640 of softmax VALU in a
// dependent chain, and the work-group reads 128 KiB (fp32 256) of LDS; a
// block's work grows with its position, so the longest prefixes start first.
// With four waves per work-group (one tile at a time, every block of a
// 2048-token pass resident at once) a pass lasted as long as its longest
// block.  Per layer at 16/4 heads of 128, 2048 tokens over fp32: 116 -> 73-88
// us.  Over fp16, where such passes ran the decode split kernel (one
// work-group per token): 512 tokens behind 1300 positions 314 + 17 us (merge)
// -> 31 + 6, 188 behind 1812 120 + 8 -> 20 + 5.  Work-groups of 128 query
// rows, each K/V fragment read once for two row groups (four waves): 70
// against 68 us at 2048 tokens over fp16, 28.8 against 26.8 at 512.
#include "attn_impl.h"
#include "lds_limit.h"

#include <algorithm>

constexpr float PA_LAZY = 2.0f;      // log2: weights stay below 4
constexpr int PA_NT = 512;
constexpr int KVT_POS = 32;          // positions per tile of the high/low copy

template <int DH>
constexpr int kvt_halves() { return KVT_POS * DH * 4; }   // K and V, high and low

template <int DH>
__global__ __launch_bounds__(256) void k_kv_hilo(AttnArgs a, int last, _Float16 *hl, int tiles)
{
#pragma clang fp contract(off)
    constexpr int KS = DH / 32, DT = DH / 16, TH = kvt_halves<DH>(), KH = TH / 2;
    const int kvh = blockIdx.x, tile = blockIdx.y, tid = threadIdx.x;
    const int p0 = tile * KVT_POS;
    const size_t off = kv_offset(a.kv, 0) + (size_t)kvh * a.max_ctx * DH;
    const float *kb = (const float *)a.kv.k_base + off;
    const float *vb = (const float *)a.kv.v_base + off;
    _Float16 *dst = hl + ((size_t)kvh * tiles + tile) * TH;
    for (int it = tid; it < 2 * KS * 64; it += 256) {
        const int lane = it & 63, cs = it >> 6, c = cs / KS, s = cs - c * KS;
        const int p = min(p0 + 16 * c + (lane & 15), last - 1);
        const float4 *src = (const float4 *)(kb + (size_t)p * DH + 32 * s + 8 * (lane >> 4));
        const float4 x0 = src[0], x1 = src[1];
        const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
        f16x8 hi, lo;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            hi[e] = (_Float16)x[e];
            lo[e] = (_Float16)((x[e] - (float)hi[e]) * 2048.0f);
        }
        *(f16x8 *)&dst[(cs * 2) * 512 + lane * 8] = hi;
        *(f16x8 *)&dst[(cs * 2 + 1) * 512 + lane * 8] = lo;
    }
    for (int it = tid; it < DT * 64; it += 256) {
        const int lane = it & 63, t = it >> 6, g = lane >> 4, col = lane & 15;
        f16x8 hi, lo;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int p = min(p0 + (e < 4 ? 4 * g + e : 16 + 4 * g + e - 4), last - 1);
            const float x = vb[(size_t)p * DH + 16 * t + col];
            hi[e] = (_Float16)x;
            lo[e] = (_Float16)((x - (float)hi[e]) * 2048.0f);
        }
        *(f16x8 *)&dst[KH + (t * 2) * 512 + lane * 8] = hi;
        *(f16x8 *)&dst[KH + (t * 2 + 1) * 512 + lane * 8] = lo;
    }
}

// Takes the V values that are not finite out of a half's staged tile, by the
// half's 256 threads (t) before a barrier of the work-group: they become 0, and
// the first value of their position's K row NaN, so that the rows that see the
// position have its weight NaN (the others mask its score).  `on`: the half has
// a tile with masked positions.
template <int DH, bool F16>
__device__ __forceinline__ void pa_take_apart(uint8_t *k, uint8_t *v, int t, bool on)
{
    constexpr int TP = F16 ? 64 : KVT_POS, KS = DH / 32;
#pragma unroll 1
    for (int q = t; on && q < TP * DH; q += 256) {
        // fp32: high piece q / 512, lane (q % 512) / 8, the low one 512 halves on
        uint16_t *p = (uint16_t *)v + (F16 ? q : (q >> 9) * 1024 + (q & 511));
        if ((*p & 0x7c00) != 0x7c00) continue;
        *p = 0;
        if (!F16) p[512] = 0;
        const int pos = F16 ? q / DH : 4 * ((q >> 7) & 3) + (q & 3) + 16 * ((q >> 2) & 1);
        *(uint16_t *)(k + (pos >> 4) * KS * (F16 ? 1024 : 2048) + (pos & 15) * 16) = 0x7e00;
    }
    __syncthreads();
}

// (d_head 64: LDS lets a CU hold two work-groups, so 128 VGPRs)
template <int DH, bool F16>
__global__ __launch_bounds__(PA_NT) __attribute__((amdgpu_waves_per_eu(DH == 64 ? 4 : 2)))
void k_attn_prompt(AttnArgs a, const _Float16 *hl, int tiles)
{
#pragma clang fp contract(off)
    constexpr int TP = F16 ? 64 : KVT_POS, CT = TP / 16;
    constexpr int KS = DH / 32, DT = DH / 16;
    constexpr int KB = F16 ? TP * DH * 2 : kvt_halves<DH>();   // K bytes of a tile (V: as many)
    constexpr int TILE = 2 * KB;
    constexpr int RPP = 1024 / (2 * DH);              // fp16: V rows per 1 KiB piece
    constexpr int VPW = TP / RPP / 4;                 // fp16: V pieces per wave
    constexpr int PIECES = TILE / 1024 / 4;           // fp32: pieces per wave
    constexpr int DH2 = DT / 2;                       // dimension tiles each half finishes
    extern __shared__ __attribute__((aligned(256))) uint8_t smem_p[];   // [stage][half][TILE]

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, col = lane & 15;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), half = wid >> 2, w4 = wid & 3;
    const int G = a.n_heads / a.n_kv, QT = 64 / G;
    // the longest prefixes first
    const int kvh = blockIdx.x, vb = (int)(gridDim.y - 1 - blockIdx.y) * QT, sp = blockIdx.z;
    const int nt = min(QT, a.n - vb);
    if (nt <= 0) return;
    const int last = min(a.seqlen[(size_t)(vb + nt - 1) * a.seqlen_stride], a.max_ctx);
    const int pa = sp * a.split, pb = min(pa + a.split, last);
    if (pa >= last) return;
    const int whole = min(min(a.seqlen[(size_t)vb * a.seqlen_stride], a.max_ctx), pb);   // visible to every row
    // scores and m stay raw dot products; a weight is 2^(t c2 - m c2) with
    // c2 = log2(e)/sqrt(d_head) on the hardware exponential (exp2(-inf) = 0)
    const float scale = 1.0f / sqrtf((float)DH), c2 = scale * 1.44269504088896341f;
    const float lazy = PA_LAZY / c2;

    const size_t off = F16 ? kv_offset(a.kv, 0) + (size_t)kvh * a.max_ctx * DH : 0;
    const uint8_t *kb = (const uint8_t *)uniform_ptr((const _Float16 *)a.kv.k_base + off);
    const uint8_t *vbp = (const uint8_t *)uniform_ptr((const _Float16 *)a.kv.v_base + off);
    // fp16: this lane's piece of a V row: row lane / (DH / 8) of the piece, LDS
    // unit u holding dimensions 16 (u ^ f(row)) .. +15
    const int vrow = lane / (DH / 8), vch = lane % (DH / 8);
    auto issue = [&](int st, int p0) {
        uint8_t *dst = smem_p + (st * 2 + half) * TILE;
        if constexpr (F16) {
            const uint32_t kp = (uint32_t)min(p0 + 16 * w4 + col, last - 1) * (2 * DH) + 16 * g;
#pragma unroll
            for (int s = 0; s < KS; s++)
                __builtin_amdgcn_global_load_lds((const gvoid_t *)(kb + kp + 64 * s),
                                                 (lvoid_t *)(dst + (w4 * KS + s) * 1024), 16, 0, 0);
#pragma unroll
            for (int i = 0; i < VPW; i++) {
                const int r = (w4 * VPW + i) * RPP + vrow;   // row of the tile
                const int f = DH == 128 ? r & 7 : (r >> 1) & 3;
                const uint32_t vp = (uint32_t)min(p0 + r, last - 1) * (2 * DH) +
                                    32 * ((vch >> 1) ^ f) + 16 * (vch & 1);
                __builtin_amdgcn_global_load_lds((const gvoid_t *)(vbp + vp),
                                                 (lvoid_t *)(dst + KB + (w4 * VPW + i) * 1024), 16, 0, 0);
            }
        } else {
            const uint8_t *src = (const uint8_t *)(hl + ((size_t)kvh * tiles + p0 / TP) * kvt_halves<DH>());
#pragma unroll
            for (int i = 0; i < PIECES; i++) {
                const int pc = w4 * PIECES + i;
                __builtin_amdgcn_global_load_lds((const gvoid_t *)(src + pc * 1024 + lane * 16),
                                                 (lvoid_t *)(dst + pc * 1024), 16, 0, 0);
            }
        }
    };
    if (pa + half * TP < pb) issue(0, pa + half * TP);

    // query operands of this lane's row 16 w4 + col = (token at, head ah)
    const int ar = 16 * w4 + col, at = ar / G, ah = ar - at * G;
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
    f32x4 o[DT], o2[DT];   // o2: products with a low part, times 2048
    float m, mk, lsum;     // mk = -m c2; a row with no visible position yet (m = -inf) has weights 0
    // fp16: transposing reads, this lane's bytes of row 4g + col/4 (+ 16 per c)
    // of dimension tile t at vaddr ^ 32t
    const int vr = 4 * g + (col >> 2);
    const uint32_t vaddr = (uint32_t)(vr * (2 * DH) + 32 * (DH == 128 ? vr & 7 : (vr >> 1) & 3) + 8 * (col & 3));

    // Masked positions are in the products with weight 0, so a V row that is not
    // finite leaves NaN (0 * inf) in the rows that do not see it, too.  Where an
    // output is not finite the walk is done again with such rows taken apart, and
    // the outputs written again (the vote on it is off the way to the first ones).
    for (bool apart = false;; apart = true) {
        m = -INFINITY;
        mk = 0.0f;
        lsum = 0.0f;
#pragma unroll
        for (int t = 0; t < DT; t++) {
            o[t] = zero4;
            o2[t] = zero4;
        }
        int st = 0;
        for (int pp = pa; pp < pb; pp += 2 * TP, st ^= 1) {
            const int p0 = pp + half * TP;   // this half's tile
            // the tiles have landed and every wave is done with the other stage
            __builtin_amdgcn_s_waitcnt(WAITCNT_VM_LGKM0(0));
            __syncthreads();
            if (p0 + 2 * TP < pb) issue(st ^ 1, p0 + 2 * TP);
            if (__builtin_expect(apart && pp + 2 * TP > whole, 0)) {   // (alike in both halves: it has a barrier)
                uint8_t *k = smem_p + (st * 2 + half) * TILE;
                pa_take_apart<DH, F16>(k, k + KB, tid & 255, p0 < pb && p0 + TP > whole);
            }
            if (p0 >= pb) continue;          // (the last pair may be one tile)
            const uint8_t *ks_ = smem_p + (st * 2 + half) * TILE, *vs_ = ks_ + KB;
            // ---- scores: sc[c][i] = position p0 + 16c + 4g + i of this lane's row
            float sc[CT][4];
#pragma unroll
            for (int c = 0; c < CT; c++) {
                f32x4 s1 = zero4, s2 = zero4;
#pragma unroll
                for (int s = 0; s < KS; s++) {
                    if constexpr (F16) {
                        const f16x8 kf = *(const f16x8 *)(ks_ + (c * KS + s) * 1024 + lane * 16);
                        s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qh[s], s1, 0, 0, 0);
                        s2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, ql[s], s2, 0, 0, 0);
                    } else {
                        const f16x8 kh = *(const f16x8 *)(ks_ + (c * KS + s) * 2048 + lane * 16);
                        const f16x8 kl = *(const f16x8 *)(ks_ + (c * KS + s) * 2048 + 1024 + lane * 16);
                        s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, qh[s], s1, 0, 0, 0);
                        s2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kl, qh[s], s2, 0, 0, 0);
                        s2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, ql[s], s2, 0, 0, 0);
                    }
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
                for (int t = 0; t < DT; t++) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        o[t][i] *= al;
                        o2[t][i] *= al;
                    }
                }
            }
            f16x8 ph[CT / 2], pl[CT / 2];
#pragma unroll
            for (int c = 0; c < CT; c++) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float e = __builtin_amdgcn_exp2f(fmaf(sc[c][i], c2, mk));
                    lsum += e;
                    const _Float16 hi = (_Float16)e;
                    ph[c >> 1][4 * (c & 1) + i] = hi;
                    pl[c >> 1][4 * (c & 1) + i] = (_Float16)((e - (float)hi) * 2048.0f);
                }
            }
            // ---- O^T += V^T P^T: k-step k covers positions 32k + 4g .. +3 and 32k + 16 + 4g .. +3
#pragma unroll
            for (int k = 0; k < CT / 2; k++) {
#pragma unroll
                for (int t = 0; t < DT; t++) {
                    if constexpr (F16) {
                        typedef short s16x4 __attribute__((ext_vector_type(4)));
                        typedef __attribute__((address_space(3))) s16x4 ls16x4;
                        const uint8_t *src = vs_ + 32 * k * (2 * DH) + (vaddr ^ (32u * t));
                        const s16x4 lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls16x4 *)src);
                        const s16x4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls16x4 *)(src + 16 * (2 * DH)));
                        const f16x8 vf = __builtin_bit_cast(f16x8, __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
                        o[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, ph[k], o[t], 0, 0, 0);
                        o2[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pl[k], o2[t], 0, 0, 0);
                    } else {
                        const f16x8 vh = *(const f16x8 *)(vs_ + t * 2048 + lane * 16);
                        const f16x8 vl = *(const f16x8 *)(vs_ + t * 2048 + 1024 + lane * 16);
                        o[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, ph[k], o[t], 0, 0, 0);
                        o2[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vl, ph[k], o2[t], 0, 0, 0);
                        o2[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, pl[k], o2[t], 0, 0, 0);
                    }
                }
            }
        }

        // The addresses below start from copies that the compiler takes as new
        // in each walk: it would compute them all before the first one and hold
        // them in registers, or spill them, during it.
        int ln = lane, tok = at, hd = ah, len = L;
        asm volatile("" : "+v"(ln), "+v"(tok), "+v"(hd), "+v"(len));
        const int gg = ln >> 4, row = 16 * w4 + (ln & 15);
        // ---- the halves meet: half 0 finishes the first DT / 2 dimension tiles of
        // each row, half 1 the others
#pragma unroll
        for (int t = 0; t < DT; t++) o[t] += o2[t] * (1.0f / 2048.0f);
        f32x4 z = zero4;   // NaN where an output of the lane is not finite
#pragma unroll
        for (int t = 0; t < DT; t++) z += o[t] * 0.0f;
        lsum += __shfl_xor(lsum, 16, 64);
        lsum += __shfl_xor(lsum, 32, 64);
        f32x4 *xo = (f32x4 *)smem_p;                        // [half][wave][DT / 2][lane]
        float *xm = (float *)(smem_p + 8 * DH2 * 64 * 16);   // [half][row] m, then [half][row] l, then a vote per wave
        const bool fin = __ballot(!(z[0] + z[1] + z[2] + z[3] == 0.0f)) == 0;
        __syncthreads();
#pragma unroll
        for (int t = 0; t < DH2; t++) xo[((half * 4 + w4) * DH2 + t) * 64 + ln] = half ? o[t] : o[DH2 + t];
        if (gg == 0) {
            xm[half * 64 + row] = m;
            xm[128 + half * 64 + row] = lsum;
        }
        if (ln == 0) xm[256 + wid] = fin ? 0.0f : 1.0f;
        __syncthreads();
        const float m1 = xm[(half ^ 1) * 64 + row], l1 = xm[128 + (half ^ 1) * 64 + row];
        const float mm = fmaxf(m, m1), mref = mm == -INFINITY ? 0.0f : mm;
        const float f0 = __builtin_amdgcn_exp2f((m - mref) * c2), f1 = __builtin_amdgcn_exp2f((m1 - mref) * c2);
        const float ls = lsum * f0 + l1 * f1;
        f32x4 r[DH2];
#pragma unroll
        for (int t = 0; t < DH2; t++) {
            const f32x4 own = half ? o[DH2 + t] : o[t], other = xo[(((half ^ 1) * 4 + w4) * DH2 + t) * 64 + ln];
            r[t] = own * f0 + other * f1;
        }

        // ---- outputs: lane (col, g) holds dimensions 16 (DH2 half + t) + 4g + i of its row
        const int nact = (len + a.split - 1) / a.split;
        const bool mine = arow && sp < nact;   // (else no positions of this token here)
        const int v = vb + tok, d0 = 16 * DH2 * half + 4 * gg;
        if (mine && nact == 1) {
            const float inv = 1.0f / ls;
            const int k0 = (kvh * G + hd) * DH + d0;
#pragma unroll
            for (int t = 0; t < DH2; t += 2) {
                const f32x4 x0 = r[t] * inv, x1 = r[t + 1] * inv;
                const int k = k0 + 16 * t;
                if (a.out) {
                    *(f32x4 *)(a.out + (size_t)v * a.out_stride + k) = x0;
                    *(f32x4 *)(a.out + (size_t)v * a.out_stride + k + 16) = x1;
                }
                if (!a.next.q) continue;
                if (a.next.dt == DT_Q8_0) {
                    act_put4(a.next, v, k, x0);
                    act_put4(a.next, v, k + 16, x1);
                } else {
                    act_put8(a.next, v, k >> 5, gg, k, k + 16, x0, x1);
                }
            }
        } else if (mine) {
            const size_t sb = (((size_t)v * a.n_kv + kvh) * a.max_splits + sp) * G + hd;
#pragma unroll
            for (int t = 0; t < DH2; t++) *(f32x4 *)&a.po[sb * DH + d0 + 16 * t] = r[t];
            if (gg == 0 && half == 0) {
                a.pm[sb] = mm * scale;   // natural units, as the merge reads them
                a.pl[sb] = ls;
            }
        }

        const f32x4 v0 = *(const f32x4 *)&xm[256], v1 = *(const f32x4 *)&xm[260], vs = v0 + v1;
        if (__builtin_expect(apart || vs[0] + vs[1] + vs[2] + vs[3] == 0.0f, 1)) break;
        __syncthreads();
        if (pa + half * TP < pb) issue(0, pa + half * TP);
    }
}

size_t attn_prompt_kv_bytes(int n_kv, int d_head, int max_ctx)
{
    const size_t tiles = (size_t)(max_ctx + KVT_POS - 1) / KVT_POS;
    return (size_t)n_kv * tiles * KVT_POS * d_head * 4 * sizeof(_Float16);
}

static int prompt_cus()
{
    static const int c = [] {
        int d = 0, n = 0;
        if (hipGetDevice(&d) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, d) != hipSuccess ||
            n < 1) {
            (void)hipGetLastError();
            n = 256;
        }
        return n;
    }();
    return c;
}

template <int DH, bool F16>
static int launch_dh(const AttnArgs &a, _Float16 *kv_hl, int last, hipStream_t s)
{
    constexpr int LDS = 4 * 64 * DH * 4;   // two stages of two tiles (64 positions fp16 or 32 high/low, K and V)
    static LdsLimit limit;
    const bool ok = limit.raise(current_device(), [] {
        return hipFuncSetAttribute((const void *)k_attn_prompt<DH, F16>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) ==
               hipSuccess;
    });
    if (!ok) {
        (void)hipGetLastError();   // (not the split kernels' launch error)
        return -4;
    }
    const int QT = 64 / (a.n_heads / a.n_kv);
    const int tiles = (a.max_ctx + KVT_POS - 1) / KVT_POS;
    if constexpr (!F16)
        hipLaunchKernelGGL(k_kv_hilo<DH>, dim3(a.n_kv, (last + KVT_POS - 1) / KVT_POS), dim3(256), 0, s, a, last,
                           kv_hl, tiles);
    const dim3 grid(a.n_kv, (a.n + QT - 1) / QT, a.max_splits);
    hipLaunchKernelGGL((k_attn_prompt<DH, F16>), grid, dim3(PA_NT), LDS, s, a, kv_hl, tiles);
    return a.max_splits > 1 ? launch_attn_merge_wave(a, s) : 0;
}

// Work-groups of one round: LDS lets a CU hold two at d_head 64, one at 128.
static long prompt_round(int d_head) { return (long)prompt_cus() * (128 / d_head); }

// Work-groups of n tokens per split.
static long prompt_blocks(int n, int n_heads, int n_kv)
{
    const int QT = 64 / (n_heads / n_kv);
    return (long)n_kv * ((n + QT - 1) / QT);
}

size_t attn_prompt_rows(int cap, int n_heads, int n_kv, int d_head, int max_ctx, int split)
{
    size_t m = 0;
    for (int n = 1; n <= cap; n++) {
        const long s = std::min((long)attn_max_splits(max_ctx, split), prompt_round(d_head) / prompt_blocks(n, n_heads, n_kv));
        if (s > 1) m = std::max(m, (size_t)n * n_heads * s);
    }
    return m;
}

int launch_attn_prompt(const AttnArgs &a, size_t part_rows, _Float16 *kv_hl, int last, hipStream_t s)
{
    const int G = a.n_heads / a.n_kv;
    if (G < 1 || G > 8 || a.n_heads % a.n_kv || a.n < 1 || (a.d_head != 64 && a.d_head != 128)) return -4;
    if (a.split < 64 || a.split % 64 || a.max_splits > ATT_MAX_MERGE) return -4;
    if ((!a.kv_f16 && !kv_hl) || last < 1 || last > a.max_ctx) return -4;
    // the pass's split: the planned one doubled until the grid fits one round
    // of the work-groups and the partials their buffers (one split has none);
    // blocks that alone exceed a round run unsplit, longest first.  At 16/4
    // heads of 128 over fp16, with merge: 512 tokens behind 1300 positions 35
    // us in 2 splits (taken), 44 in 4, 43 in 1; 188 behind 1812 24 in 4
    // (taken), 30 in 8.
    AttnArgs b = a;
    const long blocks = prompt_blocks(a.n, a.n_heads, a.n_kv);
    auto splits = [&] { return (last + b.split - 1) / b.split; };
    while (b.split < last &&
           (blocks * splits() > prompt_round(a.d_head) || (size_t)a.n * a.n_heads * splits() > part_rows))
        b.split *= 2;
    b.max_splits = splits();
    int rc;
    if (a.kv_f16) rc = a.d_head == 128 ? launch_dh<128, true>(b, kv_hl, last, s) : launch_dh<64, true>(b, kv_hl, last, s);
    else rc = a.d_head == 128 ? launch_dh<128, false>(b, kv_hl, last, s) : launch_dh<64, false>(b, kv_hl, last, s);
    if (rc) return rc;
    return hipGetLastError() == hipSuccess ? 0 : -4;
}
