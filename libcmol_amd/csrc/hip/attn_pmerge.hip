// attn_pmerge.hip — the split merge of prompt passes: a lane per four
// dimensions of a (query head, token), so a wave merges two heads of 128 or
// four of 64 and every load and store is 16 (operand: 8) bytes per lane.
// Bound by the partials it reads once.  A translation unit of its own, beside
// the decode attention kernels' code object.
#include "attn_impl.h"

// mx = max_s m_s, L = sum_s l_s e^(m_s - mx), out = sum_s o_s e^(m_s - mx) / L
// over the nact splits in ascending order.
template <int DH>
__global__ __launch_bounds__(256) void k_attn_merge_wave(AttnArgs a)
{
#pragma clang fp contract(off)
    constexpr int LPH = DH / 4;   // lanes per (head, token)
    const int sub = threadIdx.x % LPH;
    const int idx = blockIdx.x * (256 / LPH) + threadIdx.x / LPH;
    const int hq = idx % a.n_heads, n = idx / a.n_heads;
    if (n >= a.n) return;
    const int G = a.n_heads / a.n_kv, kvh = hq / G, h = hq % G;
    const int L = min(a.seqlen[n * a.seqlen_stride], a.max_ctx);
    const int nact = (L + a.split - 1) / a.split;
    if (nact <= 1) return;   // finished by the attention kernel
    const size_t hb = (((size_t)n * a.n_kv + kvh) * a.max_splits) * G + h;   // + s * G
    // eight splits at a time, their loads in one round trip (past the last
    // one: re-read, weight 0), rescaled to the largest m seen so far
    float mx = -INFINITY, Ls = 0.0f;
    f32x4 acc = {};
    for (int s0 = 0; s0 < nact; s0 += 8) {
        float pm[8], pl[8];
        f32x4 po[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const size_t o = hb + (size_t)min(s0 + u, nact - 1) * G;
            pm[u] = a.pm[o];
            pl[u] = a.pl[o];
            po[u] = *(const f32x4 *)&a.po[o * DH + 4 * sub];
        }
        float mn = mx;
#pragma unroll
        for (int u = 0; u < 8; u++) mn = fmaxf(mn, pm[u]);
        const float f = expf(mx - mn);
        mx = mn;
        Ls *= f;
        acc *= f;
#pragma unroll
        for (int u = 0; u < 8; u++) {
            if (s0 + u >= nact) break;
            const float e = expf(pm[u] - mx);
            Ls += pl[u] * e;
            acc += po[u] * e;
        }
    }
    acc /= Ls;
    const int k = hq * DH + 4 * sub;
    if (a.out) *(f32x4 *)(a.out + (size_t)n * a.out_stride + k) = acc;
    if (a.next.q) act_put4(a.next, n, k, acc);
}

int launch_attn_merge_wave(const AttnArgs &a, hipStream_t s)
{
    if (a.d_head != 64 && a.d_head != 128) return -4;
    const long per = 1024 / a.d_head;   // (head, token) pairs per work-group
    const dim3 grid((unsigned)(((long)a.n_heads * a.n + per - 1) / per)), block(256);
    if (a.d_head == 128) hipLaunchKernelGGL((k_attn_merge_wave<128>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((k_attn_merge_wave<64>), grid, block, 0, s, a);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}
