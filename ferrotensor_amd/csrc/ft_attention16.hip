// Causal / full grouped-query flash attention for whole, 16-byte aligned head dims
// (32 and 64), built from 16-row wave tiles of v_mfma_f32_16x16x4_f32.
//
// Layout as in ft_attention.hip: q/out/dO/dq [B,Sq,H,D], k/v/dk/dv [B,Sk,Hkv,D],
// stats [B*H*Sq][2] = (Delta, log-sum-exp).
//
// A wave owns 16 rows (queries in the forward and dQ kernels, keys in the dK/dV
// kernel) and keeps what belongs to them in registers; the other side streams
// through LDS. Scores are computed transposed (S^T = K Q^T for a query wave), so
// a lane's accumulator registers are keys of ONE query: softmax statistics are
// per-lane scalars plus two cross-lane steps, and the probabilities are already
// the B operand of the next product. The 16x16x4 shape keeps a wave at about a
// hundred registers (four waves per SIMD) and cuts the causal triangle in 16-row
// steps.
//
// Operand layouts of v_mfma_f32_16x16x4_f32 (lane = l16 + 16 * g):
//   A[m][k]: lane (m = l16, k = g);  B[k][n]: lane (n = l16, k = g);
//   D[m][n]: lane (n = l16), register r holds row m = 4 g + r.
// A 16-byte LDS read of four consecutive head-dim values feeds four MFMAs: the
// contraction index (or output row) of MFMA e is permuted accordingly, the same
// way on both operands.
#include "ft_attention16.h"

namespace {

template <int NG>
__global__ __launch_bounds__(4 * NG * 64) void attn16_fwd_kernel(AttnArgs p) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    attn16_fwd<NG>(p, smem);
}

template <int NG>
__global__ __launch_bounds__(4 * NG * 64) void attn16_dq_kernel(AttnArgs p) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    attn16_dq<NG>(p, smem);
}

// ---------------------------------------------------------------------------
// Backward, pass 2: dK and dV of 16 keys of one (batch, kv head), summed over the
// query heads of the group and over the 16-query blocks that can see them. The
// key block (K pre-scaled for the base-2 scores, V) sits in LDS for all eight
// waves; the (head, query block) items are dealt round-robin to the waves, which
// run without a barrier until the end: an item's Q and dO rows come from global
// memory as 16-byte quads straight into the A operands of S = Q K^T and
// dP = dO V^T (the next item's while the current one multiplies), pass through a
// wave-private LDS tile, and are read back with the head dim as the row for
// dV^T += dO^T P and dK^T += Q^T dS. The waves' partial sums are added in wave
// order through LDS (no atomics). One workgroup per (key block, batch * kv head),
// key block 0 (the most items under the causal mask) first.
// ---------------------------------------------------------------------------
template <int DP>
__global__ __launch_bounds__(512, 4) void attn16_dkdv_kernel(AttnArgs p) {
    constexpr int NB = DP / 16, EV = DP / 16, PITCH = DP, NW = 8, C4 = DP / 4;
    constexpr int BLK = 16 * PITCH;
    extern __shared__ __attribute__((aligned(16))) float smem[];  // K block, V block, 8 x (Q tile, dO tile)
    const int tid = threadIdx.x, lane = tid % 64, l16 = lane % 16, g = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);  // wave-uniform: keeps the tile bookkeeping in SGPRs
    float* ks = smem;
    float* vs = smem + BLK;
    float* qs = smem + 2 * BLK + wave * 2 * BLK;
    float* dos = qs + BLK;

    const int nhu = p.B * (p.split_g ? p.H : p.Hkv);
    const int kbi = blockIdx.x / nhu, bh = blockIdx.x % nhu;
    const int Gfull = p.H / p.Hkv;
    const int b = bh / (p.split_g ? p.H : p.Hkv);
    const int hsel = bh % (p.split_g ? p.H : p.Hkv);
    const int kvh = p.split_g ? hsel / Gfull : hsel;
    const int g0 = p.split_g ? hsel % Gfull : 0;  // first query head of this workgroup within the group
    const int G = p.split_g ? 1 : Gfull;          // and how many it covers
    const int kb0 = kbi * 16;
    const int key = kb0 + l16;
    const int key_m = key < p.Sk ? key : 0x7fffffff;  // a key past the end is visible to nobody

    const float kscale = p.scale * kLog2e;
    for (int e = tid; e < 2 * 16 * C4; e += NW * 64) {
        const int which = e / (16 * C4), r = (e / C4) % 16, c = e % C4;
        int kr = kb0 + r;
        kr = kr < p.Sk ? kr : p.Sk - 1;
        const long o = (((long)b * p.Sk + kr) * p.Hkv + kvh) * DP + 4 * c;
        if (which == 0) {
            const float4 t = *reinterpret_cast<const float4*>(p.k + o);
            *reinterpret_cast<float4*>(ks + sw(r, c)) =
                make_float4(t.x * kscale, t.y * kscale, t.z * kscale, t.w * kscale);
        } else {
            *reinterpret_cast<float4*>(vs + sw(r, c)) = *reinterpret_cast<const float4*>(p.v + o);
        }
    }

    // 16-query blocks that can see this key block
    const int nqb = (p.Sq + 15) / 16;
    int qb_start = 0;
    if (p.causal) {
        const int first_q = kb0 - p.causal_offset;  // smallest i with i + offset >= kb0
        qb_start = first_q > 0 ? first_q / 16 : 0;
    }
    const int per_head = nqb > qb_start ? nqb - qb_start : 0;
    const int items = per_head * G;

    float4 qa[NB], da[NB];
    float2 st[4];
    auto fetch = [&](int item) {
        const int gi = item / per_head;
        const int q0 = (qb_start + item % per_head) * 16;
        const int h = kvh * Gfull + g0 + gi;
        int qr = q0 + l16;
        qr = qr < p.Sq ? qr : p.Sq - 1;
        const long ro = (((long)b * p.Sq + qr) * p.H + h) * DP;
#pragma unroll
        for (int blk = 0; blk < NB; blk++) {
            qa[blk] = *reinterpret_cast<const float4*>(p.q + ro + 16 * blk + 4 * g);
            da[blk] = *reinterpret_cast<const float4*>(p.d_out + ro + 16 * blk + 4 * g);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            int qi = q0 + 4 * g + i;
            qi = qi < p.Sq ? qi : p.Sq - 1;
            st[i] = *reinterpret_cast<const float2*>(p.stats + 2 * (((long)b * p.H + h) * p.Sq + qi));
        }
    };
    if (wave < items) fetch(wave);
    __syncthreads();  // K/V block complete

    floatx4 dk[EV], dv[EV];
#pragma unroll
    for (int e = 0; e < EV; e++) {
        dk[e] = zero4();
        dv[e] = zero4();
    }

    for (int item = wave; item < items; item += NW) {
        const int q0 = (qb_start + item % per_head) * 16;
        // this item's rows -> the wave's LDS tile (for the transposed reads further down)
#pragma unroll
        for (int blk = 0; blk < NB; blk++) {
            *reinterpret_cast<float4*>(qs + sw(l16, 4 * blk + g)) = qa[blk];
            *reinterpret_cast<float4*>(dos + sw(l16, 4 * blk + g)) = da[blk];
        }
        floatx4 s = zero4(), dp = zero4();
#pragma unroll
        for (int blk = 0; blk < NB; blk++) {
            const float4 kq = *reinterpret_cast<const float4*>(ks + sw(l16, 4 * blk + g));
            const float4 vq = *reinterpret_cast<const float4*>(vs + sw(l16, 4 * blk + g));
            s = MFMA16(qa[blk].x, kq.x, s);
            dp = MFMA16(da[blk].x, vq.x, dp);
            s = MFMA16(qa[blk].y, kq.y, s);
            dp = MFMA16(da[blk].y, vq.y, dp);
            s = MFMA16(qa[blk].z, kq.z, s);
            dp = MFMA16(da[blk].z, vq.z, dp);
            s = MFMA16(qa[blk].w, kq.w, s);
            dp = MFMA16(da[blk].w, vq.w, dp);
        }
        // register i of this lane is query q0 + 4 g + i against key `key`
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // visible: a real key, a real query, and not above the diagonal; written without
            // short-circuit operators so that it stays a select (exp2(-inf) = 0)
            const int qi = q0 + 4 * g + i;
            const int lim = qi < p.Sq ? (p.causal ? qi + p.causal_offset : 0x7ffffffe) : -1;
            const float pij = exp2_fast(key_m <= lim ? s[i] - st[i].y * kLog2e : -INFINITY);
            s[i] = pij;                        // P
            dp[i] = pij * (dp[i] - st[i].x);   // dS
        }
        // the next item's rows travel while the rest of this one is computed
        fetch(item + NW < items ? item + NW : item);  // (the last item is fetched again: no branch, no copies)
        wave_lds_fence();
        float ao[4][EV], aq[4][EV];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lds_vec<EV>(dos + sw(4 * g + i, l16), ao[i]);
            lds_vec<EV>(qs + sw(4 * g + i, l16), aq[i]);
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int e = 0; e < EV; e++) {
                dv[e] = MFMA16(ao[i][e], s[i], dv[e]);
                dk[e] = MFMA16(aq[i][e], dp[i], dk[e]);
            }
        wave_lds_fence();  // the tile is rewritten by the next item
    }

    // Cross-wave sum in wave order. A wave's tile pair takes its partial dK (Q tile) and dV (dO tile)
    // as [key][head dim]; register r of accumulator e is head-dim index EV * (4 g + r) + e.
#pragma unroll
    for (int r = 0; r < 4; r++) {
        float a[EV], c[EV];
#pragma unroll
        for (int e = 0; e < EV; e++) {
            a[e] = dk[e][r];
            c[e] = dv[e][r];
        }
        store_vec<EV>(qs + sw(l16, 4 * g + r), a);
        store_vec<EV>(dos + sw(l16, 4 * g + r), c);
    }
    __syncthreads();
    const float* red = smem + 2 * BLK;
    for (int e = tid; e < 2 * 16 * C4; e += NW * 64) {
        const int which = e / (16 * C4), kk = (e / C4) % 16, c = e % C4;
        float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int wv = 0; wv < NW; wv++) {
            const float4 t = *reinterpret_cast<const float4*>(red + (wv * 2 + which) * BLK + sw(kk, c));
            sum.x += t.x; sum.y += t.y; sum.z += t.z; sum.w += t.w;
        }
        const int krow = kb0 + kk;
        const long o = (((long)b * p.Sk + krow) * p.Hkv + kvh) * DP + 4 * c;
        if (p.split_g) {
            if (krow < p.Sk) {
                const long n_all = (long)p.B * p.Sk * p.Hkv * DP;
                *reinterpret_cast<float4*>(p.part + (2 * g0 + which) * n_all + o) = sum;
            }
            continue;
        }
        if (which == 1) {
            if (krow < p.Sk) *reinterpret_cast<float4*>(p.dv + o) = sum;
            continue;
        }
        // dK = scale * sum dS Q (Q is read unscaled)
        sum.x *= p.scale; sum.y *= p.scale; sum.z *= p.scale; sum.w *= p.scale;
        if (DP == 64 && p.rope) {
            // rotated back: the partner chunk (head-dim index +- 32) is held by lane ^ 8 of this wave
            float4 oth;
            oth.x = __shfl_xor(sum.x, 8, 64);
            oth.y = __shfl_xor(sum.y, 8, 64);
            oth.z = __shfl_xor(sum.z, 8, 64);
            oth.w = __shfl_xor(sum.w, 8, 64);
            const int kc = krow < p.Sk ? krow : p.Sk - 1;
            const float2* tb = p.rope + (long)kc * 32 + ((4 * c) & 31);
            const float2 c0 = tb[0], c1 = tb[1], c2 = tb[2], c3 = tb[3];
            const float sg = c < 8 ? 1.0f : -1.0f;
            sum = make_float4(sum.x * c0.x + sg * oth.x * c0.y, sum.y * c1.x + sg * oth.y * c1.y,
                              sum.z * c2.x + sg * oth.z * c2.y, sum.w * c3.x + sg * oth.w * c3.y);
        }
        if (krow < p.Sk) *reinterpret_cast<float4*>(p.dk + o) = sum;
    }
}

template <typename K>
int set_smem(K kernel, size_t bytes) {
    FT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)bytes));
    return FT_OK;
}

template <int NG>
int launch_query_kernels(ft_context* ctx, const AttnArgs& a, bool backward) {
    constexpr int TQ = 16 * NG;
    constexpr size_t smem = (size_t)2 * 2 * TILE * sizeof(float);
    static bool attr = false;
    if (!attr) {
        FT_TRY(set_smem(&attn16_fwd_kernel<NG>, smem));
        FT_TRY(set_smem(&attn16_dq_kernel<NG>, smem));
        attr = true;
    }
    const size_t nT = ft_div_up(a.Sq, TQ);
    const dim3 grid((unsigned)(((nT + 1) / 2) * (size_t)a.B * a.H));
    if (backward)
        hipLaunchKernelGGL((attn16_dq_kernel<NG>), grid, dim3(4 * NG * 64), smem, ctx->stream, a);
    else
        hipLaunchKernelGGL((attn16_fwd_kernel<NG>), grid, dim3(4 * NG * 64), smem, ctx->stream, a);
    FT_LAUNCH_CHECK();
    return FT_OK;
}

// Which tile height the forward (backward = false) or dQ kernel should run with at this shape:
// 4 (64-row tiles, 16 waves), 2 (32-row tiles, 8 waves) or 0 (too few workgroups for either: the
// caller keeps the 32-row kernels that split the keys of a query block over waves). Thresholds
// from timings at 1-32 sequences of 15 and 9 heads x 256 tokens and at 1024 tokens.
int query_tile_groups(const ft_context* ctx, const AttnArgs& a, bool backward) {
    const size_t wgs64 = (ft_div_up(a.Sq, 64) + 1) / 2 * (size_t)a.B * a.H;
    const size_t cus = (size_t)ctx->num_cus;
    if (backward) {
        if (wgs64 * 5 >= cus * 4) return 4;
        // the 8-wave dQ kernel holds one workgroup per CU: it pays while one round covers the launch
        if (wgs64 * 4 >= cus && ((ft_div_up(a.Sq, 32) + 1) / 2) * (size_t)a.B * a.H <= cus) return 2;
        return 0;
    }
    if (wgs64 * 2 >= cus) return 4;
    if (wgs64 * 4 >= cus) return 2;
    return 0;
}

template <int DP>
int launch_dkdv(ft_context* ctx, const AttnArgs& a) {
    constexpr size_t smem = (size_t)(2 + 8 * 2) * 16 * DP * sizeof(float);
    static bool attr = false;
    if (!attr) {
        FT_TRY(set_smem(&attn16_dkdv_kernel<DP>, smem));
        attr = true;
    }
    const size_t nkb = ft_div_up(a.Sk, 16);
    const size_t G = (size_t)a.H / a.Hkv;
    const size_t n_all = (size_t)a.B * a.Sk * a.Hkv * DP;
    // Few (key block, kv head) units and a GQA group to share them out: one workgroup per query
    // head, then the ordered sum over the group.
    if (G > 1 && nkb * a.B * a.Hkv < 2 * (size_t)ctx->num_cus && 2 * G * n_all <= kAttnScratchFloats) {
        if (!ctx->attn_scratch) {
            FT_HIP(hipSetDevice(ctx->device));
            FT_HIP(hipMalloc((void**)&ctx->attn_scratch, kAttnScratchFloats * sizeof(float)));
        }
        AttnArgs s = a;
        s.part = ctx->attn_scratch;
        s.split_g = 1;
        hipLaunchKernelGGL((attn16_dkdv_kernel<DP>), dim3((unsigned)(nkb * a.B * a.H)), dim3(512), smem, ctx->stream, s);
        FT_LAUNCH_CHECK();
        return ft_attn_dkdv_combine(ctx, s, DP);
    }
    hipLaunchKernelGGL((attn16_dkdv_kernel<DP>), dim3((unsigned)(nkb * a.B * a.Hkv)), dim3(512), smem, ctx->stream, a);
    FT_LAUNCH_CHECK();
    return FT_OK;
}

}  // namespace

bool ft_attn16_usable(const AttnArgs& a) {
    auto al = [](const void* q) { return q == nullptr || (((uintptr_t)q) & 15) == 0; };
    return a.D == 64 && a.Sq > 0 && a.Sk > 0 && al(a.q) && al(a.k) && al(a.v) && al(a.out) && al(a.d_out) &&
           al(a.o) && al(a.dq) && al(a.dk) && al(a.dv) && (((uintptr_t)a.stats) & 7) == 0;
}

bool ft_attn16_forward_pays(const ft_context* ctx, const AttnArgs& a) { return query_tile_groups(ctx, a, false) != 0; }
bool ft_attn16_backward_dq_pays(const ft_context* ctx, const AttnArgs& a) { return query_tile_groups(ctx, a, true) != 0; }

int ft_attn16_forward(ft_context* ctx, const AttnArgs& a) {
    if (!ctx->f32_chain) return ft_attn_split_forward(ctx, a, query_tile_groups(ctx, a, false));
    return query_tile_groups(ctx, a, false) == 2 ? launch_query_kernels<2>(ctx, a, false)
                                                 : launch_query_kernels<4>(ctx, a, false);
}

int ft_attn16_backward_dq(ft_context* ctx, const AttnArgs& a) {
    return query_tile_groups(ctx, a, true) == 2 ? launch_query_kernels<2>(ctx, a, true)
                                                : launch_query_kernels<4>(ctx, a, true);
}

int ft_attn16_backward_dkdv(ft_context* ctx, const AttnArgs& a) { return launch_dkdv<64>(ctx, a); }
