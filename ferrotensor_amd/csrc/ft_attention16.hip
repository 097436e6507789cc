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

template <int DP>
__global__ __launch_bounds__(512, 4) void attn16_dkdv_kernel(AttnArgs p) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    attn16_dkdv<DP>(p, smem, blockIdx.x);
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

// dK/dV on bf16 parts: one workgroup per 64 keys and query head where the shares of a group fit their scratch, else per kv
// head.
struct DkdvUnits {
    bool per_head;
    size_t workgroups;
};
DkdvUnits split_dkdv_units(const AttnArgs& a) {
    const size_t G = (size_t)a.H / a.Hkv, n_all = (size_t)a.B * a.Sk * a.Hkv * a.D;
    const bool per_head = G == 1 || 2 * G * n_all <= kAttnScratchFloats;
    return {per_head, ft_div_up(a.Sk, 64) * (size_t)a.B * (per_head ? a.H : a.Hkv)};
}

// The backward on bf16 parts: its kernels hold one workgroup of 8 waves per CU and want a few rounds of them, of tiles that
// are not half empty. All three run this way or none: kernels that form the same scores with the same rounding lose less in
// the probabilities. So a line lies where forward and backward together break even (us, f32 kernels -> these, forward +
// backward, causal unless said):
//  * dQ, 480 workgroups of 128 queries (4 x 1024 tokens, 15 heads on 5) 128 -> 89, 120 (one sequence) 13 us longer;
//  * dK/dV per head: 4096 workgroups (8 x 1024, 32 heads) 360 + 1266 -> 252 + 963, 960 (4 x 1024, 15 on 5) 93 + 284 -> 66 +
//    245, 480 (8 x 256, 15 on 5) backward 60 -> 62. With a group's shares to add it takes longer queries: 4 x 384, 32 on 8
//    44 + 121 -> 31 + 111; 24 x 300, 9 on 3 52 + 139 -> 39 + 155; 8 x 256, 32 on 8 39 + 109 -> 30 + 123; without a mask
//    16 x 256, 15 on 5 64 + 156 -> 43 + 149; 20 x 200 62 + 171 -> 44 + 180;
//  * dK/dV per kv head, workgroups as long as the group is large, and under the mask unequal: 288 (6 x 384, 32 on 8) 67 + 175
//    -> 48 + 167; 264 (3 x 700) 86 + 241 -> 62 + 264, 176 (4 x 700, 32 on 4) 101 + 312 -> 73 + 450. Without a mask
//    they are equal, and one round of them is as good as several: 256 (8 x 512, 32 on 4) 158 + 538 -> 104 + 420, 132
//    (3 x 700) 140 + 498 -> 93 + 490; 88 (4 x 700, 32 on 2) 632 -> 830;
//  * tiles: 129 tokens (8 sequences, 32 heads) 23 + 70 -> 18 + 70, 90 (12) 23 + 62 -> 18 + 64, 80 21 + 54 -> 17 + 61; one tile
//    alone wants to be full: 64 (24) 24 + 72 -> 21 + 70, 48 20 + 56 -> 18 + 63.
bool split_backward_pays(const ft_context* ctx, const AttnArgs& a) {
    const size_t cus = (size_t)ctx->num_cus;
    auto full = [](int rows) { return rows <= 64 ? rows >= 56 : 3 * (size_t)rows >= 2 * 64 * (size_t)ft_div_up(rows, 64); };
    if (ctx->f32_chain || !full(a.Sq) || !full(a.Sk) || ft_div_up(a.Sq, 128) * (size_t)a.B * a.H * 2 < 3 * cus) return false;
    const DkdvUnits u = split_dkdv_units(a);
    if (!u.per_head) return u.workgroups * 8 >= 9 * cus || (!a.causal && u.workgroups * 2 >= cus && u.workgroups <= cus);
    return u.workgroups >= 3 * cus && (a.H == a.Hkv || a.Sq >= (a.causal ? 320 : 256));
}
// Alone the forward on bf16 parts beats the f32 kernels nearly everywhere, the 32-row ones too (1 x 96 tokens, 15 heads, 7.0
// us against 8.0; 2 x 160, 9 heads 8.7 against 11.4; 1 x 8, 9 heads 4.6 against 6.5), but not the 16-row ones with half a tile
// of queries (4 x 8, 32 heads 5.4 against 4.7) and not where so few workgroups have so long a row of keys that four waves
// sharing it are worth more (1 x 1024, 3 heads 31.4 against 29.2; 1 x 384 15.0 against 14.6).
bool split_forward_pays(const ft_context* ctx, const AttnArgs& a) {
    if (ctx->f32_chain) return false;
    if (a.forward_only) return query_tile_groups(ctx, a, false) != 0 ? a.Sq >= 32 : a.Sk <= 256;
    return split_backward_pays(ctx, a);
}

// One workgroup per 64 keys and query head, then the ordered sum over the group where there is one (and room for its
// shares; otherwise per kv head).
int launch_split_dkdv(ft_context* ctx, const AttnArgs& a) {
    AttnArgs s = a;
    if (a.H > a.Hkv && split_dkdv_units(a).per_head) {
        s.part = ft_scratch_or_none(ctx, &ctx->attn_scratch, kAttnScratchFloats);   // (the f32 kernels need none here)
        s.split_g = s.part != nullptr;
    }
    FT_TRY(ft_attn_split_dkdv(ctx, s));
    return s.split_g ? ft_attn_dkdv_combine(ctx, s, 64) : FT_OK;
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

bool ft_attn16_forward_pays(const ft_context* ctx, const AttnArgs& a) {
    return split_forward_pays(ctx, a) || query_tile_groups(ctx, a, false) != 0;
}
bool ft_attn16_backward_dq_pays(const ft_context* ctx, const AttnArgs& a) {
    return (!a.rope && split_backward_pays(ctx, a)) || query_tile_groups(ctx, a, true) != 0;
}

int ft_attn16_forward(ft_context* ctx, const AttnArgs& a) {
    if (split_forward_pays(ctx, a)) {
        const int groups = query_tile_groups(ctx, a, false);
        return ft_attn_split_forward(ctx, a, groups ? groups : 2);
    }
    return query_tile_groups(ctx, a, false) == 2 ? launch_query_kernels<2>(ctx, a, false)
                                                 : launch_query_kernels<4>(ctx, a, false);
}

int ft_attn16_backward_dq(ft_context* ctx, const AttnArgs& a) {
    if (!a.rope && split_backward_pays(ctx, a)) return ft_attn_split_dq(ctx, a);
    return query_tile_groups(ctx, a, true) == 2 ? launch_query_kernels<2>(ctx, a, true)
                                                : launch_query_kernels<4>(ctx, a, true);
}

int ft_attn16_backward_dkdv(ft_context* ctx, const AttnArgs& a) {
    if (!a.rope && split_backward_pays(ctx, a)) return launch_split_dkdv(ctx, a);
    return launch_dkdv<64>(ctx, a);
}

// Which call takes the kernels on bf16 parts (outside a training step, operands aligned), for callers that have no device (its
// test): the backward with the forward before it, or a forward alone.
extern "C" int ft_internal_attention_split(size_t cus, size_t B, size_t Sq, size_t Sk, size_t H, size_t Hkv, int causal,
                                           int forward_only) {
    ft_context ctx;
    ctx.num_cus = (int)cus;
    AttnArgs a{};
    a.B = (int)B, a.Sq = (int)Sq, a.Sk = (int)Sk, a.H = (int)H, a.Hkv = (int)Hkv, a.D = 64, a.causal = causal;
    a.forward_only = forward_only;
    return split_forward_pays(&ctx, a) ? 1 : 0;
}
