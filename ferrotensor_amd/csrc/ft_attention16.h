// The query-row parts of the 16-row attention kernels (see ft_attention16.hip): what a workgroup does in the forward and
// dQ kernels, for the kernels themselves and for those on bf16 parts (ft_attention_split.hip), which share the work
// decomposition and come back to these where a result is not finite.
#pragma once

#include "ft_attention.h"

#include <type_traits>

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
#define MFMA16(a, b, c) __builtin_amdgcn_mfma_f32_16x16x4f32((a), (b), (c), 0, 0, 0)

constexpr int KT = 64;  // keys per shared K/V tile (forward, dQ)
constexpr float kLog2e = 1.44269504088896340736f;
constexpr float kLn2 = 0.69314718055994530942f;

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float log2_fast(float x) { return __builtin_amdgcn_logf(x); }
__device__ __forceinline__ floatx4 zero4() { return floatx4{0.0f, 0.0f, 0.0f, 0.0f}; }

// A query's (or key's) 16 values sit in the four lanes l16, l16 + 16, l16 + 32, l16 + 48: the two
// gfx950 lane swaps bring them together without a trip through LDS. v_permlane32_swap exchanges the
// upper 32 lanes of its first operand with the lower 32 of its second, v_permlane16_swap the odd
// 16-lane rows of the first with the even rows of the second; called on (x, x) the two results
// hold a lane's own value and its partner's.
__device__ __forceinline__ float group_max(float x) {
    auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
// Sum in a fixed order: (g0 + g1) + (g2 + g3) in every lane.
__device__ __forceinline__ float group_sum(float x) {
    auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(b[0]) + __uint_as_float(b[1]);
    auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}
// The value held by the lane 32 away.
__device__ __forceinline__ float other_half(float x) {
    auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    const float lo = __uint_as_float(a[0]), hi = __uint_as_float(a[1]);
    // after the swap a[0] = (x.lo, x.lo) and a[1] = (x.hi, x.hi): lanes below 32 want x.hi
    return (threadIdx.x & 32) ? lo : hi;
}

// EV consecutive floats from LDS (EV * 4 bytes aligned).
template <int EV>
__device__ __forceinline__ void lds_vec(const float* src, float (&v)[EV]) {
    if constexpr (EV == 4) {
        const float4 t = *reinterpret_cast<const float4*>(src);
        v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
    } else if constexpr (EV == 2) {
        const float2 t = *reinterpret_cast<const float2*>(src);
        v[0] = t.x; v[1] = t.y;
    } else {
#pragma unroll
        for (int e = 0; e < EV; e++) v[e] = src[e];
    }
}
template <int EV>
__device__ __forceinline__ void store_vec(float* dst, const float (&v)[EV]) {
    if constexpr (EV == 4) {
        *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
    } else if constexpr (EV == 2) {
        *reinterpret_cast<float2*>(dst) = make_float2(v[0], v[1]);
    } else {
#pragma unroll
        for (int e = 0; e < EV; e++) dst[e] = v[e];
    }
}

// Writes of a wave to its own LDS tile become visible to its later reads.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS tiles are rows of 64 floats (16 chunks of 16 bytes) with the chunk index XOR-swizzled by
// the row. gfx950 serves a 16-byte-per-lane LDS access 16 lanes at a time, and the 16 are not
// neighbours: lanes 0-3, 12-15, 20-23, 24-27 go together (measured), i.e. half of one 16-lane row
// and the other half of the next. Both access shapes used here must spread such a group over all
// 64 banks: "column" reads (lane l16 takes row l16, all four rows of lanes one chunk each) and
// "row" reads (the 16 lanes of a lane row take the 16 chunks of one tile row, each lane row its own
// tile row 4 apart). f(r) = r ^ ((r & 4) << 1) does that for both; plain padding cannot.
__device__ __forceinline__ int sw(int row, int chunk) {
    const int r = row & 15;
    return row * 64 + (((chunk ^ r ^ ((r & 4) << 1)) & 15) << 2);
}

// ---------------------------------------------------------------------------
// Work decomposition of the forward and dQ kernels. A head's queries are cut in
// tiles of TQ = 16 * NG rows; a workgroup takes the tile pair (nT - 1 - i, i) of
// one (batch, head): under the causal mask every pair is the same amount of work,
// and both tiles walk the same K/V tiles (64 keys, staged once in LDS for all
// waves, double buffered). Sixteen query rows belong to TWO waves, one per half of
// every K/V tile (keys 0-31 and 32-63 of the tile), so the longest chain of
// dependent work is half a row block's keys; the halves meet once, through LDS,
// after the last tile. Wave order: key half, then tile of the pair, then row
// block; the row blocks of the early tile are taken in reverse, so that the four
// waves on a SIMD (waves w, w + 4, ...) add up to the same key count everywhere.
// ---------------------------------------------------------------------------
constexpr int D64 = 64;
constexpr int TILE = KT * D64;   // floats of one K or V tile in LDS
constexpr int HALF = 32 * D64;   // floats of one key half of a tile

template <int NG>
struct QueryWave {
    static constexpr int TQ = 16 * NG;
    int b, h, kvh;
    int kh;        // key half of every tile this wave multiplies
    int w2;        // index among the waves of its half
    int q0w;       // first query row of this wave
    int q;         // this lane's query row (may be >= Sq)
    int qc;        // clamped to a valid row
    bool q_ok;
    int kend_w;    // one past the last key any row of this wave may see (0: nothing to do)
    int kfull_w;   // keys below this are visible to every row of the wave
    int nkt;       // K/V tiles the workgroup walks

    __device__ __forceinline__ void init(const AttnArgs& p, int wave, int l16) {
        const int nbh = p.B * p.H;
        const int nT = (p.Sq + TQ - 1) / TQ;
        const int pi = blockIdx.x / nbh, bh = blockIdx.x % nbh;
        b = bh / p.H;
        h = bh % p.H;
        kvh = h / (p.H / p.Hkv);
        const int JA = nT - 1 - pi, JB = pi;
        kh = wave / (2 * NG);
        w2 = wave % (2 * NG);
        const int grp = w2 / NG, wr = w2 % NG;
        const bool active = grp == 0 || JB != JA;
        const int J = grp == 0 ? JA : JB;
        const int rb = grp == 0 ? wr : NG - 1 - wr;
        q0w = J * TQ + 16 * rb;
        q = q0w + l16;
        q_ok = active && q < p.Sq;
        qc = q < p.Sq ? q : p.Sq - 1;
        const int qlast_w = q0w + 15 < p.Sq ? q0w + 15 : p.Sq - 1;
        kend_w = (active && q0w < p.Sq) ? key_end(p, qlast_w) : 0;
        kfull_w = p.causal ? q0w + p.causal_offset + 1 : p.Sk;
        if (kfull_w > p.Sk) kfull_w = p.Sk;
        const int qlast_wg = ((JA + 1) * TQ < p.Sq ? (JA + 1) * TQ : p.Sq) - 1;
        nkt = (key_end(p, qlast_wg) + KT - 1) / KT;
    }
    static __device__ __forceinline__ int key_end(const AttnArgs& p, int qlast) {
        int e = p.Sk;
        if (p.causal) {
            const int c = qlast + p.causal_offset + 1;
            e = c < e ? c : e;
        }
        return e < 0 ? 0 : e;
    }
    // 16-key sub-blocks of this wave's half of the tile at key kb that some row can see (0..2)
    __device__ __forceinline__ int visible_subblocks(int kb) const {
        int n = (kend_w - kb + 15) / 16 - 2 * kh;
        n = n < 2 ? n : 2;
        return n > 0 ? n : 0;
    }
    // is every key of this wave's half of that tile visible to every row?
    __device__ __forceinline__ bool half_unmasked(int kb) const { return kb + 32 * (kh + 1) <= kfull_w; }
};

// The K/V tile of 64 keys: global -> registers (the next tile's while the current one multiplies)
// -> LDS. Defines kv_fetch(t) and kv_store(stage) over the local arrays kpre, vpre.
#define FT_ATTN16_KV_LOADER(p, w, tid, smem)                                                         \
    constexpr int LPT = KT * 16 / NT;                                                                \
    static_assert(KT * 16 % NT == 0, "a K/V tile must divide evenly over the workgroup");            \
    float4 kpre[LPT], vpre[LPT];                                                                     \
    auto kv_fetch = [&](int t) {                                                                     \
        _Pragma("unroll") for (int u = 0; u < LPT; u++) {                                            \
            const int e = tid + NT * u;                                                              \
            const int r = e / 16, c = e % 16;                                                        \
            int key = t * KT + r;                                                                    \
            key = key < p.Sk ? key : p.Sk - 1;                                                       \
            const long o = (((long)w.b * p.Sk + key) * p.Hkv + w.kvh) * D64 + 4 * c;                 \
            kpre[u] = *reinterpret_cast<const float4*>(p.k + o);                                     \
            vpre[u] = *reinterpret_cast<const float4*>(p.v + o);                                     \
        }                                                                                            \
    };                                                                                               \
    auto kv_store = [&](int stage) {                                                                 \
        float* ks_ = smem + stage * 2 * TILE;                                                        \
        _Pragma("unroll") for (int u = 0; u < LPT; u++) {                                            \
            const int e = tid + NT * u;                                                              \
            const int r = e / 16, c = e % 16;                                                        \
            *reinterpret_cast<float4*>(ks_ + sw(r, c)) =                                             \
                make_float4(kpre[u].x, kpre[u].y, kpre[u].z, kpre[u].w);                             \
            *reinterpret_cast<float4*>(ks_ + TILE + sw(r, c)) =                                      \
                make_float4(vpre[u].x, vpre[u].y, vpre[u].z, vpre[u].w);                             \
        }                                                                                            \
    }

template <int NG>
__device__ __forceinline__ void attn16_fwd(const AttnArgs& p, float* smem) {   // smem: [2 stages][K tile, V tile]
    constexpr int NT = 4 * NG * 64;
    const int tid = threadIdx.x, lane = tid % 64, l16 = lane % 16, g = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);  // wave-uniform: the tile bookkeeping stays in SGPRs

    QueryWave<NG> w;
    w.init(p, wave, l16);
    FT_ATTN16_KV_LOADER(p, w, tid, smem);
    if (w.nkt > 0) kv_fetch(0);

    // this lane's swizzled offsets into a tile: "column" reads (row l16 of a sub-block, chunk
    // 4 blk + g) and "row" reads (row 4 g + i, chunk l16), both within the wave's key half
    int off_col[4], off_row[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        off_col[j] = sw(l16, 4 * j + g) + w.kh * HALF;
        off_row[j] = sw(4 * g + j, l16) + w.kh * HALF;
    }

    // scores are kept in base 2: log2(e) / sqrt(D) goes into Q
    const float qscale = p.scale * kLog2e;
    const float* qrow = p.q + (((long)w.b * p.Sq + w.qc) * p.H + w.h) * D64;
    float4 qf[4];
#pragma unroll
    for (int blk = 0; blk < 4; blk++) {
        const float4 t = *reinterpret_cast<const float4*>(qrow + 16 * blk + 4 * g);
        qf[blk] = make_float4(t.x * qscale, t.y * qscale, t.z * qscale, t.w * qscale);
    }
    floatx4 o[4];
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] = zero4();
    float m_run = kAttnMasked, l_lane = 0.0f;
    // the last key this lane's query may see
    const int key_lim = (p.causal && w.q + p.causal_offset < p.Sk - 1) ? w.q + p.causal_offset : p.Sk - 1;

    if (w.nkt > 0) kv_store(0);
    __syncthreads();

    // This wave's half of one K/V tile against its 16 queries: NSB visible 16-key sub-blocks, MASK
    // when some key of them is hidden from some query (the diagonal, the end of the keys).
    auto tile = [&](auto nsb_tag, auto mask_tag, const float* ks, const float* vs, int kb) {
        constexpr int NSB = decltype(nsb_tag)::value;
        constexpr bool MASK = decltype(mask_tag)::value;
        floatx4 s[NSB];
#pragma unroll
        for (int u = 0; u < NSB; u++) s[u] = zero4();
#pragma unroll
        for (int blk = 0; blk < 4; blk++) {
            float4 kq[NSB];
#pragma unroll
            for (int u = 0; u < NSB; u++) kq[u] = *reinterpret_cast<const float4*>(ks + off_col[blk] + u * 16 * D64);
#pragma unroll
            for (int u = 0; u < NSB; u++) s[u] = MFMA16(kq[u].x, qf[blk].x, s[u]);
#pragma unroll
            for (int u = 0; u < NSB; u++) s[u] = MFMA16(kq[u].y, qf[blk].y, s[u]);
#pragma unroll
            for (int u = 0; u < NSB; u++) s[u] = MFMA16(kq[u].z, qf[blk].z, s[u]);
#pragma unroll
            for (int u = 0; u < NSB; u++) s[u] = MFMA16(kq[u].w, qf[blk].w, s[u]);
        }
        float tmax = kAttnMasked;
#pragma unroll
        for (int u = 0; u < NSB; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if constexpr (MASK) {
                    const int key = kb + 32 * w.kh + 16 * u + 4 * g + i;
                    s[u][i] = key <= key_lim ? s[u][i] : kAttnMasked;
                }
                tmax = fmaxf(tmax, s[u][i]);
            }
        tmax = group_max(tmax);
        const float m_new = fmaxf(m_run, tmax);
        const float corr = exp2_fast(m_run - m_new);
        float psum = 0.0f;
#pragma unroll
        for (int u = 0; u < NSB; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float pj = exp2_fast(s[u][i] - m_new);
                if constexpr (MASK) pj = s[u][i] > kAttnMasked ? pj : 0.0f;
                s[u][i] = pj;
                psum += pj;
            }
        l_lane = l_lane * corr + psum;  // this lane's keys only; the lanes of a query meet at the end
        m_run = m_new;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] *= corr;
#pragma unroll
        for (int u = 0; u < NSB; u++) {
            float4 vv[4];
#pragma unroll
            for (int i = 0; i < 4; i++) vv[i] = *reinterpret_cast<const float4*>(vs + off_row[i] + u * 16 * D64);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                o[0] = MFMA16(vv[i].x, s[u][i], o[0]);
                o[1] = MFMA16(vv[i].y, s[u][i], o[1]);
                o[2] = MFMA16(vv[i].z, s[u][i], o[2]);
                o[3] = MFMA16(vv[i].w, s[u][i], o[3]);
            }
        }
    };
    using std::integral_constant;

    for (int t = 0; t < w.nkt; t++) {
        const bool more = t + 1 < w.nkt;
        if (more) kv_fetch(t + 1);
        const float* ks = smem + (t & 1) * 2 * TILE;
        const float* vs = ks + TILE;
        const int kb = t * KT;
        const int nsb = w.visible_subblocks(kb);
        if (nsb > 0) {
            if (w.half_unmasked(kb))
                tile(integral_constant<int, 2>{}, std::false_type{}, ks, vs, kb);
            else if (nsb == 2)
                tile(integral_constant<int, 2>{}, std::true_type{}, ks, vs, kb);
            else
                tile(integral_constant<int, 1>{}, std::true_type{}, ks, vs, kb);
        }
        if (more) kv_store((t + 1) & 1);
        __syncthreads();
    }

    // The two key halves of a row block meet: the second half's (m, l, O) go through LDS (the
    // K/V stages are free now), lane for lane, and the first half finishes the softmax.
    float* mrg = smem + (w.w2 * 18) * 64 + lane;
    if (w.kh == 1) {
        mrg[0] = m_run;
        mrg[64] = l_lane;
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int r = 0; r < 4; r++) mrg[(2 + 4 * e + r) * 64] = o[e][r];
    }
    __syncthreads();
    if (w.kh == 1) return;
    {
        const float m_o = mrg[0], l_o = mrg[64];
        const float m_new = fmaxf(m_run, m_o);
        const float c0 = exp2_fast(m_run - m_new), c1 = exp2_fast(m_o - m_new);
        l_lane = l_lane * c0 + l_o * c1;
        m_run = m_new;
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int r = 0; r < 4; r++) o[e][r] = o[e][r] * c0 + mrg[(2 + 4 * e + r) * 64] * c1;
    }
    const float l_run = group_sum(l_lane);
    if (!w.q_ok) return;
    const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
    // register r of accumulator e is head-dim index 4 * (4 g + r) + e
    float* orow = p.o + (((long)w.b * p.Sq + w.q) * p.H + w.h) * D64;
#pragma unroll
    for (int r = 0; r < 4; r++)
        *reinterpret_cast<float4*>(orow + 4 * (4 * g + r)) =
            make_float4(o[0][r] * inv, o[1][r] * inv, o[2][r] * inv, o[3][r] * inv);
    if (p.stats && g == 0)
        p.stats[2 * (((long)w.b * p.H + w.h) * p.Sq + w.q) + 1] =
            l_run > 0.0f ? (m_run + log2_fast(l_run)) * kLn2 : kAttnLseEmpty;
}

// ---------------------------------------------------------------------------
// Backward, pass 1: Delta = dO.O (stats slot 0) and dQ = scale * sum_j dS_ij K_j,
// dS = P (dO.V - Delta), P = exp(S - LSE). Same decomposition as the forward; the
// two key halves of a row block add their partial dQ through LDS at the end.
// ---------------------------------------------------------------------------
template <int NG>
__device__ __forceinline__ void attn16_dq(const AttnArgs& p, float* smem) {
    constexpr int NT = 4 * NG * 64;
    const int tid = threadIdx.x, lane = tid % 64, l16 = lane % 16, g = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);

    QueryWave<NG> w;
    w.init(p, wave, l16);
    FT_ATTN16_KV_LOADER(p, w, tid, smem);
    if (w.nkt > 0) kv_fetch(0);

    int off_col[4], off_row[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        off_col[j] = sw(l16, 4 * j + g) + w.kh * HALF;
        off_row[j] = sw(4 * g + j, l16) + w.kh * HALF;
    }

    const float qscale = p.scale * kLog2e;
    const long qoff = (((long)w.b * p.Sq + w.qc) * p.H + w.h) * D64;
    const long srow = ((long)w.b * p.H + w.h) * p.Sq + w.qc;
    float4 qf[4], dof[4];
    float delta = 0.0f;
#pragma unroll
    for (int blk = 0; blk < 4; blk++) {
        const int d = 16 * blk + 4 * g;
        const float4 t = *reinterpret_cast<const float4*>(p.q + qoff + d);
        qf[blk] = make_float4(t.x * qscale, t.y * qscale, t.z * qscale, t.w * qscale);
        dof[blk] = *reinterpret_cast<const float4*>(p.d_out + qoff + d);
        const float4 ov = *reinterpret_cast<const float4*>(p.out + qoff + d);
        delta += dof[blk].x * ov.x + dof[blk].y * ov.y + dof[blk].z * ov.z + dof[blk].w * ov.w;
    }
    delta = group_sum(delta);
    const float lse2 = (w.q_ok ? p.stats[2 * srow + 1] : kAttnLseEmpty) * kLog2e;
    if (w.q_ok && g == 0 && w.kh == 0) p.stats[2 * srow] = delta;

    floatx4 acc[4];
#pragma unroll
    for (int e = 0; e < 4; e++) acc[e] = zero4();
    // the last key this lane's query may see
    const int key_lim = (p.causal && w.q + p.causal_offset < p.Sk - 1) ? w.q + p.causal_offset : p.Sk - 1;

    if (w.nkt > 0) kv_store(0);
    __syncthreads();

    auto tile = [&](auto nsb_tag, auto mask_tag, const float* ks, const float* vs, int kb) {
        constexpr int NSB = decltype(nsb_tag)::value;
        constexpr bool MASK = decltype(mask_tag)::value;
        floatx4 s[NSB], dp[NSB];
#pragma unroll
        for (int u = 0; u < NSB; u++) {
            s[u] = zero4();
            dp[u] = zero4();
        }
#pragma unroll
        for (int blk = 0; blk < 4; blk++) {
            float4 kq[NSB], vq[NSB];
#pragma unroll
            for (int u = 0; u < NSB; u++) {
                kq[u] = *reinterpret_cast<const float4*>(ks + off_col[blk] + u * 16 * D64);
                vq[u] = *reinterpret_cast<const float4*>(vs + off_col[blk] + u * 16 * D64);
            }
#pragma unroll
            for (int u = 0; u < NSB; u++) {
                s[u] = MFMA16(kq[u].x, qf[blk].x, s[u]);
                dp[u] = MFMA16(vq[u].x, dof[blk].x, dp[u]);
            }
#pragma unroll
            for (int u = 0; u < NSB; u++) {
                s[u] = MFMA16(kq[u].y, qf[blk].y, s[u]);
                dp[u] = MFMA16(vq[u].y, dof[blk].y, dp[u]);
            }
#pragma unroll
            for (int u = 0; u < NSB; u++) {
                s[u] = MFMA16(kq[u].z, qf[blk].z, s[u]);
                dp[u] = MFMA16(vq[u].z, dof[blk].z, dp[u]);
            }
#pragma unroll
            for (int u = 0; u < NSB; u++) {
                s[u] = MFMA16(kq[u].w, qf[blk].w, s[u]);
                dp[u] = MFMA16(vq[u].w, dof[blk].w, dp[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < NSB; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float pij = exp2_fast(s[u][i] - lse2);
                if constexpr (MASK) {
                    const int key = kb + 32 * w.kh + 16 * u + 4 * g + i;
                    pij = key <= key_lim ? pij : 0.0f;
                }
                s[u][i] = pij * (dp[u][i] - delta);  // dS
            }
#pragma unroll
        for (int u = 0; u < NSB; u++) {
            float4 kk[4];
#pragma unroll
            for (int i = 0; i < 4; i++) kk[i] = *reinterpret_cast<const float4*>(ks + off_row[i] + u * 16 * D64);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                acc[0] = MFMA16(kk[i].x, s[u][i], acc[0]);
                acc[1] = MFMA16(kk[i].y, s[u][i], acc[1]);
                acc[2] = MFMA16(kk[i].z, s[u][i], acc[2]);
                acc[3] = MFMA16(kk[i].w, s[u][i], acc[3]);
            }
        }
    };
    using std::integral_constant;

    for (int t = 0; t < w.nkt; t++) {
        const bool more = t + 1 < w.nkt;
        if (more) kv_fetch(t + 1);
        const float* ks = smem + (t & 1) * 2 * TILE;
        const float* vs = ks + TILE;
        const int kb = t * KT;
        const int nsb = w.visible_subblocks(kb);
        if (nsb > 0) {
            if (w.half_unmasked(kb))
                tile(integral_constant<int, 2>{}, std::false_type{}, ks, vs, kb);
            else if (nsb == 2)
                tile(integral_constant<int, 2>{}, std::true_type{}, ks, vs, kb);
            else
                tile(integral_constant<int, 1>{}, std::true_type{}, ks, vs, kb);
        }
        if (more) kv_store((t + 1) & 1);
        __syncthreads();
    }

    // the second key half's partial dQ joins the first's, lane for lane
    float* mrg = smem + (w.w2 * 16) * 64 + lane;
    if (w.kh == 1) {
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int r = 0; r < 4; r++) mrg[(4 * e + r) * 64] = acc[e][r];
    }
    __syncthreads();
    if (w.kh == 1) return;
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[e][r] += mrg[(4 * e + r) * 64];

    // K in LDS carries no scale (only Q does, for the scores): dQ = scale * dS K.
    // Register r of accumulator e is head-dim index 4 * (4 g + r) + e.
    float* drow = p.dq + qoff;
    if (p.rope) {
        // the partner of head-dim index d (d +- 32) sits in lane g ^ 2 at the same register
        const float2* tb = p.rope + (long)w.qc * 32;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float own = acc[e][r] * p.scale;
                const float other = other_half(own);
                const float2 cs = tb[(16 * g + 4 * r + e) & 31];
                v[e] = g < 2 ? own * cs.x + other * cs.y : own * cs.x - other * cs.y;
            }
            if (w.q_ok) *reinterpret_cast<float4*>(drow + 16 * g + 4 * r) = make_float4(v[0], v[1], v[2], v[3]);
        }
        return;
    }
    if (!w.q_ok) return;
#pragma unroll
    for (int r = 0; r < 4; r++)
        *reinterpret_cast<float4*>(drow + 4 * (4 * g + r)) =
            make_float4(acc[0][r] * p.scale, acc[1][r] * p.scale, acc[2][r] * p.scale, acc[3][r] * p.scale);
}

}  // namespace
