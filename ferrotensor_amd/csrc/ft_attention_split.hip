// Attention outside a training step, head dim 64: the work of the 16-row kernels (ft_attention16.hip) on
// v_mfma_f32_16x16x32_bf16. Every operand, probabilities and dS too, is the sum of three bf16 parts and a product is six
// products of parts, as in ft_split.hip: f32 operands and f32 sums at 2.7 times the rate of the f32 instruction.
//
// K and V are split once per workgroup, on their way into LDS, as three planes each: rows of a key for the products over
// the head dim, rows of a head-dim index (32 keys of a wave's half, in the order in which the probabilities leave the
// score product's registers: 16 u + 4 g + i at 8 g + 4 u + i) for the products over the keys. The probabilities then
// are the second operand of their product without leaving their lane.
//
// A score that is NaN, a result that is not finite (infinite or NaN inputs, values that round to an infinite bf16), an operand
// that three parts do not hold (below 2^-110) or a row of dQ or dK so small that its dS may be among those sends the workgroup
// through the f32 kernel's code, which says what it is. (Probabilities need no such look: their parts hold them to 2^-134,
// and exp2 makes zero of what is below 2^-126.) Looking for small ones costs the backward 3 to 5 %. The f32 code reads the
// operands again: where a result takes the place of one (o over q, dq over out, dk or dv over k or v: AttnArgs::in_place)
// the workgroup settles this before it writes, otherwise after (the vote first costs every call 1 to 4 %: 4 x 512 tokens,
// 32 heads, forward 41.0 -> 42.6 us).
//
// Relative error against f64 (2-norm), f32 kernels -> these, 4 x 1024 tokens, 15 heads on 5, normal values: o 2.8e-7 -> 2.1e-7,
// dq 4.4e-7 -> 3.6e-7, dk 5.6e-7 -> 3.4e-7, dv 5.1e-7 -> 3.0e-7; scores nine times as large (4 x 512, 32 heads): 9.3e-7 ->
// 6.0e-7, 2.1e-6 -> 1.5e-6, 2.5e-6 -> 1.5e-6, 2.0e-6 -> 1.1e-6.
//
// Bound: a tile of 64 keys costs a workgroup about 3000 cycles each of matrix unit, VALU (softmax and splitting) and LDS
// reads, and the barrier per tile keeps its waves in step, so they overlap little. us by HIP events, f32 kernel -> this:
// forward of 4 x 1024 tokens, 15 heads on 5: 93 -> 63, backward 285 -> 240; 8 x 1024, 32 heads: 363 -> 260 and 1264 ->
// 965; forward alone of 8 x 256, 15 on 5: 19.8 -> 14.8. Measured and not kept for the forward: one query tile of 64 rows per
// workgroup, two workgroups a CU (64, 272, 15.5); 32 rows a wave (61, 248, 17.5).
#include "ft_attention16.h"
#include "ft_parts.h"

namespace {

typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

constexpr int PLANE = KT * D64 * 2;   // bytes of one part of a 64-key tile

// Two values into the packed halves of their three parts.
__device__ __forceinline__ void split2(float x, float y, unsigned (&part)[3], unsigned* left = nullptr) {
#pragma unroll
    for (int t = 0; t < 3; t++) {
        if (t == 2 && left) collect_left(*left, x, y);
        const unsigned q = pack2(x, y);
        part[t] = q;
        if (t < 2) {
            x -= low_half(q);
            y -= high_half(q);
        }
    }
}
// Eight values of a lane into the operand registers of their parts.
__device__ __forceinline__ void split8(const float (&x)[8], uintx4 (&part)[3], unsigned* left = nullptr) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
        unsigned q[3];
        split2(x[2 * e], x[2 * e + 1], q, left);
#pragma unroll
        for (int t = 0; t < 3; t++) part[t][e] = q[t];
    }
}

// acc += a b over 32 k, smallest products first. SWAPPED: in the order that mfma_parts(b, a) takes.
template <bool SWAPPED = false>
__device__ __forceinline__ floatx4 mfma_parts(const uintx4 (&a)[3], const uintx4 (&b)[3], floatx4 acc) {
    constexpr int U[6] = {2, 0, 1, 1, 0, 0}, V[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int t = 0; t < 6; t++)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[SWAPPED ? V[t] : U[t]]),
                                                      __builtin_bit_cast(bf16x8, b[SWAPPED ? U[t] : V[t]]), acc, 0, 0, 0);
    return acc;
}

// A score in base 2, rounded here and nowhere else: the three kernels take the same products in the same order and
// exponentiate the same number, so what a score is off by leaves the probabilities with the log-sum-exp. (A fused
// multiply-add with what is subtracted from it would round elsewhere.)
__device__ __forceinline__ float scaled_score(float s, float scale) {
#pragma clang fp contract(off)
    return s * scale;
}

// Chunk swizzles (16 bytes) that spread the 16 lanes served together over all banks, see ft_attention16.h: rows of 128
// bytes (a key's 64 head-dim values) and of 64 bytes (a head-dim index's 32 keys).
__device__ __forceinline__ int sw_key(int row, int chunk) { return row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4); }
__device__ __forceinline__ int sw_dim(int row, int chunk) {
    const int x = (row >> 2) & 3;
    return row * 64 + ((chunk ^ (((x << 1) ^ ((x >> 1) * 3)) & 3)) << 4);
}

// One operand's tile of 64 rows (keys; queries in the dK/dV kernel) of one head on its way from global memory to LDS:
// four values a thread and round; rows past the end repeat the last.
template <int NT>
struct TileRows {       // planes [key][64]
    static constexpr int N = KT * 16 / NT;
    float4 pre[N];
    __device__ __forceinline__ float largest() const {   // of the tile's values of this thread
        float m = 0.0f;
#pragma unroll
        for (int u = 0; u < N; u++)
            m = fmaxf(fmaxf(fmaxf(fabsf(pre[u].x), fabsf(pre[u].y)), fmaxf(fabsf(pre[u].z), fabsf(pre[u].w))), m);
        return m;
    }
    __device__ __forceinline__ void fetch(const float* src, int stride, int rows, int t, int tid) {
#pragma unroll
        for (int u = 0; u < N; u++) {
            const int e = tid + NT * u;
            int row = t * KT + e / 16;
            row = row < rows ? row : rows - 1;
            pre[u] = *reinterpret_cast<const float4*>(src + (long)row * stride + 4 * (e % 16));
        }
    }
    __device__ __forceinline__ void store(char* planes, int tid, unsigned* left) const {
#pragma unroll
        for (int u = 0; u < N; u++) {
            const int e = tid + NT * u, c = e % 16;
            unsigned lo[3], hi[3];
            split2(pre[u].x, pre[u].y, lo, left);
            split2(pre[u].z, pre[u].w, hi, left);
            char* at = planes + sw_key(e / 16, c >> 1) + (c & 1) * 8;
#pragma unroll
            for (int q = 0; q < 3; q++) *reinterpret_cast<uintx2*>(at + q * PLANE) = uintx2{lo[q], hi[q]};
        }
    }
};
template <int NT>
struct TileColumns {    // planes [key half][64][32 keys]
    static constexpr int N = KT * 16 / NT;
    float pre[N][4];
    __device__ __forceinline__ void fetch(const float* src, int stride, int rows, int t, int tid) {
#pragma unroll
        for (int u = 0; u < N; u++) {
            const int e = tid + NT * u, d = e % 64, kg = e / 64;   // keys 4 kg .. 4 kg + 3
#pragma unroll
            for (int i = 0; i < 4; i++) {
                int row = t * KT + 4 * kg + i;
                row = row < rows ? row : rows - 1;
                pre[u][i] = src[(long)row * stride + d];
            }
        }
    }
    __device__ __forceinline__ void store(char* planes, int tid, unsigned* left = nullptr) const {
#pragma unroll
        for (int u = 0; u < N; u++) {
            const int e = tid + NT * u, d = e % 64, kg = e / 64;
            unsigned lo[3], hi[3];
            split2(pre[u][0], pre[u][1], lo, left);
            split2(pre[u][2], pre[u][3], hi, left);
            char* at = planes + (kg >> 3) * (PLANE / 2) + sw_dim(d, kg & 3) + ((kg >> 2) & 1) * 8;
#pragma unroll
            for (int q = 0; q < 3; q++) *reinterpret_cast<uintx2*>(at + q * PLANE) = uintx2{lo[q], hi[q]};
        }
    }
};

__device__ __forceinline__ void read_parts(const char* at, uintx4 (&part)[3]) {
#pragma unroll
    for (int q = 0; q < 3; q++) part[q] = *reinterpret_cast<const uintx4*>(at + q * PLANE);
}

// A row's 64 values (this lane's 16 of them) on their way to the two k steps' operand registers. The forward splits them
// behind its first tile and the barrier after it (before, the wait for these loads, the last ones, comes ahead of the tile:
// 33 tokens 5.6 us for 5.3); in the backward, which has no register to spare, that is slower.
struct Row {
    float4 pre[4];
    __device__ __forceinline__ void fetch(const float* row, int g) {
#pragma unroll
        for (int e = 0; e < 4; e++) pre[e] = *reinterpret_cast<const float4*>(row + 32 * (e / 2) + 8 * g + 4 * (e % 2));
    }
    __device__ __forceinline__ void parts(uintx4 (&part)[2][3], unsigned* left) const {
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            const float4 a = pre[2 * ks], b = pre[2 * ks + 1];
            const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
            split8(x, part[ks], left);
        }
    }
};

// What the backward kernels look out for, in LDS (a slot of its own per thread, so nobody waits) where their loops have no
// register to spare: what third parts leave over (split2), and the largest operand that dS is multiplied with.
struct Watch {
    unsigned left[512], most[512], all;
    __device__ __forceinline__ void start(int tid) {   // a barrier follows before join()
        left[tid] = most[tid] = 0;
        if (tid == 0) all = 0;
    }
    __device__ __forceinline__ void add(int tid, unsigned l, float m) {   // (non-negative floats compare as whole numbers)
        atomicOr(&left[tid], l);
        atomicMax(&most[tid], __float_as_uint(m));
    }
    __device__ __forceinline__ void join(int tid) {    // a barrier follows before largest()
        float m = __uint_as_float(most[tid]);
#pragma unroll
        for (int x = 1; x < 64; x *= 2) m = fmaxf(m, __shfl_xor(m, x));
        if (tid % 64 == 0) atomicMax(&all, __float_as_uint(m));
    }
    __device__ __forceinline__ float largest() const { return __uint_as_float(all); }
    __device__ __forceinline__ bool left_over(int tid) const { return ::left_over(left[tid]); }
};
// dS is a product and may be any small: its parts hold it to 2^-134 (half of bf16's smallest step). A row of a result that is
// a sum over `terms` of them times operands of at most `largest`, and that small, may be off by more than a rounding.
__device__ __forceinline__ bool too_small(const floatx4 (&row)[4], float terms, float largest, float scale) {
    float m = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
        for (int r = 0; r < 4; r++) m = fmaxf(m, fabsf(row[e][r]));
    m = group_max(m);
    return m > 0.0f && m < terms * largest * (scale * 0x1p-110f);
}

__device__ __forceinline__ bool not_finite(floatx4 v) {
    const float z = v[0] * 0.0f + v[1] * 0.0f + v[2] * 0.0f + v[3] * 0.0f;
    return !(z == 0.0f);
}

template <int NG>
__global__ __launch_bounds__(4 * NG * 64) void attn_split_fwd_kernel(AttnArgs p) {
    constexpr int NT = 4 * NG * 64, STAGE = 6 * PLANE;   // K rows, V columns
    __shared__ __attribute__((aligned(16))) char smem[2 * STAGE];
    const int tid = threadIdx.x, lane = tid % 64, l16 = lane % 16, g = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    QueryWave<NG> w;
    w.init(p, wave, l16);
    const int kv_stride = p.Hkv * D64;
    const float* const k_head = p.k + ((long)w.b * p.Sk * p.Hkv + w.kvh) * D64;
    const float* const v_head = p.v + ((long)w.b * p.Sk * p.Hkv + w.kvh) * D64;
    TileRows<NT> kl;
    TileColumns<NT> vl;
    if (w.nkt > 0) {
        kl.fetch(k_head, kv_stride, p.Sk, 0, tid);
        vl.fetch(v_head, kv_stride, p.Sk, 0, tid);
    }
    const float sscale = p.scale * kLog2e;   // scores are kept in base 2
    Row q_row;
    q_row.fetch(p.q + (((long)w.b * p.Sq + w.qc) * p.H + w.h) * D64, g);
    unsigned left = 0;
    floatx4 o[4];
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] = zero4();
    float m_run = kAttnMasked, l_lane = 0.0f;
    bool bad = false;   // something here is for the f32 code
    // the last key this lane's query may see
    const int key_lim = (p.causal && w.q + p.causal_offset < p.Sk - 1) ? w.q + p.causal_offset : p.Sk - 1;

    if (w.nkt > 0) {
        kl.store(smem, tid, &left);
        vl.store(smem + 3 * PLANE, tid, &left);
    }
    __syncthreads();
    uintx4 qp[2][3];
    q_row.parts(qp, &left);

    auto tile = [&](auto nsb_tag, auto mask_tag, const char* ks, const char* vs, int kb) {
        constexpr int NSB = decltype(nsb_tag)::value;
        constexpr bool MASK = decltype(mask_tag)::value;
        floatx4 s[2] = {zero4(), zero4()};
#pragma unroll
        for (int t = 0; t < 2; t++) {
            uintx4 kp[NSB][3];
#pragma unroll
            for (int u = 0; u < NSB; u++) read_parts(ks + sw_key(32 * w.kh + 16 * u + l16, 4 * t + g), kp[u]);
#pragma unroll
            for (int u = 0; u < NSB; u++) s[u] = mfma_parts(kp[u], qp[t], s[u]);
        }
        float tmax = kAttnMasked;
#pragma unroll
        for (int u = 0; u < NSB; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                s[u][i] = scaled_score(s[u][i], sscale);
                if constexpr (MASK) {
                    const int key = kb + 32 * w.kh + 16 * u + 4 * g + i;
                    s[u][i] = key <= key_lim ? s[u][i] : kAttnMasked;
                    bad = bad || s[u][i] != s[u][i];   // below, a NaN score counts as a masked one
                }
                tmax = fmaxf(tmax, s[u][i]);
            }
        tmax = group_max(tmax);
        const float m_new = fmaxf(m_run, tmax);
        const float corr = exp2_fast(m_run - m_new);
        float psum = 0.0f;
        float pr[8];
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float pj = 0.0f;
                if (u < NSB) {
                    pj = exp2_fast(s[u][i] - m_new);
                    if constexpr (MASK) pj = s[u][i] > kAttnMasked ? pj : 0.0f;
                    psum += pj;
                }
                pr[4 * u + i] = pj;
            }
        l_lane = l_lane * corr + psum;  // this lane's keys only; the lanes of a query meet at the end
        m_run = m_new;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] *= corr;
        uintx4 pp[3];
        split8(pr, pp);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            uintx4 vp[3];
            read_parts(vs + w.kh * (PLANE / 2) + sw_dim(16 * e + l16, g), vp);
            o[e] = mfma_parts(vp, pp, o[e]);
        }
    };
    using std::integral_constant;
    for (int t = 0; t < w.nkt; t++) {
        const bool more = t + 1 < w.nkt;
        if (more) {
            kl.fetch(k_head, kv_stride, p.Sk, t + 1, tid);
            vl.fetch(v_head, kv_stride, p.Sk, t + 1, tid);
        }
        const char* ks = smem + (t & 1) * STAGE;
        const char* vs = ks + 3 * PLANE;
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
        if (more) {
            char* next = smem + ((t + 1) & 1) * STAGE;
            kl.store(next, tid, &left);
            vl.store(next + 3 * PLANE, tid, &left);
        }
        __syncthreads();
    }

    // The two key halves of a row block meet through LDS, lane for lane.
    float* mrg = reinterpret_cast<float*>(smem) + (w.w2 * 18) * 64 + lane;
    if (w.kh == 1) {
        mrg[0] = m_run;
        mrg[64] = l_lane;
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int r = 0; r < 4; r++) mrg[(2 + 4 * e + r) * 64] = o[e][r];
    }
    __syncthreads();
    float lse = kAttnLseEmpty;
    if (w.kh == 0) {
        const float m_o = mrg[0], l_o = mrg[64];
        const float m_new = fmaxf(m_run, m_o);
        const float c0 = exp2_fast(m_run - m_new), c1 = exp2_fast(m_o - m_new);
        l_lane = l_lane * c0 + l_o * c1;
        m_run = m_new;
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int r = 0; r < 4; r++) o[e][r] = o[e][r] * c0 + mrg[(2 + 4 * e + r) * 64] * c1;
        const float l_run = group_sum(l_lane);
        const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
        if (l_run > 0.0f) lse = (m_run + log2_fast(l_run)) * kLn2;
        bad = bad || !(fabsf(lse) <= 3.0e38f) || !(l_run >= 0.0f);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            o[e] *= inv;
            bad = bad || not_finite(o[e]);
        }
    }
    bad = (bad && w.q_ok) || left_over(left);
    bool again = p.in_place && __syncthreads_or(bad);
    if (w.kh == 0 && w.q_ok && !again) {
        // register r of accumulator e is head-dim index 16 e + 4 g + r
        float* orow = p.o + (((long)w.b * p.Sq + w.q) * p.H + w.h) * D64;
#pragma unroll
        for (int e = 0; e < 4; e++) *reinterpret_cast<floatx4*>(orow + 16 * e + 4 * g) = o[e];
        if (p.stats && g == 0) p.stats[2 * (((long)w.b * p.H + w.h) * p.Sq + w.q) + 1] = lse;
    }
    if (!p.in_place) again = __syncthreads_or(bad);
    if (again) attn16_fwd<NG>(p, reinterpret_cast<float*>(smem));
}

// dQ = scale * sum_j dS_ij K_j and Delta = dO.O (stats slot 0), dS = P (dO.V - Delta), P = exp(S - LSE). A workgroup
// takes one query tile of 128 rows, the last (under the causal mask the longest) first; a wave 32 of them, against one
// half of every 64-key tile: 16 rows a wave on the forward's 16 waves need more than their 128 registers, and an operand
// read from LDS serves two blocks of rows.
__global__ __launch_bounds__(512, 2) void attn_split_dq_kernel(AttnArgs p) {
    constexpr int QB = 2;
    using Waves = QueryTile<4, QB>;
    constexpr int NT = Waves::WAVES * 64, STAGE = 9 * PLANE;   // K rows, V rows, K columns
    __shared__ __attribute__((aligned(16))) char smem[2 * STAGE];
    const int tid = threadIdx.x, lane = tid % 64, l16 = lane % 16, g = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int nbh = p.B * p.H, qtile = (p.Sq + Waves::TQ - 1) / Waves::TQ - 1 - (int)blockIdx.x / nbh, qbh = (int)blockIdx.x % nbh;
    Waves w;
    w.init(p, wave, l16, qtile, qbh);
    const int kv_stride = p.Hkv * D64;
    const float* const k_head = p.k + ((long)w.b * p.Sk * p.Hkv + w.kvh) * D64;
    const float* const v_head = p.v + ((long)w.b * p.Sk * p.Hkv + w.kvh) * D64;
    TileRows<NT> kl, vl;
    TileColumns<NT> kc;
    auto fetch = [&](int t) {
        kl.fetch(k_head, kv_stride, p.Sk, t, tid);
        vl.fetch(v_head, kv_stride, p.Sk, t, tid);
        kc.fetch(k_head, kv_stride, p.Sk, t, tid);
    };
    __shared__ Watch watch;
    watch.start(tid);
    auto store = [&](char* stage) {
        unsigned left = 0;
        kl.store(stage, tid, &left);
        vl.store(stage + 3 * PLANE, tid, &left);
        kc.store(stage + 6 * PLANE, tid);
        watch.add(tid, left, kl.largest());
    };
    unsigned left = 0;
    if (w.nkt > 0) fetch(0);
    const float sscale = p.scale * kLog2e;
    uintx4 qp[QB][2][3], dop[QB][2][3];
    float delta[QB], lse2[QB];
    int key_lim[QB];
    floatx4 acc[QB][4];
#pragma unroll
    for (int c = 0; c < QB; c++) {
        const int q = w.q + 16 * c, qc = q < p.Sq ? q : p.Sq - 1;
        const long qoff = (((long)w.b * p.Sq + qc) * p.H + w.h) * D64;
        const long srow = ((long)w.b * p.H + w.h) * p.Sq + qc;
        Row q_row, do_row;
        q_row.fetch(p.q + qoff, g);
        q_row.parts(qp[c], &left);
        do_row.fetch(p.d_out + qoff, g);
        do_row.parts(dop[c], &left);
        delta[c] = 0.0f;
#pragma unroll
        for (int blk = 0; blk < 4; blk++) {   // dO.O as the f32 kernel adds it
            const int d = 16 * blk + 4 * g;
            const float4 dv = *reinterpret_cast<const float4*>(p.d_out + qoff + d);
            const float4 ov = *reinterpret_cast<const float4*>(p.out + qoff + d);
            delta[c] += dv.x * ov.x + dv.y * ov.y + dv.z * ov.z + dv.w * ov.w;
        }
        delta[c] = group_sum(delta[c]);
        lse2[c] = (q < p.Sq ? p.stats[2 * srow + 1] : kAttnLseEmpty) * kLog2e;
        if (q < p.Sq && g == 0 && w.kh == 0) p.stats[2 * srow] = delta[c];
        key_lim[c] = (p.causal && q + p.causal_offset < p.Sk - 1) ? q + p.causal_offset : p.Sk - 1;
#pragma unroll
        for (int e = 0; e < 4; e++) acc[c][e] = zero4();
    }
    watch.add(tid, left, 0.0f);
    if (w.nkt > 0) store(smem);
    __syncthreads();

    bool bad = false;   // something here is for the f32 code
    auto tile = [&](auto nsb_tag, auto mask_tag, const char* stage, int kb) {
        constexpr int NSB = decltype(nsb_tag)::value;
        constexpr bool MASK = decltype(mask_tag)::value;
        float ds[QB][8];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            floatx4 s[QB], dp[QB];
#pragma unroll
            for (int c = 0; c < QB; c++) s[c] = dp[c] = zero4();
            if (u < NSB) {
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const int at = sw_key(32 * w.kh + 16 * u + l16, 4 * t + g);
                    uintx4 kp[3], vp[3];
                    read_parts(stage + at, kp);
                    read_parts(stage + 3 * PLANE + at, vp);
#pragma unroll
                    for (int c = 0; c < QB; c++) s[c] = mfma_parts(kp, qp[c][t], s[c]);
#pragma unroll
                    for (int c = 0; c < QB; c++) dp[c] = mfma_parts(vp, dop[c][t], dp[c]);
                }
            }
#pragma unroll
            for (int c = 0; c < QB; c++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float pij = u < NSB ? exp2_fast(scaled_score(s[c][i], sscale) - lse2[c]) : 0.0f;
                    if constexpr (MASK) {
                        const int key = kb + 32 * w.kh + 16 * u + 4 * g + i;
                        pij = key <= key_lim[c] ? pij : 0.0f;
                    }
                    ds[c][4 * u + i] = u < NSB ? pij * (dp[c][i] - delta[c]) : 0.0f;
                }
        }
        uintx4 sp[QB][3];
#pragma unroll
        for (int c = 0; c < QB; c++) split8(ds[c], sp[c]);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            uintx4 kp[3];
            read_parts(stage + 6 * PLANE + w.kh * (PLANE / 2) + sw_dim(16 * e + l16, g), kp);
#pragma unroll
            for (int c = 0; c < QB; c++) acc[c][e] = mfma_parts(kp, sp[c], acc[c][e]);
        }
    };
    using std::integral_constant;
    for (int t = 0; t < w.nkt; t++) {
        const bool more = t + 1 < w.nkt;
        if (more) fetch(t + 1);
        const char* stage = smem + (t & 1) * STAGE;
        const int kb = t * KT;
        const int nsb = w.visible_subblocks(kb);
        if (nsb > 0) {
            if (w.half_unmasked(kb))
                tile(integral_constant<int, 2>{}, std::false_type{}, stage, kb);
            else if (nsb == 2)
                tile(integral_constant<int, 2>{}, std::true_type{}, stage, kb);
            else
                tile(integral_constant<int, 1>{}, std::true_type{}, stage, kb);
        }
        if (more) store(smem + ((t + 1) & 1) * STAGE);
        __syncthreads();
    }

    watch.join(tid);
    // the second key half's partial dQ joins the first's, lane for lane
    float* mrg = reinterpret_cast<float*>(smem) + (w.w2 * 16 * QB) * 64 + lane;
    if (w.kh == 1) {
#pragma unroll
        for (int c = 0; c < QB; c++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int r = 0; r < 4; r++) mrg[(16 * c + 4 * e + r) * 64] = acc[c][e][r];
    }
    __syncthreads();
    // dQ = scale * dS K
    auto results = [&](auto write) {
#pragma unroll
        for (int c = 0; c < QB; c++) {
            const int q = w.q + 16 * c;
            float* drow = p.dq + (((long)w.b * p.Sq + q) * p.H + w.h) * D64;
            floatx4 v[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
#pragma unroll
                for (int r = 0; r < 4; r++) v[e][r] = (acc[c][e][r] + mrg[(16 * c + 4 * e + r) * 64]) * p.scale;
                if (q < p.Sq) {
                    bad = bad || not_finite(v[e]);
                    if constexpr (decltype(write)::value) *reinterpret_cast<floatx4*>(drow + 16 * e + 4 * g) = v[e];
                }
            }
            const bool small = too_small(v, (float)p.Sk, watch.largest(), p.scale);
            bad = bad || (small && q < p.Sq);
        }
    };
    bad = watch.left_over(tid);
    bool again = false;
    if (p.in_place) {
        if (w.kh == 0) results(std::false_type{});
        again = __syncthreads_or(bad);
    }
    if (w.kh == 0 && !again) results(std::true_type{});
    if (!p.in_place) again = __syncthreads_or(bad);
    if (again) {
#pragma unroll 1
        for (int c = 0; c < QB; c++) {
            if ((qtile * QB + c) * 64 < p.Sq)
                attn16_dq<4, QueryTile<4>>(p, reinterpret_cast<float*>(smem), qtile * QB + c, qbh);
            __syncthreads();
        }
    }
}

template <int NG>
dim3 query_grid(const AttnArgs& a) {
    const size_t nT = ft_div_up(a.Sq, 16 * NG);
    return dim3((unsigned)(((nT + 1) / 2) * (size_t)a.B * a.H));
}

// dK and dV of 64 keys, of one query head (split_g) or summed over a kv head's group: a wave owns 16 keys (their K and V
// in registers) against one half of every 64-query tile, whose Q and dO lie in LDS as rows and
// as columns. P and dS leave the score products as second operands of dV^T += dO^T P and dK^T += Q^T dS. Key tile 0
// (under the causal mask the most queries) first.
__global__ __launch_bounds__(512, 2) void attn_split_dkdv_kernel(AttnArgs p) {
    constexpr int NT = 512;
    __shared__ __attribute__((aligned(16))) char smem[12 * PLANE + KT * 8];   // Q rows, dO rows, Q columns, dO columns; stats
    float2* const st = reinterpret_cast<float2*>(smem + 12 * PLANE);           // (Delta, LSE in base 2) of the tile's queries
    const int tid = threadIdx.x, lane = tid % 64, l16 = lane % 16, g = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64), qh = wave / 4;
    const int nhu = p.B * (p.split_g ? p.H : p.Hkv);
    const int kt = (int)blockIdx.x / nhu, bh = (int)blockIdx.x % nhu;
    const int Gfull = p.H / p.Hkv;
    const int b = bh / (p.split_g ? p.H : p.Hkv), hsel = bh % (p.split_g ? p.H : p.Hkv);
    const int kvh = p.split_g ? hsel / Gfull : hsel, g0 = p.split_g ? hsel % Gfull : 0, G = p.split_g ? 1 : Gfull;
    const int kb0 = kt * KT + 16 * (wave % 4);
    const int key = kb0 + l16;
    const int key_m = key < p.Sk ? key : 0x7fffffff;   // a key past the end is visible to nobody
    const long krow = (((long)b * p.Sk + (key < p.Sk ? key : p.Sk - 1)) * p.Hkv + kvh) * D64;
    const float sscale = p.scale * kLog2e;
    uintx4 kp[2][3], vp[2][3];
    unsigned left = 0;
    Row k_row, v_row;
    k_row.fetch(p.k + krow, g);
    k_row.parts(kp, &left);
    v_row.fetch(p.v + krow, g);
    v_row.parts(vp, &left);

    const int nqt = (p.Sq + KT - 1) / KT;
    int qt0 = 0;
    if (p.causal) {
        const int first_q = kt * KT - p.causal_offset;   // the first query that sees the tile's first key
        qt0 = first_q > 0 ? first_q / KT : 0;
    }
    const int per_head = nqt > qt0 ? nqt - qt0 : 0, items = per_head * G;
    TileRows<NT> ql, dl;
    TileColumns<NT> qc, dc;
    float2 stat = make_float2(0.f, 0.f);
    auto fetch = [&](int item) {
        const int h = kvh * Gfull + g0 + item / per_head, t = qt0 + item % per_head;
        const long head = ((long)b * p.Sq * p.H + h) * D64;
        const int stride = p.H * D64;
        ql.fetch(p.q + head, stride, p.Sq, t, tid);
        dl.fetch(p.d_out + head, stride, p.Sq, t, tid);
        qc.fetch(p.q + head, stride, p.Sq, t, tid);
        dc.fetch(p.d_out + head, stride, p.Sq, t, tid);
        if (tid < KT) {
            int q = t * KT + tid;
            q = q < p.Sq ? q : p.Sq - 1;
            stat = *reinterpret_cast<const float2*>(p.stats + 2 * (((long)b * p.H + h) * p.Sq + q));
        }
    };
    __shared__ Watch watch;
    watch.start(tid);
    watch.add(tid, left, 0.0f);
    auto store = [&]() {
        unsigned left = 0;
        ql.store(smem, tid, &left);
        dl.store(smem + 3 * PLANE, tid, &left);
        watch.add(tid, left, ql.largest());
        qc.store(smem + 6 * PLANE, tid);
        dc.store(smem + 9 * PLANE, tid);
        if (tid < KT) st[tid] = make_float2(stat.x, stat.y * kLog2e);
    };
    floatx4 dk[4], dv[4];
#pragma unroll
    for (int e = 0; e < 4; e++) dk[e] = dv[e] = zero4();
    if (items > 0) {
        fetch(0);
        store();
    }
    __syncthreads();
    for (int item = 0; item < items; item++) {
        const bool more = item + 1 < items;
        if (more) fetch(item + 1);
        const int q0 = (qt0 + item % per_head) * KT + 32 * qh;
        // queries of this half that see some key of the wave: all of them, or none of the first ones
        const bool some = !p.causal || q0 + 31 + p.causal_offset >= kb0;
        if (some && q0 < p.Sq) {
            float pr[8], ds[8];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                floatx4 s = zero4(), dp = zero4();
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const int at = sw_key(32 * qh + 16 * u + l16, 4 * t + g);
                    uintx4 qp[3], dop[3];
                    read_parts(smem + at, qp);
                    read_parts(smem + 3 * PLANE + at, dop);
                    s = mfma_parts<true>(qp, kp[t], s);
                    dp = mfma_parts<true>(dop, vp[t], dp);
                }
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    // visible: a real key, a real query, and not above the diagonal (a select: exp2(-inf) = 0)
                    const int qi = q0 + 16 * u + 4 * g + i;
                    const float2 c = st[32 * qh + 16 * u + 4 * g + i];
                    const int lim = qi < p.Sq ? (p.causal ? qi + p.causal_offset : 0x7ffffffe) : -1;
                    const float pij = exp2_fast(key_m <= lim ? scaled_score(s[i], sscale) - c.y : -INFINITY);
                    pr[4 * u + i] = pij;
                    ds[4 * u + i] = pij * (dp[i] - c.x);
                }
            }
            uintx4 pp[3], sp[3];
            split8(pr, pp);
            split8(ds, sp);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int at = 6 * PLANE + qh * (PLANE / 2) + sw_dim(16 * e + l16, g);
                uintx4 qp[3], dop[3];
                read_parts(smem + at, qp);
                read_parts(smem + 3 * PLANE + at, dop);
                // (a tile's sum of its own first: one rounding of the running sum a tile, not six)
                dk[e] += mfma_parts(qp, sp, zero4());
                dv[e] += mfma_parts(dop, pp, zero4());
            }
        }
        __syncthreads();
        if (more) {
            store();
            __syncthreads();
        }
    }

    watch.join(tid);
    // The two query halves of a key block meet through LDS, lane for lane.
    float* mrg = reinterpret_cast<float*>(smem) + (wave % 4) * 32 * 64 + lane;
    if (qh == 1) {
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                mrg[(4 * e + r) * 64] = dk[e][r];
                mrg[(16 + 4 * e + r) * 64] = dv[e][r];
            }
    }
    __syncthreads();
    // register r of accumulator e is head-dim index 16 e + 4 g + r; dK = scale * sum dS Q (here, or where the heads
    // of the group are added)
    bool bad = watch.left_over(tid);
    auto results = [&](auto write) {
        const long n_all = (long)p.B * p.Sk * p.Hkv * D64;
        float* const dk_out = p.split_g ? p.part + 2 * g0 * n_all : p.dk;
        float* const dv_out = p.split_g ? p.part + (2 * g0 + 1) * n_all : p.dv;
        const float scale = p.split_g ? 1.0f : p.scale;
        floatx4 x[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            floatx4 y;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                x[e][r] = (dk[e][r] + mrg[(4 * e + r) * 64]) * scale;
                y[r] = dv[e][r] + mrg[(16 + 4 * e + r) * 64];
            }
            if (key < p.Sk) {
                bad = bad || not_finite(x[e]) || not_finite(y);
                if constexpr (decltype(write)::value) {
                    *reinterpret_cast<floatx4*>(dk_out + krow + 16 * e + 4 * g) = x[e];
                    *reinterpret_cast<floatx4*>(dv_out + krow + 16 * e + 4 * g) = y;
                }
            }
        }
        const bool small = too_small(x, (float)p.Sq * (float)G, watch.largest(), scale);
        bad = bad || (small && key < p.Sk);
    };
    bool again = false;
    if (p.in_place) {
        if (qh == 0) results(std::false_type{});
        again = __syncthreads_or(bad);
    }
    if (qh == 0 && !again) results(std::true_type{});
    if (!p.in_place) again = __syncthreads_or(bad);
    if (again) {
#pragma unroll 1
        for (int c = 0; c < 4; c++) {
            if (kt * KT + 16 * c < p.Sk) attn16_dkdv<64>(p, reinterpret_cast<float*>(smem), (4 * kt + c) * nhu + bh);
            __syncthreads();
        }
    }
}

}  // namespace

int ft_attn_split_forward(ft_context* ctx, const AttnArgs& args, int groups) {
    AttnArgs a = args;
    const size_t rows = (size_t)a.B * a.Sq * a.H * D64 * sizeof(float);
    a.in_place = ft_overlap(a.o, rows, a.q, rows);
    if (groups == 2) hipLaunchKernelGGL(attn_split_fwd_kernel<2>, query_grid<2>(a), dim3(512), 0, ctx->stream, a);
    else hipLaunchKernelGGL(attn_split_fwd_kernel<4>, query_grid<4>(a), dim3(1024), 0, ctx->stream, a);
    FT_LAUNCH_CHECK();
    return FT_OK;
}

int ft_attn_split_dq(ft_context* ctx, const AttnArgs& args) {
    AttnArgs a = args;
    const size_t rows = (size_t)a.B * a.Sq * a.H * D64 * sizeof(float);
    a.in_place = ft_overlap(a.dq, rows, a.out, rows);
    hipLaunchKernelGGL(attn_split_dq_kernel, dim3((unsigned)(ft_div_up(a.Sq, 128) * (size_t)a.B * a.H)), dim3(512), 0, ctx->stream, a);
    FT_LAUNCH_CHECK();
    return FT_OK;
}

int ft_attn_split_dkdv(ft_context* ctx, const AttnArgs& args) {
    AttnArgs a = args;
    const size_t heads = (size_t)a.B * (a.split_g ? a.H : a.Hkv), rows = (size_t)a.B * a.Sk * a.Hkv * D64 * sizeof(float);
    a.in_place = !a.split_g && (ft_overlap(a.dk, rows, a.k, rows) || ft_overlap(a.dk, rows, a.v, rows) ||
                                ft_overlap(a.dv, rows, a.k, rows) || ft_overlap(a.dv, rows, a.v, rows));
    hipLaunchKernelGGL(attn_split_dkdv_kernel, dim3((unsigned)(ft_div_up(a.Sk, 64) * heads)), dim3(512), 0, ctx->stream, a);
    FT_LAUNCH_CHECK();
    return FT_OK;
}
