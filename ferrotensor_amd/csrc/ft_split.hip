// f32 matrix products on the bf16 matrix instructions, without giving up f32 operands: an f32 value from 2^-110 up is the
// exact sum of three bf16 numbers (8 + 8 + 8 significant bits, f32's own exponents, so no scaling and no special rows),
// every f16 weight of two, and a product of two values is the sum of the products of their parts. With an f32 b six of
// the nine are kept, with an f16 b five of the six: what is left out is at most 2^-24 (2^-25) of the product it belongs to,
// as much as f32 may round a sum of that size by. Sums are f32, in the matrix unit, subnormals included.
// v_mfma_f32_32x32x16_bf16 does eight times the products of v_mfma_f32_32x32x2_f32 in half its cycles: 2.7 (3.2) times the
// f32 rate after six (five) of them.
//
// What the split cannot hold makes a wave do its share again with f32 products: infinities and finite values within 2^-8 of
// the largest f32, whose first part would round to infinity, leave a sum that is not finite; a value below 2^-110 (bf16
// ends at 2^-133) leaves something over after its third part, which one v_or3_b32 for two values collects. So infinities
// and NaN come out as f32 products give them, and tiny values count in full. With every wave's share made twice a product
// takes 1.7 to 2.8 times as long (8192 x 2048 x 2048, f16 b: 830 us for 328); looking for it costs 1 to 3 % (f16 b: 1 %).
// The rank-r term and what K leaves after its last whole step of 16 take the f32 instruction too.
//
// Bound: VALU and matrix unit together. 8192 x 2048 x 2048 with f16 b: 329 to 342 us (204 TFLOP/s; f32 products 518), of them
// 286 with no operand fetched at all; 2048 x 2560 x 2048 with f32 b: 129 to 134 us (160 with f32 products). Relative error
// against f64 there 3.1e-7 (8.1e-7) and 3.9e-7 (9.1e-7).
//
// Work split: the waves of a workgroup share one output tile along K (wave w takes K steps w, w + KW, ...), because an
// operand is then split into its parts by one wave only: with the usual 2 x 2 waves over the tile every value would be
// split twice, and the splitting (11 VALU instructions for two values, and one to look after them) is as long as the products
// (64 x 64 x 16: 192 VALU instructions of 4 cycles beside 24 MFMAs of 32). A wave fetches its own operand slabs (global -> registers one
// step ahead -> its own part of LDS -> MFMA operand order), so the K loop has no barrier; the KW sums meet in LDS at the
// end, in wave order. Nothing depends on alignment but the speed of the loads.
#include "ft_common.h"
#include "ft_parts.h"
#include "ft_split.h"

#include <cmath>

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
// 16 bytes from any 4-byte (f32) or 2-byte (f16) boundary
struct __attribute__((packed, aligned(4))) Load16 { uintx4 v; };
struct __attribute__((packed, aligned(2))) Load16h { uintx4 v; };

// Products that share a (q, k and v of one input) form one row of column tiles, as in gemm_async_kernel.
constexpr int kSplitProducts = 3;
struct SplitProduct {
    const char* b;
    float* out;
    const float* add;     // optional [M, N] term (may be `out` itself)
    const float* a2;      // rank-r term: [M, K2] and [K2, N] (b k-major) or [N, K2], or NULL
    const float* b2;
    const float2* rope;   // RoPE on the output, heads of 64 columns: (cos, sin) of [position][32], or NULL
    int rope_seq;         // position = row % rope_seq
    int N, ldb, K2;
    int tile_begin;       // its first column tile
};
struct SplitArgs {
    const char* a;
    int M, K, lda;
    int steps;            // K steps of 16 that may be fetched in whole 16-byte groups
    int tiles_m, tiles_n, panel, xcds, count;
    SplitProduct p[kSplitProducts];
    // EPI = kSplitGateUp: a second b of the same shape; out = a @ b, out2 = a @ b_alt, out3 = silu(out2) * out
    const char* b_alt;
    float* out2;
    float* out3;
};
constexpr int kSplitPlain = 0, kSplitGroup = 1, kSplitGateUp = 2;

// One operand: F blocks of 32 rows (of a; columns of b) by 16 k per step.
//   KM = false: element (row, k) at base[row * ld + k];  KM = true: at base[k * ld + row].
// Tile row of block f, lane l32: KM with two blocks: 2 * l32 + f (one load fetches both), else 32 * f + l32.
// A lane holds k = 8 * half + e, e = 0..7.
template <int F, bool KM, bool HALF>
struct Operand {
    using Value = typename std::conditional<HALF, _Float16, float>::type;
    static constexpr int ROWS = 32 * F;
    static constexpr int ES = HALF ? 2 : 4;
    static constexpr int LOADS = ROWS * 16 * ES / 1024;            // 16-byte loads per lane and step
    static constexpr int PAD = HALF && KM && F == 2 ? 128 : 0;     // behind k = 7: the two halves of a wave read k and k + 8
    static constexpr int BYTES = ROWS * 16 * ES + PAD;
    uintx4 g[LOADS];
    unsigned off[LOADS];   // byte offset from the step's base

    __device__ __forceinline__ static int tile_row(int f, int l32) { return KM && F == 2 ? 2 * l32 + f : 32 * f + l32; }

    __device__ __forceinline__ void set_offsets(int row0, int rows, int ld, int lane) {
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
            if constexpr (!KM) {
                constexpr int LPR = HALF ? 2 : 4;                  // lanes per row
                int row = row0 + (64 / LPR) * i + lane / LPR;
                row = row < rows ? row : rows - 1;                 // values of rows past the end are never stored
                off[i] = ((unsigned)row * (unsigned)ld + (unsigned)((lane % LPR) * (16 / ES))) * ES;
            } else {
                constexpr int LPK = ROWS * ES / 16;                // lanes per k
                int row = row0 + (lane % LPK) * (16 / ES);
                row = row < rows ? row : row0;                     // a group past the end re-reads the tile's first
                off[i] = ((unsigned)((64 / LPK) * i + lane / LPK) * (unsigned)ld + (unsigned)row) * ES;
            }
        }
    }
    __device__ __forceinline__ void fetch(const char* base) {
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
            if constexpr (HALF) g[i] = reinterpret_cast<const Load16h*>(base + off[i])->v;
            else g[i] = reinterpret_cast<const Load16*>(base + off[i])->v;
        }
    }
    __device__ __forceinline__ void stash(char* lds, int lane) const {
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
            int at;
            if constexpr (!KM && !HALF) {       // 64-byte rows, 16-byte chunk c at c ^ (row >> 2 & 3): no bank conflicts
                const int row = 16 * i + lane / 4;
                at = row * 64 + (((lane % 4) ^ ((row >> 2) & 3)) * 16);
            } else if constexpr (!KM) {         // 32-byte rows, chunk c at c ^ (row >> 3 & 1)
                const int row = 32 * i + lane / 2;
                at = row * 32 + (((lane % 2) ^ ((row >> 3) & 1)) * 16);
            } else {
                at = i * 1024 + lane * 16 + (PAD && i > 0 ? PAD : 0);
            }
            *reinterpret_cast<uintx4*>(lds + at) = g[i];
        }
    }
    __device__ __forceinline__ static void frags(const char* lds, int l32, int half, Value (&x)[F][8]) {
        if constexpr (!KM && !HALF) {
#pragma unroll
            for (int f = 0; f < F; f++) {
                const int row = 32 * f + l32;
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    const floatx4 v = *reinterpret_cast<const floatx4*>(lds + row * 64 + (((2 * half + c) ^ ((row >> 2) & 3)) * 16));
#pragma unroll
                    for (int e = 0; e < 4; e++) x[f][4 * c + e] = v[e];
                }
            }
        } else if constexpr (!KM) {
#pragma unroll
            for (int f = 0; f < F; f++) {
                const int row = 32 * f + l32;
                const halfx8 v = *reinterpret_cast<const halfx8*>(lds + row * 32 + ((half ^ ((row >> 3) & 1)) * 16));
#pragma unroll
                for (int e = 0; e < 8; e++) x[f][e] = v[e];
            }
        } else {
            const char* p = lds + half * (8 * ROWS * ES + PAD);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const char* q = p + e * (ROWS * ES);
                if constexpr (F == 2 && !HALF) {
                    const floatx2 v = *reinterpret_cast<const floatx2*>(q + l32 * 8);
                    x[0][e] = v.x;
                    x[F - 1][e] = v.y;
                } else if constexpr (F == 2) {
                    const halfx2 v = *reinterpret_cast<const halfx2*>(q + l32 * 4);
                    x[0][e] = v.x;
                    x[F - 1][e] = v.y;
                } else if constexpr (!HALF) {
                    x[0][e] = *reinterpret_cast<const float*>(q + l32 * 4);
                } else {
                    x[0][e] = *reinterpret_cast<const _Float16*>(q + l32 * 2);
                }
            }
        }
    }
};

// FM x FN blocks of 32 x 32 per wave (and workgroup), KW waves along K. EPI: kSplitGroup takes up to three products and
// rotates heads (64 columns wide); kSplitGateUp multiplies the same 32 columns of two matrices, side by side in the tile.
template <int FM, int FN, int KW, bool A_KM, bool B_KM, bool B_HALF, int EPI = kSplitPlain>
__global__ __launch_bounds__(64 * KW, 2) void gemm_split_kernel(SplitArgs g) {
    constexpr bool DUAL = EPI == kSplitGateUp;
    static_assert(!DUAL || FN == 2, "one block of columns of each matrix");
    constexpr int TM = 32 * FM, TN = 32 * FN;
    using OpA = Operand<FM, A_KM, false>;
    using OpB = Operand<DUAL ? 1 : FN, B_KM, B_HALF>;
    constexpr int NB = DUAL ? 2 : 1;
    constexpr int SLAB = OpA::BYTES + NB * OpB::BYTES;
    constexpr int REGION = SLAB > TM * TN * 4 ? SLAB : TM * TN * 4;   // a wave's slab, later its sums
    __shared__ __attribute__((aligned(16))) char lds[KW * REGION];

    // Tile order as in gemm_async_kernel: XCD x takes the x-th contiguous chunk of a panel order.
    int bid = (int)blockIdx.x;
    if (g.xcds == 8) {
        const int total = (int)gridDim.x, x = bid & 7, q = total >> 3, r = total & 7;
        bid = x * q + (x < r ? x : r) + (bid >> 3);
    }
    const int per_panel = g.tiles_m * g.panel;
    const int last = (g.tiles_n - 1) / g.panel;
    int pnl = bid / per_panel;
    pnl = pnl < last ? pnl : last;
    const int rem = bid - pnl * per_panel;
    const int width = pnl == last ? g.tiles_n - last * g.panel : g.panel;
    int tn = pnl * g.panel + rem % width;
    SplitProduct p = g.p[0];
    if constexpr (EPI == kSplitGroup) {
        if (g.count > 2 && tn >= g.p[2].tile_begin) p = g.p[2];
        else if (g.count > 1 && tn >= g.p[1].tile_begin) p = g.p[1];
        tn -= p.tile_begin;
    }
    const int m0 = (rem / width) * TM, n0 = tn * (DUAL ? 32 : TN);

    const int lane = threadIdx.x % 64, l32 = lane % 32, half = lane / 32;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / 64));
    char* const slab_a = lds + wave * REGION;
    char* const slab_b = slab_a + OpA::BYTES;

    OpA oa;
    OpB ob[NB];
    oa.set_offsets(m0, g.M, g.lda, lane);
#pragma unroll
    for (int t = 0; t < NB; t++) ob[t].set_offsets(n0, p.N, p.ldb, lane);
    const char* const bases[2] = {p.b, g.b_alt};
    const long a_step = A_KM ? 64L * g.lda : 64L;
    const long b_step = (B_KM ? 16L * p.ldb : 16L) * OpB::ES;
    const int steps = g.steps;
    using BT = typename std::conditional<B_HALF, _Float16, float>::type;
    if (wave < steps) {
        oa.fetch(g.a + wave * a_step);
#pragma unroll
        for (int t = 0; t < NB; t++) ob[t].fetch(bases[t] + wave * b_step);
    }

    floatx16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    // Up to 16 k from k0, element by element, on the f32 instruction: what K leaves after its whole steps, and the
    // rank-r term. The second half of a wave takes the odd k; a k past the end reads as zero.
    auto f32_rest = [&](const float* pa, bool a_km, int lda, const auto* pb, const auto* pb1, bool b_km, int ldb, int k0, int k_end) {
        float xa[FM][8], xb[FN][8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int k = k0 + 2 * e + half;
            const bool in = k < k_end;
            const int kc = in ? k : k0;
#pragma unroll
            for (int i = 0; i < FM; i++) {
                int row = m0 + OpA::tile_row(i, l32);
                row = row < g.M ? row : g.M - 1;
                const float v = pa[a_km ? (long)kc * lda + row : (long)row * lda + kc];
                xa[i][e] = in ? v : 0.0f;
            }
#pragma unroll
            for (int j = 0; j < FN; j++) {
                int col = n0 + (DUAL ? l32 : OpB::tile_row(j, l32));
                col = col < p.N ? col : p.N - 1;
                const float v = (float)(DUAL && j == 1 ? pb1 : pb)[b_km ? (long)kc * ldb + col : (long)col * ldb + kc];
                xb[j][e] = in ? v : 0.0f;
            }
        }
#pragma unroll
        for (int e = 0; e < 8; e++) {
            if (k0 + 2 * e >= k_end) break;
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(xa[i][e], xb[j][e], acc[i][j], 0, 0, 0);
        }
    };
    constexpr int PB = B_HALF ? 2 : 3;
    constexpr int PRODUCTS = PB == 3 ? 6 : 5, MFMAS = PRODUCTS * FM * FN;
    constexpr int PAIRS = 4 * (FM + FN);
    struct Parts {
        uintx4 a[FM][3], b[FN][PB];
    };
    // MFMA n of a step: smallest products first, the blocks of a product in turn (no two neighbours on one accumulator).
    auto mfma = [&](const Parts& p, int n) {
        constexpr int U3[6] = {2, 0, 1, 1, 0, 0}, V3[6] = {0, 2, 1, 0, 1, 0};
        constexpr int U2[6] = {2, 1, 1, 0, 0, 0}, V2[6] = {0, 1, 0, 1, 0, 0};
        const int q = n / (FM * FN), i = n / FN % FM, j = n % FN;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, p.a[i][PB == 3 ? U3[q] : U2[q]]),
                                                            __builtin_bit_cast(bf16x8, p.b[j][PB == 3 ? V3[q] : V2[q]]),
                                                            acc[i][j], 0, 0, 0);
    };
    auto stash = [&]() {
        oa.stash(slab_a, lane);
#pragma unroll
        for (int t = 0; t < NB; t++) ob[t].stash(slab_b + t * OpB::BYTES, lane);
    };
    auto frags = [&](typename OpA::Value (&xa)[FM][8], typename OpB::Value (&xb)[FN][8]) {
        OpA::frags(slab_a, l32, half, xa);
        if constexpr (DUAL) {
#pragma unroll
            for (int t = 0; t < NB; t++)
                OpB::frags(slab_b + t * OpB::BYTES, l32, half, *reinterpret_cast<typename OpB::Value(*)[1][8]>(&xb[t]));
        } else {
            OpB::frags(slab_b, l32, half, xb);
        }
    };
    auto fetch = [&](int s) {
        s = s < steps ? s : steps - 1;   // past the end: a step that nobody multiplies
        oa.fetch(g.a + s * a_step);
#pragma unroll
        for (int t = 0; t < NB; t++) ob[t].fetch(bases[t] + s * b_step);
    };
    unsigned left = 0;   // what third parts leave over
    // The slab of this wave's next step, out of LDS and into parts (`next`), beside the products of the current one
    // (`p`). A wave issues a VALU instruction every 8 cycles at best, an MFMA keeps the matrix unit for 32: they are
    // dealt out in turn, a pair of values a slot, its three stages in three slots, so that no stage waits for the one
    // before it.
    auto split = [&](Parts& next, const Parts& p, int after, auto beside) __attribute__((always_inline)) {
        constexpr bool BESIDE = decltype(beside)::value;   // false: nothing to multiply yet
        typename OpA::Value xa[FM][8];
        typename OpB::Value xb[FN][8];
        frags(xa, xb);
        float u[PAIRS], v[PAIRS];
        constexpr int SLOTS = PAIRS + 2;
        constexpr int AHEAD = FM * FN;   // MFMAs over the latency of the LDS reads
        if constexpr (BESIDE) {
#pragma unroll
            for (int n = 0; n < AHEAD; n++) mfma(p, n);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int s = 0; s < SLOTS; s++) {
            if (s == SLOTS / 3) {   // the slab has been read: the one after it, fetched a step ago, takes its place
                stash();
                fetch(after);
            }
#pragma unroll
            for (int ph = 0; ph < 3; ph++) {
                const int t = s - ph;
                if (t < 0 || t >= PAIRS) continue;
                const bool of_a = t < 4 * FM;
                const int blk = (of_a ? t : t - 4 * FM) / 4, e = t % 4;
                if (!of_a && ph >= PB) continue;
                if (ph == 2) collect_left(left, u[t], v[t]);
                if (ph == 0) {
                    u[t] = of_a ? xa[of_a ? blk : 0][2 * e] : (float)xb[of_a ? 0 : blk][2 * e];
                    v[t] = of_a ? xa[of_a ? blk : 0][2 * e + 1] : (float)xb[of_a ? 0 : blk][2 * e + 1];
                }
                const unsigned q = pack2(u[t], v[t]);
                if (of_a) next.a[blk][ph][e] = q;
                else next.b[blk][ph < PB ? ph : 0][e] = q;
                if (ph + 1 < (of_a ? 3 : PB)) {
                    u[t] -= low_half(q);
                    v[t] -= high_half(q);
                }
            }
            if constexpr (BESIDE) {
#pragma unroll
                for (int n = AHEAD + (MFMAS - AHEAD) * s / SLOTS; n < AHEAD + (MFMAS - AHEAD) * (s + 1) / SLOTS; n++) mfma(p, n);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    if (wave < steps) {
        auto finish = [&](const Parts& p) __attribute__((always_inline)) {
#pragma unroll
            for (int n = 0; n < MFMAS; n++) mfma(p, n);
        };
        Parts p0, p1;   // by turns: copying would be two VALU instructions a slot
        stash();
        fetch(wave + KW);
        split(p0, p0, wave + 2 * KW, std::false_type{});
        auto step = [&](int s, Parts& next, const Parts& now) __attribute__((always_inline)) {
            split(next, now, s + 2 * KW, std::true_type{});
            __builtin_amdgcn_sched_barrier(0);
        };
        int s = wave + KW;
#pragma unroll 1
        for (; s + KW < steps; s += 2 * KW) {
            step(s, p1, p0);
            step(s + KW, p0, p1);
        }
        if (s < steps) {
            step(s, p1, p0);
            finish(p1);
        } else {
            finish(p0);
        }
    }
    const float* const af = reinterpret_cast<const float*>(g.a);
    const BT* const b0 = reinterpret_cast<const BT*>(p.b);
    const BT* const b1 = reinterpret_cast<const BT*>(g.b_alt);
    // The waves with the fewest whole steps are the last ones.
    auto rest = [&]() {
        if (!DUAL && p.a2 && wave == KW - 1)
            for (int k = 0; k < p.K2; k += 16)
                f32_rest(p.a2, false, p.K2, p.b2, p.b2, B_KM, B_KM ? p.N : p.K2, k, p.K2);
        if (steps * 16 < g.K && wave == KW - 2)
            for (int k = steps * 16; k < g.K; k += 16) f32_rest(af, A_KM, g.lda, b0, b1, B_KM, p.ldb, k, g.K);
    };
    rest();
    // A sum that is not finite (an operand was not, or one of its parts, or the sum itself overflowed), or a value that its
    // parts do not hold: this wave's share is made again with f32 products.
    float zero = 0.0f;
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) zero = fmaf(acc[i][j][r], 0.0f, zero);
    if (__builtin_expect(__any(zero != 0.0f || left_over(left)), 0)) {
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;
        if (wave < steps) fetch(wave);
#pragma unroll 1
        for (int s = wave; s < steps; s += KW) {
            stash();
            fetch(s + KW);
            typename OpA::Value xa[FM][8];
            typename OpB::Value xb[FN][8];
            frags(xa, xb);
#pragma unroll
            for (int e = 0; e < 8; e++)   // k = e of the first half of a wave, 8 + e of the second
#pragma unroll
                for (int i = 0; i < FM; i++)
#pragma unroll
                    for (int j = 0; j < FN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(xa[i][e], (float)xb[j][e], acc[i][j], 0, 0, 0);
        }
        rest();
    }

    // Every wave's sums into its own region, then the tile in wave order.
    constexpr bool PAIRED = B_KM && FN == 2 && !DUAL;   // a lane holds two neighbouring columns
    auto swz = [](int row) { return TN == 64 && !PAIRED ? (((A_KM && FM == 2 ? row >> 3 : row >> 2) & 1) << 5) : 0; };
    float* const mine = reinterpret_cast<float*>(slab_a);
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int row = OpA::tile_row(i, (r / 4) * 8 + half * 4 + (r % 4));
            if constexpr (PAIRED) {
                *reinterpret_cast<floatx2*>(mine + row * TN + 2 * l32) = floatx2{acc[i][0][r], acc[i][FN - 1][r]};
            } else {
#pragma unroll
                for (int j = 0; j < FN; j++) mine[row * TN + ((32 * j + l32) ^ swz(row))] = acc[i][j][r];
            }
        }
    __syncthreads();
    auto sum4 = [&](int row, int c4) {
        const float* src = reinterpret_cast<const float*>(lds) + row * TN + (c4 ^ swz(row));
        floatx4 v = *reinterpret_cast<const floatx4*>(src);
#pragma unroll
        for (int w = 1; w < KW; w++) v += *reinterpret_cast<const floatx4*>(src + w * (REGION / 4));
        return v;
    };
    auto store4 = [&](float* out, long o, int n, bool vec, floatx4 v) {
        if (vec) {
            *reinterpret_cast<floatx4*>(out + o) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < p.N) out[o + e] = v[e];
        }
    };
    if constexpr (EPI != kSplitPlain) {
        // Two groups of four columns, 32 apart, per thread: the halves of a head, or the up and gate of a column.
        bool both = EPI == kSplitGateUp;
        if constexpr (EPI == kSplitGroup) both = p.rope != nullptr;
        if (both) {
            const bool vec = p.N % 4 == 0 && ((((uintptr_t)p.out) | ((uintptr_t)g.out2) | ((uintptr_t)g.out3)) & 15) == 0;
#pragma unroll 1
            for (int q = threadIdx.x; q < TM * 8; q += 64 * KW) {
                const int row = q / 8, c4 = (q % 8) * 4;
                const floatx4 x = sum4(row, c4), y = sum4(row, c4 + 32);
                const int m = m0 + row, n = n0 + c4;
                if (m >= g.M || n >= p.N) continue;
                const long o = (long)m * p.N + n;
                if constexpr (EPI == kSplitGateUp) {
                    floatx4 act;
#pragma unroll
                    for (int e = 0; e < 4; e++) act[e] = y[e] * (1.0f / (1.0f + __expf(-y[e]))) * x[e];
                    store4(p.out, o, n, vec, x);
                    store4(g.out2, o, n, vec, y);
                    store4(g.out3, o, n, vec, act);
                } else {
                    // whole heads (the host checks): x holds columns i, y columns i + 32
                    const float2* cs = p.rope + (long)(m % p.rope_seq) * 32 + c4;
                    floatx4 lo, hi;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        lo[e] = x[e] * cs[e].x - y[e] * cs[e].y;
                        hi[e] = x[e] * cs[e].y + y[e] * cs[e].x;
                    }
                    store4(p.out, o, n, vec, lo);
                    store4(p.out, o + 32, n + 32, vec, hi);
                }
            }
            return;
        }
    }
    const bool vec = p.N % 4 == 0 && ((((uintptr_t)p.out) | ((uintptr_t)p.add)) & 15) == 0;   // uniform
#pragma unroll 1
    for (int q = threadIdx.x; q < TM * TN / 4; q += 64 * KW) {
        const int row = q / (TN / 4), c4 = (q % (TN / 4)) * 4;
        floatx4 v = sum4(row, c4);
        const int m = m0 + row, n = n0 + c4;
        if (m >= g.M || n >= p.N) continue;
        const long o = (long)m * p.N + n;
        if (p.add) {
            if (vec) {
                v += *reinterpret_cast<const floatx4*>(p.add + o);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < p.N) v[e] += p.add[o + e];
            }
        }
        store4(p.out, o, n, vec, v);
    }
}

template <int FM, int FN, int KW>
void launch(ft_context* ctx, const SplitArgs& g, int layout, bool half_b) {
    const dim3 grid((unsigned)(g.tiles_m * g.tiles_n)), block(64 * KW);
    if (layout == 0 && half_b)
        hipLaunchKernelGGL((gemm_split_kernel<FM, FN, KW, false, true, true>), grid, block, 0, ctx->stream, g);
    else if (layout == 0)
        hipLaunchKernelGGL((gemm_split_kernel<FM, FN, KW, false, true, false>), grid, block, 0, ctx->stream, g);
    else if (layout == 1 && half_b)
        hipLaunchKernelGGL((gemm_split_kernel<FM, FN, KW, false, false, true>), grid, block, 0, ctx->stream, g);
    else if (layout == 1)
        hipLaunchKernelGGL((gemm_split_kernel<FM, FN, KW, false, false, false>), grid, block, 0, ctx->stream, g);
    else
        hipLaunchKernelGGL((gemm_split_kernel<FM, FN, KW, true, true, false>), grid, block, 0, ctx->stream, g);
}

// Groups and gate + up: a[M, K] @ b[K, N].
template <int FM, int KW, int EPI>
void launch_fused(ft_context* ctx, const SplitArgs& g, bool half_b) {
    const dim3 grid((unsigned)(g.tiles_m * g.tiles_n)), block(64 * KW);
    if (half_b)
        hipLaunchKernelGGL((gemm_split_kernel<FM, 2, KW, false, true, true, EPI>), grid, block, 0, ctx->stream, g);
    else
        hipLaunchKernelGGL((gemm_split_kernel<FM, 2, KW, false, true, false, EPI>), grid, block, 0, ctx->stream, g);
}

// What the products of a launch share. `whole`: see SplitArgs::steps.
SplitArgs split_args(ft_context* ctx, const float* a, size_t M, size_t K, size_t lda, bool whole) {
    SplitArgs g{};
    g.a = reinterpret_cast<const char*>(a);
    g.M = (int)M;
    g.K = (int)K;
    g.lda = (int)lda;
    // A 16-byte group that runs past its row's end reads the next row's start: not in the last step of a matrix whose
    // rows are not whole groups (its last row has no next one).
    g.steps = (int)((whole ? K : K - 1) / 16);
    g.xcds = ctx->num_cus % 8 == 0 && ctx->num_cus >= 64 ? 8 : 1;
    g.count = 1;
    return g;
}

void set_tiles(SplitArgs& g, int tm, int tiles_n) {
    g.tiles_m = (g.M + tm - 1) / tm;
    g.tiles_n = tiles_n;
    int panels = (int)((double)tiles_n / 10.0 + 0.5);
    if (panels < 1) panels = 1;
    g.panel = (tiles_n + panels - 1) / panels;
}

// Groups and gate + up, tiles 64 columns wide (32 of each matrix): as the plain products, half as high where whole
// tiles leave half of the CUs idle. 96 x 960: q/k/v of 960 + 320 + 320 columns 22 -> 10.5 us, gate + up + SiLU-gate of
// 2560 37 -> 16.6 (f32 products before).
template <int EPI>
int launch_group(ft_context* ctx, SplitArgs& g, int tiles_n, bool half_b) {
    const size_t cus = (size_t)ctx->num_cus, tiles64 = (size_t)((g.M + 63) / 64) * tiles_n;
    set_tiles(g, tiles64 * 2 > cus ? 64 : 32, tiles_n);
    if (tiles64 > cus) launch_fused<2, 4, EPI>(ctx, g, half_b);
    else if (tiles64 * 2 > cus) launch_fused<2, 8, EPI>(ctx, g, half_b);
    else launch_fused<1, 8, EPI>(ctx, g, half_b);
    FT_LAUNCH_CHECK();
    return FT_OK;
}

}  // namespace

bool ft_split_gemm_ok(int layout, size_t M, size_t K, size_t N, bool half_b) {
    if (M < 4 || N < 8 || K < 32) return false;   // whole 16-byte groups in a row of either operand
    // Per-lane operand offsets are 32-bit byte offsets from a uniform base.
    const double es = half_b ? 2.0 : 4.0, lim = 4294967296.0;
    const double a_span = 4.0 * (layout == 2 ? 17.0 * (double)M : ((double)M + 1) * (double)K);
    const double b_span = es * (layout == 1 ? ((double)N + 1) * (double)K : 17.0 * (double)N);
    return a_span < lim && b_span < lim;
}

int ft_split_gemm(ft_context* ctx, int layout, bool half_b, const float* a, const void* b, float* out, size_t M,
                  size_t K, size_t N, const float* a2, const float* b2, size_t K2, const float* add) {
    const bool whole = (layout != 2 || M % 4 == 0) && (layout == 1 || N % (half_b ? 8 : 4) == 0);
    SplitArgs g = split_args(ctx, a, M, K, layout == 2 ? M : K, whole);
    g.p[0] = SplitProduct{static_cast<const char*>(b), out, add, K2 > 0 ? a2 : nullptr, K2 > 0 ? b2 : nullptr, nullptr, 1,
                          (int)N, layout == 1 ? (int)K : (int)N, (int)K2, 0};
    const size_t cus = (size_t)ctx->num_cus;
    // Tile and waves, measured on 256 CUs (us, f16 b unless said; 64 x 64 by 4 / by 8 waves, 32 x 64 by 4, 32 x 32 by 8;
    // without the look for small values, which adds 1 % with an f16 b and 3 % with an f32 one):
    //   2048 x 960 x 960  (M x K x N, 480 tiles of 64 x 64)   24.5 / 29.1 / 27.4 / 36.1   with f32 products 35.2
    //   700 x 1024 x 1024 (176)                               15.0 / 13.6 / 15.2 / 16.0                     27.3
    //   257 x 733 x 1001  (80, f32 b)                         13.9 / 13.3 / 10.1 / 10.7                     45.5
    //   96 x 960 x 960    (30)                                13.2 / 12.4 /  9.9 /  6.9                     11.2
    // Above one tile a CU two workgroups of four waves share a CU; up to there eight waves hide a tile's latencies; with
    // half the CUs idle smaller tiles reach more of them. With under 8 K steps (8192 x 64 x 5120) two waves: 72 (four
    // 108, f32 products 76).
    const size_t tiles64 = ((M + 63) / 64) * ((N + 63) / 64), tiles32 = ((M + 31) / 32) * ((N + 31) / 32);
    const int tm = tiles64 * 2 > cus ? 64 : 32, tn = tm == 64 || tiles32 > cus ? 64 : 32;
    set_tiles(g, tm, (int)((N + tn - 1) / tn));
    char name[64];
    snprintf(name, sizeof(name), "gemm_split_kernel<%d, %d, %d, %s>", tm, tn, layout, half_b ? "true" : "false");
    ft_prof_scope prof(ctx, name, 2.0 * M * (double)N * ((double)K + (double)(g.p[0].a2 ? K2 : 0)),
                       4.0 * M * (double)K + (half_b ? 2.0 : 4.0) * N * (double)K + 4.0 * M * (double)N);
    if (tm == 64 && tiles64 > cus && g.steps < 8) launch<2, 2, 2>(ctx, g, layout, half_b);
    else if (tm == 64 && tiles64 > cus) launch<2, 2, 4>(ctx, g, layout, half_b);
    else if (tm == 64) launch<2, 2, 8>(ctx, g, layout, half_b);
    else if (tn == 64) launch<1, 2, 4>(ctx, g, layout, half_b);
    else launch<1, 1, 8>(ctx, g, layout, half_b);
    FT_LAUNCH_CHECK();
    return FT_OK;
}

int ft_split_group(ft_context* ctx, const float* x, const ft_lora_linear_desc* d, size_t count, size_t M, size_t K,
                   bool half_b) {
    bool whole = true;
    for (size_t i = 0; i < count; i++) whole = whole && d[i].N % (half_b ? 8 : 4) == 0;
    SplitArgs g = split_args(ctx, x, M, K, K, whole);
    g.count = (int)count;
    int tiles = 0;
    double flops = 0.0, bytes = 4.0 * M * (double)K;
    for (size_t i = 0; i < count; i++) {
        const bool ranked = d[i].r > 0;
        g.p[i] = SplitProduct{static_cast<const char*>(d[i].w), d[i].y, d[i].residual, ranked ? d[i].t : nullptr,
                              ranked ? d[i].b : nullptr, reinterpret_cast<const float2*>(d[i].rope_table), (int)d[i].rope_seq,
                              (int)d[i].N, (int)d[i].N, (int)d[i].r, tiles};
        tiles += (int)((d[i].N + 63) / 64);
        flops += 2.0 * M * (double)d[i].N * (double)(K + d[i].r);
        bytes += (half_b ? 2.0 : 4.0) * d[i].N * (double)K + 4.0 * M * (double)d[i].N;
    }
    ft_prof_scope prof(ctx, "gemm_split_kernel<group>", flops, bytes);
    return launch_group<kSplitGroup>(ctx, g, tiles, half_b);
}

int ft_split_gate_up(ft_context* ctx, const float* x, const void* w_gate, const void* w_up, float* gate, float* up,
                     float* act, size_t M, size_t K, size_t N, bool half_b) {
    SplitArgs g = split_args(ctx, x, M, K, K, N % (half_b ? 8 : 4) == 0);
    g.p[0] = SplitProduct{static_cast<const char*>(w_up), up, nullptr, nullptr, nullptr, nullptr, 1, (int)N, (int)N, 0, 0};
    g.b_alt = static_cast<const char*>(w_gate);
    g.out2 = gate;
    g.out3 = act;
    ft_prof_scope prof(ctx, "gemm_split_kernel<gate_up>", 4.0 * M * (double)N * (double)K,
                       4.0 * M * (double)K + (half_b ? 4.0 : 8.0) * N * (double)K + 12.0 * M * (double)N);
    return launch_group<kSplitGateUp>(ctx, g, (int)((N + 31) / 32), half_b);
}
