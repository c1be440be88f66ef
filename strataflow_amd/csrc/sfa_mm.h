// sfa_mm.h - products of several tokens with one weight matrix on the matrix
// cores: y[t][o] = sum_k W[o][k] * x[t][k] (ggml_mul_mat, engine.cpp:1883-1885,
// 1905-1906; ggml_mul_mat_id per expert, :1964-1984), for the dense products,
// the Q/K/V product with RoPE and the append, and the experts.
//
// Two kernels share one description of the work (MmArgs) and one epilogue
// (mm_emit):
//   mm_skinny_kernel  tiles of 16 (F32 weights: or 32) tokens, where those are
//                     few: bound by the read of the weights and its latency
//   mm_tile_kernel    more tokens: 128-byte k slices of W and x through LDS
// Both take the MFMA A operand from W (rows = outputs) and B from x (columns =
// tokens), so a lane's accumulator holds four consecutive outputs of one
// token.  Operands are those of the one-token kernels: F16 weights take the
// activation rounded to f16 (RNE) and sum the products in f32, F32 weights
// multiply and sum in f32; only the order of the sums differs, so a token's
// bits depend on how many it is multiplied with.
#pragma once
#include "sfa_append.h"

namespace sfa {

typedef _Float16 half4_a2 __attribute__((ext_vector_type(4), aligned(2)));  // cache rows: any half address

// What becomes of the products.
enum MmOut : int {
    kMmDense,   // y (+ residual)
    kMmQkv,     // RoPE, Q out, K and V into the cache
    kMmGateUp,  // silu(gate) * up of the routed tokens, stored as f16
    kMmDown,    // one f32 row per (token, slot)
};

// Experts: the (token, slot) pairs grouped by expert, written by
// moe_plan_kernel.  Tile T belongs to expert tile_e[T]; an expert's tiles are
// first .. first + n - 1 and split its `count` pairs from order[start].
struct MmExpert {
    int start, count, first, n;
};
struct MmPlan {
    int n_tiles;
    int pad[3];
    // then MmExpert[n_expert], int tile_e[max_tiles], int order[n_pairs]
};

struct MmBase {
    const void *w;   // [n_out][n_in], or the expert stack
    const void *w2;  // kMmGateUp: the up stack
    const void *x;   // rows of n_in
    int n_rows, n_in, n_out;
};
template <int OUT>
struct MmArgs;
template <>
struct MmArgs<kMmDense> : MmBase {
    const float *residual;
    float *y;
};
template <>
struct MmArgs<kMmQkv> : MmBase {
    float *q;
    int n_q;
    float theta_scale;
    AppendParams ap;  // k / v unused
    int kv_type;
};
struct MmExpertArgs : MmBase {
    const MmPlan *plan;
    int n_expert, max_tiles, n_used;
    void *y;  // kMmGateUp: halves [pair][n_out]; kMmDown: floats [pair][n_out]
};
template <>
struct MmArgs<kMmGateUp> : MmExpertArgs {};
template <>
struct MmArgs<kMmDown> : MmExpertArgs {};

template <int OUT>
inline constexpr bool kMmExperts = OUT == kMmGateUp || OUT == kMmDown;

__device__ inline const MmExpert *mm_experts(const MmPlan *pl) { return reinterpret_cast<const MmExpert *>(pl + 1); }
__device__ inline const int *mm_tile_e(const MmPlan *pl, int n_expert) {
    return reinterpret_cast<const int *>(mm_experts(pl) + n_expert);
}
__device__ inline const int *mm_order(const MmPlan *pl, int n_expert, int max_tiles) {
    return mm_tile_e(pl, n_expert) + max_tiles;
}

// Outputs o .. o + 3 of one token (dense, Q/K/V) or pair (experts); v2 is the
// up product beside a gate product.
template <int OUT>
__device__ inline void mm_emit(const MmArgs<OUT> &p, int t, int o, floatx4 v, floatx4 v2) {
    if constexpr (OUT == kMmDense) {
        const int64_t i = (int64_t)t * p.n_out + o;
        if (p.residual != nullptr) {
            const floatx4 r = *reinterpret_cast<const floatx4_a4 *>(p.residual + i);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = __fadd_rn(v[j], r[j]);
        }
        *reinterpret_cast<floatx4_a4 *>(p.y + i) = v;
    } else if constexpr (OUT == kMmGateUp) {
        half4 h;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            // ggml_silu_f32(x) = x / (1 + expf(-x)), times up (swiglu_split)
            const float s = __fdiv_rn(v[j], __fadd_rn(1.0f, expf(-v[j])));
            h[j] = (_Float16)__fmul_rn(s, v2[j]);
        }
        *reinterpret_cast<half4 *>(static_cast<_Float16 *>(p.y) + (int64_t)t * p.n_out + o) = h;
    } else if constexpr (OUT == kMmDown) {
        *reinterpret_cast<floatx4 *>(static_cast<float *>(p.y) + (int64_t)t * p.n_out + o) = v;
    } else {
        // rows [0, n_q) are Q, then n_kv K rows, then n_kv V rows; four
        // consecutive rows (two RoPE pairs) lie in one head
        const int hd = p.ap.head_dim, n_kv = p.ap.n_head_kv * hd;
        const bool is_q = o < p.n_q, is_k = !is_q && o < p.n_q + n_kv;
        const int r = is_q ? o : o - p.n_q - (is_k ? 0 : n_kv);
        const int ps = p.ap.pos[t];
        const bool valid = ps >= 0 && p.ap.seq[t] >= 0;
        if (valid && (is_q || is_k)) {
            const int i = (r % hd) / 2;
            float theta = (float)ps, c, s;
            for (int j = 0; j < i; ++j) theta *= p.theta_scale;
            sincosf(theta, &s, &c);
            float a0 = v[0], a1 = v[1];
            rope_rotate(a0, a1, c, s);
            theta *= p.theta_scale;
            sincosf(theta, &s, &c);
            float b0 = v[2], b1 = v[3];
            rope_rotate(b0, b1, c, s);
            v = floatx4{a0, a1, b0, b1};
        }
        if (is_q) {
            *reinterpret_cast<floatx4_a4 *>(p.q + (int64_t)t * p.n_q + o) = v;
            return;
        }
        uint8_t *dst = row_ptr(p.ap, is_k ? 0 : 1, t, r / hd);
        if (dst == nullptr) return;
        if (p.kv_type == SFA_KV_F16) {
            half4_a2 h;
#pragma unroll
            for (int j = 0; j < 4; ++j) h[j] = (_Float16)v[j];
            *reinterpret_cast<half4_a2 *>(dst + 2 * (r % hd)) = h;
        } else {
            *reinterpret_cast<floatx4_a4 *>(dst + 4 * (r % hd)) = v;
        }
    }
}

// x row of column `col` of a tile that starts at `start`, and the index
// mm_emit takes.
template <int OUT>
__device__ inline int mm_index(const MmArgs<OUT> &p, int start, int col) {
    if constexpr (kMmExperts<OUT>)
        return mm_order(p.plan, p.n_expert, p.max_tiles)[start + col];
    else
        return start + col;
}
template <int OUT>
__device__ inline int mm_x_row(const MmArgs<OUT> &p, int index) {
    if constexpr (OUT == kMmGateUp)
        return index / p.n_used;
    else
        return index;
}

__device__ inline half8 mm_half8(const floatx4 a, const floatx4 b) {
    half8 h;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        h[j] = (_Float16)a[j];
        h[4 + j] = (_Float16)b[j];
    }
    return h;
}

// Sums.  A product over thousands of k as one chain of matrix-core additions is
// off by three to seven times what the one-token kernels' 64 short lane sums
// are (k = 4096: 2.9e-7 against 0.9e-7 in f16, 8.1e-7 against 1.2e-7 in f32), so
// both kernels keep short chains.  mm_skinny_kernel adds a 256-byte block's four
// chains pairwise and the blocks of a wave with Kahan's compensated sum
// (mm_kahan); mm_tile_kernel, where that costs 30 % of the time, adds in three
// plain levels of at most kMmChain matrix-core or vector additions.
// F32 rows of kMmShortF32 values or fewer (SHORT) need shorter chains than
// that: the one-token kernels' chains of eight products meet in a tree.  There
// a chain is four products and the chains meet in pairs.  Error against 64 bits
// at 256 / 512 / 1024 values, in units of 1e-7: one token 0.81 / 0.86 / 0.99, few
// tokens 0.92 / 0.96 / 0.99 without this and 0.78 / 0.83 / 0.87 with it, 32 x 32
// tiles 0.87 / 0.91 / 0.96 and 0.79 / 0.84 / 0.89, 64 x 64 tiles 0.87 / 0.91 / 0.96
// and 0.79 / 0.85 / 0.93.  Longer rows do without: the additions cost 3-16 % of
// the time (4096 x 4096: 3 tokens 17.2 -> 18.2 us, 64 tokens 34.7 -> 40.2).
constexpr int kMmChain = 8;
constexpr int kMmShortF32 = 1024;

// One step of the compensated sum: `sum` takes `v`, `comp` keeps what the
// addition rounded away.  An infinite or NaN sum has no correction: its
// (t - sum) - y would make NaN of an infinite sum at the next step.
template <typename V>
__device__ inline void mm_kahan(V &sum, V &comp, const V &v) {
    const V y = v - comp, t = sum + y, c = (t - sum) - y;
#pragma unroll
    for (int j = 0; j < (int)(sizeof(V) / sizeof(float)); ++j) comp[j] = __builtin_isfinite(t[j]) ? c[j] : 0.0f;
    sum = t;
}

template <int N>
struct MmInt {  // a compile-time int passed to a generic lambda
    static constexpr int value = N;
};

// ---- few tokens ------------------------------------------------------------

// One workgroup per 16 output rows (of each matrix) and tile of 16 NB tokens;
// its eight waves take every eighth 256-byte block of the rows each and their
// partial sums meet in LDS, pair by pair.  The operands go straight from
// memory to registers in MFMA order (lane = row l % 16, 16-byte piece l / 16
// of each 64 bytes): the weights are read once per tile and a block's loads
// are issued before any is used.  n_in * sizeof(WT) is a multiple of
// 256.  Grid (row blocks, tiles).
template <typename WT, typename XT, bool SHORT, int OUT, int NB>
__global__ __launch_bounds__(512) void mm_skinny_kernel(MmArgs<OUT> p) {
    constexpr int NM = OUT == kMmGateUp ? 2 : 1;
    constexpr bool F16W = sizeof(WT) == 2;
    constexpr bool CVT = F16W && sizeof(XT) == 4;
    constexpr int XM = CVT ? 2 : 1;  // 16-byte loads of x per 16 bytes of weights
    __shared__ floatx4 red[8][NM * NB][64];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int r = lane & 15, kq = lane >> 4;
    const int o0 = (int)blockIdx.x * 16;

    int start = (int)blockIdx.y * 16 * NB, count = p.n_rows - start;
    int64_t mat = 0;
    if constexpr (kMmExperts<OUT>) {
        const int T = blockIdx.y;
        if (T >= p.plan->n_tiles) return;
        const int e = mm_tile_e(p.plan, p.n_expert)[T];
        const MmExpert ex = mm_experts(p.plan)[e];
        const int off = (T - ex.first) * 16 * NB;
        start = ex.start + off;
        count = ex.count - off;
        mat = (int64_t)e * p.n_out;
    }
    count = min(count, 16 * NB);

    const int64_t wb = (int64_t)p.n_in * sizeof(WT), xb = (int64_t)p.n_in * sizeof(XT);
    const int row = min(o0 + r, p.n_out - 1);
    const uint8_t *wr[NM];
    wr[0] = static_cast<const uint8_t *>(p.w) + (mat + row) * wb + 16 * kq;
    if constexpr (NM == 2) wr[1] = static_cast<const uint8_t *>(p.w2) + (mat + row) * wb + 16 * kq;
    const uint8_t *xr[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int col = min(16 * b + r, count - 1);
        xr[b] = static_cast<const uint8_t *>(p.x) + mm_x_row(p, mm_index(p, start, col)) * xb + 16 * XM * kq;
    }

    const floatx4 zero = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    floatx4 sum[NM][NB], comp[NM][NB];
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int b = 0; b < NB; ++b) sum[m][b] = comp[m][b] = zero;

    const int n_blk = (int)(wb / 256);
    for (int blk = wave; blk < n_blk; blk += 8) {
        intx4 wv[NM][4], xv[NB][4][XM];
        const int64_t off = (int64_t)blk * 256;
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int s = 0; s < 4; ++s) wv[m][s] = *reinterpret_cast<const intx4 *>(wr[m] + off + 64 * s);
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int h = 0; h < XM; ++h)
                    xv[b][s][h] = *reinterpret_cast<const intx4 *>(xr[b] + XM * (off + 64 * s) + 16 * h);
        floatx4 acc[4][NM][NB];  // a chain for each 64 bytes (SHORT: the sum of its four)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
#pragma unroll
                for (int m = 0; m < NM; ++m) acc[s][m][b] = zero;
                if constexpr (F16W) {
                    half8 xh;
                    if constexpr (CVT)
                        xh = mm_half8(__builtin_bit_cast(floatx4, xv[b][s][0]),
                                      __builtin_bit_cast(floatx4, xv[b][s][XM - 1]));
                    else
                        xh = __builtin_bit_cast(half8, xv[b][s][0]);
#pragma unroll
                    for (int m = 0; m < NM; ++m)
                        acc[s][m][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, wv[m][s]), xh,
                                                                              acc[s][m][b], 0, 0, 0);
                } else {
                    const floatx4 xf = __builtin_bit_cast(floatx4, xv[b][s][0]);
#pragma unroll
                    for (int m = 0; m < NM; ++m) {
                        const floatx4 wf = __builtin_bit_cast(floatx4, wv[m][s]);
                        [[maybe_unused]] floatx4 c[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            if constexpr (SHORT)
                                c[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[j], xf[j], zero, 0, 0, 0);
                            else
                                acc[s][m][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[j], xf[j], acc[s][m][b], 0, 0, 0);
                        }
                        if constexpr (SHORT) acc[s][m][b] = (c[0] + c[1]) + (c[2] + c[3]);
                    }
                }
            }
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int b = 0; b < NB; ++b)
                mm_kahan(sum[m][b], comp[m][b], (acc[0][m][b] + acc[1][m][b]) + (acc[2][m][b] + acc[3][m][b]));
    }

#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int b = 0; b < NB; ++b) red[wave][m * NB + b][lane] = sum[m][b];
    __syncthreads();
    for (int i = threadIdx.x; i < NB * 64; i += 512) {
        const int b = i >> 6, l = i & 63;
        const int col = 16 * b + (l & 15), o = o0 + 4 * (l >> 4);
        if (col >= count || o >= p.n_out) continue;
        floatx4 v[2];
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            floatx4 a[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) a[w] = red[2 * w][m * NB + b][l] + red[2 * w + 1][m * NB + b][l];
            v[m] = (a[0] + a[1]) + (a[2] + a[3]);
        }
        mm_emit<OUT>(p, mm_index(p, start, col), o, v[0], v[NM - 1]);
    }
}

// ---- more tokens ------------------------------------------------------------------

// One 16-byte chunk per lane from global memory straight into LDS: the
// instruction fills the 1 KB at lds_addr (wave-uniform), lane l its chunk l,
// from byte voff (per lane) of base (wave-uniform).  Issued from asm so that
// the compiler's LDS reads of other stages do not wait for it; the kernel
// waits in mm_sync, whose barrier publishes the stage.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // "m0 is reserved": intended, as above
__device__ inline void mm_dma16(const uint8_t *base, uint32_t voff, uint32_t lds_addr) {
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, %2"
        :
        : "s"(lds_addr), "v"(voff), "s"(base)
        : "memory", "m0");
}
#pragma clang diagnostic pop
// Waits until at most N of this wave's loads are in flight and its LDS reads
// are done, then for the workgroup: one asm block, so no LDS access moves
// between the two.
template <int N>
__device__ inline void mm_sync() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}

// LDS of a tile workgroup, and the waves per SIMD that its registers leave room
// for: as many workgroups of nw waves as the LDS of a CU holds, up to two.
template <typename WT, typename XT>
constexpr int mm_lds_bytes(int bm, int bn, int ks, int g, int s) {
    const int ring = (bm * 128 + bn * (sizeof(WT) == 2 && sizeof(XT) == 4 ? 256 : 128)) * g * s, tile = ks * bm * bn * 4;
    return ring > tile ? ring : tile;
}
constexpr int mm_min_waves(int nw, int lds_bytes) {
    const int wgs = lds_bytes <= 80 * 1024 ? 2 : 1;
    return nw * wgs >= 4 ? nw * wgs / 4 : 1;
}

// One workgroup per BM weight rows x BN tokens (gate/up: BM / 2 rows of each).
// A stage is G slices of 128 bytes of every weight row (64 f16 or 32 f32 k)
// and the same k of every token in LDS, S stages in a ring, loaded straight
// from memory S - 1 ahead: a weight slice comes from HBM, so one stage ahead would wait
// out its latency every time.  f32 activations beside F16 weights are staged
// as they are and rounded as they are read.  16-byte chunk c of a staged row
// sits at chunk c ^ key(row), key = row / 2 (128-byte rows) or row (256-byte
// rows): the 16 rows that a slice of an operand read touches cover all banks.
// The waves form KS groups of WR x WC over the tile; a group takes 4 / KS of
// a slice's four k steps, so that a wave keeps a tile large enough to feed
// each operand to several products while the workgroup stays small; the
// groups' products meet in LDS, from where the epilogue stores whole rows.
// The stage loop is unrolled over the ring, so that slots and chains are fixed
// and a step's operands are read from LDS while the step before it multiplies:
// read and used step by step, every product waited out an LDS read (experts of
// 512 tokens: waves waiting on counters 58 -> 42 % of their cycles, call 863 ->
// 765 us; 4096 x 4096, 64 tokens, 32 x 32 tiles 22 -> 17 us).
// 1-D grid: the token tiles of one row block follow each other on one XCD
// (XCD = L % 8), which reads its weight rows from HBM once.
template <typename WT, typename XT, bool SHORT, int BM, int BN, int WR, int WC, int KS, int G, int S, int OUT>
__global__ __launch_bounds__(64 * WR * WC * KS, mm_min_waves(WR * WC * KS, mm_lds_bytes<WT, XT>(BM, BN, KS, G, S)))
void mm_tile_kernel(MmArgs<OUT> p) {
    constexpr bool F16W = sizeof(WT) == 2;
    constexpr bool CVT = F16W && sizeof(XT) == 4;
    constexpr int NW = WR * WC * KS;                      // waves
    constexpr int XR = CVT ? 256 : 128;                   // staged bytes per token
    constexpr int FR = BM / 32 / WR, FC = BN / 32 / WC;   // 32-row, 32-column blocks per wave
    constexpr int KBW = BM / 8, KBX = BN * XR / 1024;     // KB of weights and of x a slice
    constexpr int IW = (KBW + NW - 1) / NW, IX = (KBX + NW - 1) / NW;  // loads per wave and slice
    constexpr int STAGE = BM * 128 + BN * XR;
    constexpr int NM = OUT == kMmGateUp ? 2 : 1;
    constexpr int BMO = BM / NM;                          // outputs per workgroup
    static_assert(BM % (32 * WR) == 0 && BN % (32 * WC) == 0 && 4 % KS == 0, "tile split over the waves");
    constexpr int LDS = mm_lds_bytes<WT, XT>(BM, BN, KS, G, S);
    static_assert(LDS <= 160 * 1024, "LDS of a CU");
    __shared__ __attribute__((aligned(16))) uint8_t lds[LDS];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 31, hh = lane >> 5;

    const int n_rb = (p.n_out + BMO - 1) / BMO, n_rb8 = (n_rb + 7) & ~7;
    int rb, start, count;
    int64_t mat = 0;
    if constexpr (kMmExperts<OUT>) {
        // expert by expert, so that its tokens' rows stay in L2
        const int T = (int)blockIdx.x / n_rb8;
        if (T >= p.plan->n_tiles) return;
        const int e = mm_tile_e(p.plan, p.n_expert)[T];
        const MmExpert ex = mm_experts(p.plan)[e];
        const int rem = (int)blockIdx.x - ex.first * n_rb8, grp = rem / (8 * ex.n), in = rem % (8 * ex.n);
        rb = 8 * grp + in % 8;
        const int step = (ex.count + ex.n - 1) / ex.n;  // even tiles (<= BN: n = ceil(count / BN))
        const int off = (in / 8) * step;
        start = ex.start + off;
        count = min(step, ex.count - off);
        mat = (int64_t)e * p.n_out;
        if (count <= 0) return;
    } else {
        const int nt = (p.n_rows + BN - 1) / BN, grp = (int)blockIdx.x / (8 * nt), in = (int)blockIdx.x % (8 * nt);
        rb = 8 * grp + in % 8;
        start = (in / 8) * BN;
        count = min(BN, p.n_rows - start);
    }
    if (rb >= n_rb) return;
    const int o0 = rb * BMO;

    // this wave's loads: byte offsets of the lane's chunk from the matrix's
    // first row of the tile (weights) and from x
    const int64_t wb = (int64_t)p.n_in * sizeof(WT), xb = (int64_t)p.n_in * sizeof(XT);
    const uint8_t *xbase = static_cast<const uint8_t *>(p.x);
    const uint8_t *wbase[IW];
    uint32_t w_off[IW], x_off[IX], w_lds[IW], x_lds[IX];
    // 1 KB block IW * wave + i of the slice's weights, IX * wave + i of its x
    // (blocks past the last repeat it: the same bytes to the same place)
#pragma unroll
    for (int i = 0; i < IW; ++i) {
        const int b = min(IW * wave + i, KBW - 1);
        const int lr = b * 8 + lane / 8;                      // staged row
        const int gr = min(o0 + lr % BMO, p.n_out - 1) - o0;  // its row of the matrix
        wbase[i] = static_cast<const uint8_t *>(NM == 2 && b >= KBW / 2 ? p.w2 : p.w) + (mat + o0) * wb;
        w_off[i] = (uint32_t)(gr * wb) + 16 * ((lane % 8) ^ ((lr / 2) % 8));
        w_lds[i] = 1024 * b;
    }
#pragma unroll
    for (int i = 0; i < IX; ++i) {
        constexpr int CPR = XR / 16;
        const int b = min(IX * wave + i, KBX - 1);
        const int lr = b * (64 / CPR) + lane / CPR;
        const int key = CVT ? lr % 16 : (lr / 2) % 8;
        const int xrow = mm_x_row(p, mm_index(p, start, min(lr, count - 1)));
        x_off[i] = (uint32_t)(xrow * xb) + 16 * ((lane % CPR) ^ key);
        x_lds[i] = BM * 128 + 1024 * b;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t *)(lds);
    auto issue = [&](int t, int slot) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const uint32_t at = lds0 + (slot * G + g) * STAGE;
#pragma unroll
            for (int i = 0; i < IW; ++i) mm_dma16(wbase[i] + (int64_t)(t * G + g) * 128, w_off[i], at + w_lds[i]);
#pragma unroll
            for (int i = 0; i < IX; ++i) mm_dma16(xbase + (int64_t)(t * G + g) * XR, x_off[i], at + x_lds[i]);
        }
    };

    // Sums in three levels: chains of kChain k steps in acc, kMmChain of those in
    // part, those in sum.  An F32 k step is a chain of eight products; SHORT: two
    // of four, a stage's two steps are added in acc and part takes kMmChain steps.
    constexpr int kU = 4 / KS;                         // k steps of a slice per wave
    constexpr int kSteps = G * kU;                     // .. of a stage
    constexpr int kChain = !F16W ? (SHORT ? 2 : 1) : KS == 1 ? kMmChain : kMmChain / 2;  // k steps per chain
    constexpr int kPer = kChain > kSteps ? kChain / kSteps : 1;  // stages per chain
    constexpr int kUn = S % kPer == 0 ? S : kPer % S == 0 ? kPer : S * kPer;  // stages unrolled: slot and chain are fixed in each
    static_assert(kChain % kSteps == 0 || kSteps % kChain == 0, "chains end with a stage or within it");
    static_assert(!SHORT || (!F16W && kSteps == 2), "SHORT: F32 rows, two steps a stage");
    const floatx16 zero = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f,
                           0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    floatx16 acc[FR][FC], part[FR][FC], sum[FR][FC];
#pragma unroll
    for (int a = 0; a < FR; ++a)
#pragma unroll
        for (int b = 0; b < FC; ++b) acc[a][b] = part[a][b] = sum[a][b] = zero;

    const int kg = wave / (WR * WC), wv = wave % (WR * WC);
    const int wr0 = (wv / WC) * FR * 32, wc = wv % WC;  // column blocks wc, wc + WC, ..
    const int n_stage = (int)(wb / (128 * G));
    // LDS offsets of this wave's operands of k step u in a slice: rows of
    // block 0 (the blocks' rows are 32 apart, and 32 rows keep the swizzle key)
    int a_off[kU], b_off[kU][CVT ? 2 : 1];
#pragma unroll
    for (int v = 0; v < kU; ++v) {
        const int u = KS == 1 ? v : kg * kU + v;
        const int ar = wr0 + n, br = 32 * wc + n;
        a_off[v] = ar * 128 + 16 * ((2 * u + hh) ^ ((ar / 2) % 8));
        if constexpr (CVT) {
#pragma unroll
            for (int h = 0; h < 2; ++h) b_off[v][h] = BM * 128 + br * 256 + 16 * ((4 * u + 2 * hh + h) ^ (br % 16));
        } else {
            b_off[v][0] = BM * 128 + br * 128 + 16 * ((2 * u + hh) ^ ((br / 2) % 8));
        }
    }
    // The stages with NC of the wave's column blocks (the others hold no token)
    auto run = [&](auto nc) {
        constexpr int NC = decltype(nc)::value;
        struct Operands {
            intx4 a[FR], b[NC][CVT ? 2 : 1];
        };
        auto fetch = [&](const uint8_t *st, int gv, Operands &x) {
            const uint8_t *sl = st + (gv / kU) * STAGE;
#pragma unroll
            for (int i = 0; i < FR; ++i)
                x.a[i] = *reinterpret_cast<const intx4 *>(sl + a_off[gv % kU] + 32 * 128 * i);
#pragma unroll
            for (int i = 0; i < NC; ++i)
#pragma unroll
                for (int h = 0; h < (CVT ? 2 : 1); ++h)
                    x.b[i][h] = *reinterpret_cast<const intx4 *>(sl + b_off[gv % kU][h] + 32 * XR * WC * i);
        };
        int chains = 0;
        for (int t0 = 0; t0 < n_stage; t0 += kUn) {
#pragma unroll
            for (int un = 0; un < kUn; ++un) {
                const int t = t0 + un, slot = un % S;
                if (t >= n_stage) break;
                if (t + S - 2 < n_stage)
                    mm_sync<(S - 2) * G * (IW + IX)>();
                else
                    mm_sync<0>();
                if (t + S - 1 < n_stage) issue(t + S - 1, slot == 0 ? S - 1 : slot - 1);
                const uint8_t *st = lds + slot * G * STAGE;
                Operands x[2];  // the next step's are read while this one's products run
                fetch(st, 0, x[0]);
#pragma unroll
                for (int gv = 0; gv < kSteps; ++gv) {
                    if (gv + 1 < kSteps) fetch(st, gv + 1, x[(gv + 1) & 1]);
                    const Operands &c = x[gv & 1];
                    const bool first = kSteps >= kChain ? gv % kChain == 0 : un % kPer == 0 && gv == 0;
#pragma unroll
                    for (int j = 0; j < NC; ++j) {
                        if constexpr (F16W) {
                            half8 xh;
                            if constexpr (CVT)
                                xh = mm_half8(__builtin_bit_cast(floatx4, c.b[j][0]), __builtin_bit_cast(floatx4, c.b[j][CVT ? 1 : 0]));
                            else
                                xh = __builtin_bit_cast(half8, c.b[j][0]);
#pragma unroll
                            for (int i = 0; i < FR; ++i)
                                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, c.a[i]), xh,
                                                                                   first ? zero : acc[i][j], 0, 0, 0);
                        } else {
                            const floatx4 xf = __builtin_bit_cast(floatx4, c.b[j][0]);
                            [[maybe_unused]] floatx16 half[FR][2];
#pragma unroll
                            for (int k = 0; k < 4; ++k)
#pragma unroll
                                for (int i = 0; i < FR; ++i) {
                                    floatx16 &s = SHORT ? half[i][k / 2] : acc[i][j];
                                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(
                                        __builtin_bit_cast(floatx4, c.a[i])[k], xf[k],
                                        (SHORT ? k % 2 == 0 : first && k == 0) ? zero : s, 0, 0, 0);
                                }
                            if constexpr (SHORT) {
#pragma unroll
                                for (int i = 0; i < FR; ++i) {
                                    half[i][0] += half[i][1];
                                    acc[i][j] = first ? half[i][0] : acc[i][j] + half[i][0];
                                }
                            }
                        }
                    }
                    const bool last = kSteps >= kChain ? gv % kChain == kChain - 1 : un % kPer == kPer - 1 && gv == kSteps - 1;
                    if (last) {
#pragma unroll
                        for (int i = 0; i < FR; ++i)
#pragma unroll
                            for (int j = 0; j < NC; ++j) part[i][j] += acc[i][j];
                    }
                }
                if (kSteps >= kChain || un % kPer == kPer - 1) {
                    chains += SHORT ? kSteps : kSteps >= kChain ? kSteps / kChain : 1;
                    if (chains >= kMmChain) {
                        chains = 0;
#pragma unroll
                        for (int i = 0; i < FR; ++i)
#pragma unroll
                            for (int j = 0; j < NC; ++j) {
                                sum[i][j] += part[i][j];
                                part[i][j] = zero;
                            }
                    }
                }
            }
        }
        if (kPer > 1 && n_stage % kPer != 0) {  // a chain that had not ended
#pragma unroll
            for (int i = 0; i < FR; ++i)
#pragma unroll
                for (int j = 0; j < NC; ++j) part[i][j] += acc[i][j];
        }
#pragma unroll
        for (int i = 0; i < FR; ++i)
#pragma unroll
            for (int j = 0; j < NC; ++j) sum[i][j] += part[i][j];
    };
#pragma unroll
    for (int s = 0; s < S - 1; ++s)
        if (s < n_stage) issue(s, s);
    if constexpr (kMmExperts<OUT> && FC > 1) {
        static_assert(FC == 2, "column blocks per wave");
        if (32 * (wc + WC) < count)
            run(MmInt<2>{});
        else
            run(MmInt<1>{});
    } else {
        run(MmInt<FC>{});
    }

    // the products into LDS, [group][token][row] with chunk c of a token at
    // c ^ (token % 8)
    mm_sync<0>();
    floatx4 *tile = reinterpret_cast<floatx4 *>(lds);
    constexpr int TC = BM * BN / 4;  // chunks of a group's tile
#pragma unroll
    for (int i = 0; i < FR; ++i)
#pragma unroll
        for (int j = 0; j < FC; ++j) {
            const int col = 32 * (wc + WC * j) + n;
#pragma unroll
            for (int g = 0; g < 4; ++g) {  // registers 4g .. 4g + 3: rows 8g + 4hh .. + 3
                const int c = (wr0 + 32 * i + 8 * g + 4 * hh) / 4;
                tile[kg * TC + col * (BM / 4) + (c ^ (col % 8))] =
                    floatx4{sum[i][j][4 * g], sum[i][j][4 * g + 1], sum[i][j][4 * g + 2], sum[i][j][4 * g + 3]};
            }
        }
    __syncthreads();
    auto product = [&](int col, int c) {
        floatx4 v[KS];
#pragma unroll
        for (int k = 0; k < KS; ++k) v[k] = tile[k * TC + col * (BM / 4) + (c ^ (col % 8))];
        if constexpr (KS == 4) return (v[0] + v[1]) + (v[2] + v[3]);
        else if constexpr (KS == 2) return v[0] + v[1];
        else return v[0];
    };
    constexpr int CPT = BMO / 4;  // output chunks per token
    for (int i = threadIdx.x; i < count * CPT; i += 64 * NW) {
        const int col = i / CPT, c = i % CPT, o = o0 + 4 * c;
        if (o >= p.n_out) continue;
        const floatx4 v = product(col, c);
        floatx4 v2 = v;
        if constexpr (NM == 2) v2 = product(col, c + CPT);
        mm_emit<OUT>(p, mm_index(p, start, col), o, v, v2);
    }
}

// ---- experts: grouping and the weighted sum ---------------------------------------

// Workgroup 0 groups the n_rows * n_used (token, slot) pairs by expert (ids
// outside [0, n_expert) are left out) and cuts each expert's pairs into tiles
// of at most `tile`; the others round x to f16 for the gate/up product, eight
// values a thread.  The order of an expert's pairs does not reach the
// results: a pair is a column of the product by itself.
constexpr int kPlanThreads = 1024;
constexpr int kPlanMaxExperts = 256;
__global__ __launch_bounds__(kPlanThreads) void moe_plan_kernel(const int32_t *ids, int n_pairs, int n_expert, int tile,
                                                                int max_tiles, MmPlan *plan, const float *x,
                                                                half8 *x16, int64_t n_chunk) {
    if (blockIdx.x > 0) {
        const int64_t i = ((int64_t)blockIdx.x - 1) * kPlanThreads + threadIdx.x;
        if (i < n_chunk) {
            const floatx4 *xs = reinterpret_cast<const floatx4 *>(x) + 2 * i;
            x16[i] = mm_half8(xs[0], xs[1]);
        }
        return;
    }
    __shared__ int cnt[kPlanMaxExperts], cur[kPlanMaxExperts];
    const int tid = threadIdx.x;
    MmExpert *ex = reinterpret_cast<MmExpert *>(plan + 1);
    int *tile_e = reinterpret_cast<int *>(ex + n_expert);
    int *order = tile_e + max_tiles;
    for (int e = tid; e < n_expert; e += kPlanThreads) cnt[e] = 0;
    __syncthreads();
    for (int i = tid; i < n_pairs; i += kPlanThreads) {
        const int e = ids[i];
        if (e >= 0 && e < n_expert) atomicAdd(&cnt[e], 1);
    }
    __syncthreads();
    if (tid < n_expert) {
        int start = 0, first = 0;
        for (int e = 0; e < tid; ++e) {
            start += cnt[e];
            first += (cnt[e] + tile - 1) / tile;
        }
        const int nt = (cnt[tid] + tile - 1) / tile;
        ex[tid] = MmExpert{start, cnt[tid], first, nt};
        for (int k = 0; k < nt; ++k) tile_e[first + k] = tid;
        if (tid == n_expert - 1) plan->n_tiles = first + nt;
        cur[tid] = start;
    }
    __syncthreads();
    for (int i = tid; i < n_pairs; i += kPlanThreads) {
        const int e = ids[i];
        if (e >= 0 && e < n_expert) order[atomicAdd(&cur[e], 1)] = i;
    }
}

// y[t] = (sum over slots j in order of part[t][j] * w[t][j]) + residual[t],
// slots whose id is outside the stack left out, as moe_down_kernel adds them.
// Grid (1024-value blocks of n_embd, n_rows).
__global__ __launch_bounds__(256) void moe_combine_kernel(const float *part, const int32_t *ids, const float *weights,
                                                          const float *residual, float *y, int n_embd, int n_expert,
                                                          int n_used) {
    const int t = blockIdx.y, o = ((int)blockIdx.x * 256 + threadIdx.x) * 4;
    if (o >= n_embd) return;
    floatx4 s = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int j = 0; j < n_used; ++j) {
        const int64_t i = (int64_t)t * n_used + j;
        const int e = ids[i];
        floatx4 v = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        if (e >= 0 && e < n_expert) {
            const floatx4 d = *reinterpret_cast<const floatx4 *>(part + i * n_embd + o);
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = __fmul_rn(d[k], weights[i]);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) s[k] = j == 0 ? v[k] : __fadd_rn(s[k], v[k]);
    }
    const int64_t i = (int64_t)t * n_embd + o;
    const floatx4 r = *reinterpret_cast<const floatx4_a4 *>(residual + i);
#pragma unroll
    for (int k = 0; k < 4; ++k) s[k] = __fadd_rn(s[k], r[k]);
    *reinterpret_cast<floatx4_a4 *>(y + i) = s;
}

}  // namespace sfa
