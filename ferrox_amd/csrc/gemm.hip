// Matrix products  C[m, n] = sum_k A[m, k] * W[n, k]  (weights are [out, in] as
// the checkpoint stores them; ferrox-core/src/matmul.rs:5-8) with fused epilogues,
// for plain and for expert-grouped rows.
//
//  * bfloat16: MFMA 16x16x32 tiles, float32 accumulators.
//  * float32 : MFMA 16x16x4 in float32, or every operand as the sum of three bfloat16
//    numbers on the bfloat16 instruction, with a smaller error in sums of a thousand terms (see `f32_split8`).
//
// In both, one output element's products are added in an order that the sizes of the
// weights fix, whatever the tile shape and whatever else is in the batch, so a float32
// row's result does not depend on how many rows are computed with it.
//
// Grouped mode: rows are sorted by expert; expert e owns rows
// [expert_offsets[e], expert_offsets[e+1]) and the weights at W + e * w_stride.
// Dual mode: two weight matrices (gate, up) are multiplied at once and the
// epilogue stores silu(gate) * up  (ferrox-moe/src/lib.rs:655-658).
#include "common.h"
#include <type_traits>
#include <utility>

FX_DEFINE_LAST_ERROR()

enum { EPI_STORE = 0, EPI_STORE_F32 = 1, EPI_RESID = 2, EPI_GATED = 3 };

struct GemmArgs {
    const void* A;
    long lda;
    const void* W;
    long w_stride;      // elements between experts (grouped)
    long up_offset;     // elements from the gate matrix to the up matrix (dual)
    long kb_stride;     // 0: rows of W are K long.  Else W is stored [K/64][rows][64] (64 k of every row, then the
                        // next 64 k of every row, ...) and this is rows * 64, the elements between two such slabs
    const void* bias;   // [N] or null
    int bias_dtype;
    void* C;
    long ldc;
    const float* row_scale;  // [M] or null, multiplies the product before it is added (EPI_RESID)
    const float* then_add;   // EPI_RESID of up to 16 plain rows: [M, N] at a row distance of ld_then_add, added behind the product, or null
    long ld_then_add;
    const int* a_rows;       // [M] or null: row of A to read for logical row m
    const int* c_rows;       // [M] or null: row of C to write for logical row m
    const int* expert_offsets;  // [E+1] or null
    const int* pair_ids;        // few rows, unsorted: expert of logical row ("pair") m, instead of expert_offsets
    int pair_div;               //   pair m reads row m / pair_div of A and writes row m of C
    int n_always, always_rows;  //   experts E .. E+n_always-1 take rows 0 .. always_rows-1 each: their tile s writes rows
    int always_from_a;          //   M + s*always_rows + t of C and reads row t of A (1) or that same row of A (0)
    int E;
    int M, N, K;
    const void* norm_w;  // skinny bf16 kernel only: A is the float32 residual stream and RMSNorm with these weights
    int norm_dtype;      //   is applied on the way in; norm_w is [K]
    float norm_eps;
    const float* row_ss; // skinny bf16 kernel only: row m of the product is scaled by rsqrt(sum(row_ss[m][0..row_ss_n)) / K + norm_eps)
    int row_ss_n;        //   (the rows of A are x * w of an RMSNorm whose scale is still to come)
    // skinny bf16 kernel, rope epilogue: C is [M, (nh + 2 nkv) * hd], queries | keys | values of token m at position
    // positions[m] of sequence token_seq[m].  Queries are rotated and stored in C; keys are rotated and stored in their
    // page, values in theirs (transposed), nothing of either in C.  Split-half pairs (i, i + rot/2), angle
    // pos * theta^(-2i/rot) (ferrox-core/src/attention.rs:20-32); the product is rounded to bfloat16 before it is
    // rotated, as when the rotation is a kernel of its own.
    const int* rope_positions;
    const int* rope_token_seq;
    const int* rope_table;
    int rope_max_blocks;
    void* rope_k_pages;     // null: nothing is written to pages (a layer that reads another's cache)
    void* rope_v_pages;
    int rope_nh, rope_nkv, rope_hd, rope_bs, rope_rot;
    // TURN (few rows, stored): columns come in heads of rope_hd (0: nothing is turned), and of each the rope_rot dimensions from rope_nh on are turned in pairs
    // (2i, 2i + 1), row m by rope_positions[m] * rope_inv_freq[i], and stretched by act_alpha
    const float* rope_inv_freq;       // rot/2 floats: pair i turns by (float)pos * rope_inv_freq[i]
    const float* rope_freq_factors;   // rot/2 floats or null: the angle of pair i is divided by rope_freq_factors[i]
    int stream_w;  // tiled kernel: the weights are read about once (one row tile a weight matrix): load them non-temporal
    int act;     // EPI_GATED: which activation the gate goes through (ACT_*)
    float act_limit, act_alpha;   // ACT_SWIGLU_CLAMP: the bound on gate and up, and the sigmoid's slope; SACT_SOFTCAP: the cap
    const float* pre_scale;       // EPI_GATED: [.] or null: gate and up of logical row m are multiplied by
    const int* pre_scale_rows;    //   pre_scale[pre_scale_rows ? pre_scale_rows[m] : m] before the activation (a row of A scaled)
    int store_act;   // EPI_STORE: what the product goes through before it is stored (SACT_*), 0 for nothing
    const float* out_gate;   // SACT_GATE: gate logits; row m of C belongs to row m / gate_div of it and to its columns
    long ld_gate;            //   (m % gate_div) * N + n
    int gate_div;
    int vec_ok;  // 16-byte loads are legal for A and W
    int c_vec;   // float32: so are 16-byte loads and stores of C
    int n_col_tiles, n_row_tiles;  // tiled kernels: the grid they decode block ids with
    int tile_rows;  // LDS-tiled kernels, plain rows: rows a tile takes, up to its height
    int by_row_tile;  // LDS-tiled kernels, rows sorted by expert: every eighth row tile to an XCD
};

// block -> (first logical row, end of rows, expert).  Plain: tiles of TM rows.
// Grouped: expert e has ceil(rows_e / TM) tiles, in the order of the experts; a tile past the
// last one gets r0 = -1.  Every wave finds its tile by itself, 64 experts at a time: each lane
// takes one expert's bounds, a scan over the lanes gives the tiles before it, and the lane whose
// range holds the tile tells the others.  (One load's latency instead of one per expert.)
template <int TM>
__device__ __forceinline__ void locate_rows(const GemmArgs& g, int tile, int& r0, int& r_end, int& expert) {
    if (!g.expert_offsets) {
        r0 = tile * TM;
        r_end = g.M;
        expert = 0;
        if (r0 >= g.M) r0 = -1;
        return;
    }
    const int lane = threadIdx.x & 63;
    int before = 0;
    r0 = -1;
    r_end = 0;
    expert = 0;
    for (int base = 0; base < g.E; base += 64) {
        const int e = base + lane;
        const int b = e < g.E ? g.expert_offsets[e] : 0, en = e < g.E ? g.expert_offsets[e + 1] : 0;
        const int nt = (en - b + TM - 1) / TM;
        const int incl = wave_inclusive_sum(nt);
        const int first = before + incl - nt;
        const unsigned long long hit = __ballot(tile >= first && tile < first + nt);
        if (hit) {      // (the same in every lane: what the owner knows is read from its lane, no exchange)
            const int src = __builtin_amdgcn_readfirstlane(__ffsll((long long)hit) - 1);
            r0 = __builtin_amdgcn_readlane(b + (tile - first) * TM, src);
            r_end = __builtin_amdgcn_readlane(en, src);
            expert = base + src;
            return;
        }
        before += __builtin_amdgcn_readlane(incl, 63);
    }
}

// lanes (of the 64 of a wave) whose `e` equals this lane's; e < 2^bits, e < 0 matches nothing
__device__ __forceinline__ unsigned long long same_expert_lanes(int e, int bits) {
    unsigned long long m = __ballot(e >= 0);
    for (int b = 0; b < bits; ++b) {
        const unsigned long long set = __ballot((e >> b) & 1);
        m &= ((e >> b) & 1) ? set : ~set;
    }
    return e >= 0 ? m : 0ull;
}

// Up to 64 unsorted pairs: the experts that occur, in the order of their first pairs, get one tile per 16 of
// their pairs, and a tile's rows are those pairs in their order.  Every wave works this out by itself from the
// ids (a lane per pair) with ballots and counts alone: a lane that holds an expert's first pair counts the tiles
// of the first pairs in the lanes below it (an expert has one to four tiles, so four ballots), and what the tile's
// owner knows is read from its lane directly.  (A loop over the experts that occur, two exchanges between lanes
// each, cost a wave 1-2 us before its first load.)  After those tiles come the experts that every row takes
// (n_always of them, a shared expert cut into pieces), one tile each.  Returns false for a tile past the last one;
// else the expert, and for tile row lane % 16 the rows of A and C (or -1).
__device__ __forceinline__ bool locate_pairs(const GemmArgs& g, int tile, int& expert, int& a_row, int& c_row) {
    const int lane = threadIdx.x & 63, li = lane & 15;
    int e = lane < g.M ? g.pair_ids[lane] : -1;
    if (e >= g.E) e = -1;
    int bits = 0;
    while ((1 << bits) < g.E) ++bits;
    const unsigned long long same = same_expert_lanes(e, bits);
    const bool first = e >= 0 && lane == __ffsll((long long)same) - 1;
    const int my_tiles = (__popcll(same) + 15) >> 4;
    const unsigned long long below = (1ull << lane) - 1;
    int before = 0, total = 0;      // tiles of the experts whose first pair comes earlier than this lane's; of all
#pragma unroll
    for (int t = 1; t <= 4; ++t) {
        const unsigned long long f = __ballot(first && my_tiles >= t);
        before += __popcll(f & below);
        total += __popcll(f);
    }
    a_row = c_row = -1;
    if (tile >= total) {
        const int s = tile - total;
        if (s >= g.n_always) return false;
        expert = g.E + s;
        if (li < g.always_rows) {
            c_row = g.M + s * g.always_rows + li;
            a_row = g.always_from_a ? li : c_row;
        }
        return true;
    }
    const unsigned long long sel = __ballot(first && tile >= before && tile < before + my_tiles);
    const int src = __builtin_amdgcn_readfirstlane(__ffsll((long long)sel) - 1);
    expert = __builtin_amdgcn_readlane(e, src);
    const int skip = (tile - __builtin_amdgcn_readlane(before, src)) * 16;      // pairs of this expert in its earlier tiles
    unsigned long long rows = ((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(same >> 32), src) << 32) |
                              (unsigned)__builtin_amdgcn_readlane((int)(unsigned)same, src);
    int mine = -1;                  // pair number skip + li of this expert, if it has so many
    for (int j = 0; j < skip + 16 && rows; ++j) {
        const int p = __ffsll((long long)rows) - 1;
        rows &= rows - 1;
        if (j == skip + li) mine = p;
    }
    if (mine >= 0) {
        c_row = mine;
        a_row = mine / g.pair_div;
    }
    return true;
}

// The gated epilogue stores act(gate) * up; `act` is a parameter of the call (GemmArgs::act), uniform over the
// launch, so another gated feed-forward needs no other kernel.
//   ACT_SILU       x / (1 + exp(-x))                               (ferrox-core/src/matmul.rs:268-270)
//   ACT_GELU_TANH  0.5 x (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3)))
//   ACT_GELU       0.5 x (1 + erf(x / sqrt(2)))
//   ACT_RELU       max(x, 0)
//   ACT_SWIGLU_CLAMP  g = min(gate, limit), u = clamp(up, -limit, limit): g sigmoid(alpha g) (u + 1)
enum { ACT_SILU = 0, ACT_GELU_TANH = 1, ACT_GELU = 2, ACT_RELU = 3, ACT_SWIGLU_CLAMP = 4, ACT_COUNT = 5 };
__device__ __forceinline__ float silu_f(float x) { return x / (1.0f + expf(-x)); }
// The same for several elements at once: the quotient by a reciprocal, one step of refinement and no scaling, which the divisor, 1 to
// e^80, does not need; where one of them is beyond that or infinite (inf / 1 has no remainder to refine with), as above.  The same bits for every float of either sign from
// 1e-30 to 80 (checked against the division and against 64 bits), four instructions instead of eleven an element: the epilogue of a gate/up tile is bound by them.
template <int N>
__device__ __forceinline__ void silu_n(float (&x)[N]) {
    float low = x[0], high = x[0];      // (a NaN among them is passed over and comes out of either path as one)
#pragma unroll
    for (int i = 1; i < N; ++i) low = fminf(low, x[i]), high = fmaxf(high, x[i]);
    if (low > -80.0f && high < INFINITY) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float d = 1.0f + expf(-x[i]), r = __builtin_amdgcn_rcpf(d), q = x[i] * r;
            x[i] = fmaf(fmaf(-d, q, x[i]), r, q);
        }
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] = silu_f(x[i]);
    }
}
template <int ACT>
__device__ __forceinline__ float gated_c(float gate, float up, float limit, float alpha) {
    float a;
    if constexpr (ACT == ACT_SWIGLU_CLAMP) {
        const float gc = fminf(gate, limit), uc = fminf(fmaxf(up, -limit), limit);
        return gc / (1.0f + expf(-alpha * gc)) * (uc + 1.0f);
    }
    if constexpr (ACT == ACT_GELU_TANH) a = 0.5f * gate * (1.0f + tanhf(0.7978845608028654f * (gate + 0.044715f * gate * gate * gate)));
    else if constexpr (ACT == ACT_GELU) a = 0.5f * gate * (1.0f + erff(gate * 0.7071067811865476f));
    else if constexpr (ACT == ACT_RELU) a = fmaxf(gate, 0.0f);
    else a = silu_f(gate);
    return a * up;
}
// What a stored product (EPI_STORE) may go through on its way out: the activation of a feed-forward without a gate,
// down(act(up x)).  Uniform over the launch; SACT_NONE costs one scalar compare per element.
//   SACT_RELU2    max(x, 0)^2
//   SACT_SOFTCAP  limit * tanh(x / limit)      (logits kept within +-limit)
//   SACT_GATE     x * sigmoid(gate), gate a float32 matrix of the output's elements (`out_gate`)
enum { SACT_NONE = 0, SACT_RELU2 = 1, SACT_RELU = 2, SACT_SILU = 3, SACT_GELU_TANH = 4, SACT_SOFTCAP = 5, SACT_GATE = 6, SACT_COUNT = 7 };
// the gate logit of output element (m, n); 0 without a gate
__device__ __forceinline__ float gate_of(const GemmArgs& g, int m, int n) {
    if (!g.out_gate) return 0.f;
    const int row = m / g.gate_div;
    return g.out_gate[(size_t)row * g.ld_gate + (size_t)(m - row * g.gate_div) * g.N + n];
}
__device__ __forceinline__ float stored_f(const GemmArgs& g, float x, float gate) {
    const int act = g.store_act;
    const float limit = g.act_limit;
    if (act == SACT_NONE) return x;
    if (act == SACT_GATE) return x / (1.0f + expf(-gate));
    if (act == SACT_RELU2) {
        const float r = fmaxf(x, 0.0f);
        return r * r;
    }
    if (act == SACT_RELU) return fmaxf(x, 0.0f);
    if (act == SACT_SILU) return silu_f(x);
    if (act == SACT_SOFTCAP) return limit * tanhf(x / limit);
    return 0.5f * x * (1.0f + tanhf(0.7978845608028654f * (x + 0.044715f * x * x * x)));
}
// f(what happens to an output on its way out, as a compile-time constant; SACT_COUNT: one of the rarer activations, looked
// up per element): the tiled epilogues call this once around their loops (with every activation inside the loops of a
// plain product's epilogue those were 10-16 % of the q/k/v product)
template <bool STORES, typename F>
__device__ __forceinline__ void with_stored(int act, F&& f) {
    if (!STORES || act == SACT_NONE) f(std::integral_constant<int, SACT_NONE>{});
    else if (act == SACT_RELU2) f(std::integral_constant<int, SACT_RELU2>{});
    else if (act == SACT_GATE) f(std::integral_constant<int, SACT_GATE>{});
    else f(std::integral_constant<int, SACT_COUNT>{});
}
template <int ACT>
__device__ __forceinline__ float stored_c(const GemmArgs& g, float x, float gate) {
    if constexpr (ACT == SACT_NONE) return x;
    if constexpr (ACT == SACT_GATE) return x / (1.0f + expf(-gate));
    if constexpr (ACT == SACT_RELU2) {
        const float r = fmaxf(x, 0.0f);
        return r * r;
    }
    return stored_f(g, x, gate);
}
// what gate and up of logical row m are multiplied by before the activation (1 without a pre-scale)
#define FX_PRE_SCALE(g, ml) ((g).pre_scale ? (g).pre_scale[(g).pre_scale_rows ? (g).pre_scale_rows[ml] : (ml)] : 1.0f)
// f(the activation as a compile-time constant): an epilogue calls this once around its loops, so that the choice is
// one jump per block and not work inside the loops (left inside, the compiler works out every activation for every
// element and picks one: the tiled products of a prompt were 4-10 % slower for it)
template <typename F>
__device__ __forceinline__ void with_activation(int act, F&& f) {
    switch (act) {
        case ACT_GELU_TANH: f(std::integral_constant<int, ACT_GELU_TANH>{}); break;
        case ACT_GELU: f(std::integral_constant<int, ACT_GELU>{}); break;
        case ACT_RELU: f(std::integral_constant<int, ACT_RELU>{}); break;
        case ACT_SWIGLU_CLAMP: f(std::integral_constant<int, ACT_SWIGLU_CLAMP>{}); break;
        default: f(std::integral_constant<int, ACT_SILU>{}); break;
    }
}

// ===========================================================================
// bfloat16 on MFMA
// ===========================================================================
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

#define BK 64
#define LDS_STRIDE (BK + 8)  // bf16 elements; keeps 16-byte reads of 16 rows on distinct banks

template <bool VEC>   // VEC: K is a multiple of 8 and rows are 16-byte aligned
__device__ __forceinline__ uint4 load_chunk(const bf16* row, int k, int K) {
    uint4 v = make_uint4(0, 0, 0, 0);
    if (!row || k >= K) return v;
    if (VEC) return *(const uint4*)(row + k);
    uint16_t tmp[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) tmp[i] = (k + i < K) ? row[k + i].bits : (uint16_t)0;
    v.x = tmp[0] | ((uint32_t)tmp[1] << 16);
    v.y = tmp[2] | ((uint32_t)tmp[3] << 16);
    v.z = tmp[4] | ((uint32_t)tmp[5] << 16);
    v.w = tmp[6] | ((uint32_t)tmp[7] << 16);
    return v;
}

// TM x TN block tile (TN counts weight rows: in dual mode half of them are gate
// rows and half up rows, interleaved in groups of 16), 4 waves of WM x WN.
template <int TM, int TN, int WM, int WN, bool DUAL, int EPI, bool VEC>
__global__ __launch_bounds__(256) void gemm_bf16_kernel(GemmArgs g) {
    constexpr int WAVES_N = TN / WN;
    static_assert((TM / WM) * WAVES_N == 4, "four waves per block");
    constexpr int MT = WM / 16, NT = WN / 16;
    constexpr int NA = (TM * 8 + 255) / 256, NB = (TN * 8 + 255) / 256;
    constexpr int OUT_TN = DUAL ? TN / 2 : TN;
    __shared__ __attribute__((aligned(16))) bf16 As[TM * LDS_STRIDE];
    __shared__ __attribute__((aligned(16))) bf16 Bs[TN * LDS_STRIDE];

    // Blocks go to the 8 XCDs in turn (block b runs on XCD b % 8), each with an L2 of its own: the
    // tiles are dealt out so that an XCD works through a contiguous range of column tiles, rows
    // fastest, and the weights of those columns stay in its L2.
    const int per_xcd = (g.n_col_tiles * g.n_row_tiles + 7) / 8;
    const int logical = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (logical >= g.n_col_tiles * g.n_row_tiles) return;
    int r0, r_end, expert;
    locate_rows<TM>(g, logical % g.n_row_tiles, r0, r_end, expert);
    if (r0 < 0) return;
    const int n0 = (logical / g.n_row_tiles) * OUT_TN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const bf16* Abase = (const bf16*)g.A;
    const bf16* Wbase = (const bf16*)g.W + (size_t)expert * g.w_stride;

    // the row each of this thread's chunks comes from stays the same for all k
    const bf16* a_src[NA];
    const bf16* b_src[NB];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int c = tid + i * 256, row = c >> 3;
        a_src[i] = nullptr;
        if (c < TM * 8 && r0 + row < r_end) {
            const int m = r0 + row;
            a_src[i] = Abase + (size_t)(g.a_rows ? g.a_rows[m] : m) * g.lda;
        }
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int c = tid + i * 256, row = c >> 3;
        b_src[i] = nullptr;
        if (c < TN * 8) {
            if (DUAL) {
                const int col = n0 + (row >> 5) * 16 + (row & 15);
                if (col < g.N) b_src[i] = Wbase + (size_t)col * g.K + (((row >> 4) & 1) ? g.up_offset : 0);
            } else {
                if (n0 + row < g.N) b_src[i] = Wbase + (size_t)(n0 + row) * g.K;
            }
        }
    }

    f32x4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

    // Two tiles are on their way from memory into registers while a third is multiplied out of LDS.
    uint4 a0[NA], b0[NB], a1[NA], b1[NB];
    const int kc = (tid & 7) * 8;
#define FX_FETCH(AR, BR, K0)                                                                  \
    {                                                                                         \
        _Pragma("unroll") for (int i = 0; i < NA; ++i) AR[i] = load_chunk<VEC>(a_src[i], (K0) + kc, g.K); \
        _Pragma("unroll") for (int i = 0; i < NB; ++i) BR[i] = load_chunk<VEC>(b_src[i], (K0) + kc, g.K); \
    }
#define FX_STAGE(AR, BR)                                                                      \
    {                                                                                         \
        _Pragma("unroll") for (int i = 0; i < NA; ++i) {                                      \
            const int c = tid + i * 256;                                                      \
            if (c < TM * 8) *(uint4*)(As + (c >> 3) * LDS_STRIDE + kc) = AR[i];               \
        }                                                                                     \
        _Pragma("unroll") for (int i = 0; i < NB; ++i) {                                      \
            const int c = tid + i * 256;                                                      \
            if (c < TN * 8) *(uint4*)(Bs + (c >> 3) * LDS_STRIDE + kc) = BR[i];               \
        }                                                                                     \
    }
#define FX_MULTIPLY()                                                                         \
    _Pragma("unroll") for (int ks = 0; ks < BK / 32; ++ks) {                                  \
        const int koff = ks * 32 + (lane >> 4) * 8;                                           \
        bf16x8_t af[MT], bfr[NT];                                                             \
        _Pragma("unroll") for (int i = 0; i < MT; ++i)                                        \
            af[i] = *(const bf16x8_t*)(As + (wm * WM + i * 16 + (lane & 15)) * LDS_STRIDE + koff); \
        _Pragma("unroll") for (int j = 0; j < NT; ++j)                                        \
            bfr[j] = *(const bf16x8_t*)(Bs + (wn * WN + j * 16 + (lane & 15)) * LDS_STRIDE + koff); \
        _Pragma("unroll") for (int i = 0; i < MT; ++i)                                        \
            _Pragma("unroll") for (int j = 0; j < NT; ++j)                                    \
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0); \
    }
    FX_FETCH(a0, b0, 0);
    FX_FETCH(a1, b1, BK);          // beyond K this loads zeros
    for (int k0 = 0; k0 < g.K; k0 += 2 * BK) {
        lds_barrier();  // the previous tile has been read
        FX_STAGE(a0, b0);
        lds_barrier();
        FX_FETCH(a0, b0, k0 + 2 * BK);
        FX_MULTIPLY();
        lds_barrier();
        FX_STAGE(a1, b1);           // a tile of zeros if K ends before it
        lds_barrier();
        FX_FETCH(a1, b1, k0 + 3 * BK);
        FX_MULTIPLY();
    }
#undef FX_FETCH
#undef FX_STAGE
#undef FX_MULTIPLY

    // epilogue: lane holds rows 4*(lane/16)+r, column lane%16 of each 16x16 tile
    float bias_v[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) bias_v[j] = 0.f;
    if (!DUAL && g.bias) load_strided_as_float<NT, 16>(g.bias, g.bias_dtype, n0 + wn * WN + (lane & 15), g.N, bias_v);
    if constexpr (DUAL) {
        with_activation(g.act, [&](auto ac) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int ml = r0 + wm * WM + i * 16 + (lane >> 4) * 4 + r;
                    if (ml >= r_end) continue;
                    const int m = g.c_rows ? g.c_rows[ml] : ml;
                    const float ps = FX_PRE_SCALE(g, ml);
#pragma unroll
                    for (int j = 0; j < NT; j += 2) {
                        const int n = n0 + wn * (WN / 2) + (j / 2) * 16 + (lane & 15);
                        if (n < g.N)
                            from_float((bf16*)g.C + (size_t)m * g.ldc + n, gated_c<decltype(ac)::value>(acc[i][j][r] * ps, acc[i][j + 1][r] * ps, g.act_limit, g.act_alpha));
                    }
                }
        });
        return;
    }
    with_stored<EPI == EPI_STORE || EPI == EPI_STORE_F32>(g.store_act, [&](auto kind) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int ml = r0 + wm * WM + i * 16 + (lane >> 4) * 4 + r;
            if (ml >= r_end) continue;
            const int m = g.c_rows ? g.c_rows[ml] : ml;
            {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const int n = n0 + wn * WN + j * 16 + (lane & 15);
                    if (n >= g.N) continue;
                    float v = acc[i][j][r];
                    if (g.bias) v += bias_v[j];
                    if (EPI == EPI_STORE) {
                        from_float((bf16*)g.C + (size_t)m * g.ldc + n, stored_c<decltype(kind)::value>(g, v, decltype(kind)::value == SACT_GATE ? gate_of(g, m, n) : 0.f));
                    } else if (EPI == EPI_STORE_F32) {
                        ((float*)g.C)[(size_t)m * g.ldc + n] = stored_c<decltype(kind)::value>(g, v, decltype(kind)::value == SACT_GATE ? gate_of(g, m, n) : 0.f);
                    } else {
                        if (g.row_scale) v *= g.row_scale[ml];
                        ((float*)g.C)[(size_t)m * g.ldc + n] += v;
                    }
                }
            }
        }
    }
    });
}

// ---------------------------------------------------------------------------
// Many rows, K a multiple of 64, weights that are read about once or tiles of few
// rows: tiles of up to 192 rows x TN weight rows, eight waves.  K advances in steps of 64 through a ring of NS stages in LDS; tiles
// travel from global memory straight into LDS (no registers in between), NS-1
// steps ahead of their use, and one barrier per step separates the waves that
// still read a stage from the loads that refill it.  A wave-load fills 1 KB of
// LDS, 8 rows of 64 k; inside a row the eight 16-byte chunks are stored at
// chunk ^ ((row / 2) % 8), which the loading lanes achieve by choosing which
// chunk they fetch, so that the 16 rows an MFMA operand reads fall on distinct
// banks without padding.  Waves form a 2 x 4 grid: a wave owns TN/4 weight rows
// and every second block of 16 rows (so a tile with few rows, an expert's share,
// still spreads over both halves, and the two waves of a SIMD are one of each
// half); row blocks past the tile's rows are not multiplied.  The rows' ring may
// be shallower than the weights' (NSA < NS): weights come from memory and are
// read once, so more of them are kept on their way.
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(1))) const void* fx_global_ptr;
typedef __attribute__((address_space(3))) void* fx_lds_ptr;

template <int N>
using fx_int = std::integral_constant<int, N>;
template <int... Is, typename F>
__device__ __forceinline__ void static_for(std::integer_sequence<int, Is...>, F&& f) {
    (f(std::integral_constant<int, Is>{}), ...);
}

template <int N>
__device__ __forceinline__ void wait_loads_but() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// The K loop of one wave for NA active row blocks (blocks wm, wm+2, ... of the tile).
template <int NA, int MT, int NT, int TM, int TN, int NSA, int NSB, bool STREAM>
__device__ __forceinline__ void wide_k_loop(f32x4_t (&acc)[MT][NT], const bf16* const (&a_src)[TM / 64],
                                            const bf16* const (&b_src)[TN / 64], bf16* stages, int K, int wave,
                                            int a_off, int b_off, int sw, int kq, long kb_stride) {
    static_assert(NSA >= 2 && NSB >= NSA, "the weights' ring is at least as deep as the rows'");
    const int koff0 = (kq ^ sw) * 8, koff1 = ((4 + kq) ^ sw) * 8;
    constexpr int NLA = TM / 64, NLB = TN / 64;     // wave-loads per wave and step
    bf16* const ring_b = stages + NSA * TM * 64;
    const int nk = K >> 6;
    // past the end: a tile nobody reads, so that the counts of loads in flight stay even
    auto issue_a = [&](int kt) {
        const int k0 = min(kt, nk - 1) << 6;
        bf16* st = stages + (kt % NSA) * (TM * 64);
#pragma unroll
        for (int i = 0; i < NLA; ++i)
            __builtin_amdgcn_global_load_lds((fx_global_ptr)(a_src[i] + k0), (fx_lds_ptr)(st + (wave + 8 * i) * 512), 16, 0, 0);
    };
    auto issue_b = [&](int kt) {
        const size_t w0 = kb_stride ? (size_t)min(kt, nk - 1) * kb_stride : (size_t)(min(kt, nk - 1) << 6);
        bf16* st = ring_b + (kt % NSB) * (TN * 64);
#pragma unroll
        for (int i = 0; i < NLB; ++i) {
            // weights that nothing reads twice come with the non-temporal hint (cache policy operand 2): each
            // load takes whole 128-byte lines that need no place in the caches, and memory delivers them up to a
            // tenth faster.  A compile-time choice: as a flag tested here the tiled products of a prompt, which
            // do not stream, were 3-4 % slower.
            __builtin_amdgcn_global_load_lds((fx_global_ptr)(b_src[i] + w0), (fx_lds_ptr)(st + (wave + 8 * i) * 512), 16, 0, STREAM ? 2 : 0);
        }
    };
    // Each step issues the rows of step kt + NSA - 1, then the weights of step kt + NSB - 1.  Weights come from
    // memory and nothing reads them twice, so their ring may be deeper: more of them are on their way at a time.
#pragma unroll
    for (int p = 0; p < NSB - 1; ++p) {
        if (p >= NSB - NSA) issue_a(p - (NSB - NSA));
        issue_b(p);
    }
    for (int kt = 0; kt < nk; ++kt) {
        // this wave's part of step kt has landed: what may still be on its way are the loads of the NSA - 2
        // steps issued since the rows of step kt, and the weights issued right after those rows
        wait_loads_but<(NSA - 2) * (NLA + NLB) + (NSB > NSA ? NLB : 0)>();
        __builtin_amdgcn_s_barrier();          // ... everyone's has, and the stages of step kt-1 are free
        issue_a(kt + NSA - 1);
        issue_b(kt + NSB - 1);
        const bf16* base_a = stages + (kt % NSA) * (TM * 64);
        const bf16* base_b = ring_b + (kt % NSB) * (TN * 64);
        // 2*NA units of one operand of rows against NT operands of weights; the rows' operands are
        // read from LDS a few units ahead of the products that use them
        constexpr int U = 2 * NA, D = U > 3 ? 3 : U - 1;
        bf16x8_t bfr[2][NT], fr[U];
#pragma unroll
        for (int j = 0; j < NT; ++j) bfr[0][j] = *(const bf16x8_t*)(base_b + b_off + j * 16 * 64 + koff0);
#pragma unroll
        for (int u = 0; u < D; ++u)
            fr[u] = *(const bf16x8_t*)(base_a + a_off + (u % NA) * 32 * 64 + ((u / NA) ? koff1 : koff0));
        static_for(std::make_integer_sequence<int, U>{}, [&](auto uc) {
            constexpr int u = decltype(uc)::value;
            if constexpr (u + D < U)
                fr[u + D] = *(const bf16x8_t*)(base_a + a_off + ((u + D) % NA) * 32 * 64 + (((u + D) / NA) ? koff1 : koff0));
            if constexpr (u == 0) {
#pragma unroll
                for (int j = 0; j < NT; ++j) bfr[1][j] = *(const bf16x8_t*)(base_b + b_off + j * 16 * 64 + koff1);
            }
            __builtin_amdgcn_sched_barrier(0);      // the reads above stay ahead of the products below
#pragma unroll
            for (int j = 0; j < NT; ++j)
                acc[u % NA][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[u / NA][j], fr[u], acc[u % NA][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    wait_loads_but<0>();                       // the loads past the end, before the block leaves
}

// Which tile of the output a block of the LDS-tiled kernels works on; false: none.  Blocks go to the 8 XCDs in turn (block
// b runs on XCD b % 8), each with an L2 of its own: an XCD works through a contiguous eighth of the tiles in an order that keeps
// neighbours in rows and columns together, so the operands of the tiles it has at a time stay in its L2.  That order is bands of
// 8 row tiles, rows fastest inside a band: the 32 tiles that an XCD works on at a time are 8 rows x 4 columns, and 12 operand
// tiles serve 32 products.
// Rows sorted by expert: expert after expert, each in that order; how many tiles there are is counted from the
// experts' shares (64 at a time, a lane each, as in `locate_rows`), blocks beyond them find none.  What an expert's row tiles have in
// common, its weights, is then fetched by the one or two XCDs that its tiles fall to.  (With the mapping below, the tiles in quarters took 147 us instead of 139 for the gate/up product of 2,048
// tokens on 30 of 60 experts, 236 instead of 195 for 3,500, 1,297 and 667 instead of 1,245 and 626 for both of 4,096 tokens of
// the larger model.  Eighths of equal cost, a tile's
// rows and a constant, instead of equal numbers of tiles: no better, 237 us for the 3,500.)
// `by_row_tile`: XCD x takes the row tiles x, x + 8, ... and runs through the columns of each, so weights that two row tiles
// share are fetched by two XCDs, but no XCD has many full tiles where another has nearly empty ones, and nothing is counted (the ring of 192 rows, 512 tokens
// on 40 experts, 55 against 66 us for the down product).
// SPREAD, where the caller knows that no expert has a second row tile and nothing is shared: eighths of the tiles again, equal to one, but of the row tiles in
// the order 0, 8, 16, .., 1, 9, .., so that full and nearly empty ones are dealt out (both products of 64 decoded tokens of the larger model, tiles of 64
// rows, in order 617 us, dealt out 600, of 128 tokens beside the shared expert's pieces, which all lie at the end, tiles of 128, 673 in order with tiles of 64, 635; a prompt of 64
// tokens, which takes some of the experts only, 3,550 a step either way, 3,910 with every eighth row tile, which are not equally many).  Not a flag tested here: the
// step of 117 tokens, which has second row tiles, took 0.5-1 % more for it.
// `alone`: the expert's rows are one tile (so they are taken to be with `by_row_tile` and SPREAD; either answer gives the same sums).
template <int TM, bool SPREAD = false>
__device__ __forceinline__ bool wide_tile(const GemmArgs& g, int& r0, int& r_end, int& expert, int& col_tile, bool* alone = nullptr) {
    const int lane = threadIdx.x & 63, C = g.n_col_tiles;
    if (alone) *alone = true;
    if (!SPREAD && g.by_row_tile && g.expert_offsets) {
        const int i = blockIdx.x / 8, row_tile = (i / C) * 8 + blockIdx.x % 8;
        col_tile = i % C;
        locate_rows<TM>(g, row_tile, r0, r_end, expert);       // (r0 < 0: past the last one)
        return r0 >= 0;
    }
    auto share = [&](int base, int& b, int& en) {       // row tiles of expert base + lane
        const int e = base + lane;
        b = e < g.E ? g.expert_offsets[e] : 0;
        en = e < g.E ? g.expert_offsets[e + 1] : 0;
        return (en - b + TM - 1) / TM;
    };
    auto in_bands = [&](int t, int rows, int& row) {    // tile t of rows x C tiles
        const int band = t / (8 * C), rem = t % (8 * C), band_rows = min(8, rows - band * 8);
        row = band * 8 + rem % band_rows;
        col_tile = rem / band_rows;
    };
    int rows = g.n_row_tiles, b = 0, en = 0, nt = 0, incl = 0;
    if (g.expert_offsets) {
        rows = 0;
        for (int base = 0; base < g.E; base += 64) {
            nt = share(base, b, en);
            incl = wave_inclusive_sum(nt);
            rows += __builtin_amdgcn_readlane(incl, 63);
        }
    }
    const int per_xcd = (C * rows + 7) / 8, i = blockIdx.x / 8;
    const int logical = (blockIdx.x % 8) * per_xcd + i;
    if (i >= per_xcd || logical >= C * rows) return false;
    int item = logical;                 // a tile in that order; SPREAD (rows sorted by expert): a row tile
    if constexpr (SPREAD) {
        const int s = logical / C, q = rows >> 3, m = rows & 7, longer = m * (q + 1);     // the first m of the eight have q + 1 row tiles
        item = s < longer ? s % (q + 1) * 8 + s / (q + 1) : (s - longer) % max(q, 1) * 8 + m + (s - longer) / max(q, 1);
        col_tile = logical - s * C;
    }
    if (!g.expert_offsets) {
        int row;
        in_bands(logical, rows, row);
        r0 = row * g.tile_rows;
        r_end = min(g.M, r0 + g.tile_rows);
        expert = 0;
        return true;
    }
    int before = 0;
    for (int base = 0; base < g.E; base += 64) {
        if (g.E > 64) {
            nt = share(base, b, en);
            incl = wave_inclusive_sum(nt);
        }
        const int first = (before + incl - nt) * (SPREAD ? 1 : C);
        const unsigned long long hit = __ballot(item >= first && item < first + nt * (SPREAD ? 1 : C));
        if (hit) {
            const int src = __builtin_amdgcn_readfirstlane(__ffsll((long long)hit) - 1);
            int row = item - __builtin_amdgcn_readlane(first, src);
            if constexpr (!SPREAD) in_bands(row, __builtin_amdgcn_readlane(nt, src), row);
            r0 = __builtin_amdgcn_readlane(b, src) + row * TM;
            r_end = __builtin_amdgcn_readlane(en, src);
            expert = base + src;
            if (alone) *alone = __builtin_amdgcn_readlane(nt, src) == 1;
            return true;
        }
        before += __builtin_amdgcn_readlane(incl, 63);
    }
    return false;
}

// The output column, from the tile's first on, of weight row `row` of a tile (its place in LDS).  A wave multiplies the weight rows as the
// left operand, so a lane holds columns 4*(lane/16)+r of a block of 16 and row lane%16: four columns of one row, 16 bytes of float32.  Where C is
// bfloat16 (PAIRED) two blocks' rows are dealt out so that a lane's two fours lie side by side: eight columns, 16 bytes again.  (With two matrices the
// blocks of 16 take turns between them, and two blocks of one matrix go together.)
template <int NT, bool DUAL, bool PAIRED>
__device__ __forceinline__ int wide_column(int row) {
    constexpr int NC = DUAL ? NT / 2 : NT;          // blocks of 16 columns a wave has
    const int wn = row / (16 * NT), s = row % (16 * NT), j = DUAL ? s >> 5 : s >> 4, i = s & 15;
    return wn * 16 * NC + (PAIRED && j < (NC & ~1) ? (j >> 1) * 32 + (i >> 2) * 8 + (j & 1) * 4 + (i & 3) : j * 16 + i);
}

// N values to C[at .. at + N), as far as they are columns below `left`.  Whole runs are one store (float32: one a 16 bytes) wherever the row begins, for global accesses need no
// more alignment than an element's here; rows of bfloat16 that begin between two words take three, words in the middle (one store there: 4,096 rows against 2,049 weight rows of 2,048 k
// 51 us, three 44).  A store an element touched 64 places with two bytes each: 62 us there, 2,048 rows against 50,257 532 us, now 388.
typedef f32x4_t f32x4_any_t __attribute__((aligned(4)));
template <int N, typename T>
__device__ __forceinline__ void store_columns(T* to, const float (&v)[N], int left) {
    if (left >= N) {
        if constexpr (sizeof(T) == 4) {
            if constexpr (N % 4 == 0) {
#pragma unroll
                for (int r = 0; r < N; r += 4) *(f32x4_any_t*)(to + r) = (f32x4_t){v[r], v[r + 1], v[r + 2], v[r + 3]};
            } else {
                typedef __attribute__((ext_vector_type(N))) float run_t;
                typedef run_t run_any_t __attribute__((aligned(4)));
                run_t p;
#pragma unroll
                for (int r = 0; r < N; ++r) p[r] = v[r];
                *(run_any_t*)to = p;
            }
        } else {
            typedef __attribute__((ext_vector_type(N / 2))) uint32_t packed_t;
            typedef packed_t packed_any_t __attribute__((aligned(2)));
            packed_t p;
#pragma unroll
            for (int r = 0; r < N; r += 2) p[r / 2] = pack_bf16(v[r], v[r + 1]);
            if constexpr (N >= 4) {
                if ((uintptr_t)to & 2) {
                    typedef __attribute__((ext_vector_type(N / 2 - 1))) uint32_t inner_t;
                    typedef inner_t inner_any_t __attribute__((aligned(4)));
                    inner_t in;
#pragma unroll
                    for (int r = 0; r < N / 2 - 1; ++r) in[r] = __builtin_amdgcn_alignbit(p[r + 1], p[r], 16);
                    to[0].bits = (uint16_t)p[0];
                    *(inner_any_t*)(to + 1) = in;
                    to[N - 1].bits = (uint16_t)(p[N / 2 - 1] >> 16);
                    return;
                }
            }
            *(packed_any_t*)to = p;
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < N; ++r)
        if (r < left) from_float(to + r, v[r]);
}

// What the accumulators of a wave go through on their way to C: MT row blocks (2i + wm of the tile's), NT blocks of columns.  A lane's
// row of a block is one, so its place, its scale and what is added to are few loads, and eight (or four) columns go out in
// one store.  A tile's fixed time, launch to last store, is what a short K pays: with a lane's four rows of one column (stores of two or four bytes, a
// load a row and column) and a division per gate, one round of tiles at 256 k took, us: 256 x 256 bfloat16 20.8 now 16.3, float32 20.7 20.1, added 41 30.8,
// gated 27.2 19.0; 192 x 256 gated 20.2 15.0; 128 x 128 added 12.4 10.2; at 2,048 k 63 58.5, 65 62.7, 80 72.8, 67.5 59.1; 52.5 48.8; 28.8 24.9.
template <int MT, int NT, int TM, int WN, bool DUAL, int EPI>
__device__ __forceinline__ void wide_epilogue(const GemmArgs& g, f32x4_t (&acc)[MT][NT], int r0, int r_end, int n0, int wm, int wn) {
    constexpr bool PAIRED = EPI == EPI_STORE || EPI == EPI_GATED;
    constexpr int NC = DUAL ? NT / 2 : NT, PAIRS = PAIRED ? NC / 2 : 0, RUNS = NC - PAIRS;     // runs of 8 columns, then of 4
    // (counted again, so that nothing of it is kept in registers through the loop)
    int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(lane));
    wm = __builtin_amdgcn_readfirstlane(wm);
    wn = __builtin_amdgcn_readfirstlane(wn);
    const int last = min(r_end, r0 + TM), q = lane >> 4;
    // Where each of this lane's rows goes (and its scale) is fetched for all rows at once: a load inside the loops below
    // would be waited for before the next leaves.
    int m_of[MT];
    float scale_of[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int ml = r0 + (2 * i + wm) * 16 + (lane & 15), safe = ml < last ? ml : r0;
        m_of[i] = g.c_rows ? g.c_rows[safe] : safe;
        scale_of[i] = (EPI == EPI_RESID && g.row_scale) ? g.row_scale[safe] : (DUAL ? FX_PRE_SCALE(g, safe) : 1.f);
    }
    // run u's first column
    auto column = [&](int u) { return n0 + wn * 16 * NC + (u < PAIRS ? u * 32 + q * 8 : (u + PAIRS) * 16 + q * 4); };
    // f(run, its number of columns, the first of its blocks of columns)
    auto each_run = [&](auto&& f) {
        static_for(std::make_integer_sequence<int, RUNS>{}, [&](auto uc) {
            constexpr int u = decltype(uc)::value;
            f(uc, fx_int<(u < PAIRS ? 8 : 4)>{}, fx_int<(u < PAIRS ? 2 * u : u + PAIRS)>{});
        });
    };
    if constexpr (DUAL) {
        with_activation(g.act, [&](auto ac) {
            static_for(std::make_integer_sequence<int, MT>{}, [&](auto ic) {
                constexpr int i = decltype(ic)::value;
                const int first = r0 + (2 * i + wm) * 16;
                __builtin_amdgcn_sched_barrier(0);
                if (first >= last) return;
                bf16* to = (bf16*)g.C + (size_t)m_of[i] * g.ldc;
                const float ps = scale_of[i];
                each_run([&](auto uc, auto cc, auto bc) {
                    constexpr int u = decltype(uc)::value, N = decltype(cc)::value, b = decltype(bc)::value;
                    float y[N];
                    if constexpr (decltype(ac)::value == ACT_SILU) {
#pragma unroll
                        for (int r = 0; r < N; ++r) y[r] = acc[i][2 * (b + r / 4)][r & 3] * ps;
                        silu_n(y);
#pragma unroll
                        for (int r = 0; r < N; ++r) y[r] *= acc[i][2 * (b + r / 4) + 1][r & 3] * ps;
                    } else {
#pragma unroll
                        for (int r = 0; r < N; ++r)
                            y[r] = gated_c<decltype(ac)::value>(acc[i][2 * (b + r / 4)][r & 3] * ps, acc[i][2 * (b + r / 4) + 1][r & 3] * ps, g.act_limit, g.act_alpha);
                    }
                    const int n = column(u);
                    if (first + (lane & 15) < last) store_columns<N>(to + n, y, g.N - n);
                });
            });
        });
        return;
    }
    float bias_v[NT * 4];
    if (g.bias) {
        each_run([&](auto uc, auto cc, auto bc) {
            constexpr int u = decltype(uc)::value, N = decltype(cc)::value, b = decltype(bc)::value;
            float w[N];
            load_strided_as_float<N, 1>(g.bias, g.bias_dtype, column(u), g.N, w);
#pragma unroll
            for (int r = 0; r < N; ++r) bias_v[4 * b + r] = w[r];
        });
    }
    // What a row block adds to is on its way while the blocks before it are added and stored.
    constexpr int AHEAD = 2;
    float old[EPI == EPI_RESID ? MT : 1][NT * 4];
    auto fetch_old = [&](int i) {
        if constexpr (EPI == EPI_RESID) {
            const float* from = (const float*)g.C + (size_t)m_of[i] * g.ldc;
            each_run([&](auto uc, auto cc, auto bc) {
                constexpr int u = decltype(uc)::value, N = decltype(cc)::value, b = decltype(bc)::value;
                const int n = column(u);
                if (n + N <= g.N) {
#pragma unroll
                    for (int r = 0; r < N; r += 4) {
                        const f32x4_t v = *(const f32x4_any_t*)(from + n + r);
#pragma unroll
                        for (int t = 0; t < 4; ++t) old[i][4 * b + r + t] = v[t];
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < N; ++r) old[i][4 * b + r] = from[min(n + r, g.N - 1)];
                }
            });
        }
    };
    if constexpr (EPI == EPI_RESID) {
#pragma unroll
        for (int i = 0; i < AHEAD && i < MT; ++i) fetch_old(i);
    }
    with_stored<EPI == EPI_STORE || EPI == EPI_STORE_F32>(g.store_act, [&](auto kind) {
        static_for(std::make_integer_sequence<int, MT>{}, [&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const int first = r0 + (2 * i + wm) * 16;
            __builtin_amdgcn_sched_barrier(0);
            if (first >= last) return;
            if constexpr (EPI == EPI_RESID && i + AHEAD < MT) fetch_old(i + AHEAD);
            const int m = m_of[i];
            float gates[NT * 4] = {};      // (the gates' logits of a row block, fetched together)
            if (decltype(kind)::value == SACT_GATE) {
                each_run([&](auto uc, auto cc, auto bc) {
                    constexpr int u = decltype(uc)::value, N = decltype(cc)::value, b = decltype(bc)::value;
#pragma unroll
                    for (int r = 0; r < N; ++r) gates[4 * b + r] = gate_of(g, m, min(column(u) + r, g.N - 1));
                });
            }
            each_run([&](auto uc, auto cc, auto bc) {
                constexpr int u = decltype(uc)::value, N = decltype(cc)::value, b = decltype(bc)::value;
                const int n = column(u);
                float y[N];
#pragma unroll
                for (int r = 0; r < N; ++r) {
                    float v = acc[i][b + r / 4][r & 3];
                    if (g.bias) v += bias_v[4 * b + r];
                    if constexpr (EPI == EPI_RESID) {
                        if (g.row_scale) {
                            v *= scale_of[i];
                            asm volatile("" : "+v"(v));      // rounded before it is added (no fused multiply-add)
                        }
                        y[r] = old[i][4 * b + r] + v;
                    } else {
                        y[r] = stored_c<decltype(kind)::value>(g, v, gates[4 * b + r]);
                    }
                }
                if (first + (lane & 15) < last) {
                    if constexpr (EPI == EPI_STORE) store_columns<N>((bf16*)g.C + (size_t)m * g.ldc + n, y, g.N - n);
                    else store_columns<N>((float*)g.C + (size_t)m * g.ldc + n, y, g.N - n);
                }
            });
        });
    });
}

template <int TMB, int TN, int NS, bool DUAL, int EPI, int NSA, bool STREAM>
__device__ __forceinline__ void wide_block(const GemmArgs& g, bf16* stages, int r0, int r_end, int expert, int col_tile) {
    constexpr int TM = TMB * 16;
    constexpr int MT = TMB / 2;            // row blocks per wave
    constexpr int NT = TN / 64;            // 16-row blocks of W per wave
    constexpr int WN = TN / 4;
    constexpr int OUT_TN = DUAL ? TN / 2 : TN;
    constexpr int NLA = TM / 64, NLB = TN / 64;   // wave-loads (8 rows each) per wave and K step
    static_assert(TM % 64 == 0 && TN % 64 == 0, "eight waves load 64 rows at a time");
    const int n0 = col_tile * OUT_TN;
    const int rows_here = min(TM, r_end - r0);
    const int nblk = (rows_here + 15) >> 4;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // waves w and w + 4 share a SIMD: one of each half of the rows, so that a tile with few rows loads the SIMDs evenly
    const int wm = wave >> 2, wn = wave & 3;
    const bf16* Wbase = (const bf16*)g.W + (size_t)expert * g.w_stride;

    // what this lane fetches in each of its wave-loads: row 8*j + lane/8 of the tile, chunk (lane%8) ^ ((row/2)%8)
    const bf16* a_src[NLA];
    const bf16* b_src[NLB];
#pragma unroll
    for (int i = 0; i < NLA; ++i) {
        const int j = wave + 8 * i, row = 8 * j + (lane >> 3);
        const int chunk = (lane & 7) ^ (4 * (j & 1) + (lane >> 4));
        const int m = r0 + min(row, rows_here - 1);          // rows past the end repeat the last one, unused
        a_src[i] = (const bf16*)g.A + (size_t)(g.a_rows ? g.a_rows[m] : m) * g.lda + chunk * 8;
    }
#pragma unroll
    for (int i = 0; i < NLB; ++i) {
        const int j = wave + 8 * i, row = 8 * j + (lane >> 3);
        const int chunk = (lane & 7) ^ (4 * (j & 1) + (lane >> 4));
        const int col = min(n0 + wide_column<NT, DUAL, EPI == EPI_STORE || EPI == EPI_GATED>(row), g.N - 1);
        const bool up = DUAL && ((row >> 4) & 1);
        b_src[i] = g.kb_stride ? Wbase + ((size_t)col + (up ? g.up_offset / g.K : 0)) * 64 + chunk * 8
                               : Wbase + (size_t)col * g.K + (up ? g.up_offset : 0) + chunk * 8;
    }

    f32x4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

    const int sw = (lane & 15) >> 1, kq = lane >> 4;
    const int a_off = (wm * 16 + (lane & 15)) * 64, b_off = (wn * WN + (lane & 15)) * 64;
    const int na = (nblk - wm + 1) >> 1;         // this wave's active row blocks
#define FX_LOOP(NA) \
    wide_k_loop<NA, MT, NT, TM, TN, NSA, NS, STREAM>(acc, a_src, b_src, stages, g.K, wave, a_off, b_off, sw, kq, g.kb_stride)
    if constexpr (MT >= 4) {
        if (na > 3 * MT / 4) FX_LOOP(MT);
        else if (na > MT / 2) FX_LOOP(3 * MT / 4);
        else if (na > MT / 4) FX_LOOP(MT / 2);
        else FX_LOOP(MT / 4);
    } else {
        if (na > MT / 2) FX_LOOP(MT);
        else FX_LOOP((MT + 1) / 2);
    }
#undef FX_LOOP

    wide_epilogue<MT, NT, TM, WN, DUAL, EPI>(g, acc, r0, r_end, n0, wm, wn);
}

template <int TMB, int TN, int NS, bool DUAL, int EPI, int NSA = NS, bool STREAM = false, bool SPREAD = false>
__global__ __launch_bounds__(512) void gemm_bf16_wide_kernel(GemmArgs g) {
    __shared__ __attribute__((aligned(1024))) bf16 stages[(NSA * 16 * TMB + NS * TN) * 64];    // the rows' ring, then the weights'
    int r0, r_end, expert, col_tile;
    if (!wide_tile<16 * TMB, SPREAD>(g, r0, r_end, expert, col_tile)) return;
    wide_block<TMB, TN, NS, DUAL, EPI, NSA, STREAM>(g, stages, r0, r_end, expert, col_tile);
}

// ---------------------------------------------------------------------------
// Tiles in quarters, the products of prompts: the same blocks, tiles, waves and swizzled LDS rows as above, with two
// stages only, but a step of 64 k is four phases, and the rows and the weights of a stage are two parts each, so that
// a part is refilled for the step after the next as soon as every wave has read it.  Phase by phase a wave
// multiplies part 0 of its rows with the step's first weights, then with its second, then part 1 of its rows with the second and
// with the first; while it does, it reads from LDS what the next phases multiply, one operand between every few products:
//     products              reads (this step's, ' the next one's)       refilled, for the step after the next
//  1  rows 0 x first        second weights, rows 1 (first 32 k)         -
//  2  rows 0 x second       rows 1 (second 32 k)                        rows 0, first weights
//  3  rows 1 x second       rows 0' (first 32 k)                        second weights
//  4  rows 1 x first        first weights', rows 0' (second 32 k)       rows 1
// The next step's first weights are read into the registers of this step's second ones, which phase 4 no longer
// needs, so first and second change places every step and 96 registers of operands suffice beside the 128 sums.
// Barriers stand in front of phases 2, 3 and 4: what a phase refills every wave has read (it is multiplied, so waited for,
// before the barrier), and what phases 3, 4 and 1' read has landed for every wave that waited in front of it.
// A step's stage is the number of its first weights, so every address in LDS is a register of before the loop and a constant: with the
// stage worked out from the step's number, tiles of 256 x 256 spilled up to 72 bytes a lane.
// The loop waits for loads a whole step old and never for the youngest, where the ring of two stages waited for all of them
// every step: 8,192 x 8,192 x 8,192 878 -> 758 us (1,252 -> 1,450 TFLOP/s), 4,096 rows against 40,960 weight rows of 3,584 k
// 1,047 -> 883 us, against 3,584 of 20,480 k 505 -> 432 us.  Neither a fourth barrier, nor the priority of waves that multiply, nor waves
// of a SIMD taking turns (one group reads while the other multiplies, 786 us) is any better.  An element's products are
// added in the order of k, as in every bf16 tile: the same bits.
// ---------------------------------------------------------------------------
// 16 bytes a lane from a base that all lanes share, `offset` bytes on, into 1 KB of LDS.
__device__ __forceinline__ void load_lds16(const bf16* base, unsigned offset, bf16* to) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host's pass does not know the descriptor's type)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)base, 0, -1, 0x00027000), (fx_lds_ptr)to, 16, offset, 0, 0, 0);
#endif
}

// The K loop of one wave.  MA0, MA1: its row blocks in part 0 and 1 of the tile; NA0, NA1: those of them that exist.
// NB0, NB1: its blocks of 16 weight rows in part 0 and 1.  a_src and b_base move along with the loads.
template <int NA0, int NA1, int MA0, int MA1, int NB0, int NB1>
__device__ __forceinline__ void quarters_k_loop(f32x4_t (&acc)[MA0 + MA1][NB0 + NB1], const bf16* (&a_src)[(MA0 + MA1) / 2],
                                                const bf16* (&b_base)[2], const unsigned (&b_off)[NB0 + NB1], bf16* lds, int K,
                                                int wave, int wm, int wn, int lane, long kb_stride) {
    constexpr int LA0 = MA0 / 2, LA1 = MA1 / 2, TM = 32 * (MA0 + MA1), TN = 64 * (NB0 + NB1);
    const int nk = K >> 6;
    const long b_step = kb_stride ? kb_stride : 64;
    // wave-loads FROM .. TO-1 of a step's rows or weights, steps in turn.  (The empty asm keeps the compiler from
    // holding every address twice; the weights' are 32 bits beside a base that all lanes share.  With 64 bits each
    // some of them lived in scratch memory, and the loop waited for those loads.)
    auto load_a = [&](auto from, auto to, int stage) {
        bf16* st = lds + stage * (TM * 64);
#pragma unroll
        for (int i = decltype(from)::value; i < decltype(to)::value; ++i) {
            __builtin_amdgcn_global_load_lds((fx_global_ptr)a_src[i], (fx_lds_ptr)(st + (wave + 8 * i) * 512), 16, 0, 0);
            a_src[i] += 64;
            asm volatile("" : "+v"(a_src[i]));
        }
    };
    auto load_b = [&](auto from, auto to, auto part, int stage) {
        bf16* st = lds + 2 * TM * 64 + stage * (TN * 64);
#pragma unroll
        for (int i = decltype(from)::value; i < decltype(to)::value; ++i)
            load_lds16(b_base[decltype(part)::value], b_off[i], st + (wave + 8 * i) * 512);
        b_base[decltype(part)::value] += b_step;
    };
    auto load_rows = [&](auto part, int stage) {
        if constexpr (decltype(part)::value == 0) load_a(fx_int<0>{}, fx_int<LA0>{}, stage);
        else load_a(fx_int<LA0>{}, fx_int<LA0 + LA1>{}, stage);
    };
    auto load_weights = [&](auto part, int stage) {
        if constexpr (decltype(part)::value == 0) load_b(fx_int<0>{}, fx_int<NB0>{}, part, stage);
        else load_b(fx_int<NB0>{}, fx_int<NB0 + NB1>{}, part, stage);
    };

    const int sw = (lane & 15) >> 1, kq = lane >> 4;
    const int koff[2] = {(kq ^ sw) * 8, ((4 + kq) ^ sw) * 8};
    const int a_off = (wm * 16 + (lane & 15)) * 64;
    const int b_at[2] = {2 * TM * 64 + (wn * 16 * NB0 + (lane & 15)) * 64, 2 * TM * 64 + (64 * NB0 + wn * 16 * NB1 + (lane & 15)) * 64};
    constexpr int NBX = NB0 > NB1 ? NB0 : NB1;
    bf16x8_t a[2][MA0][2], b[2][NBX][2];
    // operand u of a part's rows (the existing blocks' first 32 k, then their second) and of a part's weights
    auto read_rows = [&](auto part, auto uc, int stage) {
        constexpr int h = decltype(part)::value, u = decltype(uc)::value, na = h ? NA1 : NA0, kk = u / na, i = u % na;
        a[h][i][kk] = *(const bf16x8_t*)(lds + a_off + koff[kk] + stage * (TM * 64) + (h * MA0 + i) * 32 * 64);
    };
    auto read_weights = [&](auto part, auto uc, int stage) {
        constexpr int h = decltype(part)::value, u = decltype(uc)::value, nb = h ? NB1 : NB0, kk = u / nb, j = u % nb;
        b[h][j][kk] = *(const bf16x8_t*)(lds + b_at[h] + koff[kk] + stage * (TN * 64) + j * 16 * 64);
    };
    // a phase: the products of a part of the rows with a part of the weights, R reads spread over them
    auto phase = [&](auto rows, auto weights, auto reads, auto&& read) {
        constexpr int h = decltype(rows)::value, w = decltype(weights)::value, R = decltype(reads)::value;
        constexpr int na = h ? NA1 : NA0, nb = w ? NB1 : NB0, P = 2 * na * nb;
        if constexpr (P == 0) {
            static_for(std::make_integer_sequence<int, R>{}, read);
        } else {
            static_for(std::make_integer_sequence<int, P>{}, [&](auto qc) {
                constexpr int q = decltype(qc)::value, u0 = (q * R + P - 1) / P, u1 = ((q + 1) * R + P - 1) / P;
                if constexpr (u1 > u0) {
                    __builtin_amdgcn_sched_barrier(0);
                    static_for(std::make_integer_sequence<int, u1 - u0>{}, [&](auto uc) { read(fx_int<u0 + decltype(uc)::value>{}); });
                    __builtin_amdgcn_sched_barrier(0);
                }
                constexpr int kk = q / (na * nb), i = q / nb % na, j = q % nb;
                acc[h * MA0 + i][w * NB0 + j] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[w][j][kk], a[h][i][kk], acc[h * MA0 + i][w * NB0 + j], 0, 0, 0);
            });
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto barrier = [] {
        asm volatile("" ::: "memory");       // (the barrier alone does not keep reads of LDS on their side of it)
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
    };
    // one step; left: the steps behind it, as far as that matters (0, 1, or 2 for more).  Its stage is the number of its first weights.
    auto step = [&](auto first, auto left) {
        constexpr int f = decltype(first)::value, s = 1 - f, nb_s = s ? NB1 : NB0;
        constexpr bool next = decltype(left)::value > 0, refill = decltype(left)::value > 1;
        phase(fx_int<0>{}, fx_int<f>{}, fx_int<2 * nb_s + NA1>{}, [&](auto uc) {
            constexpr int u = decltype(uc)::value;
            if constexpr (u < 2 * nb_s) read_weights(fx_int<s>{}, uc, f);
            else read_rows(fx_int<1>{}, fx_int<u - 2 * nb_s>{}, f);
        });
        if constexpr (refill) {
            barrier();
            load_rows(fx_int<0>{}, f);
            load_weights(fx_int<f>{}, f);
        }
        phase(fx_int<0>{}, fx_int<s>{}, fx_int<NA1>{}, [&](auto uc) { read_rows(fx_int<1>{}, fx_int<decltype(uc)::value + NA1>{}, f); });
        if constexpr (next) {
            // rows 0 of the next step have landed: behind them may be its weights, its rows 1 and what phase 2 has asked for
            wait_loads_but<refill ? NB0 + NB1 + LA1 + LA0 + (f ? NB1 : NB0) : 0>();
            barrier();
        }
        if constexpr (refill) load_weights(fx_int<s>{}, f);
        phase(fx_int<1>{}, fx_int<s>{}, fx_int<next ? NA0 : 0>{}, [&](auto uc) { read_rows(fx_int<0>{}, uc, s); });
        if constexpr (refill) {
            wait_loads_but<LA0 + NB0 + NB1>();     // all of the next step has
            barrier();
            load_rows(fx_int<1>{}, f);
        }
        phase(fx_int<1>{}, fx_int<f>{}, fx_int<next ? 2 * nb_s + NA0 : 0>{}, [&](auto uc) {
            constexpr int u = decltype(uc)::value;
            if constexpr (u < 2 * nb_s) read_weights(fx_int<s>{}, uc, s);
            else read_rows(fx_int<0>{}, fx_int<u - 2 * nb_s + NA0>{}, s);
        });
    };

    // The last step's first weights are part 1 and its stage is 1, so the first step's are where the steps are an odd number.  The loads
    // go out in the order in which the loop waits for them.
    const int odd = nk & 1;
    load_rows(fx_int<0>{}, odd);
    load_weights(fx_int<0>{}, odd);
    load_weights(fx_int<1>{}, odd);
    load_rows(fx_int<1>{}, odd);
    if (nk > 1) {
        load_rows(fx_int<0>{}, odd ^ 1);
        load_weights(fx_int<0>{}, odd ^ 1);
        load_weights(fx_int<1>{}, odd ^ 1);
        load_rows(fx_int<1>{}, odd ^ 1);
        wait_loads_but<LA0 + NB0 + NB1 + LA1>();
    } else {
        wait_loads_but<0>();
    }
    barrier();
    int kt = 0;
    if (odd) {
        static_for(std::make_integer_sequence<int, 2 * NA0>{}, [&](auto uc) { read_rows(fx_int<0>{}, uc, 1); });
        static_for(std::make_integer_sequence<int, 2 * NB1>{}, [&](auto uc) { read_weights(fx_int<1>{}, uc, 1); });
        if (nk > 1) {
            step(fx_int<1>{}, fx_int<2>{});
            ++kt;
        }
    } else {
        static_for(std::make_integer_sequence<int, 2 * NA0>{}, [&](auto uc) { read_rows(fx_int<0>{}, uc, 0); });
        static_for(std::make_integer_sequence<int, 2 * NB0>{}, [&](auto uc) { read_weights(fx_int<0>{}, uc, 0); });
    }
    for (; kt + 2 < nk; kt += 2) {
        step(fx_int<0>{}, fx_int<2>{});
        step(fx_int<1>{}, fx_int<2>{});
    }
    if (nk > 1) step(fx_int<0>{}, fx_int<1>{});
    step(fx_int<1>{}, fx_int<0>{});
}

template <int TMB, int TN, bool DUAL, int EPI>
__device__ __forceinline__ void quarters_block(const GemmArgs& g, bf16* stages, int r0, int r_end, int expert, int col_tile) {
    constexpr int TM = TMB * 16, MT = TMB / 2, NT = TN / 64, WN = TN / 4, OUT_TN = DUAL ? TN / 2 : TN;
    constexpr int MA0 = MT > 4 ? 4 : MT / 2, MA1 = MT - MA0, NB0 = (NT + 1) / 2, NB1 = NT - NB0;
    constexpr int NLA = TM / 64, NLB = TN / 64;   // wave-loads (8 rows each) per wave and K step
    static_assert(MA0 % 2 == 0 && MA1 % 2 == 0 && MA1 > 0 && NB1 > 0, "eight waves load 64 rows at a time, a part at a time");
    const int n0 = col_tile * OUT_TN;
    const int rows_here = min(TM, r_end - r0);
    const int nblk = (rows_here + 15) >> 4;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3;
    const bf16* Wbase = (const bf16*)g.W + (size_t)expert * g.w_stride;

    const bf16* a_src[NLA];
#pragma unroll
    for (int i = 0; i < NLA; ++i) {
        const int j = wave + 8 * i, row = 8 * j + (lane >> 3);
        const int chunk = (lane & 7) ^ (4 * (j & 1) + (lane >> 4));
        const int m = r0 + min(row, rows_here - 1);          // rows past the end repeat the last one, unused
        a_src[i] = (const bf16*)g.A + (size_t)(g.a_rows ? g.a_rows[m] : m) * g.lda + chunk * 8;
    }
    // part 0 of the weights holds the first 16*NB0 of every wave's weight rows, part 1 the others; all that a wave loads of a
    // part are rows of one matrix where there are two (their blocks of 16 take turns)
    const bf16* b_base[2];
    unsigned b_off[NLB];
    const long ldw = g.kb_stride ? 64 : g.K;
#pragma unroll
    for (int i = 0; i < NLB; ++i) {
        const int j = wave + 8 * i, x = 8 * j + (lane >> 3);
        const int chunk = (lane & 7) ^ (4 * (j & 1) + (lane >> 4));
        const int row = i < NB0 ? x / (16 * NB0) * WN + x % (16 * NB0)
                                : (x - 64 * NB0) / (16 * NB1) * WN + 16 * NB0 + (x - 64 * NB0) % (16 * NB1);
        const int col = min(n0 + wide_column<NT, DUAL, EPI == EPI_STORE || EPI == EPI_GATED>(row), g.N - 1);
        b_off[i] = (unsigned)((col - n0) * ldw + chunk * 8) * 2;
        if (i == 0 || i == NB0) {
            const bool up = DUAL && __builtin_amdgcn_readfirstlane((row >> 4) & 1);
            b_base[i != 0] = Wbase + n0 * ldw + (up ? (g.kb_stride ? g.up_offset / g.K * 64 : g.up_offset) : 0);
        }
    }

    f32x4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

    const int na = (nblk - wm + 1) >> 1;         // this wave's row blocks that exist
#define FX_LOOP(NA0_, NA1_) quarters_k_loop<NA0_, NA1_, MA0, MA1, NB0, NB1>(acc, a_src, b_base, b_off, stages, g.K, wave, wm, wn, lane, g.kb_stride)
    if (na > MA0 + MA1 / 2) FX_LOOP(MA0, MA1);
    else if (na > MA0) FX_LOOP(MA0, MA1 / 2);
    else if (na > MA0 / 2) FX_LOOP(MA0, 0);
    else FX_LOOP(MA0 / 2, 0);
#undef FX_LOOP
    wide_epilogue<MT, NT, TM, WN, DUAL, EPI>(g, acc, r0, r_end, n0, wm, wn);
}

template <int TMB, int TN, bool DUAL, int EPI>
__global__ __launch_bounds__(512) void gemm_bf16_quarters_kernel(GemmArgs g) {
    __shared__ __attribute__((aligned(1024))) bf16 stages[2 * (16 * TMB + TN) * 64];
    int r0, r_end, expert, col_tile;
    if (!wide_tile<16 * TMB>(g, r0, r_end, expert, col_tile)) return;
    quarters_block<TMB, TN, DUAL, EPI>(g, stages, r0, r_end, expert, col_tile);
}

// Rows sorted by expert, tiles of 128 x 256, the loop by the expert's own share: one tile of rows reads its weights about once, so the ring with
// the non-temporal hint streams them; an expert of more rows takes the tiles in quarters, whose weights its other tiles find in the cache.  Either
// adds an element's products in the order of k.  Both products, us, even shares / crowded into half of the experts: tiles of 192 rows in a ring, these tiles in
// quarters whatever the share, and by the share (60 experts of 1,408, then 64 of 2,560):
//   560 tokens 194 137, 201 130, 189 128    700 203 160, 207 133, 198 139    1,000 214 181, 218 142, 211 140    1,400 235 217, 234 170, 229 171
//   300 tokens 590 420, 601 340, 579 315    400 611 455, 614 401, 597 377    600 642 525, 642 460, 627 460
// (One hot expert among many, 300 of the larger: 590, 663 and 620.)
// (With four stages of weights, all of LDS, 1 to 2 % more.)
template <int TMB, int TN, int NS, bool DUAL, int EPI, bool SPREAD>
__global__ __launch_bounds__(512) void gemm_bf16_shares_kernel(GemmArgs g) {
    constexpr int RING = 2 * 16 * TMB + NS * TN, QUARTERS = 2 * (16 * TMB + TN);
    __shared__ __attribute__((aligned(1024))) bf16 stages[(RING > QUARTERS ? RING : QUARTERS) * 64];
    int r0, r_end, expert, col_tile;
    bool alone;
    if (!wide_tile<16 * TMB, SPREAD>(g, r0, r_end, expert, col_tile, &alone)) return;
    if (alone) wide_block<TMB, TN, NS, DUAL, EPI, 2, true>(g, stages, r0, r_end, expert, col_tile);
    else quarters_block<TMB, TN, DUAL, EPI>(g, stages, r0, r_end, expert, col_tile);
}

// ---------------------------------------------------------------------------
// Few rows (decode): the weights are streamed once from memory straight into
// MFMA operands, no LDS staging.  A block owns NW sets of 16 rows of W and up
// to 16*MT logical rows; its WAVES waves split K between them in pieces of 128
// (with few accumulators, the next piece's loads are issued before this piece's
// products) and their partial sums are added in wave order through LDS.  A
// product wants lane (i = lane%16, g = lane/16) to hold 16 bytes (k 8g..8g+7 of
// every 32) of W row n0+i; they arrive in whole 128-byte lines, two loads and an
// exchange between lanes per 64 k (see `load_lines16`).  The activations use the
// same k -> lane assignment, which is all the MFMA needs to be right.
// W is the A operand: the accumulator of lane (m = lane%16, g) holds
// C[m][n0 + 4g + r], r = 0..3.
// ---------------------------------------------------------------------------
// rsqrt(mean of squares + eps) of a row from the sum of its squares.  Division and sqrtf are the correctly
// rounded ones (the compiler's default for HIP; __fsqrt_rn is NOT: it is the approximate instruction, whose
// result the compiler refines in some kernels and not in others), so every epilogue that scales its rows
// gets the same bits.
__device__ __forceinline__ float row_rstd(float total, int K, float eps) {
    const float mean = total / (float)K;
    return 1.0f / sqrtf(mean + eps);
}

// p[0] + p[1] + ... in that order; eight loads leave together (a plain loop would wait for each in turn)
__device__ __forceinline__ float sum_in_order(const float* p, int n) {
    float total = 0.f;
    for (int b0 = 0; b0 < n; b0 += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = p[min(b0 + u, n - 1)];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (b0 + u < n) total += v[u];
    }
    return total;
}

// NORM: the rows of A are float32 and are normed on the way in, y = x * rsqrt(mean(x^2) + eps) * w
// (ferrox-core/src/matmul.rs:62-69): x * w is rounded to bfloat16 and multiplied, the sums of
// squares that the waves gather over their parts of K are added up, and the product is scaled by
// the row's rsqrt before the bias is added.
__device__ __forceinline__ void load8f(const float* p, bool ok, float* v) {
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
    if (ok) {
        a = *(const float4*)p;
        b = *(const float4*)(p + 4);
    }
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// The weights come in whole lines with the non-temporal hint (`load_lines16`, `swap_halves`).  Measured at 8
// tokens of the A2.7B sizes against 16-byte loads of half lines: the experts' gate/up product 69.1 -> 64.4 us, their
// down product 36.6 -> 32.7 us, the head 132 -> 101 us (4.7 -> 6.2 TB/s).
// NW: sets of 16 weight rows per wave; in dual mode set a is the gate (a even) or up (a odd) rows of
// column group a / 2.
// TURN: some outputs of each head are turned in pairs of neighbours (see GemmArgs).
template <int MT, int WAVES, int NW, bool DUAL, int EPI, bool NORM, bool ROPE, bool HALF, int DEPTH, bool WEIGHTS_FIRST, bool TURN>
__device__ __forceinline__ void skinny_block(const GemmArgs& g, const unsigned block_x, const unsigned block_y) {
    static_assert(!TURN || (EPI == EPI_STORE && MT == 1 && !NORM && !ROPE), "turned outputs are a few plain stored rows");
    static_assert(!HALF || (MT == 1 && WAVES == 4 && !NORM && !ROPE), "sets of eight weight rows are for few plain rows");
    constexpr int CW = HALF ? 8 : 16;               // weight rows of a set, output columns of a tile
    static_assert(!DUAL || NW % 2 == 0, "dual mode multiplies two matrices");
    static_assert(!ROPE || (NW == 2 && !DUAL && !NORM && EPI == EPI_STORE), "the rope epilogue pairs two sets of columns");
    static_assert(!NORM || (!DUAL && EPI == EPI_STORE), "the fused norm feeds a plain product");
    static_assert(!WEIGHTS_FIRST || (ROPE && MT == 1), "only the rope epilogue's operands of one row tile have an order to choose");
    __shared__ float red_ss[NORM ? WAVES : 1][MT][64];
    float ss[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) ss[mt] = 0.f;
    constexpr int NACC = MT * NW;
    constexpr int COLS = (DUAL ? CW / 2 : CW) * NW;   // output columns of a block
    // K is cut into PARTS parts whose sums are added in their order: one part per wave, or, with fewer than four
    // waves, VW consecutive parts per wave with accumulators of their own, so that one, two and four waves give
    // the same bits
    constexpr int VW = WAVES < 4 ? 4 / WAVES : 1, PARTS = WAVES * VW;
    __shared__ f32x4_t red[PARTS][NACC][64];
    int r0 = 0, r_end = 0, expert = 0, pair_a = -1, pair_c = -1;
    const bool pairs = MT == 1 && g.pair_ids != nullptr;
    if (pairs) {
        if (!locate_pairs(g, block_y, expert, pair_a, pair_c)) return;
    } else {
        locate_rows<16 * MT>(g, block_y, r0, r_end, expert);
        if (r0 < 0) return;
    }
    const int n0 = block_x * COLS;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 15, grp = lane >> 4;
    const bf16* Wbase = (const bf16*)g.W + (size_t)expert * g.w_stride;
    // rope epilogue: a block takes 16 + 16 columns of one head, (16 j .. , rot/2 + 16 j ..) while they are rotated,
    // two neighbouring sets of 16 after that
    int rope_head = 0, rope_j = 0, rope_c0 = 0, rope_c1 = 0;
    bool rope_rotated = false;
    if constexpr (ROPE) {
        const int per_head = g.rope_hd >> 5;
        rope_head = block_x / per_head;
        rope_j = block_x - rope_head * per_head;
        const bool is_v = rope_head >= g.rope_nh + g.rope_nkv;
        const int n_rot = is_v ? 0 : g.rope_rot >> 5;          // blocks of this head whose columns are rotated
        rope_rotated = rope_j < n_rot;
        rope_c0 = rope_rotated ? 16 * rope_j : (is_v ? 32 * rope_j : g.rope_rot + 32 * (rope_j - n_rot));
        rope_c1 = rope_rotated ? rope_c0 + (g.rope_rot >> 1) : rope_c0 + 16;
    }
    const bf16* wrow[NW];     // this lane's place in the set's first load, and how far behind it the second is
    int wrow_b[NW];
#pragma unroll
    for (int a = 0; a < NW; ++a) {
        const int n = ROPE ? rope_head * g.rope_hd + (a ? rope_c1 : rope_c0) + li
                           : n0 + (DUAL ? a >> 1 : a) * CW + li;
        const bool up = DUAL && (a & 1);
        // whole lines per load: the lanes of a set's first load take rows li % 8, those of its second (HALF: there is none) rows
        // 8 + li % 8, both k 32 (li / 8) .. of every 64; rows past the end repeat the last one, never stored
        const int nl = n - li + (li & 7);
        const int na = min(nl, g.N - 1), nb = min(nl + 8, g.N - 1);
        const size_t rs = g.kb_stride ? 64 : (size_t)g.K;
        const size_t first = g.kb_stride ? (size_t)(up ? g.up_offset / g.K : 0) * 64 : (size_t)(up ? g.up_offset : 0);
        wrow[a] = Wbase + first + (size_t)na * rs + 32 * (li >> 3);
        wrow_b[a] = (int)((nb - na) * rs);
    }
    const size_t slab = g.kb_stride ? (size_t)g.kb_stride : 64;     // element (row, k) is at row + (k / 64) * slab + k % 64
    const bf16* xrow[MT];       // NORM: float rows, kept under the same name
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = r0 + mt * 16 + li;
        const bool live = pairs ? pair_a >= 0 : m < r_end;
        const size_t off = !live ? 0 : (size_t)(pairs ? pair_a : (g.a_rows ? g.a_rows[m] : m)) * g.lda;
        // a dead row reads the first row of A instead: its products land in rows that are never stored
        xrow[mt] = NORM ? (live ? (const bf16*)((const float*)g.A + off) : nullptr) : (const bf16*)g.A + off;
    }
    f32x4_t acc[VW][MT][NW];
#pragma unroll
    for (int p = 0; p < VW; ++p)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int a = 0; a < NW; ++a) acc[p][mt][a] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

    const int n_super = (g.K + 127) / 128;
    const int per = (n_super + PARTS - 1) / PARTS;      // pieces per part
    const int s_end = min(n_super, (wave + 1) * VW * per);
    constexpr int WL = HALF ? 2 : 4;        // loads of a set's piece
    // One piece: its loads (four per set of weight rows and per row tile), then its products.  FULL: the piece
    // lies inside K, so every load is unconditional and the compiler can count the loads in flight.
    auto load_piece = [&](auto full, int sp, uint4 (&w)[NW][WL], uint4 (&x)[MT][4]) {
        constexpr bool FULL = decltype(full)::value;
        const int kb = sp * 128 + grp * 8;     // load u of this lane: k = kb + 32u .. +7
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int kl = kb + 64 * h;                       // this lane's k without its half: 32 (li / 8) is in wrow
            const bool kin = FULL || kl + 32 * (li >> 3) < g.K;
            const size_t woff = (size_t)(kl >> 6) * slab + (kl & 63);
#pragma unroll
            for (int a = 0; a < NW; ++a) {
                w[a][HALF ? h : 2 * h] = kin ? load_lines16(wrow[a] + woff) : make_uint4(0, 0, 0, 0);
                if constexpr (!HALF) w[a][2 * h + 1] = kin ? load_lines16(wrow[a] + woff + wrow_b[a]) : make_uint4(0, 0, 0, 0);
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = kb + 32 * u;
            const bool kin = FULL || k < g.K;
            if constexpr (NORM) {
                float gv[8];
                if (g.norm_dtype == FX_F32) {
                    load8f((const float*)g.norm_w + k, kin, gv);
                } else {
                    const uint4 gw = kin ? *(const uint4*)((const bf16*)g.norm_w + k) : make_uint4(0, 0, 0, 0);
                    gv[0] = __uint_as_float(gw.x << 16); gv[1] = __uint_as_float(gw.x & 0xffff0000u);
                    gv[2] = __uint_as_float(gw.y << 16); gv[3] = __uint_as_float(gw.y & 0xffff0000u);
                    gv[4] = __uint_as_float(gw.z << 16); gv[5] = __uint_as_float(gw.z & 0xffff0000u);
                    gv[6] = __uint_as_float(gw.w << 16); gv[7] = __uint_as_float(gw.w & 0xffff0000u);
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    float xv[8];
                    load8f((const float*)xrow[mt] + k, kin && xrow[mt], xv);
#pragma unroll
                    for (int i = 0; i < 8; ++i) ss[mt] += xv[i] * xv[i];
                    x[mt][u] = make_uint4(pack_bf16(xv[0] * gv[0], xv[1] * gv[1]), pack_bf16(xv[2] * gv[2], xv[3] * gv[3]),
                                          pack_bf16(xv[4] * gv[4], xv[5] * gv[5]), pack_bf16(xv[6] * gv[6], xv[7] * gv[7]));
                }
            } else {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) x[mt][u] = kin ? *(const uint4*)(xrow[mt] + k) : make_uint4(0, 0, 0, 0);
            }
        }
    };
    auto multiply_into = [&](f32x4_t (&to)[MT][NW], const uint4 (&w)[NW][WL], const uint4 (&x)[MT][4]) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int a = 0; a < NW; ++a) {
                // low k: own first load below lane 8 of a row of 16, the other half's second load above;
                // high k: the other half's first load below, own second load above
                // (HALF: rows 8 .. 15 of the operand are the other k of rows 0 .. 7, and what they give is dropped)
                uint4 wu;
                if constexpr (HALF) wu = (u & 1) ? swap_halves<0x3>(w[a][u / 2], w[a][u / 2]) : w[a][u / 2];
                else wu = (u & 1) ? swap_halves<0x3>(w[a][u], w[a][u - 1]) : swap_halves<0xC>(w[a][u], w[a][u + 1]);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    to[mt][a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wu), __builtin_bit_cast(bf16x8_t, x[mt][u]),
                                                                        to[mt][a], 0, 0, 0);
            }
    };
    // piece sp belongs to part sp / per, the (sp / per - wave * VW)-th of this wave (the same for all its lanes)
    auto multiply_piece = [&](int sp, const uint4 (&w)[NW][WL], const uint4 (&x)[MT][4]) {
        if constexpr (VW == 1) {
            multiply_into(acc[0], w, x);
        } else {
            const int p = sp / per - wave * VW;
            if (p == 0) multiply_into(acc[0], w, x);
            else if (p == 1) multiply_into(acc[1], w, x);
            else if constexpr (VW == 4) {
                if (p == 2) multiply_into(acc[2], w, x);
                else multiply_into(acc[3], w, x);
            }
        }
    };
    constexpr std::true_type whole{};
    constexpr std::false_type masked{};
    const int s_whole = min(s_end, g.K / 128);       // pieces before this one lie inside K
    int sp = wave * VW * per;
    // Up to eight accumulators leave registers for two pieces or more (see the loop below; four row tiles and two sets of weight rows have a SIMD to a wave then, and 64 rows against
    // 6,144 weight rows of 2,048 k take 15.3 us instead of 18.4, 5,120 of 4,096 26.6 instead of 32.3, 12,288 of 2,048 27.2 instead of 28.6).  The first loads leave here,
    // and so do the old values that a block adds its product to: nothing of the epilogue waits for memory then.
    constexpr bool TWO = MT * NW <= 8 && !NORM;
    uint4 w0[TWO ? DEPTH : 1][TWO ? NW : 1][WL], x0[TWO ? DEPTH : 1][TWO ? MT : 1][4];
    const bool deep = DEPTH > 2 && s_whole - sp >= DEPTH;
    auto first_pieces = [&]() {
        if constexpr (TWO) {
            if (deep) {
#pragma unroll
                for (int d = 0; d < DEPTH; ++d) load_piece(whole, sp + d, w0[d], x0[d]);
            } else if (sp < s_whole) {
                load_piece(whole, sp, w0[0], x0[0]);
            }
        }
    };
    if constexpr (!ROPE) first_pieces();
    // The outputs of a thread: runs of V columns of a row, run tid + i * threads of the block's OUTS tiles of 16 rows x CW columns, so that all waves work.  Single elements, whose
    // rows' columns go out together, but where a thread adds to what is there, or has several row tiles of plain outputs, for what it keeps of each through the loop: as many then as
    // leave every wave its share, up to the four that a lane of the accumulators holds.  us, elements / runs: 32 rows added into 2,048 columns 8.9 / 8.2, 64 rows against 5,632
    // weight rows of 2,048 k 18.3 / 17.5, against 2,560 with a bias 13.5 / 12.6; the other way an expert's down product of one token 7.1 / 7.5, of 8 tokens 21.6 / 22.8, gate/up of
    // 1,408 and 64 rows 16.3 / 17.3.  (dual: a tile of gates and one of ups make one of outputs)
    constexpr int SETS = DUAL ? NW / 2 : NW;      // column groups of a block
    constexpr int OUTS = MT * SETS, THREADS = WAVES * 64, PER = 16 * CW, SHARE = OUTS * PER / THREADS;
    constexpr int V = EPI != EPI_RESID && (DUAL || MT == 1) ? 1 : (SHARE >= 4 ? 4 : (SHARE >= 2 ? 2 : 1)), RUNS = PER / V, IT = (OUTS * RUNS + THREADS - 1) / THREADS;
    static_assert(V == 1 || CW == 16, "runs of several columns are of whole sets");
    typedef __attribute__((ext_vector_type(V == 1 ? 2 : V))) float run_t;
    typedef run_t run_any_t __attribute__((aligned(4)));
    int m_of[IT];                                 // row of C, or -1
    constexpr bool THEN = EPI == EPI_RESID && MT == 1;
    float old[IT][V], scale_of[IT], gate[IT][V], more[THEN ? IT : 1][V];
    RawElement bias_of[IT][V];
    auto tile_of = [&](int i) { return OUTS == 1 && V == 1 ? 0 : (tid + i * THREADS) / RUNS; };
    auto row_in_tile = [&](int i) { return V == 1 ? (tid + i * THREADS) / CW % 16 : (tid + i * THREADS) % RUNS / (4 / V) % 16; };
    static_assert(V == 1 || THREADS % RUNS == 0, "the runs of a thread begin at one column");
    const int column_in_tile = V == 1 ? tid % CW : tid % RUNS / (RUNS / 4) * 4 + (V == 2 ? (tid & 1) * 2 : 0);
    auto column_of = [&](int i) { return n0 + (tile_of(i) % SETS) * CW + column_in_tile; };
    if constexpr (!ROPE) {
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const int row = row_in_tile(i), first = column_of(i);
            const int ml = pairs ? __shfl(pair_c, row) : r0 + (tile_of(i) / SETS) * 16 + row;
            const bool live = (pairs ? ml >= 0 : ml < r_end) && first < g.N && (OUTS * RUNS % THREADS == 0 || tid + i * THREADS < OUTS * RUNS);
            const int safe = live ? ml : (pairs ? 0 : r0);
            const int m = (g.c_rows && !pairs) ? g.c_rows[safe] : safe;
            m_of[i] = live ? m : -1;
            scale_of[i] = DUAL ? FX_PRE_SCALE(g, safe) : (EPI == EPI_RESID && g.row_scale ? g.row_scale[safe] : 1.f);
            if constexpr (EPI == EPI_RESID) {
                const float* from = (const float*)g.C + (size_t)m * g.ldc;
                if (V > 1 && first + V <= g.N) {
                    const run_t was = *(const run_any_t*)(from + first);
#pragma unroll
                    for (int r = 0; r < V; ++r) old[i][r] = was[r];
                } else {
#pragma unroll
                    for (int r = 0; r < V; ++r) old[i][r] = from[min(first + r, g.N - 1)];
                }
            }
            if constexpr (THEN) {
                if (g.then_add) {
                    const float* from = g.then_add + (size_t)m * g.ld_then_add;
#pragma unroll
                    for (int r = 0; r < V; ++r) more[i][r] = from[min(first + r, g.N - 1)];
                }
            }
            if constexpr (EPI == EPI_STORE || EPI == EPI_STORE_F32) {
#pragma unroll
                for (int r = 0; r < V; ++r) gate[i][r] = gate_of(g, m, min(first + r, g.N - 1));
            }
            if (!DUAL && g.bias) {
#pragma unroll
                for (int r = 0; r < V; ++r) bias_of[i][r] = fetch_element(g.bias, g.bias_dtype, min(first + r, g.N - 1));
            }
        }
    }
    // (the angle of the pair that a thread's output belongs to, worked out while the weights are on their way; 0 where it is not turned)
    float turn_cs[TURN ? IT : 1], turn_sn[TURN ? IT : 1];
    bool turned[TURN ? IT : 1];
    if constexpr (TURN) {
        static_assert(V == 1, "a lane's neighbour holds the other number of its pair");
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const int c = g.rope_hd ? column_of(i) % g.rope_hd - g.rope_nh : -1;
            turned[i] = m_of[i] >= 0 && c >= 0 && c < g.rope_rot;
            if (turned[i]) {
                sincosf((float)g.rope_positions[m_of[i]] * g.rope_inv_freq[c >> 1], &turn_sn[i], &turn_cs[i]);
                turn_cs[i] *= g.act_alpha;
                turn_sn[i] *= g.act_alpha;
            }
        }
    }
    // rope epilogue: what thread (lane, wave) needs for its pairs of outputs, rows 16 mt + lane % 16, column
    // 4 (lane / 16) + wave of the two sets, is fetched and worked out here, while the weights are on their way
    // More than two row tiles: what a row has of its own, its scale and its place in the pages, is found by one lane, asked for in front of the first weights and handed
    // to the others in LDS (a lane that finds it for all of its rows reads eight sums for each: 64 rows of 2,048 k with sums 24.0 us, so 21.4; of two tiles 32 rows 15.8
    // and 15.7, but without sums 14.3 and 15.3).
    constexpr bool LANE_PER_ROW = ROPE && MT > 2;
    __shared__ float row_scale_of[LANE_PER_ROW ? 16 * MT : 1];
    __shared__ int row_place_of[LANE_PER_ROW ? 2 : 1][LANE_PER_ROW ? 16 * MT : 1];
    float rstd_of_lane = 1.f;
    int page_of_lane = 0, slot_of_lane = 0;
    float rope_sn[MT], rope_cs[MT], rope_rstd[MT], rope_b0 = 0.f, rope_b1 = 0.f;
    size_t rope_page[MT];
    int rope_slot[MT];
    if constexpr (ROPE) {
        const int cc = grp * 4 + wave;
        const bool to_pages = rope_head >= g.rope_nh && g.rope_k_pages;
        // first every load that depends on nothing, then the page ids, which need position and sequence
        int row_of[MT], pos[MT], seq[MT];
        float total[MT];
        float squares_of_lane[8];
        int pos_of_lane = 0, seq_of_lane = 0;
        if constexpr (LANE_PER_ROW) {
            const int row = min(r0 + min(lane, 16 * MT - 1), r_end - 1), n = g.row_ss ? g.row_ss_n : 1;
            const float* ss = g.row_ss ? g.row_ss + (size_t)row * n : g.rope_inv_freq;      // (without sums the same load, not used)
            pos_of_lane = g.rope_positions[row];
            seq_of_lane = to_pages ? g.rope_token_seq[row] : 0;
            if (n > 8) squares_of_lane[0] = sum_in_order(ss, n);
            else
#pragma unroll
                for (int u = 0; u < 8; ++u) squares_of_lane[u] = ss[min(u, n - 1)];
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            row_of[mt] = min(r0 + 16 * mt + li, r_end - 1);
            pos[mt] = g.rope_positions[row_of[mt]];
            if constexpr (!LANE_PER_ROW) seq[mt] = to_pages ? g.rope_token_seq[row_of[mt]] : 0;
        }
        // (without a bias the same loads read the positions instead: a branch around them would wait for them)
        const void* bias_or = g.bias ? g.bias : (const void*)g.rope_positions;
        const int bias_dt = g.bias ? g.bias_dtype : FX_F32;
        const RawElement e0 = fetch_element(bias_or, bias_dt, g.bias ? (size_t)rope_head * g.rope_hd + rope_c0 + cc : 0);
        const RawElement e1 = fetch_element(bias_or, bias_dt, g.bias ? (size_t)rope_head * g.rope_hd + rope_c1 + cc : 0);
        // the pair's frequency from the table (columns that are not rotated read entry 0 and do not use it)
        const int p = rope_rotated ? 16 * rope_j + cc : 0;
        const float freq = g.rope_inv_freq[p];
        const float freq_div = g.rope_freq_factors ? g.rope_freq_factors[p] : 1.f;
        if constexpr (WEIGHTS_FIRST) {      // (sums of squares of one batch: asked for in front of the first weights, summed behind them)
            float squares[MT][8];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int u = 0; u < 8; ++u) squares[mt][u] = g.row_ss[(size_t)row_of[mt] * g.row_ss_n + min(u, g.row_ss_n - 1)];
            first_pieces();
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                total[mt] = 0.f;
#pragma unroll
                for (int u = 0; u < 8; ++u) total[mt] = u < g.row_ss_n ? total[mt] + squares[mt][u] : total[mt];
            }
        } else if constexpr (LANE_PER_ROW) {
            first_pieces();
            float sum = squares_of_lane[0];
            if (g.row_ss && g.row_ss_n <= 8) {
                sum = 0.f;
#pragma unroll
                for (int u = 0; u < 8; ++u) sum = u < g.row_ss_n ? sum + squares_of_lane[u] : sum;
            }
            rstd_of_lane = g.row_ss ? row_rstd(sum, g.K, g.norm_eps) : 1.f;
            slot_of_lane = pos_of_lane % g.rope_bs;
            if (to_pages) page_of_lane = g.rope_table[(size_t)seq_of_lane * g.rope_max_blocks + pos_of_lane / g.rope_bs];
        } else {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                total[mt] = g.row_ss ? sum_in_order(g.row_ss + (size_t)row_of[mt] * g.row_ss_n, g.row_ss_n) : 0.f;
        }
        rope_b0 = element_as_float(e0);
        rope_b1 = element_as_float(e1);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            rope_page[mt] = 0;
            rope_slot[mt] = 0;
            if (!LANE_PER_ROW && to_pages) {
                rope_page[mt] = (size_t)g.rope_table[(size_t)seq[mt] * g.rope_max_blocks + pos[mt] / g.rope_bs];
                rope_slot[mt] = pos[mt] % g.rope_bs;
            }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            if constexpr (!LANE_PER_ROW) rope_rstd[mt] = g.row_ss ? row_rstd(total[mt], g.K, g.norm_eps) : 1.f;
            rope_sn[mt] = 0.f;
            rope_cs[mt] = 1.f;
            if (rope_rotated) {
                float angle = (float)pos[mt] * freq;
                if (g.rope_freq_factors) angle = angle / freq_div;
                sincosf(angle, &rope_sn[mt], &rope_cs[mt]);
            }
        }
        // (what the epilogue needs first: behind the weights those short loads would wait for them)
        if constexpr (!WEIGHTS_FIRST && !LANE_PER_ROW) first_pieces();
    }
    // Few accumulators leave registers for two pieces: the loads of the next piece are then issued before the
    // products of this one, so a wave always has a piece on its way from memory.  Each product follows the
    // loads issued after its own in straight-line code.  DEPTH pieces where blocks are so few that a wave's chain of trips to
    // memory is what takes the time.
    if constexpr (TWO) {
        if (deep) {
            for (; sp + 2 * DEPTH <= s_whole; sp += DEPTH) {
#pragma unroll
                for (int d = 0; d < DEPTH; ++d) {
                    multiply_piece(sp + d, w0[d], x0[d]);
                    load_piece(whole, sp + DEPTH + d, w0[d], x0[d]);
                }
            }
            const int rest = s_whole - sp - DEPTH;       // pieces behind the ones on their way, fewer than DEPTH (what does not exist repeats the last)
            if (rest == 0) {
#pragma unroll
                for (int d = 0; d < DEPTH; ++d) multiply_piece(sp + d, w0[d], x0[d]);
            } else {
#pragma unroll
                for (int d = 0; d < DEPTH; ++d) {
                    multiply_piece(sp + d, w0[d], x0[d]);
                    if (d + 1 < DEPTH) load_piece(whole, min(sp + DEPTH + d, s_whole - 1), w0[d], x0[d]);
                }
#pragma unroll
                for (int d = 0; d + 1 < DEPTH; ++d)
                    if (d < rest) multiply_piece(sp + DEPTH + d, w0[d], x0[d]);
            }
            sp = s_whole;
        } else if (sp < s_whole) {
            for (; sp + 2 < s_whole; sp += 2) {
                load_piece(whole, sp + 1, w0[1], x0[1]);
                multiply_piece(sp, w0[0], x0[0]);
                load_piece(whole, sp + 2, w0[0], x0[0]);
                multiply_piece(sp + 1, w0[1], x0[1]);
            }
            if (sp + 1 < s_whole) {
                load_piece(whole, sp + 1, w0[1], x0[1]);
                multiply_piece(sp, w0[0], x0[0]);
                multiply_piece(sp + 1, w0[1], x0[1]);
                sp += 2;
            } else {
                multiply_piece(sp, w0[0], x0[0]);
                sp += 1;
            }
        }
    } else {
        for (; sp < s_whole; ++sp) {
            uint4 w[NW][WL], x[MT][4];
            load_piece(whole, sp, w, x);
            multiply_piece(sp, w, x);
        }
    }
    for (; sp < s_end; ++sp) {          // the piece that K ends in
        uint4 w[NW][WL], x[MT][4];
        load_piece(masked, sp, w, x);
        multiply_piece(sp, w, x);
    }
#pragma unroll
    for (int p = 0; p < VW; ++p)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int a = 0; a < NW; ++a) red[wave * VW + p][mt * NW + a][lane] = acc[p][mt][a];
    if constexpr (NORM) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) red_ss[wave][mt][lane] = ss[mt];
    }
    if constexpr (LANE_PER_ROW) {
        if (wave == 0 && lane < 16 * MT) {
            row_scale_of[lane] = rstd_of_lane;
            row_place_of[0][lane] = page_of_lane;
            row_place_of[1][lane] = slot_of_lane;
        }
    }
    __syncthreads();
    if constexpr (ROPE) {
        static_assert(!ROPE || WAVES == 4, "a wave per accumulator row");
        const int L = lane, r = wave;
        const int hd = g.rope_hd, bs = g.rope_bs, cc = (L >> 4) * 4 + r;
        const int d0 = rope_c0 + cc, d1 = rope_c1 + cc;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int ml = r0 + 16 * mt + (L & 15);
            if (ml >= r_end) continue;
            if constexpr (LANE_PER_ROW) {
                rope_rstd[mt] = row_scale_of[16 * mt + (L & 15)];
                rope_page[mt] = row_place_of[0][16 * mt + (L & 15)];
                rope_slot[mt] = row_place_of[1][16 * mt + (L & 15)];
            }
            f32x4_t v0 = (f32x4_t){0.f, 0.f, 0.f, 0.f}, v1 = v0;
#pragma unroll
            for (int w = 0; w < PARTS; ++w) {
                v0 += red[w][mt * NW][L];
                v1 += red[w][mt * NW + 1][L];
            }
            // product times scale is rounded before the bias is added, as in the plain epilogue (whose bias sits
            // behind a branch); the empty statement keeps the compiler from fusing the two here
            float o0 = v0[r] * rope_rstd[mt], o1 = v1[r] * rope_rstd[mt];
            asm volatile("" : "+v"(o0), "+v"(o1));
            if (g.bias) {
                o0 += rope_b0;
                o1 += rope_b1;
            }
            const float a = bf16_to_float(float_to_bf16(o0)), b = bf16_to_float(float_to_bf16(o1));
            float y0 = a, y1 = b;
            if (rope_rotated) rotate_pair(a, b, rope_cs[mt], rope_sn[mt], y0, y1);
            if (rope_head < g.rope_nh) {
                bf16* dst = (bf16*)g.C + (size_t)ml * g.ldc + (size_t)rope_head * hd;
                from_float(dst + d0, y0);
                from_float(dst + d1, y1);
            } else if (g.rope_k_pages) {
                if (rope_head < g.rope_nh + g.rope_nkv) {
                    bf16* dst = (bf16*)g.rope_k_pages + ((rope_page[mt] * g.rope_nkv + (rope_head - g.rope_nh)) * bs + rope_slot[mt]) * hd;
                    from_float(dst + d0, y0);
                    from_float(dst + d1, y1);
                } else {
                    bf16* dst = (bf16*)g.rope_v_pages + (rope_page[mt] * g.rope_nkv + (rope_head - g.rope_nh - g.rope_nkv)) * hd * bs + rope_slot[mt];
                    from_float(dst + (size_t)d0 * bs, y0);
                    from_float(dst + (size_t)d1 * bs, y1);
                }
            }
        }
        return;
    }
    // parts in their order; lane 16 (column / 4) + row of an accumulator holds columns 4 (column / 4) ..
    const float* sums = (const float*)red + (size_t)((column_in_tile >> 2) * 16) * 4 + (column_in_tile & 3);
    auto sum_of = [&](int acc_tile, int row, float (&v)[V]) {
#pragma unroll
        for (int r = 0; r < V; ++r) v[r] = 0.f;
#pragma unroll
        for (int w = 0; w < PARTS; ++w) {
            if constexpr (V == 1) {
                v[0] += sums[((size_t)(w * NACC + acc_tile) * 64 + row) * 4];
            } else {
                const run_t part = *(const run_t*)(sums + ((size_t)(w * NACC + acc_tile) * 64 + row) * 4);
#pragma unroll
                for (int r = 0; r < V; ++r) v[r] += part[r];
            }
        }
    };
    auto finish = [&](auto kind) {
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const int m = m_of[i];
            if (m < 0) continue;
            const int t = tile_of(i), mt = t / SETS, a = t % SETS, row = row_in_tile(i);
            const int n = column_of(i);
            float o[V];
            sum_of(mt * NW + (DUAL ? 2 * a : a), row, o);
            if constexpr (DUAL) {
                float up[V];
                sum_of(mt * NW + 2 * a + 1, row, up);
#pragma unroll
                for (int r = 0; r < V; ++r) o[r] = gated_c<decltype(kind)::value>(o[r] * scale_of[i], up[r] * scale_of[i], g.act_limit, g.act_alpha);
            } else {
                float rstd = 1.f;
                if (!NORM && g.row_ss) rstd = row_rstd(sum_in_order(g.row_ss + (size_t)m * g.row_ss_n, g.row_ss_n), g.K, g.norm_eps);
                if constexpr (NORM) {
                    float total = 0.f;
#pragma unroll
                    for (int w = 0; w < WAVES; ++w)
#pragma unroll
                        for (int q = 0; q < 4; ++q) total += red_ss[w][mt][row + 16 * q];
                    rstd = row_rstd(total, g.K, g.norm_eps);
                }
#pragma unroll
                for (int r = 0; r < V; ++r) {
                    o[r] *= rstd;
                    asm volatile("" : "+v"(o[r]));          // the product is rounded before the bias is added (no fused multiply-add)
                    if (g.bias) o[r] += element_as_float(bias_of[i][r]);
                    if constexpr (EPI == EPI_RESID) {
                        if (g.row_scale) {
                            o[r] *= scale_of[i];
                            asm volatile("" : "+v"(o[r]));
                        }
                        o[r] = old[i][r] + o[r];
                        if constexpr (THEN) {
                            if (g.then_add) o[r] += more[i][r];
                        }
                    } else {
                        o[r] = stored_c<decltype(kind)::value>(g, o[r], gate[i][r]);
                    }
                }
            }
            if constexpr (TURN) {
                if (turned[i]) {      // (rounded before it is turned, as when the rotation is a kernel of its own; a pair's two lanes are here together)
                    const float own = bf16_to_float(float_to_bf16(o[0])), other = lane_pair_other(own);
                    float y0, y1;
                    rotate_pair(n & 1 ? other : own, n & 1 ? own : other, turn_cs[i], turn_sn[i], y0, y1);
                    o[0] = n & 1 ? y1 : y0;
                }
            }
            typedef std::conditional_t<EPI == EPI_STORE || EPI == EPI_GATED, bf16, float> out_t;
            out_t* to = (out_t*)g.C + (size_t)m * g.ldc + n;
            if constexpr (V == 1) from_float(to, o[0]);
            else store_columns<V>(to, o, g.N - n);
        }
    };
    if constexpr (DUAL) with_activation(g.act, finish);
    else with_stored<EPI == EPI_STORE || EPI == EPI_STORE_F32>(g.store_act, finish);
}

template <int MT, int WAVES, int NW, bool DUAL, int EPI, bool NORM = false, bool ROPE = false, bool HALF = false, int DEPTH = 2, bool WEIGHTS_FIRST = false>
__global__ __launch_bounds__(WAVES * 64) void gemm_bf16_skinny_kernel(GemmArgs g) {
    skinny_block<MT, WAVES, NW, DUAL, EPI, NORM, ROPE, HALF, DEPTH, WEIGHTS_FIRST, false>(g, blockIdx.x, blockIdx.y);
}

// Two products of up to 16 plain rows that do not need each other, one launch: the first's blocks (gate/up, or a product that is stored in float32, in half sets of
// weight rows), then the second's (stored; in half or whole sets).  A step of few tokens is a chain of launches of 3 us and more that each wait for memory alone;
// side by side they wait together, and the streams of the larger one go on meanwhile.  The same blocks, so the same bits.  us apart -> together: gate/up of 5,632 x 2,048 and
// 1,024 x 2,048 1 row 14.6 -> 11.2, 8 rows 16.1 -> 13.2, 16 rows 18.6 -> 16.6; 2,048 x 5,632 and 4,096 x 512 with its heads turned (a launch of its own before)
// 13.5 -> 8.0, 14.1 -> 8.9, 16.3 -> 10.9.
template <bool GATED, int DEPTH, int NW2, int EPI2, bool HALF2>
__global__ __launch_bounds__(256) void gemm_bf16_skinny_pair_kernel(GemmArgs a, GemmArgs b, int first) {
    if ((int)blockIdx.x < first)
        skinny_block<1, 4, GATED ? 2 : 1, GATED, GATED ? EPI_GATED : EPI_STORE_F32, false, false, true, DEPTH, false, false>(a, blockIdx.x, 0);
    else
        skinny_block<1, 4, NW2, false, EPI2, false, false, HALF2, HALF2 ? 4 : 2, false, EPI2 == EPI_STORE>(b, blockIdx.x - first, 0);
}

// ===========================================================================
// float32 on MFMA
// ===========================================================================
// v_mfma_f32_16x16x4_f32 multiplies and adds in float32 (twice the rate of v_fma_f32, whose packed form is not used here).
// Both kernels below add an output's products in the same order, so a row's bits do not depend on which of them
// computes it: K is cut into F32_PARTS parts; inside a part 16 k at a time, four instructions of 4 k each, instruction u
// taking k = 4 g + u for g = 0..3 (the order is stated in common.h; a lane of group g holds four consecutive k in one 16-byte register group); the parts'
// sums are added in their order.  The weights are the instruction's first operand, so that a lane ends with four
// consecutive columns of one row.

// four k steps of one tile: w and x hold k = 4 g .. 4 g + 3 of the lane's weight row and activation row
template <int MT, int NT>
__device__ __forceinline__ void f32_multiply(f32x4_t (&acc)[MT][NT], const f32x4_t (&w)[NT], const f32x4_t (&x)[MT]) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j][u], x[i][u], acc[i][j], 0, 0, 0);
}
// k .. k + 3 of a row; guarded: zeros from K on (VEC: the row is 16-byte aligned and K a multiple of 4).  Inside the loops
// the loads are unconditional (a step past the end reads the last one again): behind a branch the compiler waits for them
// on the spot, and the loop has no load in flight (tiles of 64 x 64 against 2,048 k: 84 -> 47 us).
template <bool VEC>
__device__ __forceinline__ f32x4_t f32_fetch(const float* p) {
    if (VEC) return *(const f32x4_t*)p;
    return (f32x4_t){p[0], p[1], p[2], p[3]};
}
template <bool VEC>
__device__ __forceinline__ f32x4_t f32_fetch_guarded(const float* row, int k, int K) {
    f32x4_t v = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    if (VEC) {
        if (k < K) v = *(const f32x4_t*)(row + k);
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (k + r < K) v[r] = row[k + r];
    }
    return v;
}
// ---------------------------------------------------------------------------
// float32 products as bfloat16 ones
// ---------------------------------------------------------------------------
// A float32 is the sum of three bfloat16 numbers h + m + l, each the rest of the ones before it rounded to nearest (8 + 8 + 8 bits and two signs hold
// its 24 bits; Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for higher-precision computations", 2019), and a product of two such sums has six terms
// down to 2^-18 of it: hh, hm, mh, mm, hl, lh.  What is left out, ml, lm and ll, can be 2^-24 of a product (just above a power of two in both) and is of either sign: 6e-9 of a sum's norm, where
// rounding a float32 product takes 3e-8.  Of few terms the cut-off weighs more than the roundings that it saves: rows with one number that is not 0 are off by 5.0e-8 of themselves instead of 2.5e-8, with eight
// 7.2e-8 instead of 5.5e-8, from some 64 on it is level, then less.  The matrix instruction adds 32 bfloat16 products in 16 cycles where the float32 one adds
// four in 32, so six terms take 96 cycles instead of 256.
// The instruction cuts a sum off below instead of rounding it, so a step's 32 k start from zero, small terms first, and are added to the sums so far with an add that rounds; and every second step works
// out the negative and subtracts it, so that what is cut off has either sign: else outputs are low by 5e-8 of their size, which the mean over a thousand keys brings out (decoded logits at 1,030 keys: 1.3e-6
// off 64 bits instead of 0.8e-6).  Error against 64 bits, float32 instruction / taken apart: 2,048 k 2.9e-7 / 7.5e-8, 5,632 k 4.8e-7 / 7.3e-8, terms of one sign 8.9e-8 / 4.5e-8.
// Parts of K (F32_PARTS, of whole pairs of steps) are added in their order, in the kernel for few rows and in tiles alike: a row's bits do not depend on which of them computes it.
// Four columns of a row that hold an infinity, a NaN or a sum beyond float32 are worked out again on the float32 instruction: an infinity has no rest.  And so are four of which one is below 2^-64
// and not 0: bfloat16 ends where float32 does, so a number below 2^-110 loses the bits of its third part (at 2^-118 1.5e-5 of itself), at most 2^-126 of each.  Such losses come to less
// than a rounding of a sum of 2^-64 and more while the rows' absolute sums are below 2^37; what is made of such numbers alone is smaller.
__host__ __device__ __forceinline__ int f32_split_part_length(int K) { return ((K + F32_PARTS - 1) / F32_PARTS + 63) / 64 * 64; }
typedef __attribute__((ext_vector_type(8))) __bf16 f32_part8_t;
typedef __attribute__((ext_vector_type(2))) __bf16 f32_part2_t;
struct F32Split {
    f32_part8_t h, m, l;
};
// (a, b) as packed bfloat16, and what is left of both, which is exact.  A dot product with (-1, 0) or (0, -1) takes the place of moving a half into place and
// subtracting it; the two constants pass through an empty statement, in the form of inline constants the instruction reads them otherwise.  (700 x 2,048 x 5,632 160 -> 143 us.)
template <bool NEG>
__device__ __forceinline__ uint32_t f32_peel(float& a, float& b) {
    const uint32_t p = pack_bf16(NEG ? -a : a, NEG ? -b : b);
    uint32_t first = NEG ? 0x00003f80u : 0x0000bf80u, second = first << 16;
    asm("" : "+v"(first), "+v"(second));
    a = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(f32_part2_t, p), __builtin_bit_cast(f32_part2_t, first), a, false);
    b = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(f32_part2_t, p), __builtin_bit_cast(f32_part2_t, second), b, false);
    return p;
}
template <bool NEG>      // NEG: of -v
__device__ __forceinline__ void f32_split4(f32x4_t v, uint2& h, uint2& m, uint2& l) {
    float a = v[0], b = v[1], c = v[2], d = v[3];
    h.x = f32_peel<NEG>(a, b); h.y = f32_peel<NEG>(c, d);
    m.x = f32_peel<NEG>(a, b); m.y = f32_peel<NEG>(c, d);
    l.x = NEG ? pack_bf16(-a, -b) : pack_bf16(a, b); l.y = NEG ? pack_bf16(-c, -d) : pack_bf16(c, d);
}
template <bool NEG>
__device__ __forceinline__ F32Split f32_split8(f32x4_t lo, f32x4_t hi) {
    uint2 h0, m0, l0, h1, m1, l1;
    f32_split4<NEG>(lo, h0, m0, l0);
    f32_split4<NEG>(hi, h1, m1, l1);
    F32Split s;
    s.h = __builtin_bit_cast(f32_part8_t, make_uint4(h0.x, h0.y, h1.x, h1.y));
    s.m = __builtin_bit_cast(f32_part8_t, make_uint4(m0.x, m0.y, m1.x, m1.y));
    s.l = __builtin_bit_cast(f32_part8_t, make_uint4(l0.x, l0.y, l1.x, l1.y));
    return s;
}
// the operand of eight rows from a lane's four k: its own, then those of the lane that has the row's other 16 (taken apart once, then handed over)
template <bool NEG>
__device__ __forceinline__ F32Split f32_split_half(f32x4_t own) {
    uint2 h, m, l;
    f32_split4<NEG>(own, h, m, l);
    auto both = [](uint2 v) {
        const uint32_t x = __builtin_amdgcn_update_dpp(v.x, v.x, 0x128, 0xF, 0x3, false), y = __builtin_amdgcn_update_dpp(v.y, v.y, 0x128, 0xF, 0x3, false);      // (as `swap_halves<0x3>`)
        return __builtin_bit_cast(f32_part8_t, make_uint4(v.x, v.y, x, y));
    };
    F32Split s;
    s.h = both(h);
    s.m = both(m);
    s.l = both(l);
    return s;
}
// 32 k of a tile: the small terms first
#define FX_MFMA32(A, B, C) __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, B, C, 0, 0, 0)
template <bool NEG, int MT, int NT>
__device__ __forceinline__ void f32_split_multiply(f32x4_t (&acc)[MT][NT], const F32Split (&w)[NT], const F32Split (&x)[MT]) {
    f32x4_t t[MT][NT];
#define FX_TERM(W, X, C)                       \
    _Pragma("unroll") for (int i = 0; i < MT; ++i) \
        _Pragma("unroll") for (int j = 0; j < NT; ++j) t[i][j] = FX_MFMA32(w[j].W, x[i].X, C)
    FX_TERM(l, h, ((f32x4_t){0.f, 0.f, 0.f, 0.f}));
    FX_TERM(h, l, t[i][j]);
    FX_TERM(m, m, t[i][j]);
    FX_TERM(m, h, t[i][j]);
    FX_TERM(h, m, t[i][j]);
    FX_TERM(h, h, t[i][j]);
#undef FX_TERM
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = NEG ? acc[i][j] - t[i][j] : acc[i][j] + t[i][j];
}
// one tile's sums on the float32 instruction, K a multiple of 32, rows from memory
template <bool VEC>
__device__ __forceinline__ f32x4_t f32_whole_sum(int K, const float* w_row, const float* x_row, int gq) {
    const int part = f32_part_length(K);
    f32x4_t acc[1][1] = {{(f32x4_t){0.f, 0.f, 0.f, 0.f}}}, total = acc[0][0];
    for (int k = 0, end = part; k < K; k += 16) {
        if (k == end) {
            total += acc[0][0];
            acc[0][0] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
            end += part;
        }
        const f32x4_t w[1] = {f32_fetch<VEC>(w_row + k + gq * 4)}, x[1] = {f32_fetch<VEC>(x_row + k + gq * 4)};
        f32_multiply(acc, w, x);
    }
    return total + acc[0][0];
}
// Whether four sums of products taken apart stand (or eight, `other`): finite, and zero or not so small that numbers below 2^-110 may be what they are made of.  (In whole numbers, least and largest
// of all: a comparison each, with what joins them, is a chain between the vector and the scalar unit at the end of a kernel of 5 us.)
__device__ __forceinline__ bool f32_sums_stand(f32x4_t v, f32x4_t other) {
    constexpr uint32_t LEAST = 2u * (127 - 64) << 23, INFINITE = 2u * 255 << 23;      // (without the sign, one place up)
    uint32_t low = 0xffffffffu, high = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t a = __float_as_uint(v[i]) << 1, b = __float_as_uint(other[i]) << 1;
        low = min(low, min(a - 1, b - 1));        // (0 becomes the largest)
        high = max(high, max(a, b));
    }
    return (low >= LEAST - 1) & (high < INFINITE);
}

// What columns n .. n + 3 of logical row ml need on their way out besides the product: a kernel whose last wait is for its operands
// asks for it in front of them.
template <int EPI>
struct F32Out {
    int m;
    float scale;
    f32x4_t bias, old, gate;
};
template <bool DUAL, int EPI>
__device__ __forceinline__ F32Out<EPI> f32_ask(const GemmArgs& g, int ml, int n) {
    F32Out<EPI> o = {};
    o.m = g.c_rows ? g.c_rows[ml] : ml;
    o.scale = DUAL ? FX_PRE_SCALE(g, ml) : (EPI == EPI_RESID && g.row_scale ? g.row_scale[ml] : 1.0f);
    if constexpr (!DUAL) {
        if (g.bias) {
#pragma unroll
            for (int r = 0; r < 4; ++r) o.bias[r] = load_as_float(g.bias, g.bias_dtype, min(n + r, g.N - 1));
        }
        if constexpr (EPI == EPI_RESID) {
            const float* at = (const float*)g.C + (size_t)o.m * g.ldc;
            if (g.c_vec && n + 4 <= g.N) {
                o.old = *(const f32x4_t*)(at + n);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) o.old[r] = at[min(n + r, g.N - 1)];
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) o.gate[r] = gate_of(g, o.m, min(n + r, g.N - 1));
        }
    }
    return o;
}
template <bool DUAL, int EPI>
__device__ __forceinline__ void f32_store4(const GemmArgs& g, const F32Out<EPI>& o, int n, f32x4_t v, f32x4_t v2) {
    if (n >= g.N) return;
    float* out = (float*)g.C + (size_t)o.m * g.ldc + n;
    f32x4_t y;
    if constexpr (DUAL) {
        with_activation(g.act, [&](auto ac) {
#pragma unroll
            for (int r = 0; r < 4; ++r) y[r] = gated_c<decltype(ac)::value>(v[r] * o.scale, v2[r] * o.scale, g.act_limit, g.act_alpha);
        });
    } else {
        if (g.bias) {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] += o.bias[r];
        }
        if constexpr (EPI == EPI_RESID) {
            if (g.row_scale) {
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] *= o.scale;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) y[r] = o.old[r] + v[r];
        } else {
            with_stored<true>(g.store_act, [&](auto kind) {   // (the host sets store_act for stored products only)
#pragma unroll
                for (int r = 0; r < 4; ++r) y[r] = stored_c<decltype(kind)::value>(g, v[r], o.gate[r]);
            });
        }
    }
    if (g.c_vec && n + 4 <= g.N) *(f32x4_t*)out = y;
    else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (n + r < g.N) out[r] = y[r];
    }
}

// Many rows: TM x TN outputs a block (DUAL: TN / 2 columns of both matrices, their blocks of 16 in turn), four waves of
// TM/2 x TN/2, operands 32 k at a time through LDS in two stages, 16-byte pieces swizzled by the row, the loads two steps
// ahead.  Bound by the matrix units and the waits between barriers: 1,500 x 6,144 x 2,048 in 327 us, 115 of the 157
// TFLOP/s of the instruction (the FMA kernel before it: 700 x 6,144 x 2,048 in 379 us, this one 186).  Row blocks that a tile does not
// have are left out: both products of 700 tokens on 60 experts of 1,408, even shares 450 + 246 -> 404 + 238 us, crowded on half of them 393 + 216 -> 369 + 206.
template <int TM, int TN, bool DUAL, int EPI, bool VEC>
__global__ __launch_bounds__(256) void gemm_f32_tiled_kernel(GemmArgs g) {
    constexpr int MT = TM / 32, NT = TN / 32;
    static_assert(!DUAL || NT % 2 == 0, "a wave holds both matrices' blocks of its columns");
    __shared__ f32x4_t As[2][TM][8];
    __shared__ f32x4_t Bs[2][TN][8];
    int r0, r_end, expert;
    locate_rows<TM>(g, blockIdx.y, r0, r_end, expert);
    if (r0 < 0) return;
    const int n0 = blockIdx.x * (DUAL ? TN / 2 : TN);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, gq = lane >> 4;
    const int wm = wave & 1, wn = wave >> 1;
    const float* Wbase = (const float*)g.W + (size_t)expert * g.w_stride;
    // (a row or column past the end reads the last one; what comes of it is not stored)
    const int piece = tid & 7;
    const float* a_src[MT];
    const float* b_src[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        int m = r0 + (tid >> 3) + 32 * i;
        m = m < r_end ? m : r_end - 1;
        a_src[i] = (const float*)g.A + (size_t)(g.a_rows ? g.a_rows[m] : m) * g.lda;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int r = (tid >> 3) + 32 * j;
        int n = DUAL ? n0 + (r >> 5) * 16 + (r & 15) : n0 + r;
        n = n < g.N ? n : g.N - 1;
        b_src[j] = Wbase + (size_t)n * g.K + (DUAL && (r & 16) ? g.up_offset : 0);
    }
    f32x4_t ra[2][MT], rb[2][NT];
    const int n_full = g.K / 32;
    // (the rows that the tile has: `some`, as a type, the first 32 of them only)
    auto fetch = [&](auto some, int set, int step) {
        const int k = (step < n_full ? step : n_full - 1) * 32 + piece * 4;
#pragma unroll
        for (int i = 0; i < decltype(some)::value; ++i) ra[set][i] = f32_fetch<VEC>(a_src[i] + k);
#pragma unroll
        for (int j = 0; j < NT; ++j) rb[set][j] = f32_fetch<VEC>(b_src[j] + k);
    };
    auto keep = [&](auto some, int set) {
        const int row = tid >> 3, at = piece ^ (row & 7);      // (32 rows on: the same swizzle)
#pragma unroll
        for (int i = 0; i < decltype(some)::value; ++i) As[set][row + 32 * i][at] = ra[set][i];
#pragma unroll
        for (int j = 0; j < NT; ++j) Bs[set][row + 32 * j][at] = rb[set][j];
    };
    f32x4_t acc[MT][NT], total[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = total[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    const int part = f32_part_length(g.K);
    int next_end = part;
    auto multiply = [&](auto blocks, int buf, int k0) {
        constexpr int NA = decltype(blocks)::value;
        if constexpr (NA == 0) return;
        if (k0 == next_end) {
            next_end += part;
#pragma unroll
            for (int i = 0; i < NA; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    total[i][j] += acc[i][j];
                    acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
                }
        }
        f32x4_t w[2][NT], x[2][NA ? NA : 1];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int at = (s * 4 + gq) ^ (li & 7);
#pragma unroll
            for (int j = 0; j < NT; ++j) w[s][j] = Bs[buf][(wn * NT + j) * 16 + li][at];
#pragma unroll
            for (int i = 0; i < NA; ++i) x[s][i] = As[buf][(2 * i + wm) * 16 + li][at];
        }
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < NA; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[s][j][u], x[s][i][u], acc[i][j], 0, 0, 0);
    };
    // Blocks of 16 rows go to the two halves of the waves in turn, and those that do not exist are neither fetched nor multiplied (a tile of up
    // to 32 rows then takes half the time).  Every wave goes through the same barriers.
    auto loop = [&](auto blocks, auto some) {
        if (n_full > 0) {
            fetch(some, 0, 0);
            fetch(some, 1, 1);
            keep(some, 0);
            int step = 0;
            for (; step + 1 < n_full; step += 2) {
                lds_barrier();
                fetch(some, 0, step + 2);
                multiply(blocks, 0, step * 32);
                keep(some, 1);
                lds_barrier();
                fetch(some, 1, step + 3);
                multiply(blocks, 1, step * 32 + 32);
                keep(some, 0);
            }
            if (step < n_full) {
                lds_barrier();
                multiply(blocks, 0, step * 32);
            }
        }
        if (n_full * 32 < g.K) {           // the last, partial step
            const int k = n_full * 32 + piece * 4;
#pragma unroll
            for (int i = 0; i < decltype(some)::value; ++i) ra[0][i] = f32_fetch_guarded<VEC>(a_src[i], k, g.K);
#pragma unroll
            for (int j = 0; j < NT; ++j) rb[0][j] = f32_fetch_guarded<VEC>(b_src[j], k, g.K);
            lds_barrier();
            keep(some, 0);
            lds_barrier();
            multiply(blocks, 0, n_full * 32);
        }
    };
    const int n_blocks = (min(TM, r_end - r0) + 15) >> 4, mine = (n_blocks - wm + 1) >> 1;      // row blocks of the tile, of this wave
    if (mine == 0) loop(fx_int<0>{}, fx_int<1>{});
    else if (n_blocks <= 2) loop(fx_int<1>{}, fx_int<1>{});
    else if constexpr (MT > 1) {
        if (mine == 1) loop(fx_int<1>{}, fx_int<2>{});
        else loop(fx_int<2>{}, fx_int<2>{});
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int ml = r0 + (2 * i + wm) * 16 + li;
        if (ml >= r_end) continue;
#pragma unroll
        for (int j = 0; j < NT; j += DUAL ? 2 : 1) {
            const int t = wn * NT + j;
            const int n = n0 + (DUAL ? t >> 1 : t) * 16 + 4 * gq;
            f32_store4<DUAL, EPI>(g, f32_ask<DUAL, EPI>(g, ml, min(n, g.N - 1)), n, total[i][j] + acc[i][j], DUAL ? total[i][j + (DUAL ? 1 : 0)] + acc[i][j + (DUAL ? 1 : 0)] : acc[i][j]);
        }
    }
}

// Many rows, taken apart: up to TM rows x 64 NT columns a block (DUAL: 32 NT of both matrices, in each wave's blocks in turn or, ROLES, one matrix to a pair of waves), four waves that
// take 16 NT weight rows each and all the rows.  A weight row goes from memory into its wave's registers and is taken apart there, once; the rows are taken apart on their way into LDS, whose
// planes every wave reads in 16-byte pieces (swizzled by pairs of rows); two steps of 32 k between barriers, the loads of the next DEPTH such stages on their way.  LINES: the weights in whole
// lines with the non-temporal hint, where they are read about once.
// Bound by issue: of a step of 32 k of 64 x 128 outputs a wave issues 48 products of 16 cycles (23 at the clock that random values leave) and some 180 vector instructions, 84 of
// them the splitting, 32 the sums, and of these a SIMD hides up to four behind a product.  us, float32 instruction / taken apart: 700 x 6,144 x 2,048 190 / 130, 700 x 2,048 x 5,632
// 181 / 132, gate/up of 5,632 x 2,048 for 700 rows 287 / 196; both products of 700 tokens on 60 experts of 1,408, even shares 416 + 208 / 346 + 169, crowded 432 + 223 / 354 + 187;
// 1,500 x 6,144 x 2,048 321 / 230 (164 TFLOP/s; the instruction itself 153).  With a barrier a step of 32 k the tiles of few blocks took a third longer (64 x 2,048 x 2,048
// in 32 x 64 36 -> 25); the next step's splitting between this step's products 155 instead of 149 (700 x 6,144); tiles of 64 x 256 and 128 x 128 leave one wave a SIMD (214, 161).
template <int TM, int NT, int DEPTH, bool DUAL, int EPI, bool VEC, bool LINES>
__global__ __launch_bounds__(256, 2) void gemm_f32_split_kernel(GemmArgs g) {
    constexpr bool ROLES = DUAL && NT == 1;           // waves 0 and 1 take gate's rows and store, 2 and 3 up's
    constexpr int MB = TM / 16, AR = TM / 32, PER = DUAL && !ROLES ? 2 : 1;
    __shared__ uint2 Xs[2][2][3][TM][8];        // two steps of 32 k to a stage, two stages
    int r0, r_end, expert;
    if (g.expert_offsets) {
        locate_rows<TM>(g, blockIdx.y, r0, r_end, expert);
    } else {
        r0 = blockIdx.y * g.tile_rows;
        r_end = min(r0 + g.tile_rows, g.M);
        expert = 0;
    }
    if (r0 < 0) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, gq = lane >> 4;
    const int n0 = ROLES ? blockIdx.x * 32 + (wave & 1) * 16 : (blockIdx.x * 4 + wave) * (16 * NT / PER);
    const float* Wbase = (const float*)g.W + (size_t)expert * g.w_stride;
    const int piece = tid & 7, x_row = tid >> 3;
    const float* a_src[AR];
    const float* b_src[NT][LINES ? 2 : 1];      // LINES: of row li % 8, and of row li % 8 + 8
    auto a_row = [&](int i) {
        const int m = min(r0 + i, r_end - 1);
        return (const float*)g.A + (size_t)(g.a_rows ? g.a_rows[m] : m) * g.lda;
    };
    auto b_row = [&](int t, int m, int row) {
        return Wbase + (size_t)min(n0 + t * 16 + row, g.N - 1) * g.K + (m ? g.up_offset : 0);
    };
#pragma unroll
    for (int i = 0; i < AR; ++i) a_src[i] = a_row(x_row + 32 * i) + piece * 4;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int h = 0; h < (LINES ? 2 : 1); ++h)
            b_src[j][h] = b_row(j / PER, ROLES ? wave >> 1 : DUAL ? j & 1 : 0, LINES ? (li & 7) + 8 * h : li) + (LINES ? (li >> 3) * 16 : 0) + gq * 4;
    f32x4_t rx[2 * DEPTH][AR], rw[2 * DEPTH][NT][2];
    const int n_steps = g.K / 32;
    auto fetch_x = [&](auto some, int set, int step) {
        const int k = min(step, n_steps - 1) * 32;
#pragma unroll
        for (int i = 0; i < decltype(some)::value; ++i) rx[set][i] = f32_fetch<VEC>(a_src[i] + k);
    };
    auto fetch_w = [&](int set, int step) {
        const int k = min(step, n_steps - 1) * 32;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            if constexpr (LINES) {
                rw[set][j][0] = __builtin_bit_cast(f32x4_t, load_lines16(b_src[j][0] + k));
                rw[set][j][1] = __builtin_bit_cast(f32x4_t, load_lines16(b_src[j][1] + k));
            } else {
                rw[set][j][0] = f32_fetch<VEC>(b_src[j][0] + k);
                rw[set][j][1] = f32_fetch<VEC>(b_src[j][0] + k + 16);
            }
        }
    };
    // k = 4 p .. 4 p + 3 of a row are the half p >> 2 of what a lane of group p & 3 takes; 16-byte pieces swizzled by pairs of rows
    const int x_at = ((piece & 3) ^ ((x_row >> 1) & 3)) * 2 + (piece >> 2);
    auto keep = [&](auto some, auto setc, int buf) {          // (the operands of odd steps with the other sign)
        constexpr int set = decltype(setc)::value;
#pragma unroll
        for (int i = 0; i < decltype(some)::value; ++i) {
            uint2 h, m, l;
            f32_split4<(set & 1) == 1>(rx[set][i], h, m, l);
            Xs[buf][set & 1][0][x_row + 32 * i][x_at] = h;
            Xs[buf][set & 1][1][x_row + 32 * i][x_at] = m;
            Xs[buf][set & 1][2][x_row + 32 * i][x_at] = l;
        }
    };
    f32x4_t acc[MB][NT], total[MB][NT];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = total[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    const int part = f32_split_part_length(g.K) / 32;
    int next_end = part;
    const int at16 = (gq ^ ((li >> 1) & 3)) * 2;
    auto multiply = [&](auto blocks, auto setc, int buf, int step) {
        constexpr int NA = decltype(blocks)::value, set = decltype(setc)::value;
        constexpr bool NEG = (set & 1) == 1;
        if (!NEG && step == next_end) {         // (a part is an even number of steps)
            next_end += part;
#pragma unroll
            for (int i = 0; i < NA; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    total[i][j] += acc[i][j];
                    acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
                }
        }
        F32Split w[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            if constexpr (LINES) {
                const uint4 one = __builtin_bit_cast(uint4, rw[set][j][0]), two = __builtin_bit_cast(uint4, rw[set][j][1]);
                w[j] = f32_split8<false>(__builtin_bit_cast(f32x4_t, swap_halves<0xC>(one, two)), __builtin_bit_cast(f32x4_t, swap_halves<0x3>(two, one)));
            } else {
                w[j] = f32_split8<false>(rw[set][j][0], rw[set][j][1]);
            }
        }
        fetch_w(set, step + 2 * DEPTH);
        auto operand = [&](int i) {
            F32Split x;
            x.h = *(const f32_part8_t*)&Xs[buf][set & 1][0][i * 16 + li][at16];
            x.m = *(const f32_part8_t*)&Xs[buf][set & 1][1][i * 16 + li][at16];
            x.l = *(const f32_part8_t*)&Xs[buf][set & 1][2][i * 16 + li][at16];
            return x;
        };
#pragma unroll
        for (int i = 0; i + 1 < NA; i += 2) {
            const F32Split x[2] = {operand(i), operand(i + 1)};
            f32_split_multiply<NEG, 2, NT>(*(f32x4_t(*)[2][NT])&acc[i], w, x);
        }
        if constexpr (NA % 2) {
            const F32Split x[1] = {operand(NA - 1)};
            f32_split_multiply<NEG, 1, NT>(*(f32x4_t(*)[1][NT])&acc[NA - 1], w, x);
        }
    };
    auto loop = [&](auto blocks) {
        const fx_int<(decltype(blocks)::value + 1) / 2> some;
#pragma unroll
        for (int d = 0; d < 2 * DEPTH; ++d) fetch_x(some, d, d), fetch_w(d, d);
        keep(some, fx_int<0>{}, 0);
        keep(some, fx_int<1>{}, 0);
        fetch_x(some, 0, 2 * DEPTH);
        fetch_x(some, 1, 2 * DEPTH + 1);
        int buf = 0;
        auto two = [&](auto setc, int step, auto odd_too) {
            constexpr int set = decltype(setc)::value, next = (set + 2) % (2 * DEPTH);
            lds_barrier();
            multiply(blocks, setc, buf, step);
            if constexpr (decltype(odd_too)::value) {
                multiply(blocks, fx_int<set + 1>{}, buf, step + 1);
                buf ^= 1;
                keep(some, fx_int<next>{}, buf);
                keep(some, fx_int<next + 1>{}, buf);
                fetch_x(some, next, step + 2 + 2 * DEPTH);
                fetch_x(some, next + 1, step + 3 + 2 * DEPTH);
            }
        };
        int step = 0;
        for (; step + 2 * DEPTH <= n_steps; step += 2 * DEPTH)
            static_for(std::make_integer_sequence<int, DEPTH>{}, [&](auto u) { two(fx_int<2 * decltype(u)::value>{}, step + 2 * decltype(u)::value, fx_int<1>{}); });
        if (DEPTH == 2 && step + 2 <= n_steps) {
            two(fx_int<0>{}, step, fx_int<1>{});
            if (n_steps & 1) two(fx_int<2 * (DEPTH - 1)>{}, step + 2, fx_int<0>{});
        } else if (n_steps & 1) {
            two(fx_int<0>{}, step, fx_int<0>{});
        }
    };
    const int n_blocks = (min(TM, r_end - r0) + 15) >> 4;
    if (n_blocks == 1) loop(fx_int<1>{});
    else if (MB == 2 || n_blocks == 2) loop(fx_int<2>{});
    else if constexpr (MB > 2) {
        if (n_blocks == 3) loop(fx_int<3>{});
        else loop(fx_int<4>{});
    }
    f32x4_t(*other)[64] = (f32x4_t(*)[64]) & Xs[0][0][0][0][0];       // ROLES: up's sums, MB blocks of each of two waves
    if constexpr (ROLES) {
        __syncthreads();
        if (wave >= 2) {
#pragma unroll
            for (int i = 0; i < MB; ++i) other[(wave & 1) * MB + i][lane] = total[i][0] + acc[i][0];
        }
        __syncthreads();
        if (wave >= 2) return;
    }
    unsigned odd = 0;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        const int ml = r0 + i * 16 + li;
        if (ml >= r_end) continue;
#pragma unroll
        for (int j = 0; j < NT; j += PER) {
            const int n = n0 + j / PER * 16 + 4 * gq;
            const f32x4_t v = total[i][j] + acc[i][j], v2 = ROLES ? other[wave * MB + i][lane] : DUAL ? total[i][j + PER - 1] + acc[i][j + PER - 1] : v;
            if (!f32_sums_stand(v, DUAL ? v2 : v)) odd |= 1u << (i * (NT / PER) + j / PER);
            else f32_store4<DUAL, EPI>(g, f32_ask<DUAL, EPI>(g, ml, min(n, g.N - 1)), n, v, v2);
        }
    }
    if (__ballot(odd != 0) == 0) return;
#pragma unroll 1
    for (int i = 0; i < n_blocks; ++i)
#pragma unroll 1
        for (int t = 0; t < NT / PER; ++t) {
            if (__ballot(odd >> (i * (NT / PER) + t) & 1) == 0) continue;
            const float* x = a_row(i * 16 + li);
            const f32x4_t v = f32_whole_sum<VEC>(g.K, b_row(t, 0, li), x, gq), v2 = DUAL ? f32_whole_sum<VEC>(g.K, b_row(t, 1, li), x, gq) : v;
            const int n = n0 + t * 16 + 4 * gq;
            if (odd >> (i * (NT / PER) + t) & 1) f32_store4<DUAL, EPI>(g, f32_ask<DUAL, EPI>(g, r0 + i * 16 + li, min(n, g.N - 1)), n, v, v2);
        }
}

// Few rows: the weights go from memory straight into operands, every wave a part of K, 16 * MT rows and NW sets of 16
// weight rows a block (DUAL: the sets alternate between the two matrices); 32 k a step, the next step's loads issued
// before this step's products; the parts' sums meet in LDS.  LINES (rows of whole 32 k): the weights come in whole lines of 128 bytes
// with the non-temporal hint, the halves changing places before the products (`load_lines16`).  Bound by the stream of the weights: 4 rows
// against 6,144 x 2,048 15.5 us, gate/up of 5,632 24.3, 15 experts' gate/up 63 (5.5 TB/s), the head of 151,936 235 (5.3 TB/s).  With half
// lines and steps of 64 k these took 17.6, 30.0, 75 and 275: twice the registers a step leave half the waves, and it
// is waves, not deeper loads, that keep memory busy (steps of 128 k: 19.9, 33.3, 95 and 329).  SPLIT, us for 4 rows: 6,144 x 2,048 13.2, gate/up of 5,632 23.0, the head 204; with three steps on their way
// 2,048 x 2,048 8.0 instead of 7.1 and the head 277, with the next step taken apart beside this one's products 7.7 and 218.
template <int MT, int NW, bool DUAL, int EPI, bool VEC, bool LINES, bool HALF = false, bool SPLIT = false>
__global__ __launch_bounds__(512) void gemm_f32_skinny_kernel(GemmArgs g) {
    static_assert(!DUAL || NW % 2 == 0, "dual mode multiplies two matrices");
    static_assert(!HALF || (LINES && MT == 1), "sets of eight weight rows come in whole lines, for few rows");
    constexpr int CW = HALF ? 8 : 16;        // weight rows of a set
    __shared__ f32x4_t red[F32_PARTS][MT * NW][64];
    int r0, r_end, expert;
    locate_rows<16 * MT>(g, blockIdx.y, r0, r_end, expert);
    if (r0 < 0) return;
    const int n0 = blockIdx.x * (DUAL ? CW / 2 : CW) * NW;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, gq = lane >> 4;
    const float* Wbase = (const float*)g.W + (size_t)expert * g.w_stride;
    // SPLIT: the rows come in whole lines as well, the first load of 32 k with rows 0 .. 7 of a tile and the second with rows 8 .. 15, which a tile of up to eight rows does without
    // (2,048 x 5,632, 1 row 14.3 -> 13.2 us, 8 rows 15.4 -> 14.1, 32 rows 48.2 -> 44.1; 16 rows of half sets, where nothing hides that the halves change places, 18.8 and 18.9)
    constexpr bool XLINES = LINES && SPLIT;
    const float* x_src[MT][XLINES ? 2 : 1];
    constexpr int WR = LINES && !HALF ? 2 : 1;
    const float* w_src[NW][WR];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
        for (int half = 0; half < (XLINES ? 2 : 1); ++half) {
            int m = r0 + i * 16 + (XLINES ? (li & 7) + 8 * half : li);
            m = m < r_end ? m : r_end - 1;
            x_src[i][half] = (const float*)g.A + (size_t)(g.a_rows ? g.a_rows[m] : m) * g.lda + (XLINES ? (li >> 3) * 16 + gq * 4 : 0);
        }
    }
#pragma unroll
    for (int a = 0; a < NW; ++a) {
#pragma unroll
        for (int half = 0; half < WR; ++half) {
            // LINES: what the lane loads is of row li % 8, and (unless HALF) of row li % 8 + 8; else of row li
            int n = n0 + (DUAL ? a >> 1 : a) * CW + (LINES ? (li & 7) + 8 * half : li);
            n = n < g.N ? n : g.N - 1;
            w_src[a][half] = Wbase + (size_t)n * g.K + (DUAL && (a & 1) ? g.up_offset : 0) + (LINES ? (li >> 3) * 16 + gq * 4 : 0);
        }
    }
    const int part = SPLIT ? f32_split_part_length(g.K) : f32_part_length(g.K);
    const int k_first = wave * part, k_end = k_first + part < g.K ? k_first + part : g.K;
    constexpr int STEP = 2;       // groups of 16 k that are on their way together
    f32x4_t w[2][STEP][NW], x[2][STEP][MT];
    const int k_full = k_first + (k_end - k_first) / 16 * 16;
    auto fetch = [&](auto x_loads, int b, int k0) {
#pragma unroll
        for (int c = 0; c < STEP; ++c) {
            const int kc = k0 + c * 16, k = (kc < k_full ? kc : k_full - 16) + gq * 4;
#pragma unroll
            for (int a = 0; a < NW; ++a) {
                if constexpr (LINES) {
                    if (HALF && (c & 1)) continue;
                    const int pair = k0 + (c & ~1) * 16;        // 32 k, a line of each row
                    w[b][c][a] = __builtin_bit_cast(f32x4_t, load_lines16(w_src[a][HALF ? 0 : c & 1] + (pair < k_full ? pair : k_full - 32)));
                } else {
                    w[b][c][a] = f32_fetch<VEC>(w_src[a][0] + k);
                }
            }
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                if constexpr (!XLINES) x[b][c][i] = f32_fetch<VEC>(x_src[i][0] + k);
                else if (c < decltype(x_loads)::value) x[b][c][i] = f32_fetch<VEC>(x_src[i][c] + (k0 < k_full ? k0 : k_full - 32));
            }
        }
    };
    // the tile that this wave finishes, and what that needs besides the product
    constexpr int PER = DUAL ? 2 : 1;
    static_assert(MT * NW / PER <= F32_PARTS, "a wave finishes one tile at most");
    const int ti = wave * PER / NW % MT, ta = wave * PER % NW, out_row = r0 + ti * 16 + li, out_col = n0 + (DUAL ? ta >> 1 : ta) * CW + 4 * gq;
    const bool finishes = wave < MT * NW / PER && out_row < r_end && (!HALF || gq < 2) && out_col < g.N;
    F32Out<EPI> ask = {};
    if (finishes) ask = f32_ask<DUAL, EPI>(g, out_row, out_col);
    f32x4_t acc[MT][NW];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int a = 0; a < NW; ++a) acc[i][a] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    auto loop = [&](auto x_loads) {
        fetch(x_loads, 0, k_first);
        for (int k0 = k_first; k0 < k_full; k0 += 2 * STEP * 16) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int kb = k0 + b * STEP * 16;
                fetch(x_loads, b ^ 1, kb + STEP * 16);
                // what the lane multiplies of weight set a in group c of 16 k
                auto own = [&](int c, int a) -> f32x4_t {
                    if constexpr (!LINES) return w[b][c][a];
                    const uint4 keep = __builtin_bit_cast(uint4, w[b][HALF ? c & ~1 : c][a]), other = __builtin_bit_cast(uint4, w[b][HALF ? c & ~1 : c ^ 1][a]);
                    // (HALF: rows 8 .. 15 of the operand are the other k of rows 0 .. 7, and what they give is dropped)
                    if constexpr (HALF) return __builtin_bit_cast(f32x4_t, c & 1 ? swap_halves<0x3>(keep, other) : keep);
                    else return __builtin_bit_cast(f32x4_t, c & 1 ? swap_halves<0x3>(keep, other) : swap_halves<0xC>(keep, other));
                };
                if constexpr (SPLIT) {
                    if (kb < k_full) {          // (whole steps of 32 k)
                        F32Split ws[NW], xs[MT];
#pragma unroll
                        for (int a = 0; a < NW; ++a) {
                            if constexpr (HALF) ws[a] = f32_split_half<false>(w[b][0][a]);
                            else ws[a] = f32_split8<false>(own(0, a), own(1, a));
                        }
                        auto rows_of = [&](auto neg, int i) {
                            constexpr bool NEG = decltype(neg)::value;
                            if constexpr (!XLINES) return f32_split8<NEG>(x[b][0][i], x[b][1][i]);
                            else if constexpr (decltype(x_loads)::value == 1) return f32_split_half<NEG>(x[b][0][i]);
                            else {
                                const uint4 one = __builtin_bit_cast(uint4, x[b][0][i]), two = __builtin_bit_cast(uint4, x[b][1][i]);
                                return f32_split8<NEG>(__builtin_bit_cast(f32x4_t, swap_halves<0xC>(one, two)), __builtin_bit_cast(f32x4_t, swap_halves<0x3>(two, one)));
                            }
                        };
                        if (b & 1) {
#pragma unroll
                            for (int i = 0; i < MT; ++i) xs[i] = rows_of(std::true_type{}, i);
                            f32_split_multiply<true>(acc, ws, xs);
                        } else {
#pragma unroll
                            for (int i = 0; i < MT; ++i) xs[i] = rows_of(std::false_type{}, i);
                            f32_split_multiply<false>(acc, ws, xs);
                        }
                    }
                    continue;
                }
#pragma unroll
                for (int c = 0; c < STEP; ++c)
                    if (kb + c * 16 < k_full) {
                        f32x4_t ws[NW];
#pragma unroll
                        for (int a = 0; a < NW; ++a) ws[a] = own(c, a);
                        f32_multiply(acc, ws, x[b][c]);
                    }
            }
        }
    };
    if (k_first < k_full) {
        if (XLINES && MT == 1 && r_end - r0 <= 8) loop(fx_int<1>{});
        else loop(fx_int<2>{});
    }
    if (!LINES && !SPLIT && k_first < k_end && k_full < k_end) {       // the last, partial group of K
#pragma unroll
        for (int a = 0; a < NW; ++a) w[0][0][a] = f32_fetch_guarded<VEC>(w_src[a][0], k_full + gq * 4, k_end);
#pragma unroll
        for (int i = 0; i < MT; ++i) x[0][0][i] = f32_fetch_guarded<VEC>(x_src[i][0], k_full + gq * 4, k_end);
        f32_multiply(acc, w[0][0], x[0][0]);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int a = 0; a < NW; ++a) red[wave][i * NW + a][lane] = acc[i][a];
    __syncthreads();
    if (SPLIT ? wave >= MT * NW / PER : !finishes) return;
    f32x4_t v = red[0][ti * NW + ta][lane], v2 = v;
#pragma unroll
    for (int p = 1; p < F32_PARTS; ++p) v += red[p][ti * NW + ta][lane];
    if (DUAL) {
        v2 = red[0][ti * NW + ta + PER - 1][lane];
#pragma unroll
        for (int p = 1; p < F32_PARTS; ++p) v2 += red[p][ti * NW + ta + PER - 1][lane];
    }
    if constexpr (SPLIT) {
        const bool odd = finishes && !f32_sums_stand(v, DUAL ? v2 : v);
        if (__ballot(odd)) {            // (the whole wave: the products take all its lanes)
            const int m = min(r0 + ti * 16 + li, r_end - 1), n = min(n0 + (DUAL ? ta >> 1 : ta) * CW + (HALF ? li & 7 : li), g.N - 1);
            const float *x_row = (const float*)g.A + (size_t)(g.a_rows ? g.a_rows[m] : m) * g.lda, *w_row = Wbase + (size_t)n * g.K;
            const f32x4_t whole = f32_whole_sum<VEC>(g.K, w_row, x_row, gq), whole2 = DUAL ? f32_whole_sum<VEC>(g.K, w_row + g.up_offset, x_row, gq) : whole;
            if (odd) v = whole, v2 = whole2;
        }
        if (!finishes) return;
    }
    f32_store4<DUAL, EPI>(g, ask, out_col, v, v2);
}

// ===========================================================================
// host side
// ===========================================================================
template <int TM, int TN, int WM, int WN>
static void launch_bf16(GemmArgs g, int epi, int m_tiles, hipStream_t s) {
    const bool dual = epi == EPI_GATED;
    g.n_col_tiles = ceil_div(g.N, dual ? TN / 2 : TN);
    g.n_row_tiles = m_tiles;
    dim3 grid(8 * ceil_div((long)g.n_col_tiles * g.n_row_tiles, 8));
#define FX_TILED(DUAL_, EPI_)                                                                       \
    if (g.vec_ok) gemm_bf16_kernel<TM, TN, WM, WN, DUAL_, EPI_, true><<<grid, 256, 0, s>>>(g);     \
    else gemm_bf16_kernel<TM, TN, WM, WN, DUAL_, EPI_, false><<<grid, 256, 0, s>>>(g)
    switch (epi) {
        case EPI_STORE: FX_TILED(false, EPI_STORE); break;
        case EPI_STORE_F32: FX_TILED(false, EPI_STORE_F32); break;
        case EPI_RESID: FX_TILED(false, EPI_RESID); break;
        default: FX_TILED(true, EPI_GATED); break;
    }
#undef FX_TILED
}

// Switches for tests and measurement (ferrox_amd/debug.py is their one caller): they pick, whatever the sizes,
// a kernel variant that the sizes would otherwise choose.  The product path never sets them.
static int g_skinny_nw = 0;    // "skinny_sets": 1 or 2 sets of weight rows per wave of the product for few rows (0: by the sizes)
static int g_skinny_mt = 0;    // "skinny_row_tiles": 1, 2 or 4 tiles of 16 rows per block of that product (0: by the sizes)
static int g_skinny_waves = 0; // "skinny_waves": 1, 2, 4 or 8 waves that split K in a block of that product (0: by the sizes)
static int g_skinny_half = -1; // "skinny_half": 1 / 0 gives up to 16 plain rows blocks of half a set of weight rows or of whole ones (-1: by the sizes)
static int g_few_rows = 3;     // "few_rows": sorted by expert, up to this many rows an expert go to the product for few rows (at most 64)
static int g_head_rows = 16;   // "head_rows": plain rows against very many weight rows go to the tiled kernel from more than this many on
static int g_tile64_rows = 20; // "tile64_rows": experts with up to this many rows on average take tiles of 64 rows
static int g_no_wide = 0;      // "wide": 0 sends many-row products to the register-staged tiled kernel, 1 (default) by the sizes,
static int g_plain_rows = 0;   // "plain_rows": plain rows up to this many go to the product for few rows whatever the weight rows (0: by the sizes)
static int g_stream_w = -1;    // "stream_w": 1 / 0 forces the non-temporal hint on the tiled kernel's weight loads on / off; -1: by the shape
static int g_f32_split = -1;   // "f32_split": 1 / 0 works float32 products of whole 32 k out as bfloat16 ones or on the float32 instruction (-1: by the weights' size)
static int g_f32_tile = 0;     // "f32_tile": 1 sends float32 products to the kernel for few rows, 32 or 64 (taken apart also 48, 128, 144 and 160, see fx_gemm_f32_split_tile) to those tiles (0: by the sizes)
static int g_wide_grouped = 0; // "wide_grouped": as "wide", for products whose rows are sorted by expert only
static int g_wide_force = 0;   //         256, 192, 128, 64, 12 or 4 (tiles of 64 rows), 464, 4128 (64 x 64, 64 x 128), 8128 (128 x 128 in two stages), 8256 (128 x 256), 6128 or 6256 (96 rows), 1256 (sorted rows: 128 x 256 by the shares) or 1128 (128 x 128 in a ring) picks that tile of the LDS-tiled kernel
FX_API int fx_debug_set(const char* key, int value) {
    if (!strcmp(key, "skinny_sets")) { g_skinny_nw = value; return 0; }
    if (!strcmp(key, "skinny_row_tiles")) { g_skinny_mt = value; return 0; }
    if (!strcmp(key, "skinny_waves")) { g_skinny_waves = value; return 0; }
    if (!strcmp(key, "skinny_half")) { g_skinny_half = value; return 0; }
    if (!strcmp(key, "few_rows")) { g_few_rows = value < 0 ? 0 : (value > 64 ? 64 : value); return 0; }
    if (!strcmp(key, "tile64_rows")) { g_tile64_rows = value; return 0; }
    if (!strcmp(key, "head_rows")) { g_head_rows = value; return 0; }
    if (!strcmp(key, "wide")) { g_no_wide = !value; g_wide_force = value > 1 ? value : 0; return 0; }
    if (!strcmp(key, "wide_grouped")) { g_wide_grouped = value > 1 ? value : 0; return 0; }
    if (!strcmp(key, "stream_w")) { g_stream_w = value; return 0; }
    if (!strcmp(key, "f32_tile")) { g_f32_tile = value; return 0; }
    if (!strcmp(key, "f32_split")) { g_f32_split = value; return 0; }
    if (!strcmp(key, "plain_rows")) { g_plain_rows = value; return 0; }
    FX_REQUIRE(false, "gemm: no debug switch '%s' (skinny_sets, skinny_row_tiles, skinny_waves, skinny_half, few_rows, head_rows, tile64_rows, wide, wide_grouped, stream_w, plain_rows, f32_tile, f32_split)", key);
    return 1;
}

// The grid of the LDS-tiled kernels, which decode their block's tile themselves.
static dim3 wide_grid(GemmArgs& g, int epi, int tn, int m_tiles) {
    g.n_col_tiles = ceil_div(g.N, epi == EPI_GATED ? tn / 2 : tn);
    g.n_row_tiles = m_tiles;
    return dim3(g.by_row_tile && g.expert_offsets ? 8 * ceil_div(m_tiles, 8) * g.n_col_tiles : 8 * ceil_div((long)g.n_col_tiles * m_tiles, 8));
}
template <int TMB, int TN, int NS, int NSA, bool STREAM, bool SPREAD = false>
static void launch_wide(GemmArgs g, int epi, int m_tiles, hipStream_t s) {
    g.tile_rows = 16 * TMB;
    const dim3 grid = wide_grid(g, epi, TN, m_tiles);
    switch (epi) {
        case EPI_STORE: gemm_bf16_wide_kernel<TMB, TN, NS, false, EPI_STORE, NSA, STREAM, SPREAD><<<grid, 512, 0, s>>>(g); break;
        case EPI_STORE_F32: gemm_bf16_wide_kernel<TMB, TN, NS, false, EPI_STORE_F32, NSA, STREAM, SPREAD><<<grid, 512, 0, s>>>(g); break;
        case EPI_RESID: gemm_bf16_wide_kernel<TMB, TN, NS, false, EPI_RESID, NSA, STREAM, SPREAD><<<grid, 512, 0, s>>>(g); break;
        default:
            if constexpr (TN % 128 == 0) gemm_bf16_wide_kernel<TMB, TN, NS, true, EPI_GATED, NSA, STREAM, SPREAD><<<grid, 512, 0, s>>>(g);
            break;
    }
}
template <int TMB, int TN>
static void launch_quarters(GemmArgs g, int epi, int m_tiles, hipStream_t s, int rows = 16 * TMB) {
    g.tile_rows = rows;
    const dim3 grid = wide_grid(g, epi, TN, m_tiles);
    switch (epi) {
        case EPI_STORE: gemm_bf16_quarters_kernel<TMB, TN, false, EPI_STORE><<<grid, 512, 0, s>>>(g); break;
        case EPI_STORE_F32: gemm_bf16_quarters_kernel<TMB, TN, false, EPI_STORE_F32><<<grid, 512, 0, s>>>(g); break;
        case EPI_RESID: gemm_bf16_quarters_kernel<TMB, TN, false, EPI_RESID><<<grid, 512, 0, s>>>(g); break;
        default:
            if constexpr (TN % 128 == 0) gemm_bf16_quarters_kernel<TMB, TN, true, EPI_GATED><<<grid, 512, 0, s>>>(g);
            break;
    }
}
template <int TMB, int TN, int NS, bool SPREAD>
static void launch_shares(GemmArgs g, int epi, int m_tiles, hipStream_t s) {
    g.tile_rows = 16 * TMB;
    const dim3 grid = wide_grid(g, epi, TN, m_tiles);
    switch (epi) {
        case EPI_STORE: gemm_bf16_shares_kernel<TMB, TN, NS, false, EPI_STORE, SPREAD><<<grid, 512, 0, s>>>(g); break;
        case EPI_STORE_F32: gemm_bf16_shares_kernel<TMB, TN, NS, false, EPI_STORE_F32, SPREAD><<<grid, 512, 0, s>>>(g); break;
        case EPI_RESID: gemm_bf16_shares_kernel<TMB, TN, NS, false, EPI_RESID, SPREAD><<<grid, 512, 0, s>>>(g); break;
        default: gemm_bf16_shares_kernel<TMB, TN, NS, true, EPI_GATED, SPREAD><<<grid, 512, 0, s>>>(g); break;
    }
}
// Weights that are read about once go through the ring with the non-temporal hint, everything else in quarters.
template <int TMB, int TN, int NS, int NSA = NS>
static void launch_ring_or_quarters(const GemmArgs& g, int epi, int m_tiles, hipStream_t s) {
    if (g.stream_w) launch_wide<TMB, TN, NS, NSA, true>(g, epi, m_tiles, s);
    else launch_quarters<TMB, TN>(g, epi, m_tiles, s);
}
template <int TMB, int TN, int NS, int NSA = NS>
static void launch_ring(const GemmArgs& g, int epi, int m_tiles, hipStream_t s) {
    if (g.stream_w) launch_wide<TMB, TN, NS, NSA, true>(g, epi, m_tiles, s);
    else launch_wide<TMB, TN, NS, NSA, false>(g, epi, m_tiles, s);
}
template <bool DUAL, int EPI, bool VEC, bool LINES, bool SPLIT>
static void launch_f32_skinny(const GemmArgs& g, int mt, int nw, bool half, dim3 grid, hipStream_t s) {
    if constexpr (LINES) {
        if (half) {
            gemm_f32_skinny_kernel<1, DUAL ? 2 : 1, DUAL, EPI, VEC, LINES, true, SPLIT><<<grid, 512, 0, s>>>(g);
            return;
        }
    }
    if (mt == 2) gemm_f32_skinny_kernel<2, 2, DUAL, EPI, VEC, LINES, false, SPLIT><<<grid, 512, 0, s>>>(g);
    else if (nw == 2 || DUAL) gemm_f32_skinny_kernel<1, 2, DUAL, EPI, VEC, LINES, false, SPLIT><<<grid, 512, 0, s>>>(g);
    else gemm_f32_skinny_kernel<1, DUAL ? 2 : 1, DUAL, EPI, VEC, LINES, false, SPLIT><<<grid, 512, 0, s>>>(g);
}
template <bool DUAL, int EPI, bool VEC>
static void launch_f32(const GemmArgs& g, bool split, int tile, int stream, int mt, int nw, bool half, dim3 grid, hipStream_t s) {
    if (tile && split) {
        if (tile >= 128) gemm_f32_split_kernel<64, 2, 1, DUAL, EPI, VEC, false><<<grid, 256, 0, s>>>(g);
        else if (tile == 32) {
            if (VEC && stream) gemm_f32_split_kernel<32, 1, 2, DUAL, EPI, VEC, VEC><<<grid, 256, 0, s>>>(g);
            else gemm_f32_split_kernel<32, 1, 2, DUAL, EPI, VEC, false><<<grid, 256, 0, s>>>(g);
        } else if constexpr (VEC) {
            if (stream == 2) gemm_f32_split_kernel<64, 1, 2, DUAL, EPI, true, true><<<grid, 256, 0, s>>>(g);
            else if (stream) gemm_f32_split_kernel<64, 1, 1, DUAL, EPI, true, true><<<grid, 256, 0, s>>>(g);
            else gemm_f32_split_kernel<64, 1, 1, DUAL, EPI, true, false><<<grid, 256, 0, s>>>(g);
        } else {
            gemm_f32_split_kernel<64, 1, 1, DUAL, EPI, false, false><<<grid, 256, 0, s>>>(g);
        }
    } else if (tile == 64) gemm_f32_tiled_kernel<64, 64, DUAL, EPI, VEC><<<grid, 256, 0, s>>>(g);
    else if (tile == 32) gemm_f32_tiled_kernel<32, DUAL ? 64 : 32, DUAL, EPI, VEC><<<grid, 256, 0, s>>>(g);
    else if (VEC && g.K % 32 == 0) {
        if (split) launch_f32_skinny<DUAL, EPI, VEC, VEC, true>(g, mt, nw, half, grid, s);
        else launch_f32_skinny<DUAL, EPI, VEC, VEC, false>(g, mt, nw, half, grid, s);
    } else if (split) launch_f32_skinny<DUAL, EPI, VEC, false, true>(g, mt, nw, false, grid, s);
    else launch_f32_skinny<DUAL, EPI, VEC, false, false>(g, mt, nw, false, grid, s);
}

template <int MT, int WAVES, int NW, bool HALF = false, int DEPTH = 2>
static void launch_skinny_cfg(const GemmArgs& g, int epi, int m_tiles, hipStream_t s) {
    dim3 grid(ceil_div(g.N, (epi == EPI_GATED ? 8 : 16) * NW / (HALF ? 2 : 1)), m_tiles);
    if constexpr (MT * NW * WAVES <= 32) {       // the partial sums of all waves fit in LDS
        if constexpr (!HALF) {
            if (g.norm_w) {
                gemm_bf16_skinny_kernel<MT, WAVES, NW, false, EPI_STORE, true><<<grid, WAVES * 64, 0, s>>>(g);
                return;
            }
        }
        if constexpr (!(HALF && NW == 2)) {
            switch (epi) {
                case EPI_STORE: gemm_bf16_skinny_kernel<MT, WAVES, NW, false, EPI_STORE, false, false, HALF, DEPTH><<<grid, WAVES * 64, 0, s>>>(g); return;
                case EPI_STORE_F32: gemm_bf16_skinny_kernel<MT, WAVES, NW, false, EPI_STORE_F32, false, false, HALF, DEPTH><<<grid, WAVES * 64, 0, s>>>(g); return;
                case EPI_RESID: gemm_bf16_skinny_kernel<MT, WAVES, NW, false, EPI_RESID, false, false, HALF, DEPTH><<<grid, WAVES * 64, 0, s>>>(g); return;
                default: break;
            }
        }
        if constexpr (NW % 2 == 0) gemm_bf16_skinny_kernel<MT, WAVES, NW, true, EPI_GATED, false, false, HALF, DEPTH><<<grid, WAVES * 64, 0, s>>>(g);
    }
}

// mt: row tiles per block (1, 2, 4); nw: 16-row weight sets per wave; waves: 4 or 8 split K (1 or 2 with one row tile).
// half sets: four pieces on their way where that is a wave's whole part of K, or where rows are so few that their operands do not fill the way
static bool four_pieces(int M, int K) { return K <= 2048 || M <= 4; }
static void launch_skinny(const GemmArgs& g, int epi, int mt, int nw, int waves, bool half, int m_tiles, hipStream_t s) {
    if (half) {
        const bool deep = four_pieces(g.M, g.K);
        if (epi == EPI_GATED) {
            if (deep) launch_skinny_cfg<1, 4, 2, true, 4>(g, epi, m_tiles, s);
            else launch_skinny_cfg<1, 4, 2, true>(g, epi, m_tiles, s);
        } else {
            if (deep) launch_skinny_cfg<1, 4, 1, true, 4>(g, epi, m_tiles, s);
            else launch_skinny_cfg<1, 4, 1, true>(g, epi, m_tiles, s);
        }
        return;
    }
#define FX_SK(MT_, W_, NW_) launch_skinny_cfg<MT_, W_, NW_>(g, epi, m_tiles, s)
    if (waves == 8 && mt * nw <= 4) {
        if (nw == 2) {
            if (mt == 1) FX_SK(1, 8, 2);
            else FX_SK(2, 8, 2);
        } else {
            if (mt == 1) FX_SK(1, 8, 1);
            else if (mt == 2) FX_SK(2, 8, 1);
            else FX_SK(4, 8, 1);
        }
        return;
    }
    if (waves <= 2 && mt == 1) {
        if (waves == 1) {
            if (nw == 2) FX_SK(1, 1, 2);
            else FX_SK(1, 1, 1);
        } else {
            if (nw == 2) FX_SK(1, 2, 2);
            else FX_SK(1, 2, 1);
        }
        return;
    }
    if (nw == 2) {
        if (mt == 1) FX_SK(1, 4, 2);
        else if (mt == 2) FX_SK(2, 4, 2);
        else FX_SK(4, 4, 2);
    } else {
        if (mt == 1) FX_SK(1, 4, 1);
        else if (mt == 2) FX_SK(2, 4, 1);
        else FX_SK(4, 4, 1);
    }
#undef FX_SK
}

// Whether the first weights of the rotating product leave before the sums of squares of its rows have arrived.  What else its epilogue needs then waits for the weights, so it pays
// with sums of one batch and k enough, or rows (us, weights behind / first; 2,048 k and 6,144 columns, 1 row 9.1 8.7, 8 9.9 9.3, 16 11.2 10.4; 1,024 k, 16 rows 6.9 6.4; in a step of one
// sequence, where the kernel before has just written the sums, 24 layers take 1,781 us with the weights behind, so 1,763; but without sums 16 rows 10.4 10.7, 2 rows of 1,024 k 6.5
// 6.7; sums of two batches, 3,584 k, 2 rows 12.0 12.7, 17 rows 16.8 18.0; two row tiles of 2,048 k with sums 13.1 13.5).
FX_API int fx_qkv_rope_weights_first(int M, int K, int sums) { return M <= 16 && sums >= 1 && sums <= 8 && (K > 1024 || (long)M * K >= 16384); }

// Row tiles of 16 a block of the rotating product takes: the fewest with which its blocks are one round of the CUs, or else all rows' (a block fetches the operands of its row
// tiles itself and finds weights that another block has fetched in the cache; what takes the time is the CU with the most blocks).  us with sums, 1 / 2 / 3 or 4 tiles a block:
//   48 groups of columns (1,024 k)    32 rows 8.5 9.5, 48 rows 8.6 9.2 11.2, 64 rows 8.6 9.4 12.5
//   144 (3,584 k)    24 rows 24.0 18.1, 48 rows 27.7 29.8 23.9, 64 rows 37.9 32.3 28.6
//   192 (2,048 k)    24 rows 18.0 14.8, 33 rows 23.3 20.0 16.3, 48 rows 26.2 21.9 18.3, 64 rows 27.3 23.1 21.4     192 (4,096 k)    48 rows 42.6 35.4 26.3, 64 rows 44.6 37.5 31.2
// (Two tiles a block from 17 rows on, as it was, with sums found by every lane: 64 rows of the four 10.5, 35.2, 25.8 and 39.5.)  The same bits whatever the tiles.
FX_API int fx_qkv_rope_row_tiles(int M, int groups, int cus) {
    const int tiles = ceil_div(M, 16);
    for (int mt = 1; mt < tiles; ++mt)
        if ((long)groups * ceil_div(tiles, mt) <= cus) return mt;
    return tiles;
}

// The q/k/v product of up to 64 tokens with the rotation and the cache write in its epilogue (see GemmArgs):
// bfloat16, C [M, (nh + 2 nkv) hd], bias [N] or null, row_ss as in fx_gemm.  head_dim and the rotary dimension
// are multiples of 32.  k_pages [pages][nkv][bs][hd] and v_pages [pages][nkv][hd][bs], or both null.
FX_API int fx_qkv_rope(void* stream, const void* A, long lda, const void* W, long kb_rows, const void* bias, int bias_dtype,
                       void* C, long ldc, int M, int K, const float* row_ss, int row_ss_n, float eps,
                       const int* positions, const int* token_seq, const int* table, int max_blocks,
                       void* k_pages, void* v_pages, int nh, int nkv, int hd, int bs, int rot, const float* inv_freq,
                       const float* freq_factors) {
    FX_REQUIRE(M >= 1 && M <= 64 && K > 0 && K % 8 == 0 && lda % 8 == 0 && lda >= K, "qkv_rope: 1..64 rows of a multiple of 8 elements");
    FX_REQUIRE(nh > 0 && nkv > 0 && hd > 0 && hd % 32 == 0 && rot >= 0 && rot <= hd && rot % 32 == 0 && bs > 0,
               "qkv_rope: head_dim %d and rotary dimension %d must be multiples of 32", hd, rot);
    const int N = (nh + 2 * nkv) * hd;
    FX_REQUIRE(ldc >= N && (((uintptr_t)A | (uintptr_t)W) % 16) == 0, "qkv_rope: output rows too short or operands not aligned");
    FX_REQUIRE((k_pages == nullptr) == (v_pages == nullptr), "qkv_rope: key and value pages must come together");
    FX_REQUIRE(positions && token_seq && (!k_pages || (table && max_blocks > 0)), "qkv_rope: positions, sequences and block table");
    FX_REQUIRE(inv_freq || rot == 0, "qkv_rope: a rotation needs the table of its %d frequencies", rot / 2);
    FX_REQUIRE(!bias || bias_dtype == FX_F32 || bias_dtype == FX_BF16, "qkv_rope: unknown bias dtype %d", bias_dtype);
    FX_REQUIRE(kb_rows == 0 || (kb_rows == N && K % 64 == 0), "qkv_rope: weights in slabs of 64 k hold all %d rows", N);
    FX_REQUIRE(!row_ss || row_ss_n >= 1, "qkv_rope: sums of squares without their count");
    GemmArgs g = {};
    g.A = A; g.lda = lda; g.W = W; g.kb_stride = kb_rows * 64; g.bias = bias; g.bias_dtype = bias_dtype;
    g.C = C; g.ldc = ldc; g.M = M; g.N = N; g.K = K; g.vec_ok = 1;
    g.row_ss = row_ss; g.row_ss_n = row_ss_n; g.norm_eps = eps;
    g.rope_positions = positions; g.rope_token_seq = token_seq; g.rope_table = table; g.rope_max_blocks = max_blocks;
    g.rope_k_pages = k_pages; g.rope_v_pages = v_pages;
    g.rope_nh = nh; g.rope_nkv = nkv; g.rope_hd = hd; g.rope_bs = bs; g.rope_rot = rot;
    g.rope_inv_freq = inv_freq ? inv_freq : (const float*)positions;      // (rot == 0: read, never used)
    g.rope_freq_factors = freq_factors;
    dim3 grid((nh + 2 * nkv) * (hd / 32), 1);
    const int mt = fx_qkv_rope_row_tiles(M, (int)grid.x, fx_compute_units());
    grid.y = ceil_div(M, 16 * mt);
    hipStream_t s = (hipStream_t)stream;
    if (row_ss && fx_qkv_rope_weights_first(M, K, row_ss_n))
        gemm_bf16_skinny_kernel<1, 4, 2, false, EPI_STORE, false, true, false, 2, true><<<grid, 256, 0, s>>>(g);
    else if (mt == 1) gemm_bf16_skinny_kernel<1, 4, 2, false, EPI_STORE, false, true><<<grid, 256, 0, s>>>(g);
    else if (mt == 2) gemm_bf16_skinny_kernel<2, 4, 2, false, EPI_STORE, false, true><<<grid, 256, 0, s>>>(g);
    else if (mt == 3) gemm_bf16_skinny_kernel<3, 4, 2, false, EPI_STORE, false, true><<<grid, 256, 0, s>>>(g);
    else gemm_bf16_skinny_kernel<4, 4, 2, false, EPI_STORE, false, true><<<grid, 256, 0, s>>>(g);
    FX_CHECK_LAUNCH("qkv_rope");
    return 0;
}

// ---- decisions by sizes that are plain arithmetic (the compute units are an argument: they can be asked for without a GPU) ----
// 33 to 128 plain rows against so few weight rows that blocks of several row tiles are a fraction of the CUs (a router of 61
// rows as the rows, the step's tokens as the weights): whether a block takes one row tile and one set of weight rows.  Up to 64 rows,
// where the other way is four row tiles a block, while such blocks are at most one and a quarter a CU (2,048 k, 61 rows: 1,024
// weight rows 7.4 against 12.3 us, 1,280 10.2 against 12.2); beyond, where it is two, at most one a CU (96 rows: 640 weight rows 7.2 against
// 8.6 us, 768 10.4 against 8.8; 4,096 k 10.9 against 14.1 and 17.6 against 14.4).  (2,048 tokens with two row tiles a block instead of four
// took 10.6 instead of 14.9 us, but the step, whose routing runs beside the shared expert, 0.5 % longer.)
FX_API int fx_gemm_row_tile_blocks(int M, int N, int cus) {
    const long blocks = (long)ceil_div(N, 16) * ceil_div(M, 16);
    return M > 32 && M <= 128 && (M <= 64 ? 4 * blocks <= 5L * cus : blocks <= cus);
}

// Up to 16 plain rows: whether a block takes half a set of weight rows (8, or 8 of each of two matrices).  A CU gets no more than some 11 bytes a cycle from
// memory, whatever its blocks have on their way (23 MB in 128 blocks took 10.4 us, in 256 blocks of half as much 7.9), so what counts is how many rows the busiest CU
// fetches: a block's weight rows, and its rows of A, which come from the caches and count half.  us, blocks of whole / half sets, at 1, 8 and 16 rows:
//   2,048 x 2,048 5.3 4.4, 5.8 5.0, 6.3 5.7     2,048 x 5,632 10.4 7.9, 10.8 8.8, 12.6 10.4     1,024 x 2,048 5.0 3.8, 5.5 4.5, 6.0 5.3
//   gate/up of 1,408 x 2,048 6.8 5.1, 7.4 5.8, 7.9 6.5, of 5,632 12.4 11.2, 13.6 12.0, 14.3 14.0     6,144 x 2,048 7.9 7.0, 8.1 8.7, 8.6 10.3
//   the other way 2,560 x 2,048 5.3 5.3, 5.8 6.5, 6.3 8.0     3,584 x 3,584 7.7 8.0, 8.3 10.2, 9.4 12.9     4,096 x 1,024 3.9 4.1, 4.4 4.6, 4.5 5.7
// That holds where blocks of half sets are one round of the CUs.  Beyond, more blocks pay each block's start and end more often, and the rule is only taken where it was measured ahead: up
// to 24 columns a CU with two matrices, up to 40 for one or two rows of one, sums of 2,048 and more in both (`fx_gemm`: a wave's part is four pieces or more then).  Elsewhere, at 1 and 4 rows:
//   4,608 x 1,024 4.5 4.8, 4.8 5.3     5,632 x 5,632 16.9 16.6, 15.2 17.0     12,288 x 3,584 19.0 20.2, 20.1 21.1     20,480 x 1,024 10.1 12.2, 9.8 13.5     50,257 x 2,048 35.0 39.6, 35.7 44.5
//   gate/up of 4,608 x 1,024 6.6 7.5, 7.0 8.0, of 9,216 x 1,024 8.6 10.8, 9.2 11.5, x 5,632 40.4 39.1, 41.8 42.1, of 18,432 x 2,048 26.0 27.5, 25.7 28.0
FX_API int fx_gemm_half_sets(int M, int N, int dual, int sets, int cus) {
    if (ceil_div(N, 8) > cus && (dual ? N > 24 * cus : M > 2 || N > 40 * cus)) return 0;
    auto cost = [&](int columns, int weight_rows) { return ceil_div(ceil_div(N, columns), cus) * (2L * weight_rows + M); };
    return M <= 16 && (dual ? cost(8, 16) < cost(8 * sets, 16 * sets) : cost(8, 8) < cost(16 * sets, 16 * sets));
}

// Whether a float32 product is worked out from operands taken apart into bfloat16 ones (gemm_f32_split_kernel, and in the kernel for few rows): by the weights alone, so that the bits of a row
// do not depend on the rows beside it.  Whole steps of 32 k; sums of 1,024 and more, where the error is a half to a sixth of the float32 instruction's (it is level around 64); and weights of more than a million numbers, up to which the
// products are a few microseconds either way (us of 1,024 x 1,024, float32 instruction / taken apart: 1 row 4.5 4.6, 48 rows 13.4 14.4, 256 14.1 15.0, 512 18.6 16.2; of 512 x 2,048 1 row 6.1 6.2, 48 rows 23.6 23.5) and some have their sums repeated elsewhere in the float32 order (`f32_ordered_dot`).
FX_API int fx_gemm_f32_split(int N, int K) { return K % 32 == 0 && K >= 1024 && (long)N * K > 1L << 20; }

// The tile of such a product of plain rows, more than a few: its rows (32, 48 or 64) by 64 columns, or, as 128, 144 and 160, 64, 48 or 32 rows by 128
// columns (dual: half as many of both matrices).  The time goes with how many blocks the busiest CU gets: us of a first block, of each further one and beside them, of 2,048 k
// (1 to 6 blocks; up to 32 rows 32 x 64, one reading of the weights: 32 x 64 25 40 60 76 93 115; 48 x 64 34 50 70 88 104 131; 64 x 64 42 57 85 113 131 172; 32 x 128 49 70 107 137; 48 x 128 51 83 127 154 205 248; 64 x 128 59 92 141 184 229); other k in proportion.
// (whether blocks of 64 columns, of dual 32 of both matrices, are at most one a CU)
static bool fx_gemm_f32_one_round(int N, int dual, int cus) { return ceil_div(N, dual ? 32 : 64) <= cus; }
FX_API int fx_gemm_f32_split_tile(int M, int N, int dual, int cus) {
    static const struct { int code, rows, columns; float first, each, beside; } kinds[] = {
        {32, 32, 64, 25, 18.5f, 4}, {48, 48, 64, 34, 20.5f, 8}, {64, 64, 64, 42, 28.3f, 0}, {160, 32, 128, 49, 33, 5}, {144, 48, 128, 51, 41, 3}, {128, 64, 128, 59, 46, 2}};
    if (M <= 32) return 32;
    // Up to 64 rows while one row tile's blocks are one a CU: 32 x 64, two row tiles, where those are one block a CU too, else one row tile, so that the weights are read once, in whole lines and two stages ahead (us with weights from memory, float32
    // instruction / 32 x 64 / so: 33 rows and gate/up of 5,632 42.6 43.3 37.7, of 8,192 50.2 53.3 38.6, 64 rows 44.2 45.8 43.1 and 51.4 55.4 45.9, 48 rows against 9,216 40.6 39.2 36.4; gate/up of 4,096, 256
    // such blocks, 33 rows 31.0 26.9 37.4, 64 rows 31.9 27.8 43.0; with more blocks the table below is ahead of it: 64 rows against 40,960 weight rows 98 and 104).
    if (M <= 64 && fx_gemm_f32_one_round(N, dual, cus)) return 2L * ceil_div(N, dual ? 32 : 64) <= cus ? 32 : 64;
    int best = 128;
    float least = INFINITY;
    for (const auto& k : kinds) {
        const int blocks = ceil_div((long)ceil_div(N, dual ? k.columns / 2 : k.columns) * ceil_div(M, k.rows), cus);
        const float us = blocks == 1 ? k.first : k.each * blocks + k.beside;
        if (us < least) least = us, best = k.code;
    }
    return best;
}

// How the product for few rows takes up to 16 plain rows: sets of weight rows a wave has, waves a block, half sets or whole ones, pieces of K on their way (half sets only).  Two
// sets share the activations that they multiply and halve the blocks' fixed work; one where two would leave too few blocks to keep the memory busy, or where a row or two
// meet so many weight rows that the blocks are plenty either way.
struct FewRows {
    int sets, waves;
    bool half, deep;
};
static FewRows few_plain_rows(int M, int N, int K, bool dual, int cus) {
    FewRows f;
    f.sets = dual || ceil_div(N, 32) >= 160 ? 2 : 1;
    if (!dual && M <= 2 && ceil_div(N, 16) >= 4096) f.sets = 1;
    if ((g_skinny_nw == 1 && !dual) || g_skinny_nw == 2) f.sets = g_skinny_nw;
    f.waves = g_skinny_waves == 8 || g_skinny_waves == 2 || g_skinny_waves == 1 ? g_skinny_waves : 4;
    f.half = f.waves == 4 && (g_skinny_half >= 0 ? g_skinny_half != 0 : (K >= 2048 || ceil_div(N, 8) <= cus) && fx_gemm_half_sets(M, N, dual, f.sets, cus));
    f.deep = four_pieces(M, K);
    return f;
}

// A product of up to 16 plain bfloat16 rows for `fx_gemm_pair`.
struct FxProduct {
    const void *A, *W;
    void* C;
    const int* turn_positions;
    const float* turn_inv_freq;
    long lda, ldc, up_offset;
    int epi, M, N, K, act, turn_width, turn_from, turn_dims;
    float act_limit, act_alpha, turn_magnitude;
};
// Whether two such products go out in one launch: the first one's kernel is the one for half sets of weight rows (gate/up with four pieces on their way).
FX_API int fx_gemm_pairs(int M, int epi, int N, int K, int epi2, int N2, int K2, int cus) {
    const FewRows f = few_plain_rows(M, N, K, epi == EPI_GATED, cus);
    return M >= 1 && M <= 16 && K % 8 == 0 && K2 % 8 == 0 && N2 < 65536 && N < 65536 && (epi2 == EPI_STORE || epi2 == EPI_STORE_F32) &&
           f.waves == 4 && f.half && (epi == EPI_STORE_F32 || (epi == EPI_GATED && f.deep));
}
FX_API int fx_gemm_pair(void* stream, const FxProduct* first, const FxProduct* second) {
    const int cus = fx_compute_units();
    const FxProduct* products[2] = {first, second};
    FX_REQUIRE(first && second && first->M == second->M && fx_gemm_pairs(first->M, first->epi, first->N, first->K, second->epi, second->N, second->K, cus),
               "gemm_pair: up to 16 rows of a product in half sets of weight rows and of one that is stored");
    GemmArgs g[2] = {};
    for (int i = 0; i < 2; ++i) {
        const FxProduct& p = *products[i];
        FX_REQUIRE(p.A && p.W && p.C && p.N > 0 && p.K > 0 && p.lda >= p.K && p.ldc >= p.N && p.lda % 8 == 0 && p.up_offset % 8 == 0 && (((uintptr_t)p.A | (uintptr_t)p.W) % 16) == 0,
                   "gemm_pair: operands of product %d are not aligned rows", i);
        FX_REQUIRE(p.act >= 0 && p.act < ACT_COUNT && (p.act != ACT_SWIGLU_CLAMP || p.act_limit > 0.f), "gemm_pair: activation %d", p.act);
        FX_REQUIRE(p.turn_width == 0 || (i == 1 && p.epi == EPI_STORE && p.turn_positions && p.turn_inv_freq && p.turn_from >= 0 && p.turn_dims >= 0 && p.turn_from % 2 == 0 &&
                                         p.turn_dims % 2 == 0 && p.turn_width % 2 == 0 && p.turn_from + p.turn_dims <= p.turn_width && p.N % p.turn_width == 0),
                   "gemm_pair: %d turned dimensions from %d on of heads of %d", p.turn_dims, p.turn_from, p.turn_width);
        g[i].A = p.A; g[i].lda = p.lda; g[i].W = p.W; g[i].C = p.C; g[i].ldc = p.ldc; g[i].up_offset = p.up_offset;
        g[i].M = p.M; g[i].N = p.N; g[i].K = p.K; g[i].act = p.act; g[i].act_limit = p.act_limit; g[i].act_alpha = p.act_alpha; g[i].vec_ok = 1;
        if (p.turn_width) {
            g[i].rope_positions = p.turn_positions; g[i].rope_inv_freq = p.turn_inv_freq; g[i].act_alpha = p.turn_magnitude;
            g[i].rope_hd = p.turn_width; g[i].rope_nh = p.turn_from; g[i].rope_rot = p.turn_dims;
        }
    }
    FX_REQUIRE(first->turn_width == 0, "gemm_pair: the first product is not turned");
    const FewRows f = few_plain_rows(first->M, first->N, first->K, first->epi == EPI_GATED, cus), f2 = few_plain_rows(second->M, second->N, second->K, false, cus);
    const int blocks = ceil_div(first->N, 8), blocks2 = ceil_div(second->N, f2.half ? 8 : 16 * f2.sets);
    const dim3 grid(blocks + blocks2);
    hipStream_t s = (hipStream_t)stream;
    auto go = [&](auto gated, auto depth, auto sets, auto half) {
        if (second->epi == EPI_STORE) gemm_bf16_skinny_pair_kernel<decltype(gated)::value, decltype(depth)::value, decltype(sets)::value, EPI_STORE, decltype(half)::value><<<grid, 256, 0, s>>>(g[0], g[1], blocks);
        else gemm_bf16_skinny_pair_kernel<decltype(gated)::value, decltype(depth)::value, decltype(sets)::value, EPI_STORE_F32, decltype(half)::value><<<grid, 256, 0, s>>>(g[0], g[1], blocks);
    };
    auto with_second = [&](auto gated, auto depth) {
        if (f2.half) go(gated, depth, fx_int<1>{}, std::true_type{});
        else if (f2.sets == 1) go(gated, depth, fx_int<1>{}, std::false_type{});
        else go(gated, depth, fx_int<2>{}, std::false_type{});
    };
    if (first->epi == EPI_GATED) with_second(std::true_type{}, fx_int<4>{});
    else if (f.deep) with_second(std::false_type{}, fx_int<4>{});
    else with_second(std::false_type{}, fx_int<2>{});
    FX_CHECK_LAUNCH("gemm_pair");
    return 0;
}

// The tile of the LDS-tiled kernel for plain rows, as the debug switch "wide" names them; all give the same bits.  `dual`: N
// columns of two matrices.  (The times beside the lines, from 128 x 128 on, are those of tiles in rings of stages.  In quarters these take 7
// to 18 % less and what is ahead of another of them stays ahead: 4,096 rows against 4,608 weight rows of 3,584 k 149.5 -> 129 us with 256 x 192, 157 with 256 x 256;
// gate/up of 11,264, 2,048 rows 100 -> 91 with 192 x 256, 113 with 256 x 256; 2,048 rows against 2,048 of 5,632 k 55 -> 50 with 128 x 128, 62 with 128 x 256.)
FX_API int fx_gemm_plain_tile(int M, int N, int K, int dual, int cus) {
    auto tiles = [&](int tm, int tn) { return (long)ceil_div(N, dual ? tn / 2 : tn) * ceil_div(M, tm); };
    // Fewer tiles of 128 x 128 than CUs: a block's chain of K steps takes the same 23-25 us (2,048 k) whatever the rows, so
    // smaller tiles on more CUs: 64 x 64 while they are one a CU (2,048 x 2,048 weights, 512 rows 23 -> 13 us; 5,632 k 55 -> 29;
    // 6,144 weight rows, 128 rows 25 -> 14), then 64 x 128 (6,144 weight rows, 256 rows 25 -> 19; 2,048 x 5,632, 1,024 rows 56 -> 41).  Against 128 x 128 in
    // quarters as well: 512 rows against 2,048 x 2,048 19 -> 14, 5,632 k 44 -> 28; 6,144 weight rows, 128 and 300 rows 25 -> 14 and 19.0 -> 17.5; 2,048 x 5,632, 1,024 rows 46 -> 39;
    // gate/up of 11,264, 128 rows 27 -> 21, of 5,120 x 3,584, 384 rows 40 -> 30.
    if (!dual && tiles(64, 64) <= cus) return 464;
    if (tiles(64, 128) <= cus) return 4128;
    // One round of 128 x 128 in two stages, two blocks to a CU, whether half or all of it is there (2,048 k: 6,144 weight rows, 768 to
    // 1,280 rows 43 -> 34-36 us, gate/up of 11,264, 384 and 640 rows 40 -> 35 and 48 -> 38, 2,048 weight rows, 2,432 and 4,096 rows 49
    // -> 38 and 49 -> 42; 8,192 k: 3-24 % less).  But beyond 14,336 rows (of at most 512 weight rows then) of long K the
    // tiles of 256 x 128 read the rows fewer times (16,384 rows, in quarters: 4,096 k 63 against 65 us, 5,632 k 83 against 91, 8,192 k 130 against 149; 3,584 k 57 and 58,
    // where 128 x 256, which then take the place of 128 x 128, need 52).
    const long t128 = tiles(128, 128);
    if (t128 > cus && t128 <= 2L * cus && (M <= 14336 || K < 4096)) return 8128;
    // More: the widest tile that still gives the CUs (one block each) an even share of the work; a tile's score is the share of
    // its rounds that is there, of its rows that exist, and what it reaches when full.  Tiles of 192 x 256 where they divide the work more
    // evenly (2,048 rows against 11,264 weight rows: 484 tiles for two rounds of the 256 CUs instead of 352 tiles of 256 x 256).
    auto score = [&](int tm, int tn, double quality) {
        const long t = tiles(tm, tn);
        const double rows = (double)M / (double)((long)ceil_div(M, tm) * tm);
        return quality * rows * (double)t / (double)((t + cus - 1) / cus * cus);
    };
    const double s256 = score(256, 256, 1.0), s192 = dual ? 0.0 : score(256, 192, 0.92), s128 = score(256, 128, 0.85),
                 s64 = score(128, 128, 0.7), s12 = score(192, 256, 0.92);
    if (s12 > s256 && s12 > s192 && s12 > s128 && s12 > s64) return 12;
    if (s192 > s256 && s192 >= s128 && s192 >= s64) return 192;
    if (s256 >= s128 && s256 >= s64) return 256;
    if (s128 >= s64) return 128;
    // Where that is 128 x 128, several rounds of it run two blocks to a CU in two stages as well (6,144 weight rows, 2,688 rows
    // 88 -> 71 us; gate/up of 11,264, 1,337 rows 91 -> 79).  (Not ahead of the other tiles in general: four rounds' worth of tiles of 128 x 128,
    // 2,048 rows' gate/up of 8,192 73 against 67 us, 3,456 rows against 4,608 weight rows of 3,584 k 111 against 101.)
    return t128 > cus ? 8128 : 64;
}
// Plain products that take tiles of 128 x 128: whether 128 x 256 are ahead.  Two tiles of 128 x 128 on a CU take what one of twice the
// width takes (2,048 k: 31 and 29 us), so while those are one round of the CUs, or their last round is nearly full (1,000 rows
// against 6,144 weight rows 31.9 -> 30.0 us, gate/up of 11,264, 512 rows 32.1 -> 30.2 and 1,337 rows 67.9 -> 65.3, 3,001 rows against
// 2,048 of 5,632 k 75 -> 65; the other way gate/up of 11,264, 1,000 rows, 1.4 rounds, 52 against 60).
FX_API int fx_gemm_twice_as_wide(int M, int N, int dual, int cus) {
    const long t = (long)ceil_div(N, dual ? 128 : 256) * ceil_div(M, 128), rounds = ceil_div(t, (long)cus);
    return rounds == 1 || 10 * t >= 9 * rounds * cus;
}
// Plain products that are one round of tiles of 128 x 128 (64) or 128 x 256 (8256): whether tiles of 96 rows are one round as well, which
// leaves a block three quarters of the products (1,337 rows against 2,048 weight rows of 2,048 k 23.0 -> 20.9 us, of 5,632 k 45.5 -> 42.8, against
// 4,096 of 2,048 k 30.7 -> 27.3; 672 rows against 6,144 28.6 -> 25.5).
FX_API int fx_gemm_lower_tiles(int M, int N, int tile, int dual, int cus) {
    const int tn = tile == 64 ? 128 : (tile == 8256 ? 256 : 0);
    return tn && (long)ceil_div(N, dual ? tn / 2 : tn) * ceil_div(M, 96) <= cus;
}
// Plain products that are one round of tiles of 128 x 128 (64): whether a ring of four stages is ahead of the tiles in quarters, whose two stages
// do not reach as far: blocks that go through a long K drift apart, and find less of each other's operands in the caches (3,584 weight rows of 20,480 k, 800
// rows 174 -> 167 us, 1,000 rows 190 -> 177, 1,100 rows 195 -> 181; 2,048 weight rows, 1,500 rows 172 -> 168. 14,336 k: 1,000 rows 132 -> 127 to 131, 600 and 700 rows
// the other way, 116 against 121 and 118 against 120; 8,192 k: 800 rows 70 against 72; 3,584 k: 33 against 37).
FX_API int fx_gemm_ring_of_four(int tile, int K) { return tile == 64 && K >= 16384; }
// The same for rows sorted by expert.
FX_API int fx_gemm_grouped_tile(int per_group, int M, int N, int nonempty, int dual, int cus) {
    // an expert's share of up to 20 rows on average: a tile of 64 rows leaves LDS for a ring of four weight tiles
    // beside two of the rows (2-5 % less time than tiles of 192 rows with a ring of three)
    if (per_group <= g_tile64_rows) return 4;
    // up to 104 rows: tiles of 128 x 256, streamed or in quarters by each expert's own share (`gemm_bf16_shares_kernel`).  From 21 to 36 rows against tiles of 64,
    // both products, even / crowded: 176 tokens beside the shared expert's pieces 217 123 -> 196 128, 256 222 146 -> 200 129, 400 178 114 -> 180 109, 512 184 118 -> 186 127; of the larger model
    // 96 beside the pieces 662 394 -> 617 401, 200 557 353 -> 560 315, 256 569 364 -> 571 310.  Beyond 104 rows shares that are not quite
    // even spill into second tiles (nearly even / crowded against tiles of 192 rows: 104 rows 245 220 -> 239 168, 106 235 224 -> 250 177, 110 236 237 -> 247 186; of the
    // larger model 104 rows 678 577 -> 673 530, 109 674 625 -> 728 542).
    if (per_group <= 104) return 1256;
    // a share of up to 192 rows: the product streams the weights once and multiplies little, so it
    // is bound by how many of them are on their way; a ring of three weight tiles beside two of the rows, in quarters
    // from 129 rows an expert on (beyond 192 rows: tiles of 192 rows too where they leave fewer empty rows than tiles of
    // 256 do, 273 rows an expert as 2 x 192 instead of 2 x 256: the down product of a 4,096-token step 173
    // against 190 us)
    const long pad192 = ceil_div(per_group, 192) * 192L, pad256 = ceil_div(per_group, 256) * 256L;
    if (per_group <= 176 || pad192 < pad256) return 12;
    auto score = [&](int tm, int tn, double quality) {
        const long t = (long)ceil_div(N, dual ? tn / 2 : tn) * (M / tm + nonempty);
        return quality * (double)t / (double)((t + cus - 1) / cus * cus);
    };
    const double s256 = score(256, 256, 1.0), s128 = score(256, 128, 0.85), s64 = score(128, 128, 0.7);
    return s256 >= s128 && s256 >= s64 ? 256 : (s128 >= s64 ? 128 : 64);
}

// dtype: type of A and W.  C is: T for EPI_STORE and EPI_GATED, float32 otherwise.
// f32_instruction: a float32 product goes through the float32 matrix instruction whatever its sizes (a call that has its operands the other way round, rows of weights
// against tokens as "weights": the rule by the weights' sizes would go by the tokens then).
// max_share: rows sorted by expert, a number that no expert's rows exceed (0: none is known); the order of tiles depends on it, no result does.
FX_API int fx_gemm(void* stream, int dtype, int epi, const void* A, long lda, const void* W, long w_stride,
                   long up_offset, const void* bias, int bias_dtype, void* C, long ldc,
                   const float* row_scale, const int* a_rows, const int* c_rows, const int* expert_offsets,
                   int E, int M, int N, int K, const void* norm_w, int norm_dtype, float norm_eps,
                   const int* pair_ids, int pair_div, int n_always, int always_rows, int always_from_a, long kb_rows,
                   const float* row_ss, int row_ss_n, int act, int store_act, float act_limit, float act_alpha,
                   const float* pre_scale, const int* pre_scale_rows, const float* out_gate, long ld_gate, int gate_div, int max_share,
                   const float* then_add, long ld_then_add, int f32_instruction) {
    FX_REQUIRE((store_act == SACT_GATE) == (out_gate != nullptr) && (!out_gate || (gate_div >= 1 && ld_gate >= (long)gate_div * N)),
               "gemm: gated outputs need gate rows of %d x %d columns, got a row distance of %ld", gate_div, N, ld_gate);
    FX_REQUIRE(store_act >= 0 && store_act < SACT_COUNT && (store_act == 0 || ((epi == EPI_STORE || epi == EPI_STORE_F32) && !bias)),
               "gemm: a stored activation (%d) goes with the plain stored product without bias", store_act);
    FX_REQUIRE(!pre_scale || epi == EPI_GATED, "gemm: a scale in front of the activation goes with the gate/up epilogue");
    FX_REQUIRE(act != ACT_SWIGLU_CLAMP || act_limit > 0.f, "gemm: the clamped gate needs a positive limit, got %g", (double)act_limit);
    FX_REQUIRE(store_act != SACT_SOFTCAP || act_limit > 0.f, "gemm: capped outputs need a positive cap, got %g", (double)act_limit);
    FX_REQUIRE(dtype == FX_F32 || dtype == FX_BF16, "gemm: unknown dtype %d", dtype);
    FX_REQUIRE(epi >= EPI_STORE && epi <= EPI_GATED, "gemm: unknown epilogue %d", epi);
    FX_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm: bad sizes M=%d N=%d K=%d", M, N, K);
    FX_REQUIRE(lda >= K && ldc >= N, "gemm: leading dimensions lda=%ld ldc=%ld too small for K=%d N=%d", lda, ldc, K, N);
    FX_REQUIRE(!(epi == EPI_GATED && bias), "gemm: the gate/up epilogue takes no bias");
    FX_REQUIRE(act >= 0 && act < ACT_COUNT, "gemm: unknown activation %d", act);
    FX_REQUIRE(!(expert_offsets || pair_ids) || E > 0, "gemm: grouped mode needs E > 0");
    FX_REQUIRE(!pair_ids || (!expert_offsets && !a_rows && !c_rows && !row_scale && !norm_w && pair_div >= 1 && M <= 64 &&
                             dtype == FX_BF16),
               "gemm: unsorted pairs are for up to 64 bfloat16 rows without other row maps");
    FX_REQUIRE(!bias || bias_dtype == FX_F32 || bias_dtype == FX_BF16, "gemm: unknown bias dtype %d", bias_dtype);
    if (M == 0) return 0;
    if (norm_w) {
        FX_REQUIRE(dtype == FX_BF16 && epi == EPI_STORE, "gemm: the fused norm feeds a bfloat16 product that is stored");
        FX_REQUIRE(norm_dtype == FX_F32 || norm_dtype == FX_BF16, "gemm: unknown norm weight dtype %d", norm_dtype);
        FX_REQUIRE((expert_offsets ? (M + E - 1) / E : M) <= 32 && K % 8 == 0 && lda % 4 == 0 && w_stride % 8 == 0 &&
                       (((uintptr_t)A | (uintptr_t)W | (uintptr_t)norm_w) % 16 == 0),
                   "gemm: the fused norm takes up to 32 rows per group, K a multiple of 8 and 16-byte aligned rows");
    }
    GemmArgs g = {};
    g.norm_w = norm_w; g.norm_dtype = norm_dtype; g.norm_eps = norm_eps;
    g.row_ss = row_ss; g.row_ss_n = row_ss_n;
    FX_REQUIRE(!row_ss || (row_ss_n >= 1 && !norm_w && !expert_offsets && !pair_ids && !a_rows && !c_rows && dtype == FX_BF16 &&
                           epi == EPI_STORE && M <= 64 && K % 8 == 0 && lda % 8 == 0 && (((uintptr_t)A | (uintptr_t)W) % 16 == 0)),
               "gemm: a row scale from sums of squares goes with a plain stored bfloat16 product of up to 64 aligned rows");
    g.A = A; g.lda = lda; g.W = W; g.w_stride = w_stride; g.up_offset = up_offset;
    g.bias = bias; g.bias_dtype = bias_dtype; g.C = C; g.ldc = ldc; g.row_scale = row_scale;
    g.a_rows = a_rows; g.c_rows = c_rows; g.expert_offsets = expert_offsets; g.E = E; g.M = M; g.N = N; g.K = K;
    g.pair_ids = pair_ids; g.pair_div = pair_div; g.act = act; g.store_act = store_act;
    g.act_limit = act_limit; g.act_alpha = act_alpha; g.pre_scale = pre_scale; g.pre_scale_rows = pre_scale_rows;
    g.out_gate = out_gate; g.ld_gate = ld_gate; g.gate_div = gate_div;
    g.kb_stride = kb_rows * 64;
    FX_REQUIRE(kb_rows >= 0 && (kb_rows == 0 || (dtype == FX_BF16 && K % 64 == 0 && ((uintptr_t)W % 16) == 0 && lda % 8 == 0 &&
                                                 ((uintptr_t)A % 16) == 0 && (up_offset % K) == 0)),
               "gemm: weights in slabs of 64 k are bfloat16 with K a multiple of 64 and aligned operands");
    FX_REQUIRE(!then_add || (dtype == FX_BF16 && epi == EPI_RESID && M <= 16 && !expert_offsets && !pair_ids && !c_rows && ld_then_add >= N && K % 8 == 0 && lda % 8 == 0 &&
                             (((uintptr_t)A | (uintptr_t)W) % 16) == 0 && g_head_rows >= 16 && (g_plain_rows == 0 || g_plain_rows >= 16) && g_skinny_mt <= 1),
               "gemm: rows to be added behind the product go with up to 16 aligned plain bfloat16 rows that are added");
    g.then_add = then_add; g.ld_then_add = ld_then_add;
    g.n_always = n_always; g.always_rows = always_rows; g.always_from_a = always_from_a;
    FX_REQUIRE(n_always >= 0 && (n_always == 0 || (pair_ids && always_rows >= 1 && always_rows <= 16)),
               "gemm: experts that every row takes come with unsorted pairs and at most 16 rows");
    hipStream_t s = (hipStream_t)stream;
    const int nonempty = expert_offsets ? (E < M ? E : M) : 0;
    if (dtype == FX_F32) {
        g.vec_ok = K % 4 == 0 && lda % 4 == 0 && w_stride % 4 == 0 && up_offset % 4 == 0 && (((uintptr_t)A | (uintptr_t)W) % 16 == 0);
        g.c_vec = ldc % 4 == 0 && ((uintptr_t)C % 16) == 0;
        const bool dual = epi == EPI_GATED;
        const long group = expert_offsets ? (M + E - 1) / E : M, cus = fx_compute_units();
        auto row_tiles = [&](int tm) { return M / tm + (expert_offsets ? nonempty : (M % tm != 0)); };
        // Up to 32 plain rows: the kernel for few rows (2,048 x 2,048 weights, 4 rows: 9 us against 24 with tiles of 32 and 45
        // of 64; 6,144 weight rows, 30 rows: 21, 33 and 47).  Tiles of 64 once they are two and
        // a half a CU (6,144 weight rows: 512 rows 121 against 139 us, 256 rows 76 against 71; 2,048 weight rows: 1,500
        // rows 112 against 129, 700 rows 74 against 67).  Sorted rows: the kernel for few rows up to two rows an expert (60 experts' gate/up
        // products of 2,048, of 4, 16, 32 and 64 tokens: 64, 156, 197 and 220 us against 68, 173, 224 and 250 with tiles of 32, their down products 32,
        // 83, 108 and 122 against 37, 90, 115 and 129; but the tokens of one prompt crowd: 64 on 35 of the experts 163 and 91 against 169 and 86, 96 there 188 and 104
        // against 172 and 90, a prompt of 60 tokens of six layers 2,631 against 2,512), tiles of 32 up to 36 rows an expert (36 rows 419 us against 427 with tiles of 64; 47 rows 496 against 424).
        // The head's 151,936 weight rows: the kernel for few rows up to eight rows (4 rows 235 against 254 us, 16 rows 277 against 258).
        // Up to 16 plain rows take half sets of weight rows (see `fx_gemm_half_sets`) where those are at most a block a CU (2,048 x 2,048, 4 rows 8.5 -> 7.0 us, 2,048
        // x 5,632 18.5 -> 16.1, gate/up of 1,408 12.8 -> 9.1, a router of 61 8.2 -> 6.2; of 6,144 x 2,048, 768 of them, 15.9 -> 17.1).
        // Where it cannot take whole lines it stays behind tiles of 32 with sorted rows, and from three rows on with the head's.
        const bool lines = g.vec_ok && K % 32 == 0;
        const bool split = !f32_instruction && (g_f32_split >= 0 ? g_f32_split && K % 32 == 0 : fx_gemm_f32_split(N, K));
        int tile = 0, mt = 1, nw = 2;
        if (g_f32_tile) tile = g_f32_tile == 1 ? 0 : g_f32_tile;
        else if (expert_offsets) tile = lines && group <= 2 ? 0 : (group <= 36 && !split ? 32 : 64);
        else {
            const bool many_columns = ceil_div(N, 32) >= 8 * cus && M > (lines ? 8 : 2);
            if (M > 32 || many_columns) tile = split ? fx_gemm_f32_split_tile(M, N, dual, (int)cus) : M > 32 && 2 * (long)ceil_div(N, 64) * ceil_div(M, 64) >= 5 * cus ? 64 : 32;
        }
        // Sorted rows taken apart, 64 rows a tile: up to 24 an expert 64 columns (of one matrix, or 32 of both) a block and whole lines with the non-temporal hint, up to 12 with the weights
        // two stages ahead, beyond 128 columns (both products, float32 instruction / those three ways; tokens of 60 experts of 1,408: 45 373 / 374 349 407, 150 402 / 382 381 430, 300
        // 432 / 411 418 441, crowded 414 / 387 403 390, 450 crowded 507 / 470 476 431, 700 624 / 519 549 514, crowded 655 / 612 622 541).
        int stream = 0;
        if (tile) {
            if (split && expert_offsets) {
                if (!g_f32_tile) tile = group <= 24 ? 64 : 128;
                if (tile != 64) tile = 128;
                else stream = group <= 12 ? 2 : (group <= 24 ? 1 : 0);
            } else if (!(tile == 32 || (split && (tile == 48 || tile == 128 || tile == 144 || tile == 160)))) tile = 64;
            if (split && !expert_offsets && tile == 32 && M <= 32) stream = 1;
            if (split && !expert_offsets && tile == 64 && M <= 64 && fx_gemm_f32_one_round(N, dual, (int)cus)) stream = 2;
        }
        if (!tile) {
            mt = group <= 16 ? 1 : 2;
            // one set of weight rows a block where two give fewer blocks than CUs; taken apart, where a block has its rows to split besides, fewer than five eighths of them
            // (2,048 k, 4 rows: 3,072 weight rows 9.8 us with one and 12.9 with two, 4,096 10.1 and 14.4, 5,120 15.7 and 15.3, 6,144 15.6 and 13.8)
            if (mt == 1 && !dual && (long)ceil_div(N, 32) * row_tiles(16) < (split ? 5 * cus / 8 : cus)) nw = 1;
        }
        const bool half = !tile && lines && mt == 1 && !expert_offsets && M <= 16 &&
                          (g_skinny_half >= 0 ? g_skinny_half != 0 : ceil_div(N, 8) <= cus);
        if (half) nw = dual ? 2 : 1;
        if (tile && split) g.tile_rows = tile >= 128 ? 192 - tile : tile;
        const int tm = !tile ? 16 * mt : split ? g.tile_rows : tile;
        const int columns = !tile ? (half ? 8 : 16) * nw / (dual ? 2 : 1) : split ? (tile >= 128 ? 128 : 64) / (dual ? 2 : 1) : dual ? 32 : tile;
        dim3 grid(ceil_div(N, columns), row_tiles(tm));
#define FX_F32(DUAL_, EPI_)                                                            \
    if (g.vec_ok) launch_f32<DUAL_, EPI_, true>(g, split, tile, stream, mt, nw, half, grid, s);             \
    else launch_f32<DUAL_, EPI_, false>(g, split, tile, 0, mt, nw, false, grid, s)
        switch (epi) {
            case EPI_STORE:
            case EPI_STORE_F32: FX_F32(false, EPI_STORE_F32); break;
            case EPI_RESID: FX_F32(false, EPI_RESID); break;
            default: FX_F32(true, EPI_GATED); break;
        }
#undef FX_F32
        FX_CHECK_LAUNCH("gemm_f32");
        return 0;
    }
    g.vec_ok = norm_w != nullptr ||
               ((K % 8 == 0) && (lda % 8 == 0) && (w_stride % 8 == 0) && (up_offset % 8 == 0) &&
                (((uintptr_t)A | (uintptr_t)W) % 16 == 0));
    const long per_group = expert_offsets ? (M + E - 1) / E : M;
    const bool wide_ok = g.vec_ok && K % 64 == 0 && !g_no_wide;
    FX_REQUIRE(!pair_ids || g.vec_ok, "gemm: unsorted pairs need K a multiple of 8 and 16-byte aligned rows");
    // 17..64 plain rows against very many weight rows (the head): tiles of 128 rows stream the weights at the same
    // speed whatever the rows (151,936 weight rows: 131-136 us from 1 to 33 rows), the kernel for few rows slows
    // down with them (98 us at 1 row, 101 at 8; decode steps of 12 and 16 sequences are 20 us shorter with it, those
    // of 24 and 32 the same either way)
    const bool many_columns = g.vec_ok && !expert_offsets && !pair_ids && !norm_w && !row_ss && !g.kb_stride && M > g_head_rows && K % 64 == 0 &&
                              !g_no_wide && ceil_div(N, 128) >= 512;
    // Rows sorted by expert: the product for few rows only up to three rows an expert on average.  Its waves fetch
    // every row tile's operands themselves, so its time grows with the rows (512 tokens of the larger model, 64 rows
    // an expert: 1,100 us for the gate/up product), while tiles of an expert's rows stream the weights at the same speed
    // whatever the rows (128 x 256: 384 us at 6.1 TB/s).  Both products at three rows an expert 144 against 152 us with tiles of 64 rows (60 experts), 469 against 493
    // (64 of the larger model); at four rows 164 against 162 and 564 against 513.
    // 65 to 128 plain rows against few weight rows (the attention's output product): the product for few rows, 32 or 64 rows
    // a block, still streams the weights faster than tiles of 64 x 64 (2,048 x 2,048 weights 12 against 13 us, 2,048 x 5,632
    // 25 against 28-30; 3,584 x 3,584 the other way, 31 against 20)
    // (where the tiled kernel is the register-staged one, K no multiple of 64: up to 256 rows and 32 tiles of 128 x 128)
    const bool few_tiles = !expert_offsets && !pair_ids && M > 64 && !g_wide_force &&
                           (wide_ok ? M <= 128 && ceil_div(N, 128) <= 16 : M <= 256 && (long)ceil_div(N, 128) * ceil_div(M, 128) <= 32);
    // More rows against very few weight rows (a low-rank projection): tiles leave most CUs idle through the whole chain of K
    // steps, the product for few rows covers them while its blocks are one round of the CUs (K = 2,048: 1,024 rows against
    // 256 weight rows 11.2 against 12.4 us, 512 against 512 the same, 1,337 against 256 18.5 against 12.5, 768 against 512 18.7 against
    // 12.5; K = 3,584: 2,048 rows against 128 weight rows 16.9 against 18.1, 1,337 against 256 29.2 against 18.2).
    // A router's logits (float32, up to 128 outputs) stay with it up to twice as many outputs, 4,096 tokens and 65 rows of 3,584 k
    // 33 against 18.6 us beside the shared expert: which experts a token takes must not move with the tiles.
    const bool router = epi == EPI_STORE_F32 && N <= 128;
    const bool narrow = !expert_offsets && !pair_ids && M > (wide_ok ? 128 : 256) && (long)M * N <= (wide_ok && !router ? 262144 : 524288) && !g_wide_force;
    // 33 to 64 plain rows of a wide gate/up product: the product for few rows fetches every row's operands in every block,
    // tiles of 64 rows bring them to LDS once (gate/up of 11,264 x 2,048, 64 rows 27.5 -> 19 us, of 40,960 x 3,584 125 -> 70).
    // (Stored products of so many rows keep the bits of the one that rotates in its epilogue.)
    const bool tiles_of_64 = epi == EPI_GATED && !expert_offsets && !pair_ids && wide_ok && M > 32 && M <= 64 && 2 * N >= 8192;
    const long plain_limit = g_plain_rows > 0 ? g_plain_rows : (few_tiles || narrow ? M : (tiles_of_64 ? 32 : 64));
    // Groups with little weight of their own (a head's up-projection of a latent): the product for few rows up to 16 rows a
    // group, tiles of 128 x 128 beyond (tiles 256 columns wide would be half empty).  16 heads of 128 x 192: 8 rows a head
    // 5.0 against 6.9 us, 2,048 rows a head 12.6 against 21.0 us.
    const bool small_groups = expert_offsets && epi != EPI_GATED && N <= 128 && (long)N * K <= 65536;
    const long few_limit = expert_offsets ? (wide_ok ? (small_groups ? 16 : g_few_rows) : 64) : plain_limit;
    if (g.vec_ok && (per_group <= few_limit || pair_ids) && !many_columns) {
        int mt = pair_ids ? 1 : (per_group <= 16 ? 1 : (per_group <= 32 ? 2 : 4));
        if (!expert_offsets && !pair_ids && M > 64 && (long)ceil_div(N, 32) * ceil_div(M, 64) < 256) mt = 2;     // more blocks where they are few
        const bool dual = epi == EPI_GATED;
        // 33 to 64 plain rows against few weight rows (the attention's output product: 2,048): four row tiles a
        // block leave 128 blocks; a block per row tile, with two sets of weight rows, gives 256 and every block a
        // quarter of the rows' operands to fetch (13.4 -> 9.1 us at 64 rows, 11.2 -> 9.0 at 40; with 6,144 weight
        // rows the four row tiles a block stay ahead, 17.3 against 20.1 us)
        const bool spread_rows = mt == 4 && !expert_offsets && !norm_w && epi == EPI_RESID && ceil_div(N, 16) * (long)ceil_div(M, 64) < 192;
        if (spread_rows) mt = 1;
        const bool row_tile_blocks = !expert_offsets && !pair_ids && !norm_w && (epi == EPI_STORE || epi == EPI_STORE_F32) && mt > 1 &&
                                     fx_gemm_row_tile_blocks(M, N, fx_compute_units());
        if (row_tile_blocks) mt = 1;
        if (g_skinny_mt && !pair_ids) mt = g_skinny_mt;
        if (!expert_offsets && !pair_ids && !norm_w && M <= 16 && mt == 1) {
            const FewRows f = few_plain_rows(M, N, K, dual, fx_compute_units());
            launch_skinny(g, epi, 1, f.sets, f.waves, f.half, 1, s);
            FX_CHECK_LAUNCH("gemm_bf16_skinny");
            return 0;
        }
        const int m_tiles = pair_ids ? (M < E ? M : E) + M / 16 + n_always
                                     : M / (16 * mt) + (expert_offsets ? nonempty : (M % (16 * mt) != 0));
        // two sets of weight rows per wave share the activations they multiply and halve the blocks' fixed
        // work; one set when that would leave too few blocks to keep the memory busy, or when a row or two meet
        // so many weight rows that the blocks are plenty either way (measured on the sizes of the engine)
        int nw = (dual || (long)ceil_div(N, 32) * m_tiles >= 160) ? 2 : 1;
        if (!dual && (norm_w || (M <= 2 && (long)ceil_div(N, 16) * m_tiles >= 4096))) nw = 1;
        if (spread_rows) nw = 2;
        if (row_tile_blocks) nw = 1;
        if ((g_skinny_nw == 1 && !dual) || (g_skinny_nw == 2 && !norm_w)) nw = g_skinny_nw;
        // Waves per block: four, a part of K each, for unsorted pairs too.  (Those ran with one wave that went
        // through all four parts, or two, while a wave found its tile with a loop over the experts and each such
        // search cost 1-2 us; since the search is a few ballots, four waves are ahead again: decode steps of 1, 4, 8
        // and 16 sequences 1.87, 2.80, 3.70 and 5.17 ms with one or two waves, 1.84, 2.72, 3.64 and 5.06 ms with four.)
        // The sums are the same bits with one, two and four waves.
        int waves = 4;
        if (expert_offsets && mt == 1) waves = 2;      // sorted, up to 16 rows per expert: 152 against 159 us at 64 tokens
        if (g_skinny_waves == 8 || g_skinny_waves == 4 || g_skinny_waves == 2 || g_skinny_waves == 1) waves = g_skinny_waves;
        launch_skinny(g, epi, mt, nw, waves, false, m_tiles, s);
        FX_CHECK_LAUNCH("gemm_bf16_skinny");
        return 0;
    }
    FX_REQUIRE(!g.kb_stride || wide_ok, "gemm: no kernel for weights in slabs of 64 k at these sizes");
    if (per_group <= 64 && !many_columns && !wide_ok) {
        const int m_tiles = M / 64 + (expert_offsets ? nonempty : (M % 64 != 0));
        launch_bf16<64, 64, 32, 32>(g, epi, m_tiles, s);
    } else if (g.vec_ok && K % 64 == 0 && !g_no_wide && (g.kb_stride || K < (1 << 22))) {     // (32-bit offsets inside a tile of weights)
        const bool dual = epi == EPI_GATED;
        // weights that are read about once (an expert's rows fit one row tile on average; plain rows: one row tile)
        // are loaded with the non-temporal hint
        g.stream_w = g_stream_w >= 0 ? g_stream_w : (expert_offsets ? per_group <= 128 : M <= 128);
        int tile = expert_offsets && g_wide_grouped ? g_wide_grouped : g_wide_force;
        if (dual && (tile == 464 || tile == 192)) tile = 256;       // (no such tiles of two matrices)
        if (!tile && !expert_offsets) {
            tile = fx_gemm_plain_tile(M, N, K, dual, fx_compute_units());
            if (tile == 8128 && !g.stream_w && fx_gemm_twice_as_wide(M, N, dual, fx_compute_units())) tile = 8256;
            if (!g.stream_w && fx_gemm_ring_of_four(tile, K)) tile = 1128;
            else if (!g.stream_w && fx_gemm_lower_tiles(M, N, tile, dual, fx_compute_units())) tile = tile == 64 ? 6128 : 6256;
        }
        else if (!tile) tile = small_groups ? 64 : fx_gemm_grouped_tile((int)per_group, M, N, nonempty, dual, fx_compute_units());
        auto row_tiles = [&](int tm) { return M / tm + (expert_offsets ? nonempty : (M % tm != 0)); };
        // (see `wide_tile`; tiles of 64 rows seldom are two to an expert at up to five rows each)
        // (dealing them out gains nothing over tiles in order while full ones are three blocks of rows at most: prompts of 42 and 46 tokens 3,200 and 3,280 us in
        // order, 3,250 and 3,320 dealt out, of 50 and 64 level; decoding 48 sequences 9,034 -> 8,902, of the larger model 30 level, 48 3,180 -> 3,095)
        const bool one_tile = expert_offsets && (tile == 4 ? max_share >= 48 && max_share <= 64 : tile == 1256 && max_share > 0 && max_share <= 128);
        g.by_row_tile = expert_offsets && ((tile == 12 && g.stream_w) || (tile == 4 && per_group <= 5));
        switch (tile) {
            case 464: launch_ring<4, 64, 4>(g, epi, row_tiles(64), s); break;
            case 4128: launch_ring<4, 128, 3>(g, epi, row_tiles(64), s); break;
            case 4:
                if (one_tile && g.stream_w && !g.by_row_tile) launch_wide<4, 256, 4, 2, true, true>(g, epi, row_tiles(64), s);
                else launch_ring<4, 256, 4, 2>(g, epi, row_tiles(64), s);
                break;
            case 8128: launch_ring_or_quarters<8, 128, 2>(g, epi, row_tiles(128), s); break;
            case 64: launch_ring_or_quarters<8, 128, 4>(g, epi, row_tiles(128), s); break;
            case 12: launch_ring_or_quarters<12, 256, 3, 2>(g, epi, row_tiles(192), s); break;
            case 1128: launch_wide<8, 128, 4, 4, false>(g, epi, row_tiles(128), s); break;
            case 6128: launch_quarters<8, 128>(g, epi, row_tiles(96), s, 96); break;
            case 6256: launch_quarters<8, 256>(g, epi, row_tiles(96), s, 96); break;
            case 8256: launch_quarters<8, 256>(g, epi, row_tiles(128), s); break;
            case 1256:
                if (one_tile) launch_shares<8, 256, 3, true>(g, epi, row_tiles(128), s);
                else launch_shares<8, 256, 3, false>(g, epi, row_tiles(128), s);
                break;
            case 192: launch_quarters<16, 192>(g, epi, row_tiles(256), s); break;
            case 128: launch_quarters<16, 128>(g, epi, row_tiles(256), s); break;
            default: launch_quarters<16, 256>(g, epi, row_tiles(256), s); break;
        }
    } else {
        const int m_tiles = M / 128 + (expert_offsets ? nonempty : (M % 128 != 0));
        const bool dual = epi == EPI_GATED;
        // narrow outputs: tiles of 64 columns give the CUs at least two blocks each
        if (!dual && (long)ceil_div(N, 128) * m_tiles < 2L * fx_compute_units())
            launch_bf16<128, 64, 64, 32>(g, epi, m_tiles, s);
        else
            launch_bf16<128, 128, 64, 64>(g, epi, m_tiles, s);
    }
    FX_CHECK_LAUNCH("gemm_bf16");
    return 0;
}
