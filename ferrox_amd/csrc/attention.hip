// Causal grouped-query attention over the paged cache.
//
// Every kernel reads keys from pages [page][kv_head][slot][head_dim] and values
// from transposed pages [page][kv_head][head_dim][slot], through a block table
// [n_seqs, max_blocks].  A query at position p sees key t iff t <= p and, with a
// window W > 0, p - t < W (ferrox-core/src/attention.rs:441-447, 498-513), or, with a
// chunked mask of C > 0 positions, t >= floor(p / C) * C (chunks count from position 0
// of the sequence).  With a window, the first `keep_first` keys of a sequence may stay visible to
// every later query (t < keep_first), and a head may have a sink: one more term exp(sink_h) in the
// softmax's denominator, with no key and no value.  The output may be gated: out * sigmoid(gate),
// gate a matrix of out's shape.  Values may have been cached turned by their own position; the output is then turned
// back by the query's (`turns`), before the gate.  A value head may have another size (vd) than a query and key
// head (hd); the bfloat16 MFMA kernels take equal sizes, the others both.  Head
// h reads kv head h / (n_heads / n_kv_heads) (attention.rs:432-438).  Scores,
// softmax and the output sum are float32, in the one-pass form of
// attention.rs:146-175 over tiles of 64 keys that start at multiples of 64, so a
// query's result does not depend on what else is computed with it.
#include "common.h"
#include "attention.h"
#include <type_traits>
#include <utility>

FX_DEFINE_LAST_ERROR()

#define HD_MAX 256          // the widest head of the matrix-unit kernels
#define HD_MAX_ANY 512      // the widest head of the kernels for any shape (float32, or bfloat16 heads beyond HD_MAX)
#define TQ 16
#define NEG_INF (-INFINITY)

struct AttnArgs {
    const void* q;       // [tokens, n_heads * head_dim]
    long ldq;
    void* out;           // same shape
    long ldo;
    const void* k_pages;
    const void* v_pages;
    const int* block_table;
    int max_blocks;
    const int* positions;  // [tokens]
    const int* item_seq;   // per work item: sequence (row of the block table)
    const int* item_tok;   // per work item: first token
    const int* item_n;     // per work item: number of queries (prefill tiles only)
    int nh, nkv, hd, bs, window;
    int vd;              // size of a value head (and of an output head)
    int mask_chunk;      // > 0: the chunked mask
    int keep_first;      // > 0 (with a window): keys t < keep_first stay visible to every later query
    const float* sinks;  // [n_heads] or null: a logit per head that joins the softmax's denominator
    const void* gate;    // [tokens, n_heads * vd] or null (type of out, or float32): the output is multiplied by sigmoid(gate)
    long ldg;
    int gate_per_head;   // 1: the gate is [tokens, n_heads], one number for all of a head's outputs
    float softcap;       // > 0: a scaled score s becomes softcap * tanh(s / softcap)
    const float* slopes; // [n_heads] or null: the score of key t for the query at p then loses slopes[h] * (p - t)
    const float2* turns; // [tokens, vd / 2] (cos, sin) or null: output pair (2m, 2m + 1) is turned back by that angle
    int gate_f32;        // 1: the gate is float32, whatever the type of out
    const float* bias;   // or null: a number per head and distance that joins the (scaled, capped) score; see below
    int bias_n;          // distances 0 .. bias_n - 1 have a number of their own, longer ones that of bias_n - 1
    int bs_shift;        // log2(bs) if bs is a power of two, else -1
    int n_items;
    float scale;
    // decode only
    float* part_o;   // [items, nh, splits, hd]
    float* part_ml;  // [items, nh, splits, 2]
    int splits, chunk;
};

static inline int log2_or_minus_one(int v) {
    if (v <= 0 || (v & (v - 1))) return -1;
    int s = 0;
    while ((1 << s) < v) ++s;
    return s;
}

// the first key that a query at position p sees
__device__ __forceinline__ int first_visible(const AttnArgs& a, int p) {
    if (a.mask_chunk > 0) return p - p % a.mask_chunk;
    return a.window > 0 ? max(0, p - a.window + 1) : 0;
}
__host__ __device__ __forceinline__ bool shapes_scores(const AttnArgs& a) { return a.softcap > 0.f || a.slopes != nullptr || a.bias != nullptr; }
// whether queries see a bounded stretch of keys (a window or a chunk) rather than all before them
__device__ __forceinline__ bool bounded_keys(const AttnArgs& a) { return a.window > 0 || a.mask_chunk > 0; }

// The distance bias of a head is a row of BIAS_PAD + bias_n + BIAS_PAD floats that runs from far to near: the number for
// distance d stands at BIAS_PAD + bias_n - 1 - d, so the numbers of consecutive keys follow each other; in front of them
// stands the farthest one BIAS_PAD times, behind them what keys later than the query read and nobody uses.
#define BIAS_PAD 16
__host__ __device__ __forceinline__ int bias_row_len(const AttnArgs& a) { return a.bias_n + 2 * BIAS_PAD; }
__device__ __forceinline__ float bias_at(const AttnArgs& a, int h, int distance) {      // distance >= 0
    return a.bias[(size_t)h * bias_row_len(a) + BIAS_PAD + a.bias_n - 1 - min(distance, a.bias_n - 1)];
}
// A scaled score on its way into the softmax: capped, less the head's penalty for the distance p - t, plus the head's
// bias for it (keys later than the query are masked: theirs is not looked up).
__device__ __forceinline__ float shaped_score(const AttnArgs& a, int h, float slope, float s, int distance) {
    if (a.softcap > 0.f) s = a.softcap * tanhf(s / a.softcap);
    s = fmaf(-slope, (float)distance, s);
    return a.bias ? s + bias_at(a, h, max(distance, 0)) : s;
}
// where in the row the numbers of 16 consecutive keys begin, `distance` being that of the first of them (which may be
// later than the query, if all of them are)
__device__ __forceinline__ int bias_first(const AttnArgs& a, int distance) {
    return min(max(BIAS_PAD + a.bias_n - 1 - distance, 0), a.bias_n + 2 * BIAS_PAD - 16);
}
// the numbers themselves, from memory: rows start and distances fall at any multiple of four bytes
typedef float fx_f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
struct BiasRow {
    fx_f32x4_any v[4];
};
__device__ __forceinline__ BiasRow fetch_bias(const AttnArgs& a, int h, int distance) {
    const float* p = a.bias + (size_t)h * bias_row_len(a) + bias_first(a, distance);
    BiasRow b;
#pragma unroll
    for (int i = 0; i < 4; ++i) b.v[i] = *(const fx_f32x4_any*)(p + 4 * i);
    return b;
}

// The keys a block may touch: t < end and (t >= begin or t < keep), keep being the kept first keys of the
// sequence (0: none).  Pages of other keys may have been given back.
struct KeySpan {
    int begin, end, keep;
    // (`&` and `|`: with `&&` and `||` each comparison becomes a branch, 35 ns where it is taken)
    __device__ __forceinline__ bool has(int t) const { return (t < end) & ((t >= begin) | (t < keep)); }
    // whether any of the n consecutive keys from t on is one of them
    __device__ __forceinline__ bool touches(int t, int n) const { return (t < end) & ((t + n > begin) | (t < keep)); }
    // whether all of the 64 keys of the tile at t are
    __device__ __forceinline__ bool holds_tile(int t) const { return (t >= begin) & (t + 64 <= end); }
};
// The tiles of 64 keys that a block walks over, in ascending order: those that hold kept first keys and lie
// before the first tile of the span's stretch [begin, end), then that stretch's tiles.
struct TileWalk {
    int n_keep, first, n;
    __device__ __forceinline__ int start(int i) const { return i < n_keep ? 64 * i : first + 64 * (i - n_keep); }
};
__device__ __forceinline__ TileWalk tile_walk(const KeySpan& k) {
    TileWalk w;
    w.first = k.begin & ~63;
    w.n_keep = min((k.keep + 63) >> 6, w.first >> 6);
    w.n = w.n_keep + max(0, (k.end - w.first + 63) >> 6);
    return w;
}

// What a row's running maximum m and sum l become when the head's sink joins the denominator: the factor
// for the row's output, already divided by the new sum.  `m` and `sink` in the same units (natural logarithm,
// or base 2 where the caller's maximum is).
template <bool BASE2>
__device__ __forceinline__ float finish_row(const AttnArgs& a, int h, float m, float l) {
    if (!a.sinks) return 1.f / l;
    const float sk = BASE2 ? a.sinks[h] * 1.4426950408889634f : a.sinks[h];
    const float top = fmaxf(m, sk);      // (m is finite: a query sees itself)
    const float f = BASE2 ? __builtin_amdgcn_exp2f(m - top) : expf(m - top);
    const float e = BASE2 ? __builtin_amdgcn_exp2f(sk - top) : expf(sk - top);
    return f / (l * f + e);
}
// one output element on its way out: through the gate, if there is one
template <typename T>
__device__ __forceinline__ void store_out(const AttnArgs& a, int tok, int h, int d, float v) {
    if (a.gate) {
        const size_t at = (size_t)tok * a.ldg + (a.gate_per_head ? (size_t)h : (size_t)h * a.vd + d);
        const float gv = a.gate_f32 ? ((const float*)a.gate)[at] : to_float(((const T*)a.gate)[at]);
        v *= 1.f / (1.f + expf(-gv));
    }
    from_float((T*)a.out + (size_t)tok * a.ldo + (size_t)h * a.vd + d, v);
}

// Values that were cached turned by their own position (pairs 2m, 2m + 1 of a head): the output of the query at token
// tok is turned back by the query's angle, after the softmax and before any gate.  `v` is output element d, `other`
// its partner d ^ 1.
__device__ __forceinline__ float turned_back(const AttnArgs& a, int tok, int d, float v, float other) {
    const float2 cs = a.turns[(size_t)tok * (a.vd >> 1) + (d >> 1)];
    return fmaf(v, cs.x, (d & 1) ? -(other * cs.y) : other * cs.y);
}
// store_out from kernels whose lanes hold neighbouring output elements (lane l ^ 1 holds d ^ 1, and both are here)
template <typename T>
__device__ __forceinline__ void store_lane(const AttnArgs& a, int tok, int h, int d, float v) {
    if (a.turns) v = turned_back(a, tok, d, v, lane_pair_other(v));
    store_out<T>(a, tok, h, d, v);
}

// the same for a lane's elements 16 cb + li of one row, all of its angles asked for together (elements past vd are not
// stored: they read the last pair's angle)
template <int CB>
__device__ __forceinline__ void turn_back_row(const AttnArgs& a, int tok, int li, float (&y)[CB]) {
    if (!a.turns) return;
    const float2* angles = a.turns + (size_t)tok * (a.vd >> 1);
    float2 cs[CB];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) cs[cb] = angles[min(16 * cb + li, a.vd - 1) >> 1];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        const float other = lane_pair_other(y[cb]) * cs[cb].y;
        y[cb] = fmaf(y[cb], cs[cb].x, (li & 1) ? -other : other);
    }
}

// block of the table and slot in its page of key t (a shift when the page size is a power of two)
__device__ __forceinline__ void page_slot(const AttnArgs& a, int t, int& blk, int& slot) {
    if (a.bs_shift >= 0) {
        blk = t >> a.bs_shift;
        slot = t & (a.bs - 1);
    } else {
        blk = t / a.bs;
        slot = t - blk * a.bs;
    }
}

// Page ids of one sequence.  A block copies the entries of the key range it will walk into LDS once
// (stage_pages), so that finding a tile's pages is an LDS read and not a round trip to memory on
// which the tile's own loads would then wait; entries outside the copy come from memory.
#define PAGE_COPY 1024
struct PageLookup {
    const int* table;    // the sequence's row of the block table
    const int* copy;     // LDS
    int first, count;    // copy[i] = table[first + i], i < count
    __device__ __forceinline__ int page(int blk) const {
        const unsigned i = (unsigned)(blk - first);
        return i < (unsigned)count ? copy[i] : table[blk];
    }
};
// Pages and slots of N keys: one branch for how a page's number is found and one for where its entry is (every lane takes part), not one a key (decode attention, a tile a wave,
// us one a key / so: 16 heads of 128, one sequence of 2,060 keys 12.8 11.8, 8 30.6 29.4; 28 heads on 4, 8 sequences 17.0 15.9).
template <int N>
__device__ __forceinline__ void pages_of(const AttnArgs& a, const PageLookup& pl, const int (&key)[N], int (&page)[N], int (&slot)[N]) {
    int blk[N];
    if (a.bs_shift >= 0) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            blk[i] = key[i] >> a.bs_shift;
            slot[i] = key[i] & (a.bs - 1);
        }
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            blk[i] = key[i] / a.bs;
            slot[i] = key[i] - blk[i] * a.bs;
        }
    }
    unsigned farthest = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) farthest = max(farthest, (unsigned)(blk[i] - pl.first));
    if (pl.copy && __all(farthest < (unsigned)pl.count)) {
#pragma unroll
        for (int i = 0; i < N; ++i) page[i] = pl.copy[blk[i] - pl.first];
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) page[i] = pl.page(blk[i]);
    }
}
// every thread of the block calls this; blocks [first_blk, last_blk] of the table are wanted
__device__ __forceinline__ PageLookup stage_pages(const int* table, int* lds, int first_blk, int last_blk) {
    PageLookup pl;
    pl.table = table;
    pl.copy = lds;
    pl.first = first_blk;
    pl.count = min(PAGE_COPY, max(0, last_blk - first_blk + 1));
    for (int i = threadIdx.x; i < pl.count; i += blockDim.x) lds[i] = table[first_blk + i];
    __syncthreads();
    return pl;
}

template <typename T>
__device__ __forceinline__ const T* key_row(const AttnArgs& a, const int* bt, int kvh, int t) {
    const int page = bt[t / a.bs];
    return (const T*)a.k_pages + (((size_t)page * a.nkv + kvh) * a.bs + t % a.bs) * a.hd;
}
template <typename T>
__device__ __forceinline__ const T* value_col(const AttnArgs& a, const int* bt, int kvh, int t) {
    const int page = bt[t / a.bs];
    return (const T*)a.v_pages + ((size_t)page * a.nkv + kvh) * a.vd * a.bs + t % a.bs;  // + d * bs
}

// ---------------------------------------------------------------------------
// Any number of queries.  A work item is a block of up to 64 consecutive
// queries of one sequence; one wave per (quarter of an item = up to 16 queries,
// head); lanes are keys for the scores and head dimensions for the output.
// ---------------------------------------------------------------------------
// HDM: the widest head this instance takes (its queries in LDS and its outputs in registers are sized by it).
template <typename T, int HDM = HD_MAX>
__global__ __launch_bounds__(64) void attn_tile_kernel(AttnArgs a) {
    __shared__ float Qs[TQ][HDM];
    __shared__ float Ps[TQ][64];
    const int item = blockIdx.x >> 2, sub = blockIdx.x & 3, h = blockIdx.y, lane = threadIdx.x;
    const int kvh = h / (a.nh / a.nkv);
    const int tok0 = a.item_tok[item] + TQ * sub, n = min(TQ, a.item_n[item] - TQ * sub);
    if (n <= 0) return;
    const int* bt = a.block_table + (size_t)a.item_seq[item] * a.max_blocks;
    const int hd = a.hd;

    for (int idx = lane; idx < TQ * hd; idx += 64) {
        const int i = idx / hd, d = idx % hd;
        Qs[i][d] = i < n ? to_float(((const T*)a.q)[(size_t)(tok0 + i) * a.ldq + (size_t)h * hd + d]) * a.scale : 0.f;
    }
    int pos[TQ];
#pragma unroll
    for (int i = 0; i < TQ; ++i) pos[i] = i < n ? a.positions[tok0 + i] : -1;
    const int pmin = a.positions[tok0], pmax = a.positions[tok0 + n - 1];
    const int kv_begin = first_visible(a, pmin);
    const int kv_end = pmax + 1;
    const KeySpan span = {kv_begin, kv_end, a.keep_first};
    const TileWalk walk = tile_walk(span);
    const bool shaped = shapes_scores(a);
    const float slope = a.slopes ? a.slopes[h] : 0.f;

    float m[TQ], l[TQ], o[HDM / 64][TQ];
#pragma unroll
    for (int i = 0; i < TQ; ++i) {
        m[i] = NEG_INF;
        l[i] = 0.f;
#pragma unroll
        for (int dd = 0; dd < HDM / 64; ++dd) o[dd][i] = 0.f;
    }
    __syncthreads();

    for (int ti = 0; ti < walk.n; ++ti) {
        const int kt0 = walk.start(ti);
        const int t = kt0 + lane;
        const bool in_range = span.has(t);
        float s[TQ];
#pragma unroll
        for (int i = 0; i < TQ; ++i) s[i] = 0.f;
        if (in_range) {
            const T* kr = key_row<T>(a, bt, kvh, t);
            for (int d = 0; d < hd; ++d) {
                const float kv = to_float(kr[d]);
#pragma unroll
                for (int i = 0; i < TQ; ++i) s[i] = fmaf(Qs[i][d], kv, s[i]);
            }
        }
        float al[TQ];
#pragma unroll
        for (int i = 0; i < TQ; ++i) {
            const bool vis = in_range && t <= pos[i] && (t >= first_visible(a, pos[i]) || t < a.keep_first);
            if (shaped) s[i] = shaped_score(a, h, slope, s[i], pos[i] - t);
            const float sv = vis ? s[i] : NEG_INF;
            const float m_new = fmaxf(m[i], wave_max(sv));
            al[i] = (m_new == NEG_INF) ? 1.f : expf(m[i] - m_new);
            const float p = vis ? expf(sv - m_new) : 0.f;
            l[i] = l[i] * al[i] + wave_sum(p);
            m[i] = m_new;
            Ps[i][lane] = p;
        }
        __syncthreads();
#pragma unroll
        for (int dd = 0; dd < HDM / 64; ++dd) {
            const int d = dd * 64 + lane;
            if (d < a.vd) {
#pragma unroll
                for (int i = 0; i < TQ; ++i) o[dd][i] *= al[i];
                const int jn = min(64, kv_end - kt0);
                for (int j = 0; j < jn; ++j) {
                    if (!span.has(kt0 + j)) continue;
                    const float vv = to_float(value_col<T>(a, bt, kvh, kt0 + j)[(size_t)d * a.bs]);
#pragma unroll
                    for (int i = 0; i < TQ; ++i) o[dd][i] = fmaf(Ps[i][j], vv, o[dd][i]);
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int dd = 0; dd < HDM / 64; ++dd) {
        const int d = dd * 64 + lane;
        if (d < a.vd) {
#pragma unroll
            for (int i = 0; i < TQ; ++i)
                if (i < n) store_lane<T>(a, tok0 + i, h, d, o[dd][i] * finish_row<false>(a, h, m[i], l[i]));
        }
    }
}

// ---------------------------------------------------------------------------
// Single queries (decode): the keys of a sequence are cut into chunks of
// `chunk` positions; one wave per (sequence, head, chunk) writes a partial
// (max, sum, output), and a second kernel merges the chunks in ascending order.
// ---------------------------------------------------------------------------
template <typename T, int HDM>
__device__ __forceinline__ void decode_head(const AttnArgs& a, int item, int h, int split) {
    __shared__ float Qs[HDM];
    __shared__ float Ps[64];
    const int lane = threadIdx.x;
    const int kvh = h / (a.nh / a.nkv);
    const int tok = a.item_tok[item];
    const int* bt = a.block_table + (size_t)a.item_seq[item] * a.max_blocks;
    const int hd = a.hd;
    const int p = a.positions[tok];
    // the split's keys [split * chunk, (split + 1) * chunk) of which the query sees those from its window's first
    // on and the kept first ones
    const int s0 = split * a.chunk;
    const KeySpan span = {max(first_visible(a, p), s0), min(p + 1, s0 + a.chunk), a.keep_first};
    const int kv_end = span.end;
    float* po = a.part_o + (((size_t)item * a.nh + h) * a.splits + split) * a.vd;
    float* pml = a.part_ml + (((size_t)item * a.nh + h) * a.splits + split) * 2;
    if (s0 >= kv_end || !(span.begin < kv_end || s0 < span.keep)) {
        if (lane == 0) {
            pml[0] = NEG_INF;
            pml[1] = 0.f;
        }
        return;
    }
    for (int d = lane; d < hd; d += 64) Qs[d] = to_float(((const T*)a.q)[(size_t)tok * a.ldq + (size_t)h * hd + d]) * a.scale;
    __syncthreads();
    float m = NEG_INF, l = 0.f, o[HDM / 64];
#pragma unroll
    for (int dd = 0; dd < HDM / 64; ++dd) o[dd] = 0.f;
    for (int kt0 = s0; kt0 < kv_end; kt0 += 64) {
        if (!span.touches(kt0, 64)) continue;      // a tile between the kept keys and the window
        const int t = kt0 + lane;
        const bool vis = span.has(t);
        float s = 0.f;
        if (vis) {
            const T* kr = key_row<T>(a, bt, kvh, t);
            for (int d = 0; d < hd; ++d) s = fmaf(Qs[d], to_float(kr[d]), s);
        }
        if (shapes_scores(a)) s = shaped_score(a, h, a.slopes ? a.slopes[h] : 0.f, s, p - t);
        const float sv = vis ? s : NEG_INF;
        const float m_new = fmaxf(m, wave_max(sv));
        const float al = (m_new == NEG_INF) ? 1.f : expf(m - m_new);
        const float pr = vis ? expf(sv - m_new) : 0.f;
        l = l * al + wave_sum(pr);
        m = m_new;
        Ps[lane] = pr;
        __syncthreads();
#pragma unroll
        for (int dd = 0; dd < HDM / 64; ++dd) {
            const int d = dd * 64 + lane;
            if (d < a.vd) {
                float acc = o[dd] * al;
                const int jn = min(64, kv_end - kt0);
                for (int j = 0; j < jn; ++j) {
                    if (!span.has(kt0 + j)) continue;
                    acc = fmaf(Ps[j], to_float(value_col<T>(a, bt, kvh, kt0 + j)[(size_t)d * a.bs]), acc);
                }
                o[dd] = acc;
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int dd = 0; dd < HDM / 64; ++dd) {
        const int d = dd * 64 + lane;
        if (d < a.vd) po[d] = o[dd];
    }
    if (lane == 0) {
        pml[0] = m;
        pml[1] = l;
    }
}
template <typename T, int HDM = HD_MAX>
__global__ __launch_bounds__(64) void attn_decode_kernel(AttnArgs a) {
    decode_head<T, HDM>(a, blockIdx.x, blockIdx.y, blockIdx.z);
}

// Merges the chunks' partial results in ascending order.  One block per (token, head): first the weights
// exp(m_s - m) of all chunks, which LDS keeps beside the chunks' sums, then a thread per head dimension (of up to 256) adds
// its dimension up over the chunks.  What a launch of this takes is a chain of waits, so there is one for maxima and sums and one for
// outputs (asked for first, they need no weight to be fetched), loads are never behind a branch, and what is added in turn is added in stretches
// of 16 without one; chunks past the last have weight 0 (with a loop over the chunks that fetched each one's sum and outputs where its
// weight was not 0: 20 chunks of 16 heads of 192 at 8 tokens 6.3 us, 14 of 128 at one token 4.6).
#define MERGE_KEPT 7936        // chunks whose weights and sums LDS holds
#define MERGE_MOST 16384       // chunks that are merged: two million keys by 128
template <typename T, bool BEYOND>      // BEYOND: more chunks than that (an instance of its own: its loops cost the others 0.05 to 0.15 us a launch)
__global__ __launch_bounds__(256) void attn_decode_merge_kernel(AttnArgs a) {
    extern __shared__ __attribute__((aligned(16))) float wsm[];   // weights of up to MERGE_KEPT chunks, then their sums, each a multiple of 16
    __shared__ float red[4];
    const int item = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, nt = blockDim.x;
    const int tok = a.item_tok[item];
    const int hd = a.vd, S = a.splits;      // (the size of an output head)
    const float* po = a.part_o + ((size_t)item * a.nh + h) * S * hd;
    const float* pml = a.part_ml + ((size_t)item * a.nh + h) * S * 2;
    // the first chunks' outputs for this thread's first dimension (an empty chunk wrote nothing, and what is read there is dropped below)
    constexpr int STRETCH = 16;
    float early[STRETCH];
    auto fetch = [&](float (&v)[STRETCH], int s0, int d) {
#pragma unroll
        for (int s = 0; s < STRETCH; ++s) v[s] = po[(size_t)min(s0 + s, S - 1) * hd + min(d, hd - 1)];
    };
    fetch(early, 0, tid);
    const int mine = min(tid, S - 1);
    float m = pml[2 * mine];
    const float own_m = m, own_l = pml[2 * mine + 1];
    for (int s = tid + nt; s < S; s += nt) m = fmaxf(m, pml[2 * s]);
    m = wave_max(m);
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    m = fmaxf(red[0], red[1]);
    if (nt > 128) m = fmaxf(m, fmaxf(red[2], red[3]));
    auto weight_of = [&](float ms) { return (ms == NEG_INF) ? 0.f : expf(ms - m); };
    const int kept = BEYOND ? MERGE_KEPT : S, padded = (kept + STRETCH - 1) & ~(STRETCH - 1);
    float* const lsm = wsm + padded;
    for (int s = tid; s < padded; s += nt) {
        const int at = min(s, S - 1);
        const float ms = s == tid ? own_m : pml[2 * at], ls = s == tid ? own_l : pml[2 * at + 1];
        const float w = s < kept ? weight_of(ms) : 0.f;
        wsm[s] = w;
        lsm[s] = w > 0.f ? ls : 0.f;
    }
    __syncthreads();
    float l = 0.f;
    for (int s0 = 0; s0 < padded; s0 += STRETCH) {   // ascending, the same in every thread
#pragma unroll
        for (int s = 0; s < STRETCH; ++s) l = fmaf(wsm[s0 + s], lsm[s0 + s], l);
    }
    if constexpr (BEYOND) {
        for (int s = kept; s < S; ++s) {
            const float w = weight_of(pml[2 * s]);
            l = fmaf(w, (w > 0.f) ? pml[2 * s + 1] : 0.f, l);
        }
    }
    const float fin = finish_row<false>(a, h, m, l);
    for (int d = tid; d < hd; d += nt) {
        float acc = 0.f;
        for (int s0 = 0; s0 < padded; s0 += STRETCH) {
            float v[STRETCH];
            if (s0 == 0 && d == tid) {
#pragma unroll
                for (int s = 0; s < STRETCH; ++s) v[s] = early[s];
            } else {
                fetch(v, s0, d);
            }
#pragma unroll
            for (int s = 0; s < STRETCH; ++s) {
                const float w = wsm[s0 + s];
                acc = fmaf(w, w > 0.f ? v[s] : 0.f, acc);
            }
        }
        if constexpr (BEYOND) {
            for (int s = kept; s < S; ++s) {
                const float w = weight_of(pml[2 * s]);
                acc = fmaf(w, (w > 0.f) ? po[(size_t)s * hd + d] : 0.f, acc);
            }
        }
        store_lane<T>(a, tok, h, d, acc * fin);
    }
}

// ---------------------------------------------------------------------------
// bfloat16 on MFMA (head_dim and block size multiples of 16).
//
// One wave owns 16 "rows" that share one kv head: 16 consecutive queries of one
// head (prefill), or the query heads of one kv group for a single token
// (decode).  For a tile of 64 keys it computes S^T = K Q^T with K as the A
// operand, so that the accumulator of lane (row = lane%16, g = lane/16) holds 16
// scores of its own row; the softmax runs on those registers, and the same
// registers, rounded to bfloat16, are the A operand of O += P V: two 16x16x32
// MFMAs per 16 output columns, in which lane (row, g) supplies the probabilities
// of keys 16g..16g+7 and 16g+8..16g+15.  To make that work, A-row i of key block
// kb reads key 16*(i/4) + 4*kb + i%4 of the tile, and the B operand reads 16
// consecutive keys 16g..16g+15 of a transposed value row.  Keys and values come
// from memory in whole 128-byte lines with the non-temporal hint (`load_lines16`
// and `swap_halves` in common.h): 64 sequences at 2,048 keys 219 -> 171 us a layer
// (4.9 -> 6.3 TB/s), 8 sequences 36.8 -> 29.1 us, 8 at 32,768 keys 431 -> 341 us.
// ---------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

#define LOG2E 1.4426950408889634f
#define LN2 0.6931471805599453f

// Maximum and sum over the four lanes li, li + 16, li + 32, li + 48 that share a row, in every one of them, with the
// two lane-swapping moves of gfx950 (rows of 16 lanes pairwise, then the halves of the wave): the same values in the
// same order as two exchanges through the LDS crossbar (__shfl_xor by 16 and by 32) would give, without the LDS.
__device__ __forceinline__ float quad_max(float x) {
    const unsigned u = __float_as_uint(x);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const unsigned v = __float_as_uint(fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
    const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float quad_sum(float x) {
    const unsigned u = __float_as_uint(x);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const unsigned v = __float_as_uint(__uint_as_float(a[0]) + __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// The same over the two lanes l and l + 32.
__device__ __forceinline__ float half_max(float x) {
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float half_sum(float x) {
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// What the scores of a launch go through between the product and the softmax (the matrix-unit kernels have an instance for
// each: code that a launch does not run still takes registers).
enum { SHAPE_NONE = 0, SHAPE_CAP_SLOPE = 1, SHAPE_BIAS = 2 };
static inline int shape_of(const AttnArgs& a) { return a.bias ? SHAPE_BIAS : (shapes_scores(a) ? SHAPE_CAP_SLOPE : SHAPE_NONE); }

// A lane's 16 raw scores sc[kb][r] of keys key0 + 4*kb + r, scaled, capped and less the head's penalty for the
// distance from the row's query at qpos (`shaped_score` with a tanh made of one exponential and one reciprocal, whose
// error, some 1e-7 of the cap, is far below what bfloat16 operands leave of a score): afterwards they are scores in natural
// units, and the softmax step takes them with c = log2(e).
__device__ __forceinline__ void cap_and_slope(f32x4_t (&sc)[4], int key0, const AttnArgs& a, float slope, int qpos) {
    // tanh(x) = 1 - 2 / (1 + e^2x): the exponent in base 2 with the scale folded in, the quotient from the hardware's
    // reciprocal (1 ulp), cap and -2 cap as the multiply-add's constants
    const bool capped = a.softcap > 0.f;
    const float to_exp = capped ? 2.f * a.scale * LOG2E / a.softcap : 0.f;
    const float cap = a.softcap, cap2 = -2.f * a.softcap;
    const float d0 = (float)(qpos - key0);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float s;
            if (capped) s = fmaf(cap2, __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(sc[kb][r] * to_exp)), cap);
            else s = sc[kb][r] * a.scale;
            sc[kb][r] = fmaf(-slope, d0 - (float)(4 * kb + r), s);
        }
}
// the same with the head's bias for key key0 + i, `bias(i)`
template <typename B>
__device__ __forceinline__ void shape_with_bias(f32x4_t (&sc)[4], int key0, const AttnArgs& a, float slope, int qpos, B&& bias) {
    float scale = a.scale;
    if (a.softcap > 0.f || a.slopes) {
        cap_and_slope(sc, key0, a, slope, qpos);
        scale = 1.f;
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) sc[kb][r] = fmaf(sc[kb][r], scale, bias(4 * kb + r));
}

// One step of the one-pass softmax on a lane's 16 raw scores sc[kb][r] of keys key0 + 4*kb + r
// (key0 = tile start + 16g), in base 2: t = score * c with c = scale * log2(e), m and l are the
// running maximum (of t) and sum of this lane's row, shared by the row's four lanes.  MASKED: only
// keys in [lo, hi] count, and those below `keep` that are no later than hi.  Returns the factor for what was accumulated so far, and the
// probabilities rounded to bfloat16: p_lo for keys key0 .. key0+7, p_hi for key0+8 .. key0+15.
template <bool MASKED>
__device__ __forceinline__ float softmax_step(f32x4_t (&sc)[4], int key0, int lo, int hi, float c, float& m, float& l,
                                              uint4& p_lo, uint4& p_hi, int keep = 0) {
    // the maximum is taken over the raw scores and scaled once (c > 0, and rounding keeps the order); a score's
    // exponent is then one fused multiply-add, score * c - maximum
    float mt = NEG_INF;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (MASKED) {
                const int key = key0 + 4 * kb + r;
                sc[kb][r] = (((key >= lo) | (key < keep)) & (key <= hi)) ? sc[kb][r] : NEG_INF;
            }
            mt = fmaxf(mt, sc[kb][r]);
        }
    mt = quad_max(mt) * c;
    const float m_new = fmaxf(m, mt);
    const float m_use = (m_new == NEG_INF) ? 0.f : m_new;      // a row that has seen nothing yet
    const float alpha = __builtin_amdgcn_exp2f(m - m_use);      // exp2(-inf) = 0
    float ps = 0.f;
    float p[16];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            p[4 * kb + r] = __builtin_amdgcn_exp2f(fmaf(sc[kb][r], c, -m_use));
            ps += p[4 * kb + r];
        }
    p_lo = make_uint4(pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3]), pack_bf16(p[4], p[5]), pack_bf16(p[6], p[7]));
    p_hi = make_uint4(pack_bf16(p[8], p[9]), pack_bf16(p[10], p[11]), pack_bf16(p[12], p[13]), pack_bf16(p[14], p[15]));
    ps = quad_sum(ps);
    l = l * ((m_new == NEG_INF) ? 1.f : alpha) + ps;
    m = m_new;
    return (m_new == NEG_INF) ? 1.f : alpha;
}

// O = O * factor(row) + P V for one block of 16 output columns.  The accumulator holds rows
// 4g+r, so the factors come from the lanes that own those rows; `rescale` is false when every
// row's factor is 1.
__device__ __forceinline__ f32x4_t pv_step(f32x4_t acc, bool rescale, const float (&al)[4], uint4 p_lo, uint4 p_hi,
                                           uint4 v0, uint4 v1) {
    if (rescale) {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] *= al[r];
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, p_lo), __builtin_bit_cast(bf16x8_t, v0), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, p_hi), __builtin_bit_cast(bf16x8_t, v1), acc, 0, 0, 0);
    return acc;
}

// What N * 2 consecutive keys' values (first_key ..) are ANDed with: those outside the span become zeros.  Their
// probabilities are zero, but what memory holds there need not be a number.  Worked out once a tile, and selected rather than
// branched to: with a branch per key and column block the one tile at a sequence's end took 4 to 6 us longer than a whole tile
// (one sequence of 16 heads of 128: 512 keys 7.5 us, 513 11.2; 8 sequences of latent heads of 256: 512 keys 12.3, 513 17.7).
template <int N>
__device__ __forceinline__ void key_masks(uint32_t (&masks)[N], int first_key, const KeySpan& span) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int key = first_key + 2 * i;
        masks[i] &= (span.has(key) ? 0x0000ffffu : 0u) | (span.has(key + 1) ? 0xffff0000u : 0u);
    }
}

// All ones if `ok`, else zero, as a value the compiler knows nothing about: data that is loaded and then
// ANDed with it is loaded always.  With a plain `ok ? x : 0` the compiler loads only where ok holds, behind a
// branch, and waits for that load before it goes on: a tile's loads would then leave one at a time.
__device__ __forceinline__ uint32_t opaque_mask(bool ok) {
    uint32_t m = ok ? 0xffffffffu : 0u;
    asm volatile("" : "+v"(m));
    return m;
}
__device__ __forceinline__ uint4 and_mask(uint4 x, uint32_t m) { return make_uint4(x.x & m, x.y & m, x.z & m, x.w & m); }

template <int HD, int SHAPE>   // HD: compile-time bound of head_dim (a.hd <= HD)
struct WaveAttn {
    static constexpr int KS = HD / 32;   // k-steps of S^T = K Q^T
    static constexpr int CB = HD / 16;   // column blocks of O
    static constexpr bool EARLY_V = HD <= 128;   // registers allow the values to be fetched before the scores
    float m, l;                          // running max and sum of this lane's row
    f32x4_t o[CB];                       // lane (j, g): O[row 4g+r][16*cb + j]
    bf16x8_t qf[KS];                     // lane (row, g): Q[row][32u + 8g ..]

    __device__ __forceinline__ void init(const bf16* qrow, int hd) {
        m = NEG_INF;
        l = 0.f;
        const int g = threadIdx.x >> 4 & 3;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) o[cb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < KS; ++u) {
            const int d = 32 * u + 8 * g;
            uint4 v = (qrow && d < hd) ? *(const uint4*)(qrow + d) : make_uint4(0, 0, 0, 0);
            qf[u] = __builtin_bit_cast(bf16x8_t, v);
        }
    }

    // WALKS: for waves that walk many tiles (see `fx_attn_wave_walks`)
    // keys [kt0, kt0 + 64); this lane's row sees key t iff t <= hi and (lo <= t or t < span.keep) (hi < lo: row unused)
    // `slope`, `qpos`, `head`: the row's distance penalty, its query's position and its head, where the scores are shaped
    template <bool WALKS>
    __device__ __forceinline__ void tile(const AttnArgs& a, const PageLookup& pl, int kvh, int kt0, const KeySpan& span,
                                         int lo, int hi, float slope, int qpos, int head) {
        const int kv_end = span.end;
        const int lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
        const int l8 = li & 7, lh = li >> 3;
        const int hd = a.hd, bs = a.bs, vd = a.vd;      // (vd <= hd: the value heads may be narrower than the key heads)
        // Loads are issued without branches: a key outside [kv_begin, kv_end) (its page may have been
        // given back) reads from a group of keys that is inside, and its data is replaced by zeros.
        const int safe_group = (kv_end - 1) & ~15;
        // values first, so that they arrive while the scores are computed: 16 consecutive keys
        // kt0 + 16g .. of transposed row d = 16*cb + li
        const int kg = kt0 + 16 * g;
        const bool edge = !span.holds_tile(kt0);      // some key of the tile is outside
        const bool vlive = span.touches(kg, 16);
        const int vkey = vlive ? kg : safe_group;
        // every page id of the tile is looked up before the first load leaves: a lookup that stands between two
        // groups of loads makes the second group wait for the first
        constexpr int KP = KS & ~1;      // k-steps that are loaded in pairs, whole lines of eight keys at a time
        constexpr int NP = KP < KS ? 13 : 9;
        int key_of[NP], page_of[NP], slot_of[NP];
        bool klives[4];
        // rows li % 8 and 8 + li % 8 of the block's 16 keys (row i is key 16 (i / 4) + 4 kb + i % 4 of the tile)
        const int row0 = 16 * (li >> 2) + (li & 3), row_a = 16 * (l8 >> 2) + (l8 & 3), row_b = row_a + 32;
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) klives[kb] = (WALKS && !edge) || span.has(kt0 + row0 + 4 * kb);
        if ((!WALKS || !edge) && a.bs_shift >= 6) {
            // the tile is on one page, which is there, as some key of it is: one lookup, and slots that follow each other (what stands in those of other keys is masked below).
            // Nine lookups a tile took 16 heads of 128 and one sequence of 2,060 keys in a trace of the step 10.1 us a launch, this 9.7; four waves of heads of 128 with values of 64, 8 sequences, 26.3 and 25.5.
            // In waves that walk many tiles it is for tiles whose keys are all there.
            const int page = pl.page(kt0 >> a.bs_shift), slot = kt0 & (a.bs - 1);
#pragma unroll
            for (int i = 0; i < NP; ++i) page_of[i] = page;
            slot_of[0] = slot + 16 * g;
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
                slot_of[1 + kb] = slot + row_a + 4 * kb;
                slot_of[5 + kb] = slot + row_b + 4 * kb;
                if constexpr (KP < KS) slot_of[9 + kb] = slot + row0 + 4 * kb;
            }
        } else {
            key_of[0] = vkey;
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
                const int key0 = kt0 + row0 + 4 * kb, key_a = kt0 + row_a + 4 * kb, key_b = kt0 + row_b + 4 * kb;
                key_of[1 + kb] = span.has(key_a) ? key_a : safe_group;
                key_of[5 + kb] = span.has(key_b) ? key_b : safe_group;
                if constexpr (KP < KS) key_of[9 + kb] = klives[kb] ? key0 : safe_group;
            }
            pages_of(a, pl, key_of, page_of, slot_of);
        }
        const int *kpage_a = page_of + 1, *kslots_a = slot_of + 1, *kpage_b = page_of + 5, *kslots_b = slot_of + 5;
        const bf16* vbase = (const bf16*)a.v_pages + ((size_t)page_of[0] * a.nkv + kvh) * vd * bs + slot_of[0];
        uint4 vv[EARLY_V ? CB : 1][2];
        const uint32_t vmask = opaque_mask(vlive);
        if (EARLY_V) {
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                // whole lines: the first load's lanes take rows 16 cb + li % 8, the second's the eight after them, both
                // the keys 8 (li / 8) .. of the lane's 16; the halves change places before the products
                const int d1 = 16 * cb + l8, d2 = d1 + 8;
                vv[cb][0] = load_lines16(vbase + (size_t)(d1 < vd ? d1 : 0) * bs + 8 * lh);
                vv[cb][1] = load_lines16(vbase + (size_t)(d2 < vd ? d2 : 0) * bs + 8 * lh);
            }
        }
        f32x4_t sc[4];
        uint4 kf[4][KS];
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            const bf16* kra = (const bf16*)a.k_pages + (((size_t)kpage_a[kb] * a.nkv + kvh) * bs + kslots_a[kb]) * hd;
            const bf16* krb = (const bf16*)a.k_pages + (((size_t)kpage_b[kb] * a.nkv + kvh) * bs + kslots_b[kb]) * hd;
#pragma unroll
            for (int u = 0; u < KP; u += 2) {
                if (HD > 128 && 32 * u >= hd) continue;           // (the same in every lane: k-steps past the head's size)
                const int d = 32 * u + 32 * lh + 8 * g;           // the low or the high 32 of the pair's 64
                kf[kb][u] = load_lines16(kra + (d < hd ? d : 0));
                kf[kb][u + 1] = load_lines16(krb + (d < hd ? d : 0));
            }
            if (KP < KS) {
                const bf16* kr = (const bf16*)a.k_pages + (((size_t)page_of[NP - 4 + kb] * a.nkv + kvh) * bs + slot_of[NP - 4 + kb]) * hd;
                const uint32_t kmask = opaque_mask(klives[kb]);
#pragma unroll
                for (int u = KP; u < KS; ++u) {
                    const int d = 32 * u + 8 * g;
                    const uint4 x = *(const uint4*)(kr + (d < hd ? d : 0));
                    kf[kb][u] = and_mask(x, kmask & opaque_mask(d < hd));
                }
            }
        }
        BiasRow bias = {};      // (behind the keys: in front of them it would take the registers that their addresses need)
        if (SHAPE == SHAPE_BIAS) bias = fetch_bias(a, head, qpos - (kt0 + 16 * g));
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            sc[kb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
            const uint32_t kmask = opaque_mask(klives[kb]);
#pragma unroll
            for (int u = 0; u < KS; ++u) {
                if (HD > 128 && 32 * u >= hd) continue;
                uint4 ku = kf[kb][u];
                if (u < KP) {
                    // low 32: own first load below lane 8 of a row of 16, the other half's second load above;
                    // high 32: the other half's first load below, own second load above
                    ku = (u & 1) ? swap_halves<0x3>(kf[kb][u], kf[kb][u - 1]) : swap_halves<0xC>(kf[kb][u], kf[kb][u + 1]);
                    ku = and_mask(ku, kmask & opaque_mask(32 * u + 8 * g < hd));
                }
                sc[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, ku), qf[u], sc[kb], 0, 0, 0);
            }
        }
        // Heads too wide for their values to be fetched before the scores: the values arrive in groups of VG column
        // blocks, a group's loads issued together and a group ahead of the products that use them (the first one before
        // the softmax), so that a tile waits for memory CB / VG times and not once per column block.
        constexpr int VG = CB < 4 ? CB : (EARLY_V ? 4 : 8);      // (wide heads, groups of four / eight: 8 sequences of 2,060 latent keys 18.1 / 17.5 us, 64 41.1 / 38.7)
        uint4 ahead[EARLY_V ? 1 : VG][2];
        auto fetch_values = [&](int c0) {
#pragma unroll
            for (int j = 0; j < VG; ++j) {
                const int d1 = 16 * (c0 + j) + l8, d2 = d1 + 8;
                ahead[EARLY_V ? 0 : j][0] = load_lines16(vbase + (size_t)(d1 < vd ? d1 : 0) * bs + 8 * lh);
                ahead[EARLY_V ? 0 : j][1] = load_lines16(vbase + (size_t)(d2 < vd ? d2 : 0) * bs + 8 * lh);
            }
        };
        if (!EARLY_V) fetch_values(0);
        // softmax on this lane's 16 scores (keys kt0 + 16g + 4kb + r); the row's four lanes share max and sum
        uint4 p_lo, p_hi;
        constexpr bool shaped = SHAPE != SHAPE_NONE;
        if (SHAPE == SHAPE_CAP_SLOPE) cap_and_slope(sc, kt0 + 16 * g, a, slope, qpos);
        if (SHAPE == SHAPE_BIAS) shape_with_bias(sc, kt0 + 16 * g, a, slope, qpos, [&](int i) { return bias.v[i >> 2][i & 3]; });
        const float alpha = softmax_step<true>(sc, kt0 + 16 * g, lo, hi, shaped ? LOG2E : a.scale * LOG2E, m, l, p_lo, p_hi, span.keep);
        const bool rescale = __builtin_amdgcn_ballot_w64(alpha != 1.f) != 0;
        float al[4] = {1.f, 1.f, 1.f, 1.f};
        if (rescale) {
#pragma unroll
            for (int r = 0; r < 4; ++r) al[r] = __shfl(alpha, 4 * g + r, 64);
        }
        // (Narrow heads whose scores are shaped ask for the edge at each column block: 64 sequences of 2,060 keys, 16 heads of 64 with biases, 125 us with masks in every tile, 112 so; 8 of
        // them capped 23.4 and 21.4.  In the others a branch a column block costs 1 % on average.)
        constexpr bool APART = HD <= 64 && SHAPE != SHAPE_NONE;
        uint32_t kept[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) kept[i] = vmask;
        if (edge) key_masks(kept, kg, span);
#pragma unroll
        for (int c0 = 0; c0 < CB; c0 += VG) {
            if (HD > 128 && 16 * c0 >= vd) break;                 // (the same in every lane: columns past the value head's size)
            uint4 now[EARLY_V ? 1 : VG][2];
            if (!EARLY_V) {
#pragma unroll
                for (int j = 0; j < VG; ++j) {
                    now[j][0] = ahead[j][0];
                    now[j][1] = ahead[j][1];
                }
                if (c0 + VG < CB && 16 * (c0 + VG) < vd) fetch_values(c0 + VG);
            }
#pragma unroll
            for (int j = 0; j < VG; ++j) {
                const int cb = c0 + j;
                const uint4 t1 = EARLY_V ? vv[EARLY_V ? cb : 0][0] : now[EARLY_V ? 0 : j][0];
                const uint4 t2 = EARLY_V ? vv[EARLY_V ? cb : 0][1] : now[EARLY_V ? 0 : j][1];
                uint4 v0 = swap_halves<0xC>(t1, t2), v1 = swap_halves<0x3>(t2, t1);
                if (APART) {
                    v0 = and_mask(v0, vmask);
                    v1 = and_mask(v1, vmask);
                }
                if (!APART || edge) {
                    v0 = make_uint4(v0.x & kept[0], v0.y & kept[1], v0.z & kept[2], v0.w & kept[3]);
                    v1 = make_uint4(v1.x & kept[4], v1.y & kept[5], v1.z & kept[6], v1.w & kept[7]);
                }
                o[cb] = pv_step(o[cb], rescale, al, p_lo, p_hi, v0, v1);      // (columns past vd: row 0's values, never stored)
            }
        }
    }
};

// ---------------------------------------------------------------------------
// float32 on MFMA (head sizes that are multiples of 4 up to 256, pages of a multiple of 4 keys): one wave owns 16 rows
// that share a kv head, 16 consecutive queries of a head (prefill) or the query heads of a kv group at one token
// (decode).  v_mfma_f32_16x16x4_f32 multiplies and adds in float32.  S^T = K Q^T with keys as the first operand leaves
// lane (row = lane % 16, g = lane / 16) the scores of keys 16 kb + 4 g + r of its own row, and the same registers are the
// second operand of O^T += V^T P^T, whose first operand is four consecutive keys of a transposed value row: keys and
// values go from memory straight into operands, no LDS and no barrier.  A unit (16 keys x up to 128 numbers, or 32 value
// rows x 64 keys) is on its way while the one before it is multiplied; page ids are asked for a tile ahead.
// (A lane per key that reads its row number by number, as the kernels for any shape do, took 514 us a layer for 700
// tokens of 16 heads and 124 us for four single queries at 1,030 keys; these take 88 and 22 us.  What bounds them now is
// one wave's chain: 256 products of 32 cycles a tile of 64 keys x 128 numbers, 3.4 of the 5.8 us that a tile takes where the other SIMDs are idle, and where four waves
// of a block read the same tile, 8 us, the CU's L1: half lines, 64 KB a tile and wave.  Masks and pages without branches: 700 tokens 94.5 -> 88.2 us, 300 46.9 -> 38.7,
// 64 17.9 -> 16.1, 20 at 3,000 keys 345 -> 271, 1,500 under a window of 128 74.5 -> 62.0; four single queries at 1,030 keys 24.9 -> 21.7; heads of 64, 700 tokens 64.7 -> 47.2, single queries 17.3 -> 13.7.)
// ---------------------------------------------------------------------------
template <int HDM>
struct F32Attention {
    static constexpr int NC = HDM / 16;                         // groups of 16 numbers in a row
    static constexpr int UC = NC < 8 ? NC : 8, NU = NC / UC;    // a unit's groups, units of a key block
    f32x4_t q[NC];     // the row's query, scaled: numbers 16 c + 4 g + u
    f32x4_t o[NC];     // the row's outputs 16 c + 4 g + u
    float m, l;

    // `query`: the row's query, of a row that exists (`there`) or of any other.  The loads are unconditional, the choice comes after
    // them: behind a branch each load was waited for before the next one, up to 64 waits in a row in front of the first key (a single
    // query of 16 heads over 64 keys, merge included: heads of 64 12.8 -> 11.2 us, of 128 16.9 -> 14.2).
    __device__ __forceinline__ void begin(const AttnArgs& a, const float* query, bool there, int g) {
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int u = 0; u < 4; ++u) q[c][u] = query[min(16 * c + 4 * g, a.hd - 4) + u];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const bool real = there && 16 * c + 4 * g < a.hd;
            o[c] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < 4; ++u) q[c][u] = real ? q[c][u] * a.scale : 0.f;
        }
        m = NEG_INF;
        l = 0.f;
    }
    __device__ __forceinline__ static int next_tile(const KeySpan& span, int kt0) {
        return (kt0 >= span.keep && kt0 + 64 <= span.begin) ? span.begin & ~63 : kt0;
    }
    // Tiles of 64 keys from `first` (a multiple of 64) to the span's end.  The row stands at `pos`, head `h`, and sees keys
    // from `lo` on (and the kept first ones).
    __device__ __forceinline__ void walk(const AttnArgs& a, const int* bt, int kvh, const KeySpan& span, int first, int pos, int lo, int h) {
        const int lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
        const bool shaped = shapes_scores(a);
        const float slope = a.slopes ? a.slopes[h] : 0.f;
        // (a key outside the span may have lost its page: its lane reads a key of the span instead, and its score is masked)
        const int safe = span.begin < span.end ? span.end - 1 : min(span.keep, span.end) - 1;
        const float* kp[4];       // the tile's key rows of this lane, from number 4 g on
        const float* vp[4];       // row li of the values, at keys 16 c + 4 g
        int page_ids[8], page_slots[8];      // of the keys, then of the values
        auto ask_pages = [&](int kt0) {
            int t[8], blk[8];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int k = kt0 + 16 * c + li, v = kt0 + 16 * c + 4 * g;
                t[c] = span.has(k) ? k : safe;
                // (four keys of one page: the page is there if any of them is in the span)
                t[4 + c] = span.touches(v, 4) ? v : safe & ~3;
            }
            int (&slot)[8] = page_slots;
            if (a.bs_shift >= 0) {
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    blk[c] = t[c] >> a.bs_shift;
                    slot[c] = t[c] & (a.bs - 1);
                }
            } else {
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    blk[c] = t[c] / a.bs;
                    slot[c] = t[c] - blk[c] * a.bs;
                }
            }
#pragma unroll
            for (int c = 0; c < 8; ++c) page_ids[c] = bt[blk[c]];
        };
        auto point_keys = [&]() {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                kp[c] = (const float*)a.k_pages + (((size_t)page_ids[c] * a.nkv + kvh) * a.bs + page_slots[c]) * a.hd + min(4 * g, a.hd - 4);
        };
        auto point_values = [&]() {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                vp[c] = (const float*)a.v_pages + (((size_t)page_ids[4 + c] * a.nkv + kvh) * a.vd + min(li, a.vd - 1)) * a.bs + page_slots[4 + c];
        };
        f32x4_t kb[2][UC];
        auto fetch_keys = [&](int set, int unit) {       // unit: key block, then the part of its numbers
            const int c0 = unit % NU * UC;
            const int at = min(4 * g, a.hd - 4);
#pragma unroll
            for (int i = 0; i < UC; ++i) kb[set][i] = *(const f32x4_t*)(kp[unit / NU] + (min(16 * (c0 + i) + 4 * g, a.hd - 4) - at));
        };
        f32x4_t vb[2][8];
        auto fetch_values = [&](int set, int pair) {     // value rows 32 pair .. 32 pair + 31
            const int v0 = min(li, a.vd - 1);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int c = 0; c < 4; ++c) vb[set][4 * i + c] = *(const f32x4_t*)(vp[c] + (size_t)(min(32 * pair + 16 * i + li, a.vd - 1) - v0) * a.bs);
        };
        int kt0 = next_tile(span, first);
        if (kt0 >= span.end) return;
        ask_pages(kt0);
        point_keys();
        point_values();
        fetch_keys(0, 0);
        while (true) {
            const int after = next_tile(span, kt0 + 64);
            const bool more = after < span.end;
            ask_pages(more ? after : kt0);
            f32x4_t s[4];
#pragma unroll
            for (int unit = 0; unit < 4 * NU; ++unit) {
                if (unit + 1 < 4 * NU) fetch_keys((unit + 1) & 1, unit + 1);
                else fetch_values(0, 0);
                if (a.hd < HDM) {      // numbers that the head does not have: zeros, for 0 (the query's) times infinity is none
#pragma unroll
                    for (int i = 0; i < UC; ++i)
                        if (16 * (unit % NU * UC + i) + 4 * g >= a.hd) kb[unit & 1][i] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
                }
                // (two chains of sums: an instruction that waits for the one before it takes longer than its turn)
                f32x4_t part[2] = {(f32x4_t){0.f, 0.f, 0.f, 0.f}, (f32x4_t){0.f, 0.f, 0.f, 0.f}};
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int i = 0; i < UC; ++i)
                        part[i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kb[unit & 1][i][u], q[unit % NU * UC + i][u], part[i & 1], 0, 0, 0);
                s[unit / NU] = unit % NU == 0 ? part[0] + part[1] : s[unit / NU] + (part[0] + part[1]);
            }
            if (shaped) {
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[c][r] = shaped_score(a, h, slope, s[c][r], pos - (kt0 + 16 * c + 4 * g + r));
            }
            // (masks as one number each, and none for a tile that all rows see whole: in `&&` and `||` a score's was up to four branches of some 35 ns)
            const bool whole = span.holds_tile(kt0);
            if (!whole || !__all((kt0 >= lo) & (kt0 + 63 <= pos))) {
                const int from = max(lo, span.begin), to = min(pos, span.end - 1);
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int t = kt0 + 16 * c + 4 * g + r;
                        s[c][r] = ((t <= to) & ((t >= from) | (t < a.keep_first))) ? s[c][r] : NEG_INF;
                    }
            }
            float top = NEG_INF;
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) top = fmaxf(top, s[c][r]);
            const float m_new = fmaxf(m, quad_max(top));
            const float al = m_new == NEG_INF ? 1.f : expf(m - m_new), from_m = m_new == NEG_INF ? 0.f : m_new;
            float sum = 0.f;
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    s[c][r] = expf(s[c][r] - from_m);       // (minus infinity: 0)
                    sum += s[c][r];
                }
            l = l * al + quad_sum(sum);
            m = m_new;
            int inside = 0;      // bit 4 c + r: key 16 c + 4 g + r of the tile is in the span
            if (!whole) {
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r) inside |= (span.has(kt0 + 16 * c + 4 * g + r) ? 1 : 0) << (4 * c + r);
            }
#pragma unroll
            for (int pair = 0; pair < (NC + 1) / 2; ++pair) {
                if (pair + 1 < (NC + 1) / 2) fetch_values((pair + 1) & 1, pair + 1);
                f32x4_t (&v)[8] = vb[pair & 1];
                if (!whole) {          // memory of keys outside the span may hold anything
#pragma unroll
                    for (int c = 0; c < 4; ++c)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (!(inside >> (4 * c + r) & 1)) v[c][r] = v[4 + c][r] = 0.f;
                }
                o[2 * pair] *= al;
                o[2 * pair + 1] *= al;
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        o[2 * pair] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[c][r], s[c][r], o[2 * pair], 0, 0, 0);
                        o[2 * pair + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[4 + c][r], s[c][r], o[2 * pair + 1], 0, 0, 0);
                    }
                if (pair == 0) {
                    // (the next tile's first keys: their pages were asked for a tile ago)
                    point_keys();
                    fetch_keys(0, 0);
                }
            }
            if (!more) return;
            point_values();
            kt0 = after;
        }
    }
};

// prefill: block = (item of up to 64 queries, head), a wave per 16 queries
template <int HDM>
__global__ __launch_bounds__(256) void attn_f32_block_kernel(AttnArgs a) {
    const int item = blockIdx.x, h = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
    const int kvh = h / (a.nh / a.nkv);
    const int tok0 = a.item_tok[item] + 16 * wave, n = min(16, a.item_n[item] - 16 * wave);
    if (n <= 0) return;
    const int* bt = a.block_table + (size_t)a.item_seq[item] * a.max_blocks;
    const int tok = tok0 + min(li, n - 1);
    const int pos = a.positions[tok], pmin = a.positions[tok0], pmax = a.positions[tok0 + n - 1];
    const KeySpan span = {first_visible(a, pmin), pmax + 1, a.keep_first};
    F32Attention<HDM> w;
    w.begin(a, (const float*)a.q + (size_t)tok * a.ldq + (size_t)h * a.hd, li < n, g);
    w.walk(a, bt, kvh, span, 0, pos, first_visible(a, pos), h);
    if (li >= n) return;
    const float fin = finish_row<false>(a, h, w.m, w.l);
#pragma unroll
    for (int c = 0; c < HDM / 16; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int d = 16 * c + 4 * g + r;
            if (d >= a.vd) continue;
            float v = w.o[c][r] * fin;
            if (a.turns) v = turned_back(a, tok, d, v, w.o[c][r ^ 1] * fin);
            store_out<float>(a, tok, h, d, v);
        }
}
// decode: block = one wave = (item, kv head x block of 16 of its query heads, chunk of keys); results merge as those of
// attn_decode_kernel do.  Queries below position FEW_KEYS go a wave per head as in that kernel: it is through with so few keys before a
// tile's chain of waits is, which takes the same for any number of keys (merge included, 16 heads of 128: 5 keys 10.0 against 14.0 us, 12 12.4, 16 13.9, 20 15.4; 16 of 64 in groups
// of four: 5 keys 8.0 against 11.0, 16 10.1, 20 10.8, 24 11.6; 16 of 256 in groups of eight: 5 keys 14.1 against 20.5, 12 19.4, 14 20.9.  By time
// alone the line would be at 20, 16 and 12 keys for heads of 64, 128 and 256; it is where these positions have had the bits of the kernels for any shape).
// The waves for a group's other heads come behind the chunks' blocks (a wave per head in every chunk, most of which leave again: 16
// sequences of 3,000 keys, heads of 64, 30 -> 42 us).  The choice is the position's alone, so a query's bits do not depend on the step.
template <int HDM>
__global__ __launch_bounds__(64) void attn_f32_decode_kernel(AttnArgs a) {
    constexpr int FEW_KEYS = HDM == 128 ? 24 : 32;
    const int item = blockIdx.x, split = blockIdx.z, lane = threadIdx.x, li = lane & 15, g = lane >> 4;
    const int group = a.nh / a.nkv, group_blocks = (group + 15) / 16;
    const int kvh = blockIdx.y / group_blocks, first = blockIdx.y % group_blocks * 16, row = first + li;
    if (split == 0 || split >= a.splits) {
        const int own = split ? first + 1 + split - a.splits : first;
        const bool few = a.positions[a.item_tok[item]] < FEW_KEYS;
        if (few && own < group) decode_head<float, HDM>(a, item, kvh * group + own, 0);
        if (few || split) return;
    }
    const bool there = row < group;
    const int h = kvh * group + min(row, group - 1);
    const int tok = a.item_tok[item];
    const int* bt = a.block_table + (size_t)a.item_seq[item] * a.max_blocks;
    const int p = a.positions[tok], s0 = split * a.chunk, lo = first_visible(a, p);
    const KeySpan span = {max(lo, s0), min(p + 1, s0 + a.chunk), a.keep_first};
    F32Attention<HDM> w;
    w.m = NEG_INF;
    w.l = 0.f;
    if (s0 < span.end && (span.begin < span.end || s0 < span.keep)) {
        w.begin(a, (const float*)a.q + (size_t)tok * a.ldq + (size_t)h * a.hd, there, g);
        w.walk(a, bt, kvh, span, s0, p, lo, h);
    }
    if (!there) return;
    const size_t at = ((size_t)item * a.nh + h) * a.splits + split;
    if (g == 0) {
        a.part_ml[2 * at] = w.m;
        a.part_ml[2 * at + 1] = w.l;
    }
    if (w.m == NEG_INF) return;
#pragma unroll
    for (int c = 0; c < HDM / 16; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int d = 16 * c + 4 * g + r;
            if (d < a.vd) a.part_o[at * a.vd + d] = w.o[c][r];
        }
}

// prefill: item = up to 16 consecutive queries of one sequence; block = one wave = (item, head)
template <int HD, int SHAPE>
__global__ __launch_bounds__(64) void attn_mfma_tile_kernel(AttnArgs a) {
    const int item = blockIdx.x >> 2, sub = blockIdx.x & 3, h = blockIdx.y, lane = threadIdx.x, li = lane & 15, g = lane >> 4;
    const int kvh = h / (a.nh / a.nkv);
    const int tok0 = a.item_tok[item] + 16 * sub, n = min(16, a.item_n[item] - 16 * sub);
    if (n <= 0) return;
    const int* bt = a.block_table + (size_t)a.item_seq[item] * a.max_blocks;
    const int hd = a.hd;
    const int pmin = a.positions[tok0], pmax = a.positions[tok0 + n - 1];
    const int kv_begin = first_visible(a, pmin);
    const int kv_end = pmax + 1;
    int lo = 1, hi = 0;
    const bf16* qrow = nullptr;
    if (li < n) {
        hi = a.positions[tok0 + li];
        lo = first_visible(a, hi);
        qrow = (const bf16*)a.q + (size_t)(tok0 + li) * a.ldq + (size_t)h * hd;
    }
    WaveAttn<HD, SHAPE> w;
    w.init(qrow, hd);
    const PageLookup pl = {bt, nullptr, 0, 0};
    const KeySpan span = {kv_begin, kv_end, a.keep_first};
    const TileWalk walk = tile_walk(span);
    const float slope = a.slopes ? a.slopes[h] : 0.f;
    for (int ti = 0; ti < walk.n; ++ti) w.template tile<false>(a, pl, kvh, walk.start(ti), span, lo, hi, slope, max(hi, 0), h);
    const float fin = li < n ? finish_row<true>(a, h, w.m, w.l) : 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 4 * g + r;
        const float fr = __shfl(fin, row, 64);
        if (row < n) {
#pragma unroll
            for (int cb = 0; cb < WaveAttn<HD, SHAPE>::CB; ++cb) {
                const int d = 16 * cb + li;
                if (d < a.vd) store_lane<bf16>(a, tok0 + row, h, d, w.o[cb][r] * fr);
            }
        }
    }
}

// decode, several waves per block: block = (item, kv head x group block of 16 query heads, split);
// its waves take the split's tiles of 64 keys in turn and their results are merged through LDS in
// wave order.  With one split the block writes the output itself, no second launch.
template <int HD, int MAX_THREADS, int SHAPE, bool WALKS = false>
__global__ __launch_bounds__(MAX_THREADS) void attn_mfma_decode_block_kernel(AttnArgs a) {
    extern __shared__ float wave_out[];      // [waves][rows][HD + 2]: o, then m and l
    // The grid is (heads, items, splits): blocks go to the eight XCDs in turn, so with the heads fastest every
    // item's blocks are spread over all of them, and with the splits slowest a sequence's last, shorter chunks start
    // last.  (With the items fastest and their number a multiple of eight, as a recorded step's is, an item's blocks
    // all land on one XCD, and 17 live sequences beside 7 stand-ins give one XCD three sequences and the others
    // two: 73 against 57 us.)
    const int item = blockIdx.y, split = blockIdx.z;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n_waves = blockDim.x >> 6;
    const int li = lane & 15, g = lane >> 4;
    const int group = a.nh / a.nkv, gblocks = (group + 15) / 16;
    const int kvh = blockIdx.x / gblocks, hb = blockIdx.x % gblocks;
    const int tok = a.item_tok[item];
    const int* bt = a.block_table + (size_t)a.item_seq[item] * a.max_blocks;
    const int hd = a.hd;
    const int p = a.positions[tok];
    // The keys this query sees, from the tile of 64 that holds the first of them on, go to the splits in equal
    // chunks of whole tiles: a sequence shorter than the launch's bound, or a window far into a long sequence,
    // still keeps every split busy.  (a.chunk is the longest chunk any sequence of the launch can have.)
    __shared__ int page_copy[PAGE_COPY];
    int first_blk, last_blk, unused;
    PageLookup pl;
    if (!bounded_keys(a)) {
        // the page ids that the split can need, whatever the position turns out to be, are copied before the
        // position has arrived (entries past the sequence's pages are read and never used)
        page_slot(a, (split + 1) * a.chunk - 1, last_blk, unused);
        last_blk = min(last_blk, a.max_blocks - 1);
        pl = stage_pages(bt, page_copy, max(0, last_blk - PAGE_COPY + 1), last_blk);
    }
    const int first_key = first_visible(a, p);
    const int base = first_key & ~63;
    const int chunk = (((p + 1 - base + a.splits - 1) / a.splits) + 63) & ~63;
    const int kv_begin = max(first_key, base + split * chunk);
    const int kv_end = min(p + 1, base + (split + 1) * chunk);
    if (bounded_keys(a)) {
        page_slot(a, min(kv_begin, p), first_blk, unused);
        page_slot(a, max(kv_end - 1, 0), last_blk, unused);
        first_blk = min(first_blk, a.max_blocks - 1);
        last_blk = min(last_blk, a.max_blocks - 1);
        pl = stage_pages(bt, page_copy, first_blk, last_blk);
    }
    const int n = min(16, group - hb * 16);        // query heads in this block
    const int h0 = kvh * group + hb * 16;
    const bool empty = kv_begin >= kv_end;
    WaveAttn<HD, SHAPE> w;
    const bool row_ok = li < n;
    w.init(row_ok && !empty ? (const bf16*)a.q + (size_t)tok * a.ldq + (size_t)(h0 + li) * hd : nullptr, hd);
    if (!empty) {
        // (the kept first keys of the sequence, where they lie before the window, go with the first split)
        const KeySpan span = {kv_begin, kv_end, split == 0 ? min(a.keep_first, kv_begin) : 0};
        const TileWalk walk = tile_walk(span);
        const int lo = row_ok ? kv_begin : 1, hi = row_ok ? kv_end - 1 : 0;
        const float slope = (a.slopes && row_ok) ? a.slopes[h0 + li] : 0.f;      // (a row is a query head here)
        for (int ti = wave; ti < walk.n; ti += n_waves) w.template tile<WALKS>(a, pl, kvh, walk.start(ti), span, lo, hi, slope, p, h0 + min(li, n - 1));
    }
    if (n_waves == 1) {
        // one wave: nothing to merge, the rows go out from the registers that hold them (lane (li, g) has rows
        // 4g .. 4g + 3 of columns 16 cb + li; a row's maximum and sum sit in the lanes whose li is the row).  Without gate and turns through a buffer whose end drops the
        // columns past the value head and the rows past the group: a block's only tile is little longer than this end of it, and with a branch around each of the stores
        // (and two more inside) 40 keys of 16 heads on one kv head of
        // 256 took 14.3 us, so 11.0 (8 sequences of 2,060 keys 17.5 and 16.3; 28 heads of 128 on 4, 40 keys 8.7 and 6.9).
        // A block of one row leaves out the three that lanes hold beside it (16 heads of 128, one sequence of 300 keys, scores capped, 10.6 -> 10.1 us; 16 of 64, 64 sequences of 300 keys
        // 22.2 -> 21.9, and 21.1 with branches here and in front of the loads: a wave of narrow heads walks five tiles there, and asks for its keys' pages together in each).
        constexpr int CB = WaveAttn<HD, SHAPE>::CB;
        constexpr uint32_t OUTSIDE = 1u << 30;       // (a row and a column that do not exist: 2^31, past any end)
        const int vd = a.vd;
        const bool parts = a.splits > 1;
        auto store_rows = [&](auto rows) {
            constexpr int R = decltype(rows)::value;
            const size_t first = parts ? (((size_t)item * a.nh + h0) * a.splits + split) * vd : (size_t)tok * a.ldo + (size_t)h0 * vd;
            const int row_len = parts ? a.splits * vd : vd, size = parts ? 4 : 2;
            const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc(parts ? (void*)(a.part_o + first) : (void*)((bf16*)a.out + first), 0, ((n - 1) * row_len + vd) * size, 0x00027000);
            float m[R], l[R];
            uint32_t at[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                m[r] = __shfl(w.m, 4 * g + r, 64);
                l[r] = __shfl(w.l, 4 * g + r, 64);
                at[r] = 4 * g + r < n ? (4 * g + r) * row_len * size : OUTSIDE;
            }
            if (parts) {
#pragma unroll
                for (int cb = 0; cb < CB; ++cb) {
                    const uint32_t column = 16 * cb + li < vd ? 4 * (16 * cb + li) : OUTSIDE;
#pragma unroll
                    for (int r = 0; r < R; ++r) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(m[r] == NEG_INF ? 0.f : w.o[cb][r]), to, at[r] + column, 0, 0);
                }
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (li == 0 && 4 * g + r < n) {
                        float* pml = a.part_ml + (((size_t)item * a.nh + h0 + 4 * g + r) * a.splits + split) * 2;
                        pml[0] = m[r] == NEG_INF ? NEG_INF : m[r] * LN2;
                        pml[1] = m[r] == NEG_INF ? 0.f : l[r];
                    }
                return;
            }
            float fin[R];
#pragma unroll
            for (int r = 0; r < R; ++r) fin[r] = finish_row<true>(a, h0 + min(4 * g + r, n - 1), m[r], l[r]);
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const uint32_t column = 16 * cb + li < vd ? 2 * (16 * cb + li) : OUTSIDE;
#pragma unroll
                for (int r = 0; r < R; ++r) __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, float_to_bf16(w.o[cb][r] * fin[r])), to, at[r] + column, 0, 0);
            }
        };
        if (parts || !(a.gate || a.turns)) {
            if (n == 1) store_rows(std::integral_constant<int, 1>{});
            else store_rows(std::integral_constant<int, 4>{});
            return;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 4 * g + r;
            const float m = __shfl(w.m, row, 64), l = __shfl(w.l, row, 64);
            if (row >= n) continue;
            const int h = h0 + row;
            const float fin = finish_row<true>(a, h, m, l);
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const int d = 16 * cb + li;
                if (d < vd) store_lane<bf16>(a, tok, h, d, w.o[cb][r] * fin);
            }
        }
        return;
    }
    const int stride = HD + 2;
    float* mine = wave_out + (size_t)wave * n * stride;
    if (row_ok && g == 0) {
        mine[li * stride + HD] = w.m;            // base 2
        mine[li * stride + HD + 1] = w.l;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 4 * g + r;
        if (row < n) {
#pragma unroll
            for (int cb = 0; cb < WaveAttn<HD, SHAPE>::CB; ++cb) mine[row * stride + 16 * cb + li] = w.o[cb][r];
        }
    }
    __syncthreads();
    // the block's threads are dealt out to the rows in equal shares: each works out its row's maximum, the waves'
    // weights and the sum once, then takes every per_row-th column
    const int vd = a.vd;
    const int per_row = blockDim.x / n;
    const int row = threadIdx.x / per_row, sub = threadIdx.x - row * per_row;
    if (row >= n) return;
    // (up to four waves or up to eight; waves past the last stand for it with weight 0: all reads of a step of this on their way together.  In loops over the waves that there are each
    // read was waited for, us: 16 heads of 128, one sequence of 2,060 keys 11.9, so 11.3, 8 29.8 and 29.0; 28 heads on 4, 8 sequences 16.0 and 15.3.)
    auto merge = [&](auto most) {
        constexpr int W = decltype(most)::value;
        const float* from[W];
        float ms[W], ls[W], f[W], m = NEG_INF, l = 0.f;
#pragma unroll
        for (int u = 0; u < W; ++u) {
            from[u] = wave_out + ((size_t)min(u, n_waves - 1) * n + row) * stride;
            ms[u] = from[u][HD];
            ls[u] = from[u][HD + 1];
        }
#pragma unroll
        for (int u = 0; u < W; ++u) m = fmaxf(m, ms[u]);
#pragma unroll
        for (int u = 0; u < W; ++u) {
            const float e = __builtin_amdgcn_exp2f(ms[u] - m);
            f[u] = ((u < n_waves) & (ms[u] != NEG_INF)) ? e : 0.f;
            l += f[u] * (u < n_waves ? ls[u] : 0.f);
        }
        auto value = [&](int u, int d) {      // (of a wave that is there: the last one's sum may be infinite, and an infinity with weight 0 is no 0)
            const float v = from[u][d];
            return u < n_waves ? v : 0.f;
        };
        const int h = h0 + row;
        const bool last = a.splits == 1;
        const float fin = last ? finish_row<true>(a, h, m, l) : 1.f;
        float* po = a.part_o + (((size_t)item * a.nh + h) * a.splits + split) * vd;
        if (last && a.turns) {      // pairs of columns, which are turned back together
            for (int d = 2 * sub; d < vd; d += 2 * per_row) {
                float o0 = 0.f, o1 = 0.f;
#pragma unroll
                for (int u = 0; u < W; ++u) {
                    o0 += f[u] * value(u, d);
                    o1 += f[u] * value(u, d + 1);
                }
                o0 *= fin;
                o1 *= fin;
                store_out<bf16>(a, tok, h, d, turned_back(a, tok, d, o0, o1));
                store_out<bf16>(a, tok, h, d + 1, turned_back(a, tok, d + 1, o1, o0));
            }
            return;
        }
        for (int d = sub; d < vd; d += per_row) {
            float o = 0.f;
#pragma unroll
            for (int u = 0; u < W; ++u) o += f[u] * value(u, d);
            if (last) store_out<bf16>(a, tok, h, d, o * fin);
            else po[d] = o;
        }
        if (!last && sub == 0) {
            float* pml = a.part_ml + (((size_t)item * a.nh + h) * a.splits + split) * 2;
            pml[0] = m == NEG_INF ? NEG_INF : m * LN2;
            pml[1] = l;
        }
    };
    if (n_waves <= 4) merge(std::integral_constant<int, 4>{});
    else merge(std::integral_constant<int, 8>{});
}

// A head's row of biases for a block that walks over many tiles is copied to LDS (dynamic, sized by the launch): a load from
// memory inside the walk would be waited for behind the tiles that are on their way.  Rows longer than this are for the
// kernels for any shape (beside the stages of the widest of these kernels, 132 KB, they would not fit).
#define BIAS_LDS_MAX 6144      // floats
__device__ __forceinline__ void stage_bias(const AttnArgs& a, int h, float* lds) {      // every thread; a barrier follows before its use
    const float* row = a.bias + (size_t)h * bias_row_len(a);
    for (int i = threadIdx.x; i < bias_row_len(a); i += blockDim.x) lds[i] = row[i];
}
static size_t bias_lds_bytes(const AttnArgs& a) { return a.bias ? (size_t)bias_row_len(a) * sizeof(float) : 0; }

// Which item and head a block of a prompt takes.  Blocks go to the 8 XCDs in turn, each with an L2 of its own: block b runs on XCD b % 8, as number j = b / 8 there.
// Later items of a prompt see more keys, so every XCD takes the items from the last to the first, each for the heads that are its own: an eighth of them, so
// that their keys and values stay in its L2 (the eight, and the 32 CUs below, are this GPU's; another would lose balance, no item).  Where that is no whole number, the lines between the XCDs shift from item to item, through the eighths of a
// head in turn, and eight items make nh blocks for each.  PAIRED: two blocks fit a CU, and as the first 64 of an XCD are handed out to its 32 CUs in turn the
// second half of them runs the other way, so that a CU's two have the same work together.  (Before, an XCD took an eighth of the pairs, heads outermost: with 28 heads half of an XCD's
// last head was the long half, 7 % more than its share, and every other head's longest item came last.)
__host__ __device__ constexpr int place_shift(int row) { return ((row & 1) << 2) | (row & 2) | ((row >> 2) & 1); }       // 0 4 2 6 1 5 3 7
__host__ __device__ constexpr int place_head(int nh, int xcd, int row) { return (nh * xcd - place_shift(row & 7) + 7) >> 3; }      // the first of an XCD's heads in that row
template <bool PAIRED>
__host__ __device__ inline bool block_place(int b, int nh, int n_items, int& item, int& head) {
    const int x = b & 7;
    int j = b >> 3;
    if (PAIRED && j >= 32 && j < 64) {
        int n = n_items / 8 * nh;
        for (int row = 0; row < n_items % 8; ++row) n += place_head(nh, x + 1, row) - place_head(nh, x, row);
        if (j < n) j = 31 + min(n, 64) - j;
    }
    int row = j / nh * 8;
    j %= nh;
    for (int k = 0; k < 8; ++k, ++row) {
        const int first = place_head(nh, x, k), n = place_head(nh, x + 1, k) - first;
        if (j < n) {
            head = first + j;
            break;
        }
        j -= n;
    }
    item = n_items - 1 - row;
    return item >= 0;
}
static int place_blocks(int nh, int n_items) { return 8 * (n_items / 8 * nh + n_items % 8 * ceil_div(nh, 8)); }      // (the last ones of an XCD may have nothing)

// Prefill with the keys and values of a tile shared through LDS: a block of four waves owns up
// to 64 consecutive queries of one head (16 each); per tile of 64 keys the block stages K
// (rows permuted so that the 16 keys an MFMA operand needs lie in consecutive rows) and the
// transposed V once, and every wave takes its operands from there.  While a tile is multiplied
// the next one is already on its way from memory into registers.
template <int HD, int SHAPE>
__global__ __launch_bounds__(256, HD > 128 ? 2 : 1) void attn_mfma_block_kernel(AttnArgs a) {
    constexpr int KS = HD / 32, CB = HD / 16;
    constexpr int KROW = HD + 8;          // bf16 elements per staged key row (16 bytes of padding)
    constexpr int VROW = 64 + 8;          // bf16 elements per staged value row
    constexpr int KCH = 64 * (HD / 8), VCH = HD * 8;      // 16-byte chunks per tile
    constexpr int NK = (KCH + 255) / 256, NV = (VCH + 255) / 256;
    __shared__ __attribute__((aligned(16))) bf16 Ks[64 * KROW];
    __shared__ __attribute__((aligned(16))) bf16 Vs[HD * VROW];
    extern __shared__ float bias_lds[];
    int item, h;
    if (!block_place<false>(blockIdx.x, a.nh, a.n_items, item, h)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 15, g = lane >> 4;
    const int kvh = h / (a.nh / a.nkv);
    const int tok_first = a.item_tok[item], n_all = a.item_n[item];
    const int* bt = a.block_table + (size_t)a.item_seq[item] * a.max_blocks;
    const int hd = a.hd, bs = a.bs, vd = a.vd;      // (vd <= hd: the value heads may be narrower than the key heads)
    const int pmin = a.positions[tok_first], pmax = a.positions[tok_first + n_all - 1];
    const int kv_begin = first_visible(a, pmin);
    const int kv_end = pmax + 1;
    // this wave's 16 rows
    const int tok0 = tok_first + 16 * wave, n = min(16, n_all - 16 * wave);
    int lo = 1, hi = 0;
    const bf16* qrow = nullptr;
    if (li < n) {
        hi = a.positions[tok0 + li];
        lo = first_visible(a, hi);
        qrow = (const bf16*)a.q + (size_t)(tok0 + li) * a.ldq + (size_t)h * hd;
    }
    int w_lo = 0x7fffffff, w_hi = -1;     // keys any row of this wave can see
    int w_lo_max = 0x7fffffff, w_hi_min = -1;   // keys every row of this wave sees: [w_lo_max, w_hi_min]
    if (n > 0) {
        w_hi = a.positions[tok0 + n - 1];
        w_lo = first_visible(a, a.positions[tok0]);
        if (n == 16) {                    // a wave with idle rows masks always
            w_hi_min = a.positions[tok0];
            w_lo_max = first_visible(a, w_hi);
        }
    }
    constexpr bool shaped = SHAPE != SHAPE_NONE;
    const float slope = a.slopes ? a.slopes[h] : 0.f;
    const float cs = shaped ? LOG2E : a.scale * LOG2E;
    float m = NEG_INF, l = 0.f;
    f32x4_t o[CB];
    bf16x8_t qf[KS];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) o[cb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < KS; ++u) {
        const int d = 32 * u + 8 * g;
        uint4 v = (qrow && d < hd) ? *(const uint4*)(qrow + d) : make_uint4(0, 0, 0, 0);
        qf[u] = __builtin_bit_cast(bf16x8_t, v);
    }

    // Two tiles on their way from memory; the widest heads keep one (DEEP false): their registers then allow two blocks
    // on a CU, whose waves fill each other's waits, and a tile's products take longer than its loads.
    constexpr bool DEEP = HD <= 128;
    uint4 kreg_a[NK], vreg_a[NV], kreg_b[DEEP ? NK : 1], vreg_b[DEEP ? NV : 1];
    // Loads are issued without branches: a key outside [kv_begin, kv_end) (its page may have been
    // given back) reads from a group of keys that is inside, and its data is replaced by zeros.
    const int safe_group = (kv_end - 1) & ~15;
    const KeySpan span = {kv_begin, kv_end, a.keep_first};
    const TileWalk walk = tile_walk(span);
    __shared__ int page_copy[PAGE_COPY];
    int first_blk, last_blk, unused;
    page_slot(a, kv_begin, first_blk, unused);
    page_slot(a, kv_end - 1, last_blk, unused);
    if (SHAPE == SHAPE_BIAS) stage_bias(a, h, bias_lds);
    const PageLookup pl = stage_pages(bt, page_copy, first_blk, last_blk);
    auto fetch = [&](uint4* kreg, uint4* vreg, int kt0) {
        size_t kbase[4], vbase[4];     // page and slot of each group of 16 keys of the tile (the same for all threads)
        bool live[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int key0 = kt0 + 16 * j;
            live[j] = span.touches(key0, 16);
            int blk, slot;
            page_slot(a, live[j] ? key0 : safe_group, blk, slot);
            const size_t page = pl.page(blk);
            kbase[j] = ((page * a.nkv + kvh) * bs + slot) * hd;
            vbase[j] = (page * a.nkv + kvh) * vd * bs + slot;
        }
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const int c = tid + i * 256;
            if (c < KCH) {
                const int r = c / (HD / 8), d = (c % (HD / 8)) * 8;
                const int key = kt0 + r;
                const bool ok = span.has(key) && d < hd;
                const uint4 v = *(const uint4*)((const bf16*)a.k_pages + kbase[r >> 4] + (size_t)(r & 15) * hd + (d < hd ? d : 0));
                kreg[i] = ok ? v : make_uint4(0, 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = tid + i * 256;
            if (c < VCH) {
                const int d = c >> 3, k8 = (c & 7) * 8;
                if (HD > 128 && d >= vd) {       // (whole groups of 32 rows past the value head's size: nothing to load)
                    vreg[i] = make_uint4(0, 0, 0, 0);
                    continue;
                }
                const bool ok = d < vd && live[k8 >> 4];
                uint4 v = *(const uint4*)((const bf16*)a.v_pages + vbase[k8 >> 4] + (size_t)(d < vd ? d : 0) * bs + (k8 & 15));
                if (!span.holds_tile(kt0)) {
                    uint32_t kept[4] = {v.x, v.y, v.z, v.w};
                    key_masks(kept, kt0 + k8, span);
                    v = make_uint4(kept[0], kept[1], kept[2], kept[3]);
                }
                vreg[i] = ok ? v : make_uint4(0, 0, 0, 0);
            }
        }
    };
    auto stage = [&](const uint4* kreg, const uint4* vreg) {
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const int c = tid + i * 256;
            if (c < KCH) {
                const int r = c / (HD / 8), d = (c % (HD / 8)) * 8;
                const int row = ((r >> 2) & 3) * 16 + (r >> 4) * 4 + (r & 3);     // key 16a + 4kb + b -> row 16kb + 4a + b
                *(uint4*)(Ks + row * KROW + d) = kreg[i];
            }
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = tid + i * 256;
            if (c < VCH) *(uint4*)(Vs + (c >> 3) * VROW + (c & 7) * 8) = vreg[i];
        }
    };

    fetch(kreg_a, vreg_a, walk.start(0));
    if (DEEP && 1 < walk.n) fetch(kreg_b, vreg_b, walk.start(1));
    int parity = 0;
    for (int ti = 0; ti < walk.n; ++ti, parity ^= 1) {
        const int kt0 = walk.start(ti);
        lds_barrier();            // the previous tile has been read by every wave
        if (!DEEP || parity == 0) stage(kreg_a, vreg_a); else stage(kreg_b, vreg_b);
        lds_barrier();
        if (DEEP) {
            if (ti + 2 < walk.n) {     // the registers just emptied take the tile after the next
                if (parity == 0) fetch(kreg_a, vreg_a, walk.start(ti + 2)); else fetch(kreg_b, vreg_b, walk.start(ti + 2));
            }
        } else if (ti + 1 < walk.n) {
            fetch(kreg_a, vreg_a, walk.start(ti + 1));
        }
        if (kt0 > w_hi || (kt0 + 64 <= w_lo && kt0 >= span.keep)) continue;      // nothing in this tile for this wave's rows
        f32x4_t sc[4];
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            sc[kb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < KS; ++u) {
                if (HD > 128 && 32 * u >= hd) continue;           // (the same in every lane: k-steps past the head's size)
                const bf16x8_t kf = *(const bf16x8_t*)(Ks + (kb * 16 + li) * KROW + 32 * u + 8 * g);
                sc[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[u], sc[kb], 0, 0, 0);
            }
        }
        // tiles that every row of this wave sees whole need no mask
        const bool whole = kt0 >= w_lo_max && kt0 + 63 <= w_hi_min && kt0 >= kv_begin;
        uint4 p_lo, p_hi;
        if (SHAPE == SHAPE_CAP_SLOPE) cap_and_slope(sc, kt0 + 16 * g, a, slope, hi);
        if (SHAPE == SHAPE_BIAS) {
            const float* bias = bias_lds + bias_first(a, max(hi, 0) - (kt0 + 16 * g));
            shape_with_bias(sc, kt0 + 16 * g, a, slope, hi, [&](int i) { return bias[i]; });
        }
        const float alpha = whole ? softmax_step<false>(sc, kt0 + 16 * g, lo, hi, cs, m, l, p_lo, p_hi)
                                  : softmax_step<true>(sc, kt0 + 16 * g, lo, hi, cs, m, l, p_lo, p_hi, span.keep);
        const bool rescale = __builtin_amdgcn_ballot_w64(alpha != 1.f) != 0;
        float al[4] = {1.f, 1.f, 1.f, 1.f};
        if (rescale) {
#pragma unroll
            for (int r = 0; r < 4; ++r) al[r] = __shfl(alpha, 4 * g + r, 64);
        }
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            if (HD > 128 && 16 * cb >= vd) continue;              // (the same in every lane: columns past the value head's size)
            const bf16* vr = Vs + (16 * cb + li) * VROW + 16 * g;
            o[cb] = pv_step(o[cb], rescale, al, p_lo, p_hi, *(const uint4*)vr, *(const uint4*)(vr + 8));
        }
    }
    const float fin = li < n ? finish_row<true>(a, h, m, l) : 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 4 * g + r;
        const float fr = __shfl(fin, row, 64);
        if (row < n) {
            float y[CB];
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) y[cb] = o[cb][r] * fr;
            turn_back_row(a, tok0 + row, li, y);
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const int d = 16 * cb + li;
                if (d < vd) store_out<bf16>(a, tok0 + row, h, d, y[cb]);
            }
        }
    }
}

// Prefill when head_dim is exactly 64 or 128 and a page holds a multiple of 64 keys: a tile of 64
// keys then lies in one page, 64 * HD contiguous elements of keys and as many of transposed values,
// and travels from global memory straight into LDS (no registers in between, nothing to unpack),
// two stages, one barrier per tile.  (The next tile's loads are asked for in front of this one's products, but not in flight
// beside them: the compiler cannot tell the reads of LDS from what these loads write there, and waits for all of them, s_waitcnt
// vmcnt(0), in front of the first read behind them.  What a second stage hides is the way to that read, and other waves.)
// A wave-load fills 1 KB: 1024 / (2 HD) key rows, or eight value rows of 64 keys.  Key row
// 16 kb + 4 a + b of LDS holds key 16 a + 4 kb + b (what the MFMA operands want, see above; four
// such keys follow each other in memory and in LDS alike), and inside a row the 16-byte chunks
// stand at chunk ^ (row % 16) for key rows of 256 bytes, chunk ^ ((row / 2) % 8) for those of 128 and chunk ^ value_turn(row) for value rows, which the loading
// lanes achieve by choosing which chunk they fetch: the 16 rows an operand reads then fall on
// distinct banks without padding.  Keys outside [kv_begin, kv_end) come along as whatever memory
// holds: their scores are masked, and their values are zeroed in LDS before the product.
typedef __attribute__((address_space(1))) const void* fx_global_ptr;
typedef __attribute__((address_space(3))) void* fx_lds_ptr;

// What value row d's 16-byte chunks stand at, chunk ^ value_turn(d): lanes 0 - 3, 12 - 15 and 20 - 27 are served together in a 16-byte read (and so on), the
// lanes of two neighbouring g, which read chunks 2 apart, so the pairs of rows 2, 3, 4, 5 of their sixteen must not stand where 0, 1, 6, 7 do with 2 turned.
__host__ __device__ constexpr int value_turn(int d) {
    const int p = (d >> 1) & 7;
    return (p & 1) | ((p >> 2) << 1) | (((p >> 2) ^ ((p >> 1) & 1)) << 2);
}

// f(0), .. f(N - 1), each number a compile-time one
template <int N>
using fx_int = std::integral_constant<int, N>;
template <typename F, int... Is>
__device__ __forceinline__ void each_of(std::integer_sequence<int, Is...>, F&& f) {
    (f(fx_int<Is>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) {
    each_of(std::make_integer_sequence<int, N>{}, f);
}

// W waves per block, 16 queries each: an item is up to 16 W queries.  Eight waves share every tile that the block
// brings into LDS between twice as many queries, and four of them per SIMD (two blocks on a CU) hide each other's
// waits; four waves (items of 64) are for prompt portions too short to fill the GPU with larger items.
// G = 2: two such groups of W waves share the item's queries and take its tiles of keys in turn (group 0 the even
// ones, group 1 the odd ones), each with stages, running maxima, sums and outputs of its own; group 1 hands its
// results over through LDS at the end and group 0 merges them.  An item's chain of tiles is then half as long,
// which is what bounds a prompt portion of few items over many keys.
// HD = 256 (a latent that all heads read): the stages take 128 KB, one block on a CU, and value heads may be narrower than key heads (vd a multiple of
// 16).  The same bits as the kernel that stages through registers.
// With one or two waves a SIMD nothing hides a product that waits for its operand, so operands are then read from LDS six products ahead (keys) and
// four column blocks ahead (values).  us left to the compiler / so / with value_turn and the pairs of keys that an edge masks, 16 heads of 256 and 192 numbers: 1,337
// tokens 69 / 53 / 51, 2,048 104 / 83 / 82, at 4,096 keys 295 / 233 / 229, 4,000 210 / 171 / 166; left to the compiler / all of it, items of 64 of 16 heads of 128: 497
// tokens 16.7 / 16.1, at 2,048 keys 51.5 / 49.1, 28 heads over 4, 60 tokens at 2,048 43.4 / 42.0; without read-ahead, items of 128 of 16 heads of 128, 1,000 tokens 33.5 / 31.0.
// What is left of a tile (2.2 us at 256) is neither LDS (1.3 us) nor the matrix units (0.8) but a wave's own chain, in which the next tile's way into LDS is waited for (above).
template <int HD, int NS, int W, int G, int SHAPE>
__global__ __launch_bounds__(W * G * 64, HD > 128 ? W / 4 : HD == 64 && G == 1 ? 4 : W / 2) void attn_mfma_direct_kernel(AttnArgs a) {      // two blocks on a CU (heads of 64: four), or one of two groups
    const int vd = HD > 128 ? a.vd : HD;
    constexpr bool AHEAD = HD > 128 || W == 4;      // no more than two waves on a SIMD (heads of 64, whose four blocks fit a CU: up to four, but few where it counts)
    static_assert(G == 1 || (G == 2 && NS == 2), "one group, or two with two stages each");
    // (heads of 64 in items of 128 keep the plain order: 16 over 4, 1,500 tokens at 8,192 keys 176 us with value_turn, 170 so; in items of 64 value_turn is ahead, 90 -> 78)
    auto turn_of = [](int d) { return HD == 64 && W == 8 ? (d >> 1) & 7 : value_turn(d); };
    constexpr int KS = HD / 32, CB = HD / 16;
    constexpr int NCH = HD / 8;                 // 16-byte chunks of a key row
    constexpr int KROWS = 1024 / (2 * HD);      // key rows of a wave-load
    constexpr int NLOAD = HD / (8 * W);         // wave-loads per wave for the keys of a tile, and as many for the values
    constexpr int TILE = 2 * 64 * HD;           // elements of a stage: keys, then values
    static_assert(NS == 2 || NS == 3, "two or three stages");
    __shared__ __attribute__((aligned(1024))) bf16 tiles[G * NS * TILE];
    extern __shared__ float bias_lds[];
    __shared__ int page_copy[PAGE_COPY];
    int item, h;
    if (!block_place<G == 1 && HD <= 128>(blockIdx.x, a.nh, a.n_items, item, h)) return;
    const int tid = G == 1 ? (int)threadIdx.x : (int)threadIdx.x % (W * 64), lane = tid & 63, wave = tid >> 6;      // within the group
    const int grp = G == 1 ? 0 : (int)threadIdx.x / (W * 64);
    const int li = lane & 15, g = lane >> 4;
    const int kvh = h / (a.nh / a.nkv);
    const int tok_first = a.item_tok[item], n_all = a.item_n[item];
    const int* bt = a.block_table + (size_t)a.item_seq[item] * a.max_blocks;
    const int bs = a.bs;
    const int pmin = a.positions[tok_first], pmax = a.positions[tok_first + n_all - 1];
    const int kv_begin = first_visible(a, pmin);
    const int kv_end = pmax + 1;
    const int tok0 = tok_first + 16 * wave, n = min(16, n_all - 16 * wave);
    int lo = 1, hi = 0;
    const bf16* qrow = nullptr;
    if (li < n) {
        hi = a.positions[tok0 + li];
        lo = first_visible(a, hi);
        qrow = (const bf16*)a.q + (size_t)(tok0 + li) * a.ldq + (size_t)h * HD;
    }
    int w_lo = 0x7fffffff, w_hi = -1;
    int w_lo_max = 0x7fffffff, w_hi_min = -1;
    if (n > 0) {
        w_hi = a.positions[tok0 + n - 1];
        w_lo = first_visible(a, a.positions[tok0]);
        if (n == 16) {
            w_hi_min = a.positions[tok0];
            w_lo_max = first_visible(a, w_hi);
        }
    }
    constexpr bool shaped = SHAPE != SHAPE_NONE;
    const float slope = a.slopes ? a.slopes[h] : 0.f;
    const float cs = shaped ? LOG2E : a.scale * LOG2E;
    float m = NEG_INF, l = 0.f;
    f32x4_t o[CB];
    bf16x8_t qf[KS];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) o[cb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < KS; ++u) {
        const uint4 v = qrow ? *(const uint4*)(qrow + 32 * u + 8 * g) : make_uint4(0, 0, 0, 0);
        qf[u] = __builtin_bit_cast(bf16x8_t, v);
    }
    int first_blk, last_blk, unused;
    page_slot(a, kv_begin, first_blk, unused);
    page_slot(a, kv_end - 1, last_blk, unused);
    if (SHAPE == SHAPE_BIAS) stage_bias(a, h, bias_lds);
    const PageLookup pl = stage_pages(bt, page_copy, first_blk, last_blk);
    const KeySpan span = {kv_begin, kv_end, a.keep_first};
    const TileWalk walk = tile_walk(span);

    // what this lane fetches in each of its wave-loads, relative to the tile's first key / value row 0
    int k_src[NLOAD], v_src[NLOAD];
#pragma unroll
    for (int i = 0; i < NLOAD; ++i) {
        const int j = wave + W * i;                          // wave-load j of HD / 8
        const int row = KROWS * j + lane / NCH;              // LDS key row 16 kb + 4 a + b
        const int key = 16 * ((row >> 2) & 3) + 4 * (row >> 4) + (row & 3);
        k_src[i] = key * HD + (((lane % NCH) ^ (NCH >= 16 ? (row & 15) : ((row >> 1) & 7))) * 8);
        const int d = 8 * j + (lane >> 3);                   // value row
        v_src[i] = d * bs + (((lane & 7) ^ turn_of(d)) * 8);
    }
    auto issue = [&](int kt0, int stage) {
        int blk, slot;
        page_slot(a, kt0, blk, slot);
        const size_t page = (size_t)__builtin_amdgcn_readfirstlane(pl.page(blk));
        const bf16* kbase = (const bf16*)a.k_pages + ((page * a.nkv + kvh) * bs + slot) * HD;
        const bf16* vbase = (const bf16*)a.v_pages + (page * a.nkv + kvh) * vd * bs + slot;
        bf16* st = tiles + (grp * NS + stage) * TILE;
#pragma unroll
        for (int i = 0; i < NLOAD; ++i)
            __builtin_amdgcn_global_load_lds((fx_global_ptr)(kbase + k_src[i]), (fx_lds_ptr)(st + (wave + W * i) * 512), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < NLOAD; ++i)
            if (HD <= 128 || 8 * (wave + W * i) < vd)          // (value rows that exist)
                __builtin_amdgcn_global_load_lds((fx_global_ptr)(vbase + v_src[i]),
                                             (fx_lds_ptr)(st + 64 * HD + (wave + W * i) * 512), 16, 0, 0);
    };
    // operands: key row 16 kb + li, chunk 4 u + g; value row 16 cb + li, chunks 2 g and 2 g + 1
    const int k_at = li * HD, v_at = 64 * HD + li * 64;
    const int ksw = NCH >= 16 ? li : (li >> 1) & 7, vsw = turn_of(li);

    // Every wave of the block goes through the same barriers: the loop runs over rounds of G tiles, of which group
    // grp takes tile grp (a round's last tiles may not exist: that group then only keeps step).
    // (tiles are counted along the block's walk: the kept first keys' tiles, then the window's)
    if (grp < walk.n) issue(walk.start(grp), 0);
    if (NS == 3 && 1 < walk.n) issue(walk.start(1), 1);
    int stage = 0;
    for (int round = 0; round < walk.n; round += G, stage = (stage + 1 == NS ? 0 : stage + 1)) {
        const int ti = round + grp;
        const int kt0 = ti < walk.n ? walk.start(ti) : kv_end;      // (no such tile: past the keys)
        // this wave's part of the tile has landed (with three stages the next tile's loads may still fly)
        if (NS == 3 && ti + 1 < walk.n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NLOAD) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();                           // ... everyone's has, and the stage read last is free
        if (ti + G * (NS - 1) < walk.n) issue(walk.start(ti + G * (NS - 1)), (stage + NS - 1) % NS);
        bf16* st = tiles + (grp * NS + stage) * TILE;
        // a tile at the edge: values of keys outside become zeros.  Whether any tile of the round is one is the
        // same for all waves, so all of them meet at the barrier behind the zeros.
        bool any_edge = false;
#pragma unroll
        for (int q = 0; q < G; ++q)
            any_edge = any_edge || (round + q < walk.n && !span.holds_tile(walk.start(round + q)));
        if (any_edge) {
            if (kt0 < kv_end && !span.holds_tile(kt0)) {
                if constexpr (W == 8 && G == 1 && HD <= 128) {
                    // (two such blocks on a CU fill LDS with their reads: stores alone, of one key in all rows that a thread takes.  16 heads of 128 over 4 with biases, 4,096 tokens 145 us with pairs read and
                    // written, 134 so; capped, 4,096 175 and 168, 8,000 450 and 438; two groups on a CU 46 and 49 for 1,337, one block of heads of 256 31.8 and 32.9 for 700)
                    const int key = tid & 63;                  // the same in all rows that this thread takes
                    if (!span.has(kt0 + key))
                        for (int d = tid >> 6; d < vd; d += W) st[64 * HD + d * 64 + (((key >> 3) ^ turn_of(d)) * 8) + (key & 7)].bits = 0;
                } else {
                    uint32_t* v = (uint32_t*)(st + 64 * HD);
                    const int pair = tid & 31;                 // of keys, the same in all rows that this thread takes
                    uint32_t kept[1] = {0xffffffffu};
                    key_masks(kept, kt0 + 2 * pair, span);
                    if (kept[0] != 0xffffffffu) {
                        // (with few waves beside it a wave has eight reads on their way at once: one after the other 16 of them took a microsecond of a launch, 16 heads of 128,
                        // 60 tokens 9.6 us, so 8.1, with a window of 256 at 2,048 keys 15.7 and 12.5; items of 128, whose waves hide each other's reads, are behind with several)
                        constexpr int B = W == 4 ? 8 : 1;
                        for (int r = 0; r < vd; r += 2 * W * B) {
                            uint32_t was[B], *at[B];
#pragma unroll
                            for (int i = 0; i < B; ++i) {
                                const int d = r + 2 * W * i + (tid >> 5);
                                at[i] = v + d * 32 + ((pair >> 2) ^ turn_of(d)) * 4 + (pair & 3);
                                if (r + 2 * W * i < vd) was[i] = *at[i];
                            }
#pragma unroll
                            for (int i = 0; i < B; ++i)
                                if (r + 2 * W * i < vd) *at[i] = was[i] & kept[0];
                        }
                    }
                }
            }
            lds_barrier();      // the zeros are in LDS (a bare s_barrier does not wait for this wave's stores) before any wave reads values
        }
        if (kt0 >= kv_end || kt0 > w_hi || (kt0 + 64 <= w_lo && kt0 >= span.keep)) continue;      // no such tile, or nothing in it for this wave's rows
        f32x4_t sc[4];
        constexpr int VG = 4;                              // (the widest heads: column blocks whose values are on their way together)
        uint4 vv[AHEAD ? 2 : 1][VG][2];
        auto read_value = [&](int cb, int half) {
            vv[cb / VG & 1][cb % VG][half] = *(const uint4*)(st + v_at + cb * 16 * 64 + (((2 * g + half) ^ vsw) * 8));
        };
        auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
        if constexpr (AHEAD) {
            // (heads of 64, one group: four, in 128 registers.  With 131 three blocks fitted a CU instead of four, 32 heads over 8, 2,048 tokens at 8,192 keys 295 us, so 260; a window of 1,024 46 and 40)
            constexpr int D = HD == 64 && G == 1 ? 4 : 6, N = 4 * KS;
            bf16x8_t ring[D + 1];
            auto read_key = [&](auto qc) {
                constexpr int q = decltype(qc)::value;
                ring[q % (D + 1)] = *(const bf16x8_t*)(st + k_at + (q & 3) * 16 * HD + (((4 * (q >> 2) + g) ^ ksw) * 8));
            };
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) sc[kb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
            fence();
            each<D>(read_key);
            each<N>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                fence();
                if constexpr (q + D < N) read_key(fx_int<q + D>{});
                else read_value((q + D - N) / 2, (q + D - N) % 2);
                fence();
                sc[q & 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[q % (D + 1)], qf[q >> 2], sc[q & 3], 0, 0, 0);
            });
            fence();
#pragma unroll
            for (int i = D; i < 2 * VG; ++i) read_value(i / 2, i % 2);
            fence();
        } else {
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
                sc[kb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int u = 0; u < KS; ++u) {
                    const bf16x8_t kf = *(const bf16x8_t*)(st + k_at + kb * 16 * HD + (((4 * u + g) ^ ksw) * 8));
                    sc[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[u], sc[kb], 0, 0, 0);
                }
            }
        }
        const bool whole = kt0 >= w_lo_max && kt0 + 63 <= w_hi_min && kt0 >= kv_begin;
        uint4 p_lo, p_hi;
        if (SHAPE == SHAPE_CAP_SLOPE) cap_and_slope(sc, kt0 + 16 * g, a, slope, hi);
        if (SHAPE == SHAPE_BIAS) {
            const float* bias = bias_lds + bias_first(a, max(hi, 0) - (kt0 + 16 * g));
            shape_with_bias(sc, kt0 + 16 * g, a, slope, hi, [&](int i) { return bias[i]; });
        }
        const float alpha = whole ? softmax_step<false>(sc, kt0 + 16 * g, lo, hi, cs, m, l, p_lo, p_hi)
                                  : softmax_step<true>(sc, kt0 + 16 * g, lo, hi, cs, m, l, p_lo, p_hi, span.keep);
        const bool rescale = __builtin_amdgcn_ballot_w64(alpha != 1.f) != 0;
        float al[4] = {1.f, 1.f, 1.f, 1.f};
        if (rescale) {
#pragma unroll
            for (int r = 0; r < 4; ++r) al[r] = __shfl(alpha, 4 * g + r, 64);
        }
        if constexpr (AHEAD) {
            each<CB / VG>([&](auto gc) {
                constexpr int c0 = VG * decltype(gc)::value;
                if (16 * c0 >= vd) return;                 // (columns past vd inside a group: whatever LDS holds, never stored)
                fence();
                if constexpr (c0 + VG < CB) {
#pragma unroll
                    for (int i = 0; i < 2 * VG; ++i) read_value(c0 + VG + i / 2, i % 2);
                }
                fence();
#pragma unroll
                for (int j = 0; j < VG; ++j) o[c0 + j] = pv_step(o[c0 + j], rescale, al, p_lo, p_hi, vv[c0 / VG & 1][j][0], vv[c0 / VG & 1][j][1]);
            });
        } else {
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const bf16* vr = st + v_at + cb * 16 * 64;
                o[cb] = pv_step(o[cb], rescale, al, p_lo, p_hi, *(const uint4*)(vr + (((2 * g) ^ vsw) * 8)),
                                *(const uint4*)(vr + (((2 * g + 1) ^ vsw) * 8)));
            }
        }
    }
    if constexpr (G == 2) {
        // group 1 hands over maximum, sum and outputs, lane for lane, through the LDS that the tiles no longer need
        __syncthreads();
        float* hand = (float*)tiles + (size_t)wave * ((2 + 4 * CB) * 64);
        if (grp == 1) {
            hand[lane] = m;
            hand[64 + lane] = l;
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                for (int r = 0; r < 4; ++r) hand[(2 + 4 * cb + r) * 64 + lane] = o[cb][r];
        }
        __syncthreads();
        if (grp == 1) return;
        const float m1 = hand[lane], l1 = hand[64 + lane];
        const float mn = fmaxf(m, m1), mu = (mn == NEG_INF) ? 0.f : mn;
        const float f0 = __builtin_amdgcn_exp2f(m - mu), f1 = __builtin_amdgcn_exp2f(m1 - mu);
        l = l * f0 + l1 * f1;
        m = mn;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float a0 = __shfl(f0, 4 * g + r, 64), a1 = __shfl(f1, 4 * g + r, 64);      // of the accumulator's row 4 g + r
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) o[cb][r] = o[cb][r] * a0 + hand[(2 + 4 * cb + r) * 64 + lane] * a1;
        }
    }
    const float fin = li < n ? finish_row<true>(a, h, m, l) : 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 4 * g + r;
        const float fr = __shfl(fin, row, 64);
        if (row < n) {
            float y[CB];
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) y[cb] = o[cb][r] * fr;
            turn_back_row(a, tok0 + row, li, y);
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
                if (HD <= 128 || 16 * cb < vd) store_out<bf16>(a, tok0 + row, h, 16 * cb + li, y[cb]);
        }
    }
}

// The same for heads of 128 in items of up to 128 queries, without anything that shapes a score or turns an output: a wave takes 32 queries, so that what it reads
// out of LDS serves twice as many products as in the kernel above, which LDS bounds (every 16 queries read whole tiles of keys and values: 4,096 cycles of LDS a
// tile of 64 keys and 256 queries, against 2,048 of the matrix units and as many of exponentials; here all three are about 2,100).  Products are 32 x 32 x 16 with a
// query a lane (lane % 32): scores are S^T = K Q^T, keys in rows, and the outputs O^T += V^T P^T, so a query's maximum, sum and rescaling are a lane's own, but for
// one exchange between the halves of the wave.  The accumulator of lane (q, h = lane / 32) holds rows 8 (i / 4) + 4 h + i % 4; key row 16 s + 8 a + 4 h + b of LDS
// (within 32) holds key 16 s + 8 h + 4 a + b, so that a lane's scores 8 s .. 8 s + 7 are of the eight keys 16 s + 8 h .. that it supplies to
// the second product, whose other operand is then 16 bytes of a value row.
// 250 registers (256 and 36 bytes a lane in scratch memory with two groups, of which an edge tile reloads some), two waves a SIMD: two blocks of four waves on a CU, or one
// whose two groups take the tiles in turn (fx_attn_rows32 has the line and its figures).  us, waves of 16 / of 32 queries: 28 heads over 4, 4,096 queries at 0 168 / 140, at 4,096
// 456 / 379, at 12,288 1,070 / 857 (787 / 982 TFLOP/s), 12,000 at 0 1,213 / 1,028; 16 heads, 2,048 at 0 51 / 47, 8,000 337 / 278.  What is left of a round are waits in a wave's own chain (a wave
// alone on its SIMD takes 1.9 us a tile, two take 2.3), a whole trip of the loads for the next two tiles among them, which are waited for in front of the round's first read of LDS as in the kernel
// above.  A register more a tile to touch lines two and three rounds ahead: slower (907 -> 1,082).
template <int G>
__global__ __launch_bounds__(256 * G, 2) void attn_mfma_rows32_kernel(AttnArgs a) {
    constexpr int HD = 128, W = 4, NS = 2, NLOAD = 4, TILE = 2 * 64 * HD;
    typedef __attribute__((ext_vector_type(16))) float f32x16_t;
    __shared__ __attribute__((aligned(1024))) bf16 tiles[G * NS * TILE];
    __shared__ int page_copy[PAGE_COPY];
    int item, hd_i;
    if (!block_place<G == 1>(blockIdx.x, a.nh, a.n_items, item, hd_i)) return;
    const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), grp = G == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);
    const int li = lane & 31, hl = lane >> 5;
    const int kvh = hd_i / (a.nh / a.nkv);
    const int tok_first = a.item_tok[item], n_all = a.item_n[item];
    const int* bt = a.block_table + (size_t)a.item_seq[item] * a.max_blocks;
    const int bs = a.bs;
    const int pmin = a.positions[tok_first], pmax = a.positions[tok_first + n_all - 1];
    const int kv_begin = first_visible(a, pmin), kv_end = pmax + 1;
    const int tok0 = tok_first + 32 * wave, n = min(32, n_all - 32 * wave);
    // (rows that do not exist are the last existing one again and are not stored, so a wave with some of them still takes whole tiles unmasked: with rows that saw no key a
    // portion's last item masked every tile, and 16 heads, 6,000 tokens at 8,192 keys with a window of 1,024 took 96 us where 6,016 took 85)
    const int tok = tok_first + min(32 * wave + li, n_all - 1);
    const int hi = a.positions[tok], lo = first_visible(a, hi);
    int w_lo = 0x7fffffff, w_hi = -1;               // keys any row of the wave can see (the same in every lane, and kept as such)
    int w_lo_max = 0x7fffffff, w_hi_min = -1;       // keys that all of them see
    if (n > 0) {
        const int first_pos = __builtin_amdgcn_readfirstlane(a.positions[tok0]), last_pos = __builtin_amdgcn_readfirstlane(a.positions[tok0 + n - 1]);
        w_hi = last_pos;
        w_lo = first_visible(a, first_pos);
        w_lo_max = first_visible(a, last_pos);
        w_hi_min = first_pos;
    }
    const float cs = a.scale * LOG2E;
    float m = NEG_INF, l = 0.f;
    f32x16_t o[4];
    bf16x8_t qf[8];
    const bf16* qrow = (const bf16*)a.q + (size_t)tok * a.ldq + (size_t)hd_i * HD + 8 * hl;
#pragma unroll
    for (int u = 0; u < 8; ++u) qf[u] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(qrow + 16 * u));
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
    int first_blk, last_blk, unused;
    page_slot(a, kv_begin, first_blk, unused);
    page_slot(a, kv_end - 1, last_blk, unused);
    const PageLookup pl = stage_pages(bt, page_copy, first_blk, last_blk);
    const KeySpan span = {kv_begin, kv_end, a.keep_first};
    const TileWalk walk = tile_walk(span);

    int k_src[NLOAD], v_src[NLOAD];
#pragma unroll
    for (int i = 0; i < NLOAD; ++i) {
        const int j = wave + W * i, row = 4 * j + (lane >> 4);
        const int key = (row & ~12) | ((row & 4) << 1) | ((row & 8) >> 1);
        k_src[i] = key * HD + (((lane & 15) ^ (row & 15)) * 8);
        const int d = 8 * j + (lane >> 3);
        v_src[i] = d * bs + (((lane & 7) ^ ((d >> 1) & 7)) * 8);
    }
    // Where tile ti lies (the last one, past it), from its page: looked up in front of a round's wait, for the join behind the lookup waits for
    // all loads on their way (the kernel's rounds took 2 us longer with a lookup between two groups of them).  Keys of tile ti go into stage ti / G % 2, and its
    // values into theirs a round later.
    struct Place {
        const bf16 *k, *v;
    };
    auto place_of = [&](int ti) {
        const int kt0 = walk.start(min(ti, walk.n - 1));
        int blk, slot;
        page_slot(a, kt0, blk, slot);
        const size_t page = (size_t)__builtin_amdgcn_readfirstlane(pl.page(blk));
        return Place{(const bf16*)a.k_pages + ((page * a.nkv + kvh) * bs + slot) * HD, (const bf16*)a.v_pages + (page * a.nkv + kvh) * HD * bs + slot};
    };
    auto issue_keys = [&](const Place& at, int stage) {
#pragma unroll
        for (int i = 0; i < NLOAD; ++i)
            __builtin_amdgcn_global_load_lds((fx_global_ptr)(at.k + k_src[i]), (fx_lds_ptr)(tiles + (grp * NS + stage) * TILE + (wave + W * i) * 512), 16, 0, 0);
    };
    auto issue_values = [&](const Place& at, int stage) {
#pragma unroll
        for (int i = 0; i < NLOAD; ++i)
            __builtin_amdgcn_global_load_lds((fx_global_ptr)(at.v + v_src[i]), (fx_lds_ptr)(tiles + (grp * NS + stage) * TILE + 64 * HD + (wave + W * i) * 512), 16, 0, 0);
    };
    // operands: key row 32 b + li, chunk 2 u + hl; value row 32 db + li, chunk 2 t + hl
    const int k_at = li * HD, v_at = 64 * HD + li * 64, ksw = li & 15, vsw = (li >> 1) & 7;
    auto scores = [&](f32x16_t (&sc)[2], int stage) {
        const bf16* st = tiles + (grp * NS + stage) * TILE;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) sc[b][i] = 0.f;
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const bf16x8_t kf = *(const bf16x8_t*)(st + k_at + b * 32 * HD + (((2 * u + hl) ^ ksw) * 8));
                sc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[u], sc[b], 0, 0, 0);
            }
    };
    auto start = [&](int ti) { return ti < walk.n ? walk.start(ti) : kv_end; };      // (no such tile: past the keys)
    auto landed = [] {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    const Place first = place_of(grp);
    Place ahead = place_of(grp + G);           // (of the tile behind the one that a round works on)
    issue_keys(first, 0);
    landed();
    issue_keys(ahead, 1);
    issue_values(first, 0);
    f32x16_t sc[2], next[2];
    scores(sc, 0);
    // A round: the products of the next tile's keys run under this tile's softmax, then come its values.  Both were asked for a round ago and landed then; what this
    // round asks for has landed before its first product too (see above).
    auto one = [&](auto sg, int round, f32x16_t (&now)[2], f32x16_t (&then)[2]) {
        constexpr int stage = decltype(sg)::value;
        const int kt0 = start(round + grp);
        const Place behind = place_of(round + 2 * G + grp);
        landed();                              // this tile's values and the next one's keys, for everyone
        issue_keys(behind, stage);             // (past the last tile: the last one again, never used)
        issue_values(ahead, stage ^ 1);
        ahead = behind;
        // a tile at the edge: values of keys outside become zeros (whether any tile of the round is one is the same for all waves)
        bool any_edge = false;
#pragma unroll
        for (int q = 0; q < G; ++q) any_edge = any_edge || (round + q < walk.n && !span.holds_tile(walk.start(round + q)));
        if (any_edge) {
            if (kt0 < kv_end && !span.holds_tile(kt0)) {
                uint32_t* v = (uint32_t*)(tiles + (grp * NS + stage) * TILE + 64 * HD);
                for (int idx = tid; idx < HD * 32; idx += 256) {
                    const int d = idx >> 5, pair = idx & 31;
                    uint32_t kept[1] = {0xffffffffu};
                    key_masks(kept, kt0 + 2 * pair, span);
                    v[d * 32 + ((pair >> 2) ^ ((d >> 1) & 7)) * 4 + (pair & 3)] &= kept[0];
                }
            }
            lds_barrier();
        }
        // one step of the softmax in base 2 (see softmax_step): score i of block b is of key kt0 + 32 b + 16 (i / 8) + 8 hl + i % 8
        if (!(kt0 >= w_lo_max && kt0 + 63 <= w_hi_min && kt0 >= kv_begin)) {
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int key = kt0 + 32 * b + 16 * (i >> 3) + 8 * hl + (i & 7);
                    now[b][i] = ((key >= lo || key < span.keep) && key <= hi) ? now[b][i] : NEG_INF;
                }
        }
        // From here on operands are read from LDS three products ahead of their use, and the softmax runs between the products, a score (a multiply-add, an
        // exponential, an addition) at a time: the first two of its four parts under the next tile's scores, the others under the first values' products.
        // (Left to the compiler every product waited for its own operand.)
        const bf16 *kst = tiles + (grp * NS + (stage ^ 1)) * TILE + k_at, *vst = tiles + (grp * NS + stage) * TILE + v_at;
        constexpr int D = 3;
        bf16x8_t ring[D + 1];
        auto read_key = [&](auto qc) {
            constexpr int q = decltype(qc)::value;
            ring[q % (D + 1)] = *(const bf16x8_t*)(kst + (q & 1) * 32 * HD + (((2 * (q >> 1) + hl) ^ ksw) * 8));
        };
        auto read_value = [&](auto qc) {
            constexpr int q = decltype(qc)::value;
            ring[q % (D + 1)] = *(const bf16x8_t*)(vst + (q & 3) * 32 * 64 + (((2 * (q >> 2) + hl) ^ vsw) * 8));
        };
        auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
        fence();
        each<D>([&](auto qc) { read_key(qc); });
        fence();
        float mt = NEG_INF;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) mt = fmaxf(mt, now[b][i]);
        mt = half_max(mt) * cs;
        const float m_new = fmaxf(m, mt);
        const float m_use = (m_new == NEG_INF) ? 0.f : m_new;      // a row that has seen nothing yet
        const float alpha = (m_new == NEG_INF) ? 1.f : __builtin_amdgcn_exp2f(m - m_use);
        m = m_new;
        float ps = 0.f, p[8];
        uint4 pf[4];
        auto weight = [&](auto xc) {               // score x of 32; a part is packed when its eighth is there
            constexpr int x = decltype(xc)::value, e = x & 7;
            p[e] = __builtin_amdgcn_exp2f(fmaf(now[x >> 4][x & 15], cs, -m_use));
            asm volatile("" : "+v"(p[e]));       // (here, not behind the branch below)
            ps += p[e];
            if constexpr (e == 7) pf[x >> 3] = make_uint4(pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3]), pack_bf16(p[4], p[5]), pack_bf16(p[6], p[7]));
        };
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) then[b][i] = 0.f;
        // the next tile's scores (past the last tile: of what the stage holds, never used)
        each<16>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            fence();
            if constexpr (q + D < 16) read_key(fx_int<q + D>{});
            else read_value(fx_int<q + D - 16>{});
            fence();
            then[q & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[q % (D + 1)], qf[q >> 1], then[q & 1], 0, 0, 0);
            fence();
            weight(qc);
        });
        fence();
        // Nothing in this tile for this wave's rows, or no such tile (which begins at kv_end): the weights are zeros and nothing would change, but values need not be
        // numbers, and a product with them would be none either (an infinite value of a later token then reached every query of the item).
        if (kt0 > w_hi || (kt0 + 64 <= w_lo && kt0 >= span.keep)) return;
        if (__builtin_amdgcn_ballot_w64(alpha != 1.f)) {
#pragma unroll
            for (int db = 0; db < 4; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
        }
        each<16>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            fence();
            if constexpr (q + D < 16) read_value(fx_int<q + D>{});
            fence();
            o[q & 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[q % (D + 1)], __builtin_bit_cast(bf16x8_t, pf[q >> 2]), o[q & 3], 0, 0, 0);
            fence();
            if constexpr (q < 8) weight(fx_int<16 + q>{});
            else if constexpr (q < 12) {
                weight(fx_int<24 + 2 * (q - 8)>{});
                weight(fx_int<25 + 2 * (q - 8)>{});
            }
        });
        fence();
        l = l * alpha + half_sum(ps);
    };
    for (int round = 0; round < walk.n; round += 2 * G) {
        one(std::integral_constant<int, 0>{}, round, sc, next);
        if (round + G < walk.n) one(std::integral_constant<int, 1>{}, round + G, next, sc);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // the loads past the end, before the block leaves or uses its LDS otherwise
    if constexpr (G == 2) {
        // group 1 hands over maximum, sum and outputs, lane for lane, through the LDS that the tiles no longer need
        __syncthreads();
        float* hand = (float*)tiles + (size_t)wave * (66 * 64);
        if (grp == 1) {
            hand[lane] = m;
            hand[64 + lane] = l;
#pragma unroll
            for (int db = 0; db < 4; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) hand[(2 + 16 * db + i) * 64 + lane] = o[db][i];
        }
        __syncthreads();
        if (grp == 1) return;
        const float m1 = hand[lane], l1 = hand[64 + lane];
        const float mn = fmaxf(m, m1), mu = (mn == NEG_INF) ? 0.f : mn;
        const float f0 = __builtin_amdgcn_exp2f(m - mu), f1 = __builtin_amdgcn_exp2f(m1 - mu);
        l = l * f0 + l1 * f1;
        m = mn;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[db][i] = o[db][i] * f0 + hand[(2 + 16 * db + i) * 64 + lane] * f1;
    }
    if (li >= n) return;
    const float fin = finish_row<true>(a, hd_i, m, l);
    bf16* out = (bf16*)a.out + (size_t)tok * a.ldo + (size_t)hd_i * HD;
    const bool whole = !a.gate && ((uintptr_t)a.out % 8) == 0 && a.ldo % 4 == 0;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int d = 32 * db + 8 * c + 4 * hl;
            if (whole) {
                *(uint2*)(out + d) = make_uint2(pack_bf16(o[db][4 * c] * fin, o[db][4 * c + 1] * fin), pack_bf16(o[db][4 * c + 2] * fin, o[db][4 * c + 3] * fin));
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) store_out<bf16>(a, tok, hd_i, d + r, o[db][4 * c + r] * fin);
            }
        }
}

// Switch for tests and measurement (ferrox_amd/debug.py is its one caller); the product path never sets it.
static int g_direct = 2;     // "direct_stages": 0 keeps prefill on the kernel that stages tiles through registers; 2 (default), 3: stages
static int g_groups = 0;     // "direct_groups": 1 or 2 groups of waves per block of 64 queries in that kernel (0: by the number of blocks)
static int g_rows32 = 1;     // "rows32": items of 128 queries with heads of 128 never (0), always (2) or by the number of blocks (1) on waves of 32 queries
FX_API int fx_debug_set(const char* key, int value) {
    if (!strcmp(key, "rows32")) { g_rows32 = value; return 0; }
    if (!strcmp(key, "direct_stages")) { g_direct = value; return 0; }
    if (!strcmp(key, "direct_groups")) { g_groups = value; return 0; }
    FX_REQUIRE(false, "attention: no debug switch '%s' (direct_stages, direct_groups, rows32)", key);
    return 1;
}

// (value heads narrower than key heads, vd < hd in multiples of 16: attn_mfma_tile_kernel and
// attn_mfma_decode_block_kernel, in which a wave fetches its own operands, and for heads wider than 128
// attn_mfma_block_kernel<256>, which stages them in LDS; heads beyond HD_MAX go to the kernels for any shape)
static bool mfma_ok(int dtype, int hd, int bs, const void* q, long ldq, const void* k_pages, const void* v_pages, int vd = 0) {
    return hd <= HD_MAX && (vd == 0 || vd == hd || (vd < hd && vd % 16 == 0)) && dtype == FX_BF16 && hd % 16 == 0 && bs % 16 == 0 && hd % 8 == 0 && ldq % 8 == 0 &&
           (((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages) % 16 == 0);
}

// f(the launch's shape as a compile-time constant)
template <typename F>
static void by_shape(const AttnArgs& a, F&& f) {
    switch (shape_of(a)) {
        case SHAPE_BIAS: f(std::integral_constant<int, SHAPE_BIAS>{}); break;
        case SHAPE_CAP_SLOPE: f(std::integral_constant<int, SHAPE_CAP_SLOPE>{}); break;
        default: f(std::integral_constant<int, SHAPE_NONE>{}); break;
    }
}

// ---------------------------------------------------------------------------
static int check_common(const char* who, int dtype, int nh, int nkv, int hd, int bs, int window, float scale, int vd = 0, int mask_chunk = 0,
                        int keep_first = 0) {
    FX_REQUIRE(keep_first >= 0 && !(keep_first > 0 && mask_chunk > 0), "%s: kept first keys (%d) go with a window, not with a chunked mask (%d)", who, keep_first, mask_chunk);
    FX_REQUIRE(vd >= 0 && vd <= HD_MAX_ANY, "%s: value head size %d is outside 1..%d", who, vd, HD_MAX_ANY);
    FX_REQUIRE(mask_chunk >= 0 && !(mask_chunk > 0 && window > 0), "%s: a window (%d) or a chunked mask (%d), not both", who, window, mask_chunk);
    // (the bfloat16 kernels take a row's maximum over the raw scores and scale it once, which is the maximum of
    // the scaled scores only under a positive scale)
    FX_REQUIRE(scale > 0.f && scale < INFINITY, "%s: the scale of the scores must be positive and finite, got %g", who, (double)scale);
    FX_REQUIRE(dtype == FX_F32 || dtype == FX_BF16, "%s: unknown dtype %d", who, dtype);
    FX_REQUIRE(nh > 0 && nkv > 0 && nh % nkv == 0, "%s: n_heads %d must be a multiple of n_kv_heads %d", who, nh, nkv);
    FX_REQUIRE(hd > 0 && hd <= HD_MAX_ANY, "%s: head_dim %d is outside 1..%d", who, hd, HD_MAX_ANY);
    FX_REQUIRE(bs > 0, "%s: block size %d", who, bs);
    FX_REQUIRE(window >= 0, "%s: window %d", who, window);
    return 0;
}

// float32 heads that the matrix-unit kernels take: keys and values in 16-byte pieces, a head's numbers in registers
static bool f32_mfma_ok(int hd, int vd, int bs, const void* k_pages, const void* v_pages) {
    return hd % 4 == 0 && bs % 4 == 0 && hd <= HD_MAX && vd <= HD_MAX && (((uintptr_t)k_pages | (uintptr_t)v_pages) % 16) == 0;
}

// Items of up to 128 queries are for bfloat16 with head_dim 64, 128 or 256 and pages of a multiple of 64 keys.
static bool wide_items_ok(int dtype, int hd, int bs) {
    return dtype == FX_BF16 && bs % 64 == 0 && (hd == 64 || hd == 128 || hd == 256) && g_direct == 2;
}
FX_API int fx_attn_tile_queries(int dtype, int hd, int bs) { return wide_items_ok(dtype, hd, bs) ? 128 : 64; }

// The pair that block b of a prompt's launch takes (see block_place), as item * nh + head, or -1; -2 past the launch.
FX_API int fx_attn_block_place(int b, int nh, int n_items, int paired) {
    int item, head;
    if (b < 0 || b >= place_blocks(nh, n_items)) return -2;
    return (paired ? block_place<true>(b, nh, n_items, item, head) : block_place<false>(b, nh, n_items, item, head)) ? item * nh + head : -1;
}

// Groups of waves of 32 queries for that many blocks, or 0: waves of 16.  us with 16 (the better of one and two groups) / 32 one group / 32 two groups, 28 heads over 4 and
// (*) 16 heads: 160 blocks* 36 / 36 / 31, 168 25 / 25 / 24, 176* 37 / 38 / 33, at 8,192 keys 215 / 233 / 175; 192* 40 / 41 / 35, 196 at 8,192 206 / 221 / 166, 224 30 / 31 / 28, 256* 51 / 54 / 47,
// 336 41 / 44 / 38, 448 59 / 59 / 55, at 8,192 353 / 289 / 334, 512* 111 / 111 / 96, 640* 166 / 145 / 154, at 8,192 676 / 558 / 562, 752* 200 / 177 / 199; 784 133 / 111 / 137, at 8,192
// 718 / 574 / 686, 896 168 / 140 / 167, at 12,288 1,070 / 855 / 987, 1,008* 337 / 279 / 323.  So two blocks of one group on a CU from three a CU on, where
// they even out, and before, two groups.  The line was drawn when a wave still multiplied tiles that it does not see, at 3/4 of a block a CU for waves of 16 queries and three a CU for one
// group: since then the columns say two groups from 160 blocks on and one from some 600, which is not done yet.
FX_API int fx_attn_rows32(long blocks, int cus) { return 4 * blocks < 3L * cus ? 0 : blocks <= 3L * cus ? 2 : 1; }

// The same where a mask, a window of `span` keys or chunks of that many, bounds the keys that a query sees.  Items of a few tiles are what the longer start and end of waves of 32 queries take; and behind
// the first span all items of a window have the same work, so from a block a CU on one group, which leaves no wave without a tile.  us with 16 (one group; up to a block a CU two) / 32 one / 32 two, at
// 8,192 keys: 16 heads, 2,048 tokens (256 blocks), a window of 256 19 / 23 / 22, 1,024 36 / 40 / 36, 2,048 60 / 65 / 56; 4,096 (512) 256 30 / 31 / 42, 512 39 / 40 / 50, 1,024 60 / 57 / 68, 4,096 187 / 160 / 175;
// 6,000 (752) 512 57 / 60 / 73, 700 70 / 72 / 88, 1,024 89 / 86 / 99; 28 heads over 4, 1,500 (336) 256 26 / 26 / 38, 1,024 53 / 49 / 63, 4,096 167 / 145 / 164; 4,096 (896) 256 47 / 53 / 73.  Chunks, whose
// items see from none to all of one, at 9,000 keys: 2,048 tokens, chunks of 2,048 59 / 77 / 61, 4,096 72 / 79 / 66; 4,096 (512) 1,024 54 / 54 / 73, 1,536 69 / 70 / 85, 4,096 140 / 149 / 121; 1,500 (336) 1,024 45 / 49 / 54,
// 1,536 72 / 72 / 70; 3,000 (672) 2,048 93 / 94 / 112, 8,192 152 / 134 / 159.  Two groups where most of the launch's tokens can lie in front of the span, as in a prompt without a mask (4,096 tokens at 0, a window
// of 4,096 129 / 111 / 96, chunks 125 / 114 / 101), up to 5/2 blocks a CU (5,000 at 0 143 / 132 / 143); with windows and fewer than two, only portions behind a long context come in items of 128.
FX_API int fx_attn_rows32_masked(long blocks, int cus, long span, int chunked, long tokens) {
    if (4 * blocks < 3L * cus || span <= (chunked ? 1024 : 768)) return 0;
    if (blocks <= cus) return span > (chunked ? 2048 : 1024) ? 2 : 0;
    return 2 * blocks < 5L * cus && 4 * span > 3 * tokens && (chunked || blocks >= 2L * cus) ? 2 : 1;
}

// Queries in blocks: item i covers item_n[i] <= tile_q consecutive tokens of one sequence; tile_q is 64, or what
// fx_attn_tile_queries gives for these sizes.
FX_API int fx_attn_tiles(void* stream, int dtype, const void* q, long ldq, void* out, long ldo,
                         const void* k_pages, const void* v_pages, const int* block_table, int max_blocks,
                         const int* positions, const int* item_seq, const int* item_tok, const int* item_n,
                         int n_items, int nh, int nkv, int hd, int bs, int window, float scale, int tile_q,
                         int vd, int mask_chunk, int keep_first, const float* sinks, const void* gate, long ldg,
                         float softcap, const float* slopes, int gate_per_head, const float* turns, int gate_f32, const float* bias,
                         int bias_n) {
    if (vd <= 0) vd = hd;
    FX_REQUIRE(!bias || bias_n >= 1, "attn_tiles: a distance bias for %d distances", bias_n);
    FX_REQUIRE(!turns || vd % 2 == 0, "attn_tiles: outputs that are turned back come in pairs, a value head has %d", vd);
    FX_REQUIRE(softcap >= 0.f && softcap < INFINITY, "attn_tiles: a cap of %g on the scores", (double)softcap);
    if (check_common("attn_tiles", dtype, nh, nkv, hd, bs, window, scale, vd, mask_chunk, keep_first)) return 1;
    FX_REQUIRE(tile_q == 64 || (tile_q == 128 && (vd == hd || hd == 256) && wide_items_ok(dtype, hd, bs) && mfma_ok(dtype, hd, bs, q, ldq, k_pages, v_pages, vd)),
               "attn_tiles: items of %d queries (64, or 128 where fx_attn_tile_queries says so)", tile_q);
    FX_REQUIRE(tile_q == 64 || !bias || bias_n + 2 * BIAS_PAD <= BIAS_LDS_MAX, "attn_tiles: items of %d queries with biases for %d distances", tile_q, bias_n);
    if (n_items <= 0) return 0;
    AttnArgs a = {};
    a.q = q; a.ldq = ldq; a.out = out; a.ldo = ldo; a.k_pages = k_pages; a.v_pages = v_pages;
    a.block_table = block_table; a.max_blocks = max_blocks; a.positions = positions;
    a.item_seq = item_seq; a.item_tok = item_tok; a.item_n = item_n;
    a.nh = nh; a.nkv = nkv; a.hd = hd; a.bs = bs; a.window = window; a.scale = scale;
    a.vd = vd; a.mask_chunk = mask_chunk;
    a.keep_first = window > 0 ? keep_first : 0; a.sinks = sinks; a.gate = gate; a.ldg = ldg;
    a.gate_per_head = gate_per_head ? 1 : 0;
    a.softcap = softcap; a.slopes = slopes; a.turns = (const float2*)turns;
    a.gate_f32 = gate_f32 ? 1 : 0; a.bias = bias; a.bias_n = bias_n;
    a.bs_shift = log2_or_minus_one(bs);
    a.n_items = n_items;
    dim3 grid(n_items * 4, nh), grid_blocks(place_blocks(nh, n_items));     // a wave per 16 queries / a block per item
    hipStream_t s = (hipStream_t)stream;
    const size_t shm = bias_lds_bytes(a);
    // no more blocks than CUs: a block's chain of tiles is what takes the time, and two groups of waves halve it
    // (measured: 512-token portions at depth 8k-24k 130 and 360 us against 214 and 616 us; from 448 blocks on, one
    // group and two blocks to a CU are as fast or faster)
    const bool two_groups = g_groups ? g_groups == 2 : (long)n_items * nh <= fx_compute_units();
    const long span = window > 0 ? window : mask_chunk, blocks = (long)n_items * nh;
    const int rows32 = span > 0 ? fx_attn_rows32_masked(blocks, fx_compute_units(), span, window <= 0, 128L * n_items) : fx_attn_rows32(blocks, fx_compute_units());
    const bool beyond = hd > HD_MAX || vd > HD_MAX;      // heads wider than the matrix-unit kernels take
    if (dtype == FX_F32 && f32_mfma_ok(hd, vd, bs, k_pages, v_pages)) {
        const dim3 grid_items(n_items, nh);
        if (hd <= 64 && vd <= 64) attn_f32_block_kernel<64><<<grid_items, 256, 0, s>>>(a);
        else if (hd <= 128 && vd <= 128) attn_f32_block_kernel<128><<<grid_items, 256, 0, s>>>(a);
        else attn_f32_block_kernel<256><<<grid_items, 256, 0, s>>>(a);
    } else if (dtype == FX_F32 && beyond)
        attn_tile_kernel<float, HD_MAX_ANY><<<grid, 64, 0, s>>>(a);
    else if (dtype == FX_F32)
        attn_tile_kernel<float><<<grid, 64, 0, s>>>(a);
    else if (beyond)
        attn_tile_kernel<bf16, HD_MAX_ANY><<<grid, 64, 0, s>>>(a);
    else if (mfma_ok(dtype, hd, bs, q, ldq, k_pages, v_pages, vd) && shm <= BIAS_LDS_MAX * sizeof(float)) by_shape(a, [&](auto shape) {
        constexpr int SH = decltype(shape)::value;
        // the widest heads: items of up to 64 queries go on four waves where tiles can travel straight into LDS (us on the kernel that stages through registers / so, 16
        // heads of 256 and 192 numbers: 20 tokens 14.6 / 10.9, 117 20.8 / 13.3, 128 at 2,048 keys 189 / 77; two such blocks for an item of 128 instead of its eight waves: 700
        // tokens 30.6 -> 35.9, 1,337 53 -> 60, level where the last item has no second half), else through registers, tiles of 64 keys (34 KB) and their values (36 KB)
        if (hd > 128 && tile_q == 128) attn_mfma_direct_kernel<256, 2, 8, 1, SH><<<grid_blocks, 512, shm, s>>>(a);
        else if (hd == 256 && bs % 64 == 0 && g_direct == 2) attn_mfma_direct_kernel<256, 2, 4, 1, SH><<<grid_blocks, 256, shm, s>>>(a);
        else if (hd > 128) attn_mfma_block_kernel<256, SH><<<grid_blocks, 256, shm, s>>>(a);
        else if (vd != hd && hd <= 64) attn_mfma_tile_kernel<64, SH><<<grid, 64, 0, s>>>(a);
        else if (vd != hd) attn_mfma_tile_kernel<128, SH><<<grid, 64, 0, s>>>(a);
        else if (SH == SHAPE_NONE && tile_q == 128 && hd == 128 && !turns &&
                 (g_rows32 == 2 || (g_rows32 && rows32))) {
            if (g_groups ? g_groups == 2 : rows32 != 1) attn_mfma_rows32_kernel<2><<<grid_blocks, 512, 0, s>>>(a);
            else attn_mfma_rows32_kernel<1><<<grid_blocks, 256, 0, s>>>(a);
        }
        else if (tile_q == 128 && hd == 128 && two_groups) attn_mfma_direct_kernel<128, 2, 8, 2, SH><<<grid_blocks, 1024, shm, s>>>(a);
        else if (tile_q == 128 && hd == 64 && two_groups) attn_mfma_direct_kernel<64, 2, 8, 2, SH><<<grid_blocks, 1024, shm, s>>>(a);
        else if (tile_q == 128 && hd == 128) attn_mfma_direct_kernel<128, 2, 8, 1, SH><<<grid_blocks, 512, shm, s>>>(a);
        else if (tile_q == 128) attn_mfma_direct_kernel<64, 2, 8, 1, SH><<<grid_blocks, 512, shm, s>>>(a);
        else if (bs % 64 == 0 && hd == 128 && g_direct == 2 && two_groups) attn_mfma_direct_kernel<128, 2, 4, 2, SH><<<grid_blocks, 512, shm, s>>>(a);
        else if (bs % 64 == 0 && hd == 64 && g_direct == 2 && two_groups) attn_mfma_direct_kernel<64, 2, 4, 2, SH><<<grid_blocks, 512, shm, s>>>(a);
        else if (bs % 64 == 0 && hd == 128 && g_direct == 3) attn_mfma_direct_kernel<128, 3, 4, 1, SH><<<grid_blocks, 256, shm, s>>>(a);
        else if (bs % 64 == 0 && hd == 128 && g_direct) attn_mfma_direct_kernel<128, 2, 4, 1, SH><<<grid_blocks, 256, shm, s>>>(a);
        else if (bs % 64 == 0 && hd == 64 && g_direct) attn_mfma_direct_kernel<64, 2, 4, 1, SH><<<grid_blocks, 256, shm, s>>>(a);
        else if (hd <= 32) attn_mfma_block_kernel<32, SH><<<grid_blocks, 256, shm, s>>>(a);
        else if (hd <= 64) attn_mfma_block_kernel<64, SH><<<grid_blocks, 256, shm, s>>>(a);
        else attn_mfma_block_kernel<128, SH><<<grid_blocks, 256, shm, s>>>(a);
    });
    else
        attn_tile_kernel<bf16><<<grid, 64, 0, s>>>(a);
    FX_CHECK_LAUNCH("attn_tiles");
    return 0;
}

// Single queries.  part_o has n_items*nh*splits*hd floats, part_ml n_items*nh*splits*2;
// splits * chunk must cover every position + 1.
template <typename T>
static void launch_merge(const AttnArgs& a, dim3 grid, hipStream_t s) {
    const int threads = a.vd <= 128 ? 128 : 256;
    if (a.splits > MERGE_KEPT) attn_decode_merge_kernel<T, true><<<grid, threads, 2 * MERGE_KEPT * sizeof(float), s>>>(a);
    else attn_decode_merge_kernel<T, false><<<grid, threads, 2 * ((a.splits + 15) & ~15) * sizeof(float), s>>>(a);
}

// Whether a decode block's waves walk many tiles of plain scores: 16 and more each of the longest sequence that the launch can have, of heads of up to 64 five.  They look a page up apart from the tiles at the span's ends,
// which costs a wave of few tiles the time to fetch that code (8 sequences of 2,050 keys in a trace of the step 31.1 us a launch, 34.6) and is ahead where a launch is at the
// rate of memory (us without / with: 16 heads of 128 64 sequences in a trace 192 and 168, 72 sequences of 2,054 keys 223 and 207; heads of 64 64 sequences 90.8 and 86.6, 128 of 200 keys 26.1 and 24.6; the other way 96 sequences of 2,060 keys
// 223 and 228; from nine tiles on 12 sequences of 8,000 keys 123.2 and 125.7).
FX_API int fx_attn_wave_walks(long keys, int waves, int hd) { return (keys + 63) / 64 >= (hd <= 64 ? 5L : 16L) * waves; }

static int attn_decode_launch(void* stream, int dtype, const void* q, long ldq, void* out, long ldo,
                              const void* k_pages, const void* v_pages, const int* block_table, int max_blocks,
                              const int* positions, const int* item_seq, const int* item_tok, int n_items,
                              int nh, int nkv, int hd, int bs, int window, float scale,
                              float* part_o, float* part_ml, int splits, int chunk, int waves, int vd = 0, int mask_chunk = 0,
                              int keep_first = 0, const float* sinks = nullptr, const void* gate = nullptr, long ldg = 0,
                              float softcap = 0.f, const float* slopes = nullptr, int gate_per_head = 0, const float* turns = nullptr,
                              int gate_f32 = 0, const float* bias = nullptr, int bias_n = 0) {
    if (vd <= 0) vd = hd;
    AttnArgs a = {};
    a.gate_f32 = gate_f32 ? 1 : 0; a.bias = bias; a.bias_n = bias_n;
    a.softcap = softcap; a.slopes = slopes; a.gate_per_head = gate_per_head ? 1 : 0; a.turns = (const float2*)turns;
    a.q = q; a.ldq = ldq; a.out = out; a.ldo = ldo; a.k_pages = k_pages; a.v_pages = v_pages;
    a.block_table = block_table; a.max_blocks = max_blocks; a.positions = positions;
    a.item_seq = item_seq; a.item_tok = item_tok; a.item_n = nullptr;
    a.nh = nh; a.nkv = nkv; a.hd = hd; a.bs = bs; a.window = window; a.scale = scale;
    a.vd = vd; a.mask_chunk = mask_chunk;
    a.keep_first = window > 0 ? keep_first : 0; a.sinks = sinks; a.gate = gate; a.ldg = ldg;
    a.bs_shift = log2_or_minus_one(bs);
    a.part_o = part_o; a.part_ml = part_ml; a.splits = splits; a.chunk = chunk;
    dim3 grid(n_items, nh, splits), grid2(n_items, nh);
    hipStream_t s = (hipStream_t)stream;
    const bool beyond = hd > HD_MAX || vd > HD_MAX;      // heads wider than the matrix-unit kernels take
    if (dtype == FX_F32) {
        if (f32_mfma_ok(hd, vd, bs, k_pages, v_pages)) {
            const int group = nh / nkv;
            const dim3 gridf(n_items, nkv * ((group + 15) / 16), splits + (group < 16 ? group : 16) - 1);
            if (hd <= 64 && vd <= 64) attn_f32_decode_kernel<64><<<gridf, 64, 0, s>>>(a);
            else if (hd <= 128 && vd <= 128) attn_f32_decode_kernel<128><<<gridf, 64, 0, s>>>(a);
            else attn_f32_decode_kernel<256><<<gridf, 64, 0, s>>>(a);
        } else if (beyond) attn_decode_kernel<float, HD_MAX_ANY><<<grid, 64, 0, s>>>(a);
        else attn_decode_kernel<float><<<grid, 64, 0, s>>>(a);
        launch_merge<float>(a, grid2, s);
    } else if (beyond) {
        attn_decode_kernel<bf16, HD_MAX_ANY><<<grid, 64, 0, s>>>(a);
        launch_merge<bf16>(a, grid2, s);
    } else if (mfma_ok(dtype, hd, bs, q, ldq, k_pages, v_pages, vd)) {
        const int group = nh / nkv;
        dim3 gridm(nkv * ((group + 15) / 16), n_items, splits);
        // as many waves per block (up to 8, and no more than a split has tiles) as their results fit in LDS
        const int rows = group < 16 ? group : 16;
        const int hdc = hd <= 32 ? 32 : (hd <= 64 ? 64 : (hd <= 128 ? 128 : 256));
        const int nw_max = hd <= 128 ? 8 : 4;      // the widest heads need the registers of half a block
        int nw = nw_max;
        FX_REQUIRE(waves >= 0 && waves <= nw_max, "attn_decode: %d waves per block, this head size takes up to %d", waves, nw_max);
        const long n_blocks = (long)n_items * gridm.x * splits;
        FX_REQUIRE(n_items <= 65535 && splits <= 65535, "attn_decode: %d single queries in %d chunks each are more than a launch takes", n_items, splits);
        // fewer waves per block when there are blocks enough: a chunk's tiles then divide more evenly.  Whole
        // sequences (one chunk) keep four waves a block, or get one each once the blocks number half the GPU's wave
        // slots; two waves a block are behind both (decode steps of 72, 96 and 128 sequences of 16 kv heads: 12.3,
        // 14.3 and 16.1 ms with two waves a block, 11.9, 13.5 and 15.9 with four, 11.7, 13.3 and 15.6 with one).
        const long slots = 8L * fx_compute_units();
        const int nw_min = splits > 1 ? 1 : 4;
        // (wide heads under a mask: a sequence's own chunks hold its span's tiles, however long the sequences are.  17 chunks of one tile, 16 sequences of 16 heads on one
        // kv head: a second wave that has nothing to do 22.6 us, without it 20.1)
        const long span = hd > 128 ? (window > 0 ? window : mask_chunk) : 0;
        const long own = span > 0 ? std::min<long>(chunk, ((span + 63 + splits - 1) / splits + 63) / 64 * 64 + (keep_first + 63L) / 64 * 64) : chunk;
        while (nw > 1 && ((size_t)nw * rows * (hdc + 2) * 4 > 48 * 1024 || nw * 64 >= 2 * own)) nw >>= 1;
        while (nw > nw_min && n_blocks * (nw / 2) >= slots) nw >>= 1;
        if (splits == 1 && 2 * n_blocks >= slots) nw = 1;
        // heads wider than 128: a wave has a SIMD to itself, and waves beyond one round of the SIMDs cost a whole one more
        // (32 sequences of 2,060 keys in chunks of 128, two waves a block 39 us, one 27)
        while (hd > 128 && splits > 1 && nw > 1 && n_blocks * nw > slots / 2) nw >>= 1;
        if (waves > 0 && (size_t)waves * rows * (hdc + 2) * 4 <= 48 * 1024) nw = waves;      // the caller's choice
        const size_t shm = (size_t)nw * rows * (hdc + 2) * 4;
        by_shape(a, [&](auto shape) {
            constexpr int SH = decltype(shape)::value;
            if constexpr (SH == 0) {
                if (hd > 32 && hd <= 128 && fx_attn_wave_walks(own, nw, hd)) {
                    if (hd <= 64) attn_mfma_decode_block_kernel<64, 512, SH, true><<<gridm, nw * 64, shm, s>>>(a);
                    else attn_mfma_decode_block_kernel<128, 512, SH, true><<<gridm, nw * 64, shm, s>>>(a);
                    return;
                }
            }
            if (hd <= 32) attn_mfma_decode_block_kernel<32, 512, SH><<<gridm, nw * 64, shm, s>>>(a);
            else if (hd <= 64) attn_mfma_decode_block_kernel<64, 512, SH><<<gridm, nw * 64, shm, s>>>(a);
            else if (hd <= 128) attn_mfma_decode_block_kernel<128, 512, SH><<<gridm, nw * 64, shm, s>>>(a);
            else attn_mfma_decode_block_kernel<256, 256, SH><<<gridm, nw * 64, shm, s>>>(a);
        });
        if (splits > 1) launch_merge<bf16>(a, grid2, s);
    } else {
        attn_decode_kernel<bf16><<<grid, 64, 0, s>>>(a);
        launch_merge<bf16>(a, grid2, s);
    }
    FX_CHECK_LAUNCH("attn_decode");
    return 0;
}

static int attn_decode_check(int dtype, int nh, int nkv, int hd, int bs, int window, float scale, int splits, int chunk) {
    if (check_common("attn_decode", dtype, nh, nkv, hd, bs, window, scale)) return 1;
    FX_REQUIRE(splits > 0 && chunk > 0 && chunk % 64 == 0, "attn_decode: chunk %d must be a positive multiple of 64", chunk);
    FX_REQUIRE(splits <= MERGE_MOST, "attn_decode: %d chunks are more than the merge kernel takes (%d)", splits, MERGE_MOST);
    return 0;
}

FX_API int fx_attn_decode(void* stream, int dtype, const void* q, long ldq, void* out, long ldo,
                          const void* k_pages, const void* v_pages, const int* block_table, int max_blocks,
                          const int* positions, const int* item_seq, const int* item_tok, int n_items,
                          int nh, int nkv, int hd, int bs, int window, float scale,
                          float* part_o, float* part_ml, int splits, int chunk, int waves, int vd, int mask_chunk,
                          int keep_first, const float* sinks, const void* gate, long ldg, float softcap, const float* slopes,
                          int gate_per_head, const float* turns, int gate_f32, const float* bias, int bias_n) {
    FX_REQUIRE(!bias || bias_n >= 1, "attn_decode: a distance bias for %d distances", bias_n);
    FX_REQUIRE(!turns || (vd > 0 ? vd : hd) % 2 == 0, "attn_decode: outputs that are turned back come in pairs, a value head has %d", vd > 0 ? vd : hd);
    if (attn_decode_check(dtype, nh, nkv, hd, bs, window, scale, splits, chunk)) return 1;
    FX_REQUIRE(softcap >= 0.f && softcap < INFINITY, "attn_decode: a cap of %g on the scores", (double)softcap);
    if (check_common("attn_decode", dtype, nh, nkv, hd, bs, window, scale, vd, mask_chunk, keep_first)) return 1;
    if (n_items <= 0) return 0;
    return attn_decode_launch(stream, dtype, q, ldq, out, ldo, k_pages, v_pages, block_table, max_blocks, positions,
                              item_seq, item_tok, n_items, nh, nkv, hd, bs, window, scale, part_o, part_ml, splits,
                              chunk, waves, vd, mask_chunk, keep_first, sinks, gate, ldg, softcap, slopes, gate_per_head, turns,
                              gate_f32, bias, bias_n);
}

// ---------------------------------------------------------------------------
// fx_attn_decode_static: fx_attn_decode for callers that cannot allocate (see attention.h).  The chunks' partial
// results, which fx_attn_decode's caller brings in part_o and part_ml, live in this array instead.  Each GPU that
// the library runs on holds its own copy until the process ends.  Every call on a GPU uses that GPU's copy from its
// start: two calls that overlap on one GPU (two streams, two threads) race; calls that follow each other on one
// stream do not.  Nothing in it has to start at zero: every chunk writes its (m, l) and its outputs before the merge
// reads them, and the merge reads no chunk of another call's larger shape.
// ---------------------------------------------------------------------------
#define FX_ATTN_STATIC_FLOATS (4u << 20)       // 16 MiB: e.g. 64 queries x 16 heads x 31 chunks x (128 + 2) floats
static __device__ __align__(256) float fx_attn_scratch[FX_ATTN_STATIC_FLOATS];

#define FX_MAX_DEVICES 64
static float* g_attn_scratch_ptr[FX_MAX_DEVICES];    // per device: the address of that device's copy (null: not asked yet)

// The array's name is only a host-side stand-in; its memory on a device is found with hipGetSymbolAddress, once
// per device, with that device current.  `stream`: the stream a call is for (its device is the one whose copy is
// used; null: the current device).  While `stream` is being captured nothing is looked up: the address must be
// known by then, through fx_attn_static_init() or an earlier call on that device.
static int attn_scratch_of(hipStream_t stream, float** out) {
    int current = -1, dev = -1;
    hipError_t e = hipGetDevice(&current);
    FX_REQUIRE(e == hipSuccess, "attn_decode_static: hipGetDevice: %s", hipGetErrorString(e));
    dev = current;
    if (stream) {
        e = hipStreamGetDevice(stream, &dev);
        FX_REQUIRE(e == hipSuccess, "attn_decode_static: hipStreamGetDevice: %s", hipGetErrorString(e));
    }
    FX_REQUIRE(dev >= 0 && dev < FX_MAX_DEVICES, "attn_decode_static: device %d is beyond the %d this library keeps", dev, FX_MAX_DEVICES);
    float* p = __atomic_load_n(&g_attn_scratch_ptr[dev], __ATOMIC_ACQUIRE);
    if (!p) {
        if (stream) {
            hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
            e = hipStreamIsCapturing(stream, &capturing);
            FX_REQUIRE(e == hipSuccess, "attn_decode_static: hipStreamIsCapturing: %s", hipGetErrorString(e));
            FX_REQUIRE(capturing == hipStreamCaptureStatusNone,
                       "attn_decode_static: the stream is being captured and device %d's array has not been looked up yet; "
                       "call fx_attn_static_init() with that device current before the capture begins", dev);
        }
        if (dev != current) {
            e = hipSetDevice(dev);
            FX_REQUIRE(e == hipSuccess, "attn_decode_static: hipSetDevice(%d): %s", dev, hipGetErrorString(e));
        }
        void* sym = nullptr;
        e = hipGetSymbolAddress(&sym, HIP_SYMBOL(fx_attn_scratch));
        if (dev != current) (void)hipSetDevice(current);
        FX_REQUIRE(e == hipSuccess && sym, "attn_decode_static: hipGetSymbolAddress: %s", hipGetErrorString(e));
        p = (float*)sym;
        __atomic_store_n(&g_attn_scratch_ptr[dev], p, __ATOMIC_RELEASE);     // (two threads would store the same address)
    }
    *out = p;
    return 0;
}

// The array's address on the current device, looked up now (no allocation; call it once per device before calls
// that are captured into a graph).
FX_API int fx_attn_static_init(void) {
    float* p;
    return attn_scratch_of(nullptr, &p);
}

FX_API long fx_attn_static_capacity(void) { return (long)FX_ATTN_STATIC_FLOATS; }

FX_API int fx_attn_decode_static(void* stream, int dtype, const void* q, long ldq, void* out, long ldo,
                                 const void* k_pages, const void* v_pages, const int* block_table, int max_blocks,
                                 const int* positions, const int* item_seq, const int* item_tok, int n_items,
                                 int nh, int nkv, int hd, int bs, int window, float scale, int splits, int chunk, int waves) {
    if (attn_decode_check(dtype, nh, nkv, hd, bs, window, scale, splits, chunk)) return 1;
    if (n_items <= 0) return 0;
    const size_t n_o = (size_t)n_items * nh * splits * hd, n_ml = (size_t)n_items * nh * splits * 2;
    FX_REQUIRE(n_o + n_ml <= FX_ATTN_STATIC_FLOATS,
               "attn_decode_static: %d queries x %d heads x %d chunks x (%d + 2) floats = %zu are more than the %u this entry "
               "point holds; use fewer chunks or fx_attn_decode with buffers of your own",
               n_items, nh, splits, hd, n_o + n_ml, FX_ATTN_STATIC_FLOATS);
    float* scratch = nullptr;
    if (attn_scratch_of((hipStream_t)stream, &scratch)) return 1;
    return attn_decode_launch(stream, dtype, q, ldq, out, ldo, k_pages, v_pages, block_table, max_blocks, positions,
                              item_seq, item_tok, n_items, nh, nkv, hd, bs, window, scale, scratch, scratch + n_o, splits,
                              chunk, waves);
}
