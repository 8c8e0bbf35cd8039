// M tokens through one MoE layer with every selected expert's weights read once.
//
// The reference batches M tokens as M*k (token, expert) pairs and re-reads an expert's weights for
// every pair that names it (src/qwen38_moe.cuh:1316-1437, :2743-3237).  Here a pass is two dispatches:
//   AB router, selection and shared gate/up of every token side by side, and the routed gate/up + SwiGLU over the union of the
//      selected experts: a weight row is fetched and decoded once and applied to the activation of every token that selected the
//      expert.  The routed workgroups set themselves up while the router runs and wait for the ids inside the dispatch, as in the
//      one-token dispatch AB; with ids that are known before, and for the site profiler, the two parts (A and B) are launched apart.
//   C  down projections over the union (a member's rows are loaded once and applied to the activations of its
//      tokens) and the ordered combine per token.
// AB and C each work the union out for themselves from the T*k ids (one wave per workgroup, in LDS); nothing about
// it goes through global memory.  Per token, the arithmetic and its order are those of the one-token kernels, so the
// results are bit-identical to M separate passes.
#pragma once

#include "wd_fused.cuh"

namespace wd {

constexpr int kMaxTokens = 8;

constexpr int kPairEntries = 128;  // entries of a pointer table (wd_moe_layer_tokens_pairs_f32)

// Tensor T of "expert" e when the pass was given a table of pointers instead of tensors that hold every expert: e is
// then an index into the table ([entry][tensors per entry]).  The host fills every one of the kPairEntries entries
// (those past the caller's with entry 0), and a number outside the table reads entry 0 (so do numbers past the caller's
// entries: token_pair_id): a wrong id in the scratch gives a wrong result, never a load through a pointer nobody set.
template <int T>
WD_DEV const uint8_t *mat_ptr_entry(const MatSrc &s, int e) {
    if (s.table) return s.table[(static_cast<unsigned>(e) < static_cast<unsigned>(kPairEntries) ? e : 0) * s.per_expert + T];
    return mat_ptr_expert<T>(s, e);
}

template <int T>
WD_DEV const uint8_t *mat_ptr_entry_uniform(const MatSrc &s, int e) {  // e the same in every lane: through the scalar path
    if (s.table) {
        const uint8_t *const *p = s.table + (static_cast<unsigned>(e) < static_cast<unsigned>(kPairEntries) ? e : 0) * s.per_expert + T;
        const uint32_t lo = static_cast<uint32_t>(sld_i32(reinterpret_cast<const int32_t *>(p))), hi = static_cast<uint32_t>(sld_i32(reinterpret_cast<const int32_t *>(p) + 1));
        return reinterpret_cast<const uint8_t *>((static_cast<uintptr_t>(hi) << 32) | lo);
    }
    return mat_ptr_expert_uniform<T>(s, e);
}

struct TokenSlots {
    const float *x;
    float *logits;
    int32_t *ids;
    float *weights;
    float *act;          // [k+1][F]
    float *shared_gate;  // [1]
    uint32_t *hand;      // (LayerArgs),
    int hand_side;
    float *expert_out;   // null or [k][H]
    float *accum, *down_f32, *out;
    uint32_t *tagged;    // selected ids published inside dispatch AB (ids_tagged, LayerArgs),
    int tag_side;
    unsigned *status;    // [0] set to 1 when a wait for the ids or the logits ran out
};

struct TokenArgs {
    LayerArgs common;  // the layer; the per-token members are taken from tok[]
    int T;
    int front_wgs;     // workgroups of dispatch AB that take its first part
    int wait_ids;      // the ids come out of the same dispatch (otherwise they are in the scratches)
    TokenSlots tok[kMaxTokens];
};

// ---- dispatch AB for T tokens, first part (A) --------------------------------------------------------------
// T * (router_stride + shared_stride) + kTokensSelectWgs (none where the ids are given) workgroups, 512 threads, the strides being the router and the
// shared workgroups of a token rounded up to a multiple of 8 (tokens_a_grid): first the router workgroups of every token, token by token, then the workgroups
// that select, one per token, then the shared ones.  The router workgroups are on the pass's critical path and start first; and workgroup w of every
// token - the same weight rows - lands on the same XCD (workgroups go to the eight XCDs in turn), so its L2 serves the
// rows to the tokens after the first.  The padding workgroups return at once.  Per token this is the front of the
// one-token merged dispatch: router rows one per wave, the token's selecting workgroup waits for them, selects its experts
// and publishes the ids, the other workgroups run the shared expert's gate/up.
// lds: 4 * H + 16 bytes, x as f32 for the router rows (the shared workgroups use H + H/16 of it); s_work: kTokensWorkBytes of the
// routed part's tables, for the selection; tiles: the shared rows' eight.
constexpr int kTokensSelectWgs = kMaxTokens;
static_assert(kTokensSelectWgs % 8 == 0, "the workgroups behind keep their XCDs");
struct TokensAGrid {
    int router_stride, shared_stride;
    __host__ __device__ int total(int tokens, bool selects) const { return (selects ? kTokensSelectWgs : 0) + tokens * (router_stride + shared_stride); }
};
__host__ __device__ inline TokensAGrid tokens_a_grid(int n_router_wgs, int n_shared_wgs) {
    return TokensAGrid{(n_router_wgs + 7) & ~7, (n_shared_wgs + 7) & ~7};
}
constexpr int kTokensWorkBytes = kTopkLdsBytes2 + 128;
// Selects token t's experts as the selecting workgroup of the one-token dispatch does.
WD_DEV void tokens_select(const TokenArgs &ta, int t, uint8_t *s_work, int lane, int wave) {
    const LayerArgs &a = ta.common;
    const TokenSlots &s = ta.tok[t];
    int32_t *lds_ids = reinterpret_cast<int32_t *>(s_work + kTopkLdsBytes2);  // behind the selection's own scratch
    float *lds_w = reinterpret_cast<float *>(s_work + kTopkLdsBytes2 + 64);
    if (wave == 0) __builtin_amdgcn_s_setprio(3);
    const uint32_t *const hand = hand_copy(s.hand, s.hand_side);
    const bool there = topk_block(HandRow{hand, a.E, a.E, a.sh_inp != nullptr, a.hand_limit}, a.k, a.w_scale, lds_ids, lds_w, nullptr, s_work, lane, wave, nullptr,
                                  ta.wait_ids ? s.tagged : nullptr, s.tag_side);
    if (!there && lane == 0) __hip_atomic_store(s.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (a.sh_inp && wave == 5 && lane == 0) s.shared_gate[0] = sigmoid_ggml(bits_f(hand_load(hand + a.E)));
    if (wave == 0) {
        wave_lds_fence();
        if (lane < a.k) {
            s.ids[lane] = lds_ids[lane];
            s.weights[lane] = lds_w[lane];
        }
    }
}
// WIDE: router rows of 2049..4096 columns, two waves each (n_router_wgs is then for four rows per workgroup).
// HIDDEN: 2048, where it is known (0: it is not).  With it the dispatch for five and more tokens spills 11 registers instead of 18; us per layer,
// unknown / known: two tokens 28.3 / 28.3, four 41.1 / 40.3, eight 69.5 / 67.9.  (2560 known: nothing, 55.0 / 55.0 and 84.6 / 84.5.)
template <bool WIDE, int HIDDEN>
WD_DEV void tokens_front(const TokenArgs &ta, uint8_t *lds_ta, uint8_t *s_work, Q8RowTile *tiles) {
    const LayerArgs &a = ta.common;
    const int H = HIDDEN ? HIDDEN : a.H;
    const int n_shared_wgs = a.sh_inp ? (a.F + 7) / 8 : 0;
    const TokensAGrid gr = tokens_a_grid(a.n_router_wgs, n_shared_wgs);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int token, wg;
    {
        const int router_part = ta.T * gr.router_stride, selecting = a.preselected ? 0 : kTokensSelectWgs;
        int b = blockIdx.x;
        if (b < router_part) {
            token = b / gr.router_stride, wg = b - token * gr.router_stride;
            if (wg >= a.n_router_wgs) return;
        } else if (b < router_part + selecting) {
            token = b - router_part, wg = -1;
            if (token >= ta.T) return;
        } else {
            b -= router_part + selecting;
            token = b / gr.shared_stride;
            const int w = b - token * gr.shared_stride;
            if (w >= n_shared_wgs) return;
            wg = a.n_router_wgs + w;
        }
    }
    const TokenSlots &s = ta.tok[token];
    if (wg >= 0 && wg < a.n_router_wgs) {
        const int rows = a.preselected ? 0 : a.E;
        int row;
        float logit;
        if (WIDE)
            logit = router_rows_wave_pair(a.router, s.x, reinterpret_cast<float *>(lds_ta), reinterpret_cast<float *>(s_work), s.hand, s.hand_side, rows, H, a.sh_inp, a.E, wg, row);
        else
            logit = router_rows_wave(a.router, s.x, reinterpret_cast<float *>(lds_ta), s.hand, s.hand_side, rows, H, a.sh_inp, a.E, wg, row);
        if (lane == 32 && row >= 0 && row < rows) s.logits[row] = logit;  // (the caller's view)
        // (no selection: the one wave with the shared gate's row)
        if (a.preselected && row == a.E && lane == 32) s.shared_gate[0] = sigmoid_ggml(bits_f(hand_word_bits(f_bits(logit))));
        return;
    }
    if (wg < 0) return tokens_select(ta, token, s_work, lane, wave);
    int8_t *xq = reinterpret_cast<int8_t *>(lds_ta);
    uint16_t *xd = reinterpret_cast<uint16_t *>(lds_ta + H);
    const int r = (wg - a.n_router_wgs) * 8 + wave;
    const int nb = H >> 5;
    const size_t rb = static_cast<size_t>(nb) * 34;
    const size_t off = static_cast<size_t>(min(r, a.F - 1)) * rb;
    const uint8_t *const rows[2] = {uniform_ptr(a.sh_gate + off), uniform_ptr(a.sh_up + off)};  // one row pair per wave
    float gu[2];
    q8_row_pair<0, WIDE>(rows, nb, xq, xd, tiles[wave], lane, gu, [&]() {
        lds_quantize_q8_0(s.x, H, xq, xd, threadIdx.x, 512);
        __syncthreads();
    });
    if (lane == 0 && r < a.F) s.act[static_cast<size_t>(a.k) * a.F + r] = silu_ggml(gu[0]) * gu[1];
}

// The id of pair `pair` (= token * k + rank; at most the last pair's) as it stands in the scratch.
WD_DEV int token_pair_raw(const TokenArgs &ta, int pair) {
    const int k = ta.common.k, n = ta.T * k;
    const int pc = min(pair, n - 1);  // the load is unconditional (no branch, so that it can overlap with others)
    int t = 0;
    const int32_t *p = ta.tok[0].ids;
#pragma unroll
    for (int q = 1; q < kMaxTokens; ++q) {
        const bool past = pc >= q * k;
        t += past ? 1 : 0;
        p = past ? ta.tok[q].ids : p;
    }
    return p[pc - t * k];
}
// The same for lane-parallel comparisons; pairs past the end get distinct negative values that match nothing.  An id outside
// the layer's experts (only a selection that the caller left in the scratches can hold one) counts as expert 0, as in
// checked_expert: it also indexes the union's tables.  (checked_expert in this place, a branch between the load and the union,
// takes 0.8 us per layer: another wave reports it, token_ids_report.)
WD_DEV int token_pair_id(const TokenArgs &ta, int pair) {
    const int v = token_pair_raw(ta, pair);
    return pair < ta.T * ta.common.k ? (static_cast<unsigned>(v) < ta.common.down.n_experts ? v : 0) : -1 - pair;
}

// One wave: reports an id outside the layer's experts through the status word.
WD_DEV void token_ids_report(const TokenArgs &ta, int lane) {
    for (int pair = lane; pair < ta.T * ta.common.k; pair += 64) checked_expert(ta.common.down, token_pair_raw(ta, pair));
}

// The union of the T*k routed ids, in order of first appearance, with the rank at which every token selected
// each member (-1: not selected).  Lives in LDS; built by one full wave (T*k <= 128, expert ids < 1024).
struct TokenUnion {
    int count;
    int expert[128];
    int upos[128];                   // scratch of the build: union index of a first occurrence
    int8_t rank[128][kMaxTokens];
    int first_pair[1024];            // scratch of the build: lowest pair naming an expert
};

// The ids of pairs `lane` and `lane + 64` as the first part of the same dispatch publishes them; false: the wait ran out.
WD_DEV bool token_pairs_wait(const TokenArgs &ta, int lane, int &id_lo, int &id_hi) {
    const int k = ta.common.k, n = ta.T * k;
    auto word_of = [&](int pair) {
        const int pc = min(pair, n - 1);
        int t = 0;
        const uint32_t *p = tag_copy(ta.tok[0].tagged, ta.tok[0].tag_side, static_cast<int>(blockIdx.x));
#pragma unroll
        for (int q = 1; q < kMaxTokens; ++q) {
            const bool past = pc >= q * k;
            t += past ? 1 : 0;
            p = past ? tag_copy(ta.tok[q].tagged, ta.tok[q].tag_side, static_cast<int>(blockIdx.x)) : p;
        }
        return p + (pc - t * k);
    };
    const uint32_t *const lo = word_of(lane), *const hi = word_of(lane + 64);
    for (unsigned polls = 1;; ++polls) {
        const uint32_t v = __hip_atomic_load(lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), w = __hip_atomic_load(hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__builtin_amdgcn_ballot_w64(v == kTagInvalid || w == kTagInvalid) == 0ull) {
            id_lo = lane < n ? static_cast<int>(v) : -1 - lane, id_hi = lane + 64 < n ? static_cast<int>(w) : -65 - lane;
            return true;
        }
        if (polls >= ta.common.spin_limit) return false;
        __builtin_amdgcn_s_sleep(4);
    }
}
// Returns with un.count < 0 when the ids did not come (the status word is set).
WD_DEV void token_union_build(const TokenArgs &ta, TokenUnion &un, int lane) {
    const int k = ta.common.k, n = ta.T * k;
    int id_lo, id_hi;
    if (!ta.wait_ids) {
        id_lo = token_pair_id(ta, lane), id_hi = token_pair_id(ta, lane + 64);
    } else if (!token_pairs_wait(ta, lane, id_lo, id_hi)) {
        if (lane == 0) {
#pragma unroll
            for (int q = 0; q < kMaxTokens; ++q)
                if (q < ta.T) __hip_atomic_store(ta.tok[q].status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            un.count = -1;
        }
        return;
    }
    const bool on_lo = lane < n, on_hi = lane + 64 < n;
    for (int i = lane; i < 128 * kMaxTokens / 4; i += 64) reinterpret_cast<uint32_t *>(&un.rank[0][0])[i] = 0xffffffffu;
    // lowest pair that names the same expert, through a table indexed by expert id
    if (on_lo) un.first_pair[id_lo] = 0x7fffffff;
    if (on_hi) un.first_pair[id_hi] = 0x7fffffff;
    wave_lds_fence();
    if (on_lo) atomicMin(&un.first_pair[id_lo], lane);
    if (on_hi) atomicMin(&un.first_pair[id_hi], lane + 64);
    wave_lds_fence();
    const int fq_lo = on_lo ? un.first_pair[id_lo] : -1, fq_hi = on_hi ? un.first_pair[id_hi] : -1;
    const bool first_lo = on_lo && fq_lo == lane, first_hi = on_hi && fq_hi == lane + 64;
    const unsigned long long m_lo = __builtin_amdgcn_ballot_w64(first_lo), m_hi = __builtin_amdgcn_ballot_w64(first_hi);
    const unsigned long long below = (1ull << lane) - 1ull;
    const int u_lo = __builtin_popcountll(m_lo & below);
    const int u_hi = __builtin_popcountll(m_lo) + __builtin_popcountll(m_hi & below);
    if (first_lo) {
        un.upos[lane] = u_lo;
        un.expert[u_lo] = id_lo;
    }
    if (first_hi) {
        un.upos[lane + 64] = u_hi;
        un.expert[u_hi] = id_hi;
    }
    if (lane == 0) un.count = __builtin_popcountll(m_lo) + __builtin_popcountll(m_hi);
    wave_lds_fence();
    // (token, rank) of a pair without a division: tokens are k pairs apart
    int t_lo = 0, t_hi = 0;
#pragma unroll
    for (int q = 1; q < kMaxTokens; ++q) {
        t_lo += (lane >= q * k) ? 1 : 0;
        t_hi += (lane + 64 >= q * k) ? 1 : 0;
    }
    if (on_lo) un.rank[un.upos[fq_lo]][t_lo] = static_cast<int8_t>(lane - t_lo * k);
    if (on_hi) un.rank[un.upos[fq_hi]][t_hi] = static_cast<int8_t>(lane + 64 - t_hi * k);
    wave_lds_fence();
}

// ---- dispatch AB for T tokens ---------------------------------------------------------------------------
// grid = front_wgs (the first part, tokens_front) + min(T * k * ceil(F / 8), a few workgroups per compute unit), 512 threads.
// Every workgroup of the second part (B) stages the codebooks and quantises the T inputs once, builds the union (wave 0) - when the
// ids come out of this dispatch, behind the set-up, with a bounded wait -, then walks the items (union member, group of 8 rows) in
// turn with the stride of their number; a wave takes one (gate, up) row pair of the item, decodes it once and applies it to every
// token that selected the expert.  As a dispatch of its own this part began 2.6 us after the ids and spent 3.5 more on its set-up.
// MAXT: token capacity of the instantiation (4 or kMaxTokens).
// dynamic LDS: T * (H bytes + H/256 floats), the Q8_K copies of the T inputs; at least what tokens_front takes (tokens_ab_lds).
// FETCH: 0, or how the rows come in when they can be fetched as aligned words (IqRowWords): 8 and 10 rows of that many
// super-blocks, 1 and 2 others of one or two words per lane.  The row pair of the wave's next item is then requested before the
// current one is worked on.  dynamic LDS then has 8 * 2 * iq_cover_bytes more bytes behind the activations (16-byte aligned).
// As many workgroups per compute unit as the registers allow without spilling in the routed part (eight tokens and rows of eight
// super-blocks spill eleven in all: 73.1 us per layer, 75.7 as two dispatches of which one spilled two).
// The shared rows' tiles of the first part lie behind the quantised x of the same workgroup: in the static area they would make it 2.9 KB larger
// than the tables and the union, which is what the inputs of eight tokens of 17920 columns leave (162128 of 163840 bytes).
__host__ __device__ inline uint32_t tokens_front_tiles(int H) { return static_cast<uint32_t>(H + H / 16 + 15) & ~15u; }
// activations: the T inputs, and the staging behind them.
inline size_t tokens_ab_lds(int H, size_t activations) {
    return std::max({activations, sizeof(float) * static_cast<size_t>(H) + 16, tokens_front_tiles(H) + 8 * sizeof(Q8RowTile)});
}
template <int TYPE, int MAXT, int FETCH>
constexpr int kTokensBPerCu = FETCH == 8 || (FETCH == 10 && TYPE == 22 && MAXT <= 4) ? 3 : 2;
template <int TYPE, int MAXT, int FETCH = 0>
__global__ __launch_bounds__(512, (2 * kTokensBPerCu<TYPE, MAXT, FETCH>)) void k_tokens_ab(TokenArgs ta) {
    extern __shared__ __align__(16) uint8_t lds_tb[];
    struct Routed {
        IqTables tables;
        TokenUnion un;
    };
    static_assert(sizeof(Routed) >= kTokensWorkBytes, "the selection works in the place of the tables and the union");
    __shared__ __align__(16) uint8_t s_area[sizeof(Routed)];
    const LayerArgs &a = ta.common;
    if (static_cast<int>(blockIdx.x) < ta.front_wgs) {
        const bool wide = a.H > 2048 && a.H <= 4096;
        Q8RowTile *const tiles = reinterpret_cast<Q8RowTile *>(lds_tb + tokens_front_tiles(a.H));
        if (FETCH != 8 && (FETCH == 10 || FETCH == 2 || wide)) tokens_front<true, 0>(ta, lds_tb, s_area, tiles);
        else tokens_front<false, FETCH == 8 ? 2048 : 0>(ta, lds_tb, s_area, tiles);
        return;
    }
    IqTables &tables = reinterpret_cast<Routed *>(s_area)->tables;
    // (IQ2_S, ten super-blocks, three workgroups per compute unit: with all look-ups of a block at once 11 registers are spilled, half by half 5.  2560 / 640, two
    // tokens 31.8 us per layer, so 31.1, three 41.6, 41.0, four 49.1, 49.0.)
    const auto &look_up = static_cast<const typename std::conditional<TYPE == 22 && FETCH == 10 && kTokensBPerCu<TYPE, MAXT, FETCH> == 3, IqTablesTight, IqTables>::type &>(tables);
    TokenUnion &un = reinterpret_cast<Routed *>(s_area)->un;
    const int wg = static_cast<int>(blockIdx.x) - ta.front_wgs, n_wgs = static_cast<int>(gridDim.x) - ta.front_wgs;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int groups = (a.F + 7) / 8;
    int8_t *xq = reinterpret_cast<int8_t *>(lds_tb);
    float *xd = reinterpret_cast<float *>(lds_tb + static_cast<size_t>(ta.T) * a.H);
    constexpr int kBlk = (TYPE == 21) ? 110 : 82;
    const int nb = FETCH >= 8 ? FETCH : a.H >> 8;
    const size_t rb = static_cast<size_t>(nb) * kBlk;
    mark(a, 1, 0);
    // the T inputs as Q8_K: a wave's blocks (wave, wave + 8, ...) are requested four at a time, the first four before
    // anything else so that the union build and the codebook staging run under their latency
    constexpr int kMaxBlocks = 4;
    float4 xv[kMaxBlocks];
    auto load_blocks = [&](int b0) {
#pragma unroll
        for (int i = 0; i < kMaxBlocks; ++i) {
            const int b = min(b0 + 8 * i, ta.T * nb - 1);
            const int t = __builtin_amdgcn_readfirstlane(b / nb), bb = b - t * nb;  // uniform index into the argument block
            xv[i] = reinterpret_cast<const float4 *>(ta.tok[t].x + bb * 256)[lane];
        }
    };
    auto quantise_blocks = [&](int b0) {
#pragma unroll
        for (int i = 0; i < kMaxBlocks; ++i) {
            const int b = b0 + 8 * i;
            if (b < ta.T * nb) {
                const int t = b / nb, bb = b - t * nb;
                wave_quantize_q8_k_regs(xv[i], xq + static_cast<size_t>(t) * a.H + bb * 256, xd + t * nb + bb, lane);
            }
        }
    };
    load_blocks(wave);
    if (!ta.wait_ids && wave == 0) token_union_build(ta, un, lane);
    if (a.preselected && wg == 0 && wave == 1) token_ids_report(ta, lane);  // (ahead of the loads: 0.4 us)
    mark(a, 1, 1);
    stage_tables<TYPE == 21, TYPE == 22>(tables, threadIdx.x, 512);
    quantise_blocks(wave);
    for (int b0 = wave + 8 * kMaxBlocks; b0 < ta.T * nb; b0 += 8 * kMaxBlocks) {
        load_blocks(b0);
        quantise_blocks(b0);
    }
    if (ta.wait_ids && wave == 0) token_union_build(ta, un, lane);
    __syncthreads();
    if (un.count < 0) return;  // the wait ran out
    mark(a, 1, 2);
    const int n_items = un.count * groups;
    // the aligned forms use the lane layout of iq_rows8_coal_dots (a chain's lanes two apart inside a row, no lane excluded from
    // a chain step), rows of ten super-blocks with the last two of both rows in one shared pass, as in iq_rows10_coal
    constexpr bool kPairs = FETCH != 0;
    constexpr int kLoads = FETCH == 2 || (FETCH == 10 && TYPE == 21) ? 2 : 1;
    const int ib = kPairs ? ((lane >> 4) << 1) | (lane & 1) : lane >> 3, sbl = kPairs ? (lane >> 1) & 7 : lane & 7;
    const bool first = sbl == 0;
    const uint32_t kStage = iq_cover_bytes<TYPE>(nb);
    uint8_t *stage = lds_tb + ((static_cast<size_t>(ta.T) * (a.H + sizeof(float) * nb) + 15) & ~static_cast<size_t>(15)) +
                     static_cast<size_t>(wave) * 2 * kStage;
    IqRowWords<TYPE, kLoads> fetch[2];
    auto row_pair = [&](int item, const uint8_t *(&rows)[2]) {
        const int u = item / groups, rg = item - u * groups;
        const int e = un.expert[u];
        const size_t off = static_cast<size_t>(min(rg * 8 + wave, a.F - 1)) * rb;
        rows[0] = uniform_ptr(mat_ptr_entry<0>(a.gate_up, e) + off), rows[1] = uniform_ptr(mat_ptr_entry<1>(a.gate_up, e) + off);
    };
    if (FETCH != 0 && wg < n_items) {
        const uint8_t *rows[2];
        row_pair(wg, rows);
        fetch[0].request(rows[0], nb, lane), fetch[1].request(rows[1], nb, lane);
    }
    for (int item = wg; item < n_items; item += n_wgs) {
        const int u = item / groups, rg = item - u * groups;
        int rank[MAXT];
#pragma unroll
        for (int t = 0; t < MAXT; ++t) rank[t] = __builtin_amdgcn_readfirstlane(static_cast<int>(un.rank[u][t]));
        const int r = rg * 8 + wave;
        const uint8_t *rows[2];  // one row pair per wave
        row_pair(item, rows);
        uint32_t lead[2] = {0, 0};
        if (FETCH != 0) {
            wave_lds_fence();  // the previous item's rows have been read
            fetch[0].store(stage, lane), fetch[1].store(stage + kStage, lane);
            lead[0] = fetch[0].lead, lead[1] = fetch[1].lead;
            wave_lds_fence();
            if (item + n_wgs < n_items) {  // the next item's rows, into the registers just written out
                const uint8_t *next[2];
                row_pair(item + n_wgs, next);
                fetch[0].request(next[0], nb, lane), fetch[1].request(next[1], nb, lane);
            }
        }
        float acc[MAXT][2];
#pragma unroll
        for (int t = 0; t < MAXT; ++t) acc[t][0] = acc[t][1] = 0.0f;
        for (int base = 0; base < (FETCH == 10 ? 8 : nb); base += 8) {
            // (aligned forms: positions past the row's end work on its last super-block and contribute zero)
            const bool in_row = FETCH >= 8 || base + sbl < nb, on = kPairs || in_row;
            const int sb = FETCH >= 8 ? base + sbl : min(base + sbl, nb - 1);
            uint32_t w[2][8];
            int ls[2][2];
            float dw[2] = {0.0f, 0.0f};
            if (on) {
                IqFields f[2];
                if (FETCH != 0) {
                    const uint32_t o0 = lead[0] + sb * kBlk, o1 = lead[1] + sb * kBlk;
                    f[0] = iq_fields_shifted<TYPE>(stage + o0, ib, (o0 + 2) & 2u);
                    f[1] = iq_fields_shifted<TYPE>(stage + kStage + o1, ib, (o1 + 2) & 2u);
                } else {
                    f[0] = iq_load<TYPE>(rows[0] + static_cast<size_t>(sb) * kBlk, ib);
                    f[1] = iq_load<TYPE>(rows[1] + static_cast<size_t>(sb) * kBlk, ib);
                }
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    iq_decode<TYPE>(f[i], ib, look_up, w[i], ls[i]);
                    dw[i] = h2f(f[i].d);
                }
            }
#pragma unroll
            for (int t = 0; t < MAXT; ++t) {
                if (rank[t] < 0) continue;  // uniform
                uint32_t av[8];
                float dx = 0.0f;
                if (on) {
                    const int8_t *aq = xq + static_cast<size_t>(t) * a.H + sb * 256 + ib * 32;
                    const uint4 a0 = *reinterpret_cast<const uint4 *>(aq);
                    const uint4 a1 = *reinterpret_cast<const uint4 *>(aq + 16);
                    av[0] = a0.x, av[1] = a0.y, av[2] = a0.z, av[3] = a0.w, av[4] = a1.x, av[5] = a1.y, av[6] = a1.z, av[7] = a1.w;
                    dx = in_row ? xd[t * nb + sb] : 0.0f;
                }
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    int p[8];
                    float ds = 0.0f;
                    if (on) {
                        iq_dot_decoded(w[i], ls[i], av, p);
                        ds = dw[i] * dx;
                    } else {
#pragma unroll
                        for (int c = 0; c < 8; ++c) p[c] = 0;
                    }
                    if (kPairs) {
                        const float pf = static_cast<float>(reduce_scatter_ib_pairs(p, lane));
                        // the chain's value of the pass before moves to the first position, which keeps it while the others
                        // converge; past the row's end it passes through, fma(0, finite, acc) == acc
                        float up = FETCH >= 8 || base == 0 ? 0.0f : dpp_f<kDppShl14>(0.0f, acc[t][i]);
                        float v = __builtin_fmaf(ds, pf, up);
#pragma unroll
                        for (int s = 1; s < 8; ++s) {
                            up = FETCH >= 8 ? dpp_f<kDppShr2, 0xf, 0xf, true>(0.0f, v) : dpp_f<kDppShr2>(up, v);
                            v = __builtin_fmaf(ds, pf, up);
                        }
                        acc[t][i] = v;
                        continue;
                    }
                    const float pf = static_cast<float>(reduce_scatter_ib(p, lane));
                    const float carry = dpp_f<kDppShl7>(0.0f, acc[t][i]);
                    float v = __builtin_fmaf(ds, pf, base == 0 ? 0.0f : carry);
#pragma unroll
                    for (int s = 1; s < 8; ++s) {
                        const float up = dpp_f<kDppShr1>(0.0f, v);
                        const float nxt = __builtin_fmaf(ds, pf, up);
                        v = first ? v : nxt;
                    }
                    acc[t][i] = v;
                }
            }
        }
        if (FETCH == 10) {
            // super-blocks 8 and 9: position 0/1 of the pass = row 0, position 2/3 = row 1 (positions 4..7 idle)
            const int ri = min(sbl >> 1, 1), sb = 8 + (sbl & 1);
            const bool on = sbl < 4;
            const IqFields f = iq_fields_lds<TYPE>(stage + ri * kStage + (ri ? lead[1] : lead[0]) + sb * kBlk, ib, sb);
            uint32_t w[8];
            int ls[2];
            iq_decode<TYPE>(f, ib, look_up, w, ls);
            const float dw = h2f(f.d);
#pragma unroll
            for (int t = 0; t < MAXT; ++t) {
                if (rank[t] < 0) continue;  // uniform
                const int8_t *aq = xq + static_cast<size_t>(t) * a.H + sb * 256 + ib * 32;
                const uint4 a0 = *reinterpret_cast<const uint4 *>(aq);
                const uint4 a1 = *reinterpret_cast<const uint4 *>(aq + 16);
                const uint32_t av[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
                int p[8];
                iq_dot_decoded(w, ls, av, p);
                const float ds = on ? dw * xd[t * nb + sb] : 0.0f;
                const int P = reduce_scatter_ib_pairs(p, lane);
                const float pf = on ? static_cast<float>(P) : 0.0f;
                float carry = dpp_f<0x10E, 0xf, 0x1>(0.0f, acc[t][0]);  // row 0's chain: position 7 -> position 0
                carry = dpp_f<0x10A, 0xf, 0x2>(carry, acc[t][1]);       // row 1's chain: position 7 -> position 2
                const float v8 = __builtin_fmaf(ds, pf, carry);
                const float v9 = __builtin_fmaf(ds, pf, dpp_f<kDppShr2, 0xf, 0xf, true>(0.0f, v8));
                acc[t][0] = dpp_f<0x11C>(0.0f, v9);  // back to position 7 for the closing tree
                acc[t][1] = dpp_f<0x118>(0.0f, v9);
            }
        }
#pragma unroll
        for (int t = 0; t < MAXT; ++t) {
            if (rank[t] < 0) continue;
            float g = kPairs ? close_chains_pairs(acc[t][0]) : close_lanes8_strided(acc[t][0]);
            float up = kPairs ? close_chains_pairs(acc[t][1]) : close_lanes8_strided(acc[t][1]);
            if (TYPE == 22) {
                g = 0.125f * g;
                up = 0.125f * up;
            }
            if (lane == 0 && r < a.F) ta.tok[t].act[static_cast<size_t>(rank[t]) * a.F + r] = silu_ggml(g) * up;
        }
        mark(a, 1, item == wg ? 3 : 4);
    }
    mark(a, 1, 5);
}

// The same for Q8_0 (KIND 0) and IQ4_NL (KIND 1) gate/up rows.  The waves of the grid take the items (union member, group of
// four rows) in turn: four gate rows and the same four up rows are the eight rows of q8_rows8_pass, 32 blocks of each in
// registers at a time and applied to every token that selected the expert.
// (One row pair per wave with a block per lane runs the chains of two rows on all 64 lanes, 64 steps each, for every token: 61 us
// for eight tokens, top-5, hidden 3584, ffn 512, against 30.)
// dynamic LDS: T * (H bytes + H/32 halves), the Q8_0 copies of the T inputs, and 4 * H + 16 bytes at least (tokens_front).
template <int KIND>
__global__ __launch_bounds__(512, 4) void k_tokens_ab_q8(TokenArgs ta) {
    extern __shared__ __align__(16) uint8_t lds_tq[];
    struct Routed {
        Q8Tile8 tiles[8];
        TokenUnion un;
    };
    static_assert(sizeof(Routed) >= kTokensWorkBytes && sizeof(Routed) >= 8 * sizeof(Q8RowTile), "the first part works in the place of the tiles and the union");
    __shared__ __align__(16) uint8_t s_area[sizeof(Routed)];
    const LayerArgs &a = ta.common;
    if (static_cast<int>(blockIdx.x) < ta.front_wgs) {
        Q8RowTile *const tiles = reinterpret_cast<Q8RowTile *>(s_area);
        if (a.H > 2048) tokens_front<true, 0>(ta, lds_tq, s_area, tiles);  // (hidden 4096 at most)
        else tokens_front<false, 0>(ta, lds_tq, s_area, tiles);
        return;
    }
    Q8Tile8 *const tiles = reinterpret_cast<Routed *>(s_area)->tiles;
    TokenUnion &un = reinterpret_cast<Routed *>(s_area)->un;
    const int wg = static_cast<int>(blockIdx.x) - ta.front_wgs, n_wgs = static_cast<int>(gridDim.x) - ta.front_wgs;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int groups = a.F >> 2, nb = a.H >> 5;  // (F is a multiple of 32, H of 256)
    constexpr int kBlk = (KIND == 0) ? 34 : 18, kChunk = 4;  // passes of eight blocks
    const size_t rb = static_cast<size_t>(nb) * kBlk;
    int8_t *xq = reinterpret_cast<int8_t *>(lds_tq);
    uint16_t *xd = reinterpret_cast<uint16_t *>(lds_tq + static_cast<size_t>(ta.T) * a.H);
    if (!ta.wait_ids && wave == 0) token_union_build(ta, un, lane);
    if (a.preselected && wg == 0 && wave == 1) token_ids_report(ta, lane);
    for (int t = 0; t < ta.T; ++t) lds_quantize_q8_0(ta.tok[t].x, a.H, xq + static_cast<size_t>(t) * a.H, xd + t * nb, threadIdx.x, 512);
    if (ta.wait_ids && wave == 0) token_union_build(ta, un, lane);
    __syncthreads();
    if (un.count < 0) return;  // the wait ran out
    const int n_items = un.count * groups, row = lane >> 3, b = lane & 7;
    // (neighbouring workgroups take neighbouring items, a workgroup's waves items far apart: every wave of the grid gets one
    // before any gets a second)
    for (int item = wave * n_wgs + wg; item < n_items; item += 8 * n_wgs) {
        const int u = item / groups, r0 = 4 * (item - u * groups);
        const int e = __builtin_amdgcn_readfirstlane(un.expert[u]);
        const uint8_t *const gate = mat_ptr_entry<0>(a.gate_up, e), *const up = mat_ptr_entry<1>(a.gate_up, e);
        const uint8_t *const mine = (row < 4 ? gate : up) + static_cast<size_t>(r0 + (row & 3)) * rb;
        int rank[kMaxTokens];
#pragma unroll
        for (int t = 0; t < kMaxTokens; ++t) rank[t] = __builtin_amdgcn_readfirstlane(static_cast<int>(un.rank[u][t]));
        Q8Chain ch[kMaxTokens];
        for (int base = 0; base < nb; base += 8 * kChunk) {
            Q8Block w[kChunk];
#pragma unroll
            for (int q = 0; q < kChunk; ++q) w[q] = q8_load<KIND>(mine + static_cast<size_t>(min(base + 8 * q + b, nb - 1)) * kBlk);
#pragma unroll
            for (int t = 0; t < kMaxTokens; ++t) {
                if (rank[t] < 0) continue;  // uniform
#pragma unroll
                for (int q = 0; q < kChunk; ++q)
                    if (base + 8 * q < nb)
                        q8_rows8_pass<KIND, false>(w[q], base + 8 * q, nb, xq + static_cast<size_t>(t) * a.H, xd + t * nb, tiles[wave], lane, ch[t], nullptr);
            }
        }
#pragma unroll
        for (int t = 0; t < kMaxTokens; ++t) {
            if (rank[t] < 0) continue;
            const float y = q8_rows8_close<KIND>(ch[t], nb, tiles[wave], lane);
            const wd_uint2v h = __builtin_amdgcn_permlane32_swap(f_bits(y), f_bits(y), false, false);  // .y in lanes 0..31: the value 32 lanes up
            if (b == 0 && row < 4) ta.tok[t].act[static_cast<size_t>(rank[t]) * a.F + r0 + row] = silu_ggml(y) * bits_f(h.y);
        }
    }
}

// ---- dispatch C for T tokens ----------------------------------------------------------------------------
// As layer_clear_handed: workgroup t for token t, by its last wave, which has the fewest items.
WD_DEV void tokens_clear_handed(const TokenArgs &ta, int waves, int tw, int lane) {
    if (static_cast<int>(blockIdx.x) >= ta.T || tw != waves - 1) return;
    const TokenSlots &s = ta.tok[blockIdx.x];
    for (int i = lane; i < kTagCopies * 8; i += 64) {
        __hip_atomic_store(s.tagged + i, kTagInvalid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(s.tagged + s.tag_side + i, kTagInvalid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    hand_clear(s.hand, s.hand_side, ta.common.E + 1, lane, 64);
}
// grid = H / 8: a workgroup owns eight output rows, as the one-token k_layer_c8 does.  Work items are (token, matrix) with
// matrix = the token's k routed down tensors, then the shared one (always Q8_0); the waves take them in turn: the
// activation, then the eight rows, one block per lane and pass.  Items that name the same expert read the same rows within one
// workgroup, so memory sees them once.  Waves 0..T-1 finally fold token t's results in its own top-k order.
// One item in flight per wave and as many waves as the registers allow - two workgroups of sixteen waves per compute unit for
// rows of 16 blocks, two of eight for longer ones -, so that grids of more than 256 workgroups (hidden > 2048) still run in one round: with two
// or three items per wave and one workgroup of sixteen waves per compute unit, hidden 2304 took twice the time of 2048.
// KIND: down tensor kind; PASSES: of eight blocks per row (F <= 256 PASSES).
// dynamic LDS (layer_c_lds): [T][k+1][8] floats, then per wave the tile and the quantised activation (layer_c8_wave_bytes<false>).
template <int PASSES>
constexpr int kTokensCWaves = PASSES <= 2 ? 16 : 8;
template <int KIND, int PASSES>
__global__ __launch_bounds__(64 * kTokensCWaves<PASSES>) __attribute__((amdgpu_waves_per_eu(PASSES <= 2 ? 8 : (PASSES == 3 ? 5 : 4))))
void k_tokens_c(TokenArgs ta) {
    extern __shared__ __align__(16) uint8_t lds_tc[];
    const LayerArgs &a = ta.common;
    const int lane = threadIdx.x & 63, tw = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    constexpr int kWaves = kTokensCWaves<PASSES>, kActs = (PASSES + 1) / 2;
    const uint32_t per_wave = layer_c8_wave_bytes<false>(a.F);
    float *ybuf = reinterpret_cast<float *>(lds_tc);  // [T][k+1][8]
    uint8_t *const own = lds_tc + 32 * ta.T * (a.k + 1) + tw * per_wave;
    Q8Tile8 &tile = *reinterpret_cast<Q8Tile8 *>(own);
    int8_t *aq = reinterpret_cast<int8_t *>(own + sizeof(Q8Tile8));
    uint16_t *ad = reinterpret_cast<uint16_t *>(aq + a.F);
    const bool shared = a.sh_down != nullptr;
    const int per_token = a.k + (shared ? 1 : 0), n_items = ta.T * per_token;
    const int r0 = blockIdx.x * 8, nb = a.F >> 5;  // hidden is a multiple of 8
    mark(a, 2, 0);
    tokens_clear_handed(ta, kWaves, tw, lane);
    // every routed id of the pass, one vector load per wave; an item's id is then a lane read
    const int id_lo = token_pair_id(ta, lane), id_hi = token_pair_id(ta, lane + 64);
    // combine operands of token `tw`, requested early: lane j keeps router weight j, lane 16 the shared gate
    float wreg;
    const unsigned bad = __hip_atomic_load(ta.tok[min(tw, ta.T - 1)].status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // 1: a wait of dispatch AB ran out
    {
        const TokenSlots &s = ta.tok[min(tw, ta.T - 1)];
        const float *src = (lane == 16 && shared) ? s.shared_gate : s.weights + min(lane, a.k - 1);
        wreg = *src;
    }
    for (int item = tw; item < n_items; item += kWaves) {
        const int t = item / per_token, j = item - t * per_token;
        const bool is_shared = j == a.k;
        float4 v[2 * kActs];
#pragma unroll
        for (int q = 0; q < kActs; ++q) {
            const float *p = ta.tok[t].act + static_cast<size_t>(j) * a.F + min(512 * q + lane * 8, a.F - 8);
            v[2 * q] = *reinterpret_cast<const float4 *>(p), v[2 * q + 1] = *reinterpret_cast<const float4 *>(p + 4);
        }
        const int pair = t * a.k + (is_shared ? 0 : j);
        const int e = pair < 64 ? __builtin_amdgcn_readlane(id_lo, pair) : __builtin_amdgcn_readlane(id_hi, pair - 64);
        const uint8_t *const rows = uniform_ptr((is_shared ? a.sh_down : mat_ptr_entry<0>(a.down, e)) + static_cast<size_t>(r0) * nb * (KIND == 0 || is_shared ? 34 : 18));
        auto run = [&](auto kind) {
            constexpr int K = decltype(kind)::value;
            Q8Rows8Blocks<K, PASSES> blocks;
            // (the longest rows leave no registers to hold the activation beside the blocks: quantised ahead of their request)
            constexpr bool kActFirst = PASSES > 4;
            if (!kActFirst) blocks.request(rows, nb, lane);
            wave_lds_fence();
#pragma unroll
            for (int q = 0; q < kActs; ++q)
                lds_quantize_q8_0_step<false>(v[2 * q], v[2 * q + 1], 512 * q + lane * 8 < a.F, 512 * q + lane * 8, aq, ad, lane);
            wave_lds_fence();
            if (kActFirst) blocks.request(rows, nb, lane);
            Q8Chain ch;
#pragma unroll
            for (int q = 0; q < PASSES; ++q)
                if (8 * q < nb) q8_rows8_pass<K, false>(blocks.w[q], 8 * q, nb, aq, ad, tile, lane, ch, nullptr);
            return q8_rows8_close<K>(ch, nb, tile, lane);
        };
        const float y = (KIND == 0 || is_shared) ? run(std::integral_constant<int, 0>{}) : run(std::integral_constant<int, KIND>{});
        if ((lane & 7) == 0) ybuf[(t * (a.k + 1) + j) * 8 + (lane >> 3)] = y;
        mark(a, 2, item == tw ? 2 : 3);
    }
    __syncthreads();
    mark(a, 2, 5);
    if (tw < ta.T) {
        const TokenSlots &s = ta.tok[tw];
        const int t = tw;
        const int row = r0 + lane;
        const bool row_on = lane < 8 && row < a.H;
        const float *const mine = ybuf + t * (a.k + 1) * 8 + (lane & 7);
        const float y_shared = shared ? mine[a.k * 8] : 0.0f;
        const float acc = fold_in_order<8>(mine, wreg, a.k);
        const float gate = readlane_f(wreg, 16);
        if (row_on) {
            float o = acc;
            if (s.expert_out)
                for (int j = 0; j < a.k; ++j) s.expert_out[static_cast<size_t>(j) * a.H + row] = mine[j * 8];
            if (shared) {
                const float prod = y_shared * gate;
                o = acc + prod;
                s.down_f32[row] = y_shared;
            }
            s.accum[row] = bad == 1u ? __builtin_nanf("") : acc;
            s.out[row] = bad == 1u ? __builtin_nanf("") : o;
        }
    }
    mark(a, 2, 6);
}

// The same with one workgroup of sixteen waves for every compute unit, hidden / 256 rows each, as in k_layer_c_even: a work item is
// (token, matrix, group of up to 64 / LPR rows).  (The next item's activation and rows requested while this one is worked on: 2560 / 640,
// four tokens 63.8 us per layer instead of 61.7, 4096 / 1536 128.8 instead of 119.2.)  Where it is taken and what it measures: tokens_c_even_lanes.
// grid = 256.  dynamic LDS (layer_c_lds): [T][k+1][16] floats, then per wave the tile and the quantised activation (layer_c_even_wave_bytes).
constexpr int kTokensCEvenWaves = 16;
template <int KIND, int LPR, int PASSES>
__global__ __launch_bounds__(64 * kTokensCEvenWaves) void k_tokens_c_even(TokenArgs ta) {
    constexpr int kWaves = kTokensCEvenWaves, kActs = LPR * PASSES <= 48 ? (LPR * PASSES + 15) / 16 : 3;
    extern __shared__ __align__(16) uint8_t lds_tc[];
    const LayerArgs &a = ta.common;
    const int lane = threadIdx.x & 63, tw = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const uint32_t per_wave = layer_c_even_wave_bytes<LPR>(a.F);
    float *ybuf = reinterpret_cast<float *>(lds_tc);  // [T][k+1][16]
    uint8_t *const own = lds_tc + 64 * ta.T * (a.k + 1) + tw * per_wave;
    Q8TileN<LPR> &tile = *reinterpret_cast<Q8TileN<LPR> *>(own);
    int8_t *aq = reinterpret_cast<int8_t *>(own + ((sizeof(Q8TileN<LPR>) + 15) & ~15u));
    uint16_t *ad = reinterpret_cast<uint16_t *>(aq + a.F);
    const bool shared = a.sh_down != nullptr;
    const int rows_per_wg = a.H >> 8, r0 = blockIdx.x * rows_per_wg, nb = a.F >> 5;
    const int n_groups = rows_per_wg * LPR > 64 ? 2 : 1, rows0 = n_groups == 2 ? (rows_per_wg + 1) >> 1 : rows_per_wg;
    mark(a, 2, 0);
    tokens_clear_handed(ta, kWaves, tw, lane);
    // every routed id of the pass, one vector load per wave; an item's id is then a lane read
    const int id_lo = token_pair_id(ta, lane), id_hi = token_pair_id(ta, lane + 64);
    // combine operands of token `tw`, requested early: lane j keeps router weight j, lane 16 the shared gate
    float wreg;
    const unsigned bad = __hip_atomic_load(ta.tok[min(tw, ta.T - 1)].status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // 1: a wait of dispatch AB ran out
    {
        const TokenSlots &s = ta.tok[min(tw, ta.T - 1)];
        const float *src = (lane == 16 && shared) ? s.shared_gate : s.weights + min(lane, a.k - 1);
        wreg = *src;
    }
    // items [begin, end): of `per_token` matrices from number `first` on for every token
    auto run = [&](auto kind, int first, int per_token, int begin, int end) {
        constexpr int K = decltype(kind)::value, kBlk = K == 0 ? 34 : 18;
        struct Item {
            const float *act;
            const uint8_t *rows;
            int nrows, y;  // y: where the results go in ybuf
        };
        auto item_at = [&](int i) {
            const int g = n_groups == 2 ? i & 1 : 0, pair = n_groups == 2 ? i >> 1 : i;
            const int t = pair / per_token, j = first + (pair - t * per_token);
            const int p = t * a.k + min(j, a.k - 1);
            const int e = p < 64 ? __builtin_amdgcn_readlane(id_lo, p) : __builtin_amdgcn_readlane(id_hi, p - 64);
            Item it;
            it.nrows = g ? rows_per_wg - rows0 : rows0;
            it.act = ta.tok[t].act + static_cast<size_t>(j) * a.F;
            it.rows = uniform_ptr((j == a.k ? a.sh_down : mat_ptr_entry_uniform<0>(a.down, e)) + static_cast<size_t>(r0 + g * rows0) * nb * kBlk);
            it.y = (t * (a.k + 1) + j) * 16 + g * rows0;
            return it;
        };
        for (int i = begin; i < end; i += kWaves) {
            const Item it = item_at(i);
            float4 v[2 * kActs];
#pragma unroll
            for (int q = 0; q < kActs; ++q) {
                const float *p = it.act + min(512 * q + lane * 8, a.F - 8);
                v[2 * q] = *reinterpret_cast<const float4 *>(p), v[2 * q + 1] = *reinterpret_cast<const float4 *>(p + 4);
            }
            const Q8RowsNAt<K, LPR> at(lane, it.nrows);
            Q8Block w[PASSES];
#pragma unroll
            for (int q = 0; q < PASSES; ++q) w[q] = q8_rowsn_load<K, LPR>(it.rows, q * LPR, nb, it.nrows, at);
            wave_lds_fence();
#pragma unroll
            for (int q = 0; q < kActs; ++q)
                lds_quantize_q8_0_step<false>(v[2 * q], v[2 * q + 1], 512 * q + lane * 8 < a.F, 512 * q + lane * 8, aq, ad, lane);
            wave_lds_fence();
            Q8Chain ch;
#pragma unroll
            for (int q = 0; q < PASSES; ++q)
                if (q == 0 || q * LPR < nb) q8_rowsn_pass<K, LPR>(w[q], q * LPR, nb, aq, ad, tile, at, ch);
            const float y = q8_rowsn_close<K, LPR>(ch, nb, tile, at);
            if ((lane & 7) == 0 && (lane >> 3) < it.nrows) ybuf[it.y + (lane >> 3)] = y;
            mark(a, 2, i == tw ? 2 : 3);
        }
    };
    if (KIND == 0) {
        run(std::integral_constant<int, 0>{}, 0, a.k + (shared ? 1 : 0), tw, ta.T * (a.k + (shared ? 1 : 0)) * n_groups);
    } else {
        const int routed = ta.T * a.k * n_groups;
        run(std::integral_constant<int, KIND>{}, 0, a.k, tw, routed);
        // the waves that have one routed item less begin with the shared ones
        if (shared) run(std::integral_constant<int, 0>{}, a.k, 1, (tw - routed) & (kWaves - 1), ta.T * n_groups);
    }
    __syncthreads();
    mark(a, 2, 5);
    if (tw < ta.T) {
        const TokenSlots &s = ta.tok[tw];
        const int t = tw;
        const int row = r0 + lane;
        const bool row_on = lane < rows_per_wg;
        const float *const mine = ybuf + t * (a.k + 1) * 16 + (lane & 15);
        const float y_shared = shared ? mine[a.k * 16] : 0.0f;
        const float acc = fold_in_order<16>(mine, wreg, a.k);
        const float gate = readlane_f(wreg, 16);
        if (row_on) {
            float o = acc;
            if (s.expert_out)
                for (int j = 0; j < a.k; ++j) s.expert_out[static_cast<size_t>(j) * a.H + row] = mine[j * 16];
            if (shared) {
                const float prod = y_shared * gate;
                o = acc + prod;
                s.down_f32[row] = y_shared;
            }
            s.accum[row] = bad == 1u ? __builtin_nanf("") : acc;
            s.out[row] = bad == 1u ? __builtin_nanf("") : o;
        }
    }
    mark(a, 2, 6);
}

}  // namespace wd
