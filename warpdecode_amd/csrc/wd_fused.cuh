// Fused MoE layer: two dispatches per layer (three when the caller asks for the split form).
//   AB router logits (+ shared-expert gate logit), a wave or two per row; a workgroup behind them waits for
//      them, runs softmax/top-k and publishes the ids inside the dispatch; the shared expert's gate/up + SwiGLU and
//      the routed gate/up + SwiGLU run in the same launch: the routed workgroups quantise x and stage the
//      codebooks while the router runs and pick the ids up as soon as they appear - or request their weights at
//      once when the ids are known before the launch (given by the caller, or by a routing trace).
//      The same kernel with only the first or only the last of these parts is the split form.
//   C  Q8_0 re-quantisation of the k+1 activations, all down projections, the ordered weighted
//      sum, the gated shared branch and the optional residual update
// Activation quantisation is redone by every workgroup that needs it (8 KB of f32 from L2 and a
// few dozen instructions per lane) instead of being a dispatch of its own.
#pragma once
#include <type_traits>

#include "wd_handword.hpp"
#include "wd_kernels.cuh"

namespace wd {

struct LayerArgs {
    int H, F, E, k;
    float w_scale;
    const float *x;
    const float *router;
    MatSrc gate_up, down;        // resolved through ids (global scratch)
    const float *sh_inp;         // null = no shared expert
    const uint8_t *sh_gate, *sh_up, *sh_down;
    float *logits;               // [E]
    int32_t *ids;                // [k]
    float *weights;              // [k]
    const int32_t *ids_override; // null or [k]
    float *act;                  // [k+1][F]
    float *shared_gate;          // [1]: logit after A, sigmoid after B
    float *expert_out;           // null or [k][H]
    float *accum, *down_f32, *out;
    float *residual;             // null, [H] (residual += out * residual_scale), or [hc][H] when hc > 0
    float residual_scale;
    const float *hc_inject;      // hc > 0: [hc] inject projections; residual[c] += out * 2 sigmoid(inject[c] / hc)
    int hc, hc_round_half;
    int dry;                     // measurement aid: every workgroup returns at once
    int preselected;
    int n_router_wgs;            // workgroups of dispatch AB that take router rows,
    int n_select_wgs;            // those that wait for these and select: one, or none,
    int n_shared_wgs;            // those that take the shared expert's gate/up (the rest: routed gate/up)
    int n_routed_items;          // (expert rung, group of eight rows) items shared by the routed workgroups
    const int32_t *ids_known;    // null, or the k ids where they are known before the launch
    uint32_t *hand;              // [E + 2]: the router's logits and the shared gate's on their way to the selection, for side 0, and the count of hand_close; kHandEmpty between passes
    int hand_side;               // so many words on from these the logits for side 1 (0: one copy for both)
    uint32_t *ids_tagged;        // selected ids published inside the merged dispatch (kTagInvalid = not yet): [kTagCopies / 2][16] for side 0,
    int tag_side;                // so many words on from these for side 1 (tag_copy)
    int clear_tagged;            // dispatch C resets ids_tagged when it is done with the layer
    int close_hand;              // no dispatch C follows: the router and the selecting workgroups set `hand` back themselves (hand_close)
    unsigned *status;            // [0] set to 1 when a bounded wait inside a dispatch ran out
    unsigned spin_limit;         // polls (about half a microsecond each) before such a wait gives up,
    unsigned hand_limit;         // and before the selection's for the logits does (hand_gather)
    unsigned long long *trace;   // profiling aid: null, or [3][16][8] time stamps (100 MHz) of workgroup trace_wg
    int trace_wg;
    // the PART variants of the dispatches also store the exact int32 chunk sums of the routed rows:
    int32_t *gup_part;           // [k][2][F][8 * H / 256]
    int32_t *down_part;          // [k][H][8 * F / 32]
    uint32_t *host_ids;          // null, or [k] in host memory: dispatch AB reports its selection
};

constexpr int kTagCopies = 16;           // replicas of the published ids, 64 bytes apart, so that pollers spread over lines
constexpr uint32_t kTagInvalid = 0xffffffffu;

// Sides.  A word that workgroups hand on has a home in one half of the device's memory, and the XCDs of that half reach it sooner: a device-scope
// load that misses the L2 takes 350 to 450 clocks near its home and 580 to 700 from the other half (stores 370 to 500 and 600 to 760), a word from
// XCD 0 to XCD 1 360 ns by way of the near half and 575 by the far one.  Memory alternates between the halves in pieces of kSidePiece bytes; which
// of two neighbours is whose is measured when a scratch is made (side_vote).  XCDs 0..3 are side 0, the others side 1.
// What has readers on either side is written once for each, and a reader takes the copy of the side of the XCD that it does run on (HW_REG XCC_ID) and not of
// its block number: block 0 of a dispatch is on the XCD at which its hardware queue begins, 0 for one stream and 7 for another.
constexpr int kSidePiece = 8192;
constexpr unsigned kSideChunk = 2u << 20;  // within which the halves keep their order
WD_DEV unsigned xcc_id() { return static_cast<unsigned>(__builtin_amdgcn_s_getreg(20 | (3 << 11))) & 7u; }
WD_DEV int xcc_side() { return static_cast<int>(xcc_id() >> 2); }
// The replica of the published ids that workgroup `wg` of the waiting ones polls.
WD_DEV const uint32_t *tag_copy(const uint32_t *tagged, int tag_side, int wg) {
    return tagged + (xcc_side() ? tag_side : 0) + ((wg >> 3) & (kTagCopies / 2 - 1)) * 16;
}
constexpr unsigned kSpinLimit = 1u << 16;  // default number of polls before a wait gives up (tens of milliseconds; a wait lasts microseconds)

// Time stamp `i` of dispatch `d` (0 = A, 1 = B, 2 = C) for the traced workgroup; lane 0 of every wave.
// TRACE false: compiled out (the kernels that take the stamps as a template parameter run without their tests then).
template <bool TRACE = true>
WD_DEV void mark(const LayerArgs &a, int d, int i) {
    if (!TRACE) return;
    if (a.trace && static_cast<int>(blockIdx.x) == a.trace_wg && (threadIdx.x & 63) == 0 && (threadIdx.x >> 6) < 15)
        a.trace[(d * 16 + (threadIdx.x >> 6)) * 8 + i] = wall_clock64();
}

// ---- in-workgroup quantisers (results in LDS) ------------------------------------------------
// Q8_0 of n values (multiple of 32): four threads per block, eight values per thread.
// The general form of the step on eight loaded values (v0, v1 = x[base .. base + 8)); all four threads of a block must call it.  The quants, and the scale's bits.
WD_DEV uint2 quantize_q8_0_general(const float4 &v0, const float4 &v1, uint16_t &scale) {
    float amax = __builtin_fmaxf(
        __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(v0.x), __builtin_fabsf(v0.y)),
                        __builtin_fmaxf(__builtin_fabsf(v0.z), __builtin_fabsf(v0.w))),
        __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(v1.x), __builtin_fabsf(v1.y)),
                        __builtin_fmaxf(__builtin_fabsf(v1.z), __builtin_fabsf(v1.w))));
    amax = quad_max_nonneg(amax);
    uint2 packed = make_uint2(0u, 0u);
    if (amax != 0.0f) {  // (one division for the eight values)
        const float inv = 127.0f / amax;
        packed.x = q8_0_pack4_scaled(v0, inv);
        packed.y = q8_0_pack4_scaled(v1, inv);
    }
    scale = f2h_ref(amax / 127.0f);
    return packed;
}
// The step, for what comes between a dispatch's activations and its dot products (on: the thread's values are of a block; the whole wave must call it).
// ORDINARY false: the general form only, which takes fewer registers.
template <bool ORDINARY = true>
WD_DEV void lds_quantize_q8_0_step(const float4 &v0, const float4 &v1, bool on, int base, int8_t *qs, uint16_t *d, int tid) {
    uint2 packed;
    uint16_t scale;
    if constexpr (ORDINARY) {
        uint32_t m = umax_step<kDppXor1>(f_bits(max3_abs(max3_abs(max3_abs(v0.x, v0.y, v0.z), v0.w, v1.x), max3_abs(v1.y, v1.z, v1.w), 0.0f)));
        m = umax_step<kDppXor2>(m);
        const float most = bits_f(m), inverse = quot_ordinary(127.0f, most);
        uint32_t worst = 0u;
        packed.x = quants_ordinary(v0, inverse, worst);
        packed.y = quants_ordinary(v1, inverse, worst);
        scale = f2h_number(over_127(most));
        if (__builtin_expect(quants_not_ordinary(worst, m, on), 0)) packed = quantize_q8_0_general(v0, v1, scale);
    } else {
        packed = quantize_q8_0_general(v0, v1, scale);
    }
    if (on) {
        *reinterpret_cast<uint2 *>(qs + base) = packed;
        if ((tid & 3) == 0) d[base >> 5] = scale;
    }
}
WD_DEV void lds_quantize_q8_0(const float *__restrict__ x, int n, int8_t *qs, uint16_t *d, int tid, int nthreads) {
    const int per_pass = nthreads * 8;
    for (int base0 = 0; base0 < n; base0 += per_pass) {
        const int base = base0 + tid * 8;
        const bool on = base < n;
        float4 v0 = make_float4(0.f, 0.f, 0.f, 0.f), v1 = v0;
        if (on) {
            v0 = *reinterpret_cast<const float4 *>(x + base);
            v1 = *reinterpret_cast<const float4 *>(x + base + 4);
        }
        lds_quantize_q8_0_step<false>(v0, v1, on, base, qs, d, tid);  // (beside other things that nobody waits for)
    }
}

// Q8_K of one 256-value block by one wave (four values per lane).
WD_DEV void wave_quantize_q8_k_regs(const float4 &v, int8_t *qs256, float *d, int lane);
WD_DEV void wave_quantize_q8_k_block(const float *__restrict__ x256, int8_t *qs256, float *d, int lane) {
    wave_quantize_q8_k_regs(reinterpret_cast<const float4 *>(x256)[lane], qs256, d, lane);
}
// The same on four loaded values per lane (v = x256[4 * lane .. 4 * lane + 4)).
WD_DEV void wave_quantize_q8_k_regs(const float4 &v, int8_t *qs256, float *d, int lane) {
    float amax = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(v.x), __builtin_fabsf(v.y)),
                                 __builtin_fmaxf(__builtin_fabsf(v.z), __builtin_fabsf(v.w)));
    amax = wave_max_nonneg(amax);
    uint32_t packed = 0;
    float dv = 0.0f;
    if (amax != 0.0f) {
        const float iscale = -127.0f / amax;
        const int q0 = min(127, static_cast<int>(__builtin_rintf(v.x * iscale)));
        const int q1 = min(127, static_cast<int>(__builtin_rintf(v.y * iscale)));
        const int q2 = min(127, static_cast<int>(__builtin_rintf(v.z * iscale)));
        const int q3 = min(127, static_cast<int>(__builtin_rintf(v.w * iscale)));
        packed = (q0 & 0xff) | ((q1 & 0xff) << 8) | ((q2 & 0xff) << 16) | (static_cast<uint32_t>(q3 & 0xff) << 24);
        dv = 1.0f / iscale;
    }
    reinterpret_cast<uint32_t *>(qs256)[lane] = packed;
    if (lane == 0) *d = dv;
}

// ---- softmax + top-k by one wave, probabilities kept in registers --------------------------------
// Lane l owns the 8-expert groups l (and l + 64 when M == 2, i.e. more than 512 experts).
// Lanes 0..k-1 write ids/weights through the given pointers (LDS or global).
// src/qwen38_moe.cuh:711-818: softmax over all experts with the per-8 sums accumulated in a double in
// ascending order, k rungs of "largest remaining probability, lowest index on ties", renormalise.
// Wave-wide exact sum of doubles (any order gives the same bits when the caller has made sure that the sum is
// exact); the result is uniform.
WD_DEV double wave_sum_exact_f64(double v) {
    auto step = [](double x, auto mover) {
        const uint64_t b = __builtin_bit_cast(uint64_t, x);
        const int lo = mover(static_cast<int>(b & 0xffffffffu)), hi = mover(static_cast<int>(b >> 32));
        return x + __builtin_bit_cast(double, (static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) | static_cast<uint32_t>(lo));
    };
    v = step(v, [](int w) { return dpp_i<kDppXor1>(0, w); });
    v = step(v, [](int w) { return dpp_i<kDppXor2>(0, w); });
    v = step(v, [](int w) { return dpp_i<0x141>(0, w); });                     // row_half_mirror: quads 0/1, 2/3 of a row
    v = step(v, [](int w) { return dpp_i<0x140>(0, w); });                     // row_mirror: the two halves of a row
    v = step(v, [](int w) { return dpp_i<kDppBcast15, 0xa, 0xf, true>(0, w); });  // rows 1, 3 += lane 15 of rows 0, 2
    v = step(v, [](int w) { return dpp_i<kDppBcast31, 0xc, 0xf, true>(0, w); });  // rows 2, 3 += lane 31
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(b & 0xffffffffu), 63));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(b >> 32), 63));
    return __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
}

// Sum of the group sums as the reference takes it (a double accumulated in ascending group order); gs[m] of lane
// l is the sum of group l + 64 m.  When every non-zero group sum is within a factor 2^20 of the largest, all of
// them are multiples of one power of two and every partial sum fits 53 bits, so the result is exact and the same
// in any order: a lane tree then replaces the chain of dependent double additions.
template <int M>
WD_DEV double sum_groups(const float (&gs)[M], int groups, int lane) {
    float gmax = 0.0f, gmin = INFINITY;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        gmax = __builtin_fmaxf(gmax, gs[m]);
        gmin = __builtin_fminf(gmin, gs[m] > 0.0f ? gs[m] : INFINITY);
    }
    gmax = wave_max(gmax);
    gmin = -wave_max(-gmin);
    double sum = 0.0;
    if (gmin >= gmax * 0x1p-20f && gmax < INFINITY) {
        double part = 0.0;
#pragma unroll
        for (int m = 0; m < M; ++m) part += static_cast<double>(gs[m]);
        sum = wave_sum_exact_f64(part);
    } else {
#pragma unroll
        for (int m = 0; m < M; ++m) {
#pragma unroll
            for (int l = 0; l < 64; ++l) {
                const float gl = readlane_f(gs[m], l);
                if (l + 64 * m < groups) sum += static_cast<double>(gl);
            }
        }
    }
    return sum;
}

// Softmax of the row: lane l ends up with the probabilities of its 8-expert group(s) in v (or -inf everywhere
// when every exponential vanished: `dead`).
template <int M>
WD_DEV void softmax_probs(const float *logits, int n, int lane, float (&v)[8 * M], bool &dead) {
    const int groups = n >> 3;
    float mx = -INFINITY;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int g = lane + 64 * m;
        if (g < groups) {
            const float4 a = *reinterpret_cast<const float4 *>(logits + g * 8);
            const float4 b = *reinterpret_cast<const float4 *>(logits + g * 8 + 4);
            v[8 * m + 0] = a.x, v[8 * m + 1] = a.y, v[8 * m + 2] = a.z, v[8 * m + 3] = a.w;
            v[8 * m + 4] = b.x, v[8 * m + 5] = b.y, v[8 * m + 6] = b.z, v[8 * m + 7] = b.w;
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[8 * m + i] = -INFINITY;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) mx = __builtin_fmaxf(mx, v[8 * m + i]);
    }
    mx = wave_max(mx);
    float gs[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const bool on = lane + 64 * m < groups;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[8 * m + i] = on ? exp_ggml(v[8 * m + i] - mx) : 0.0f;
        const float lo = v[8 * m + 0] + v[8 * m + 4], lh = v[8 * m + 2] + v[8 * m + 6];
        const float hi = v[8 * m + 1] + v[8 * m + 5], hh = v[8 * m + 3] + v[8 * m + 7];
        gs[m] = (lo + lh) + (hi + hh);
    }
    const double sum = sum_groups<M>(gs, groups, lane);
    dead = (sum == 0.0);
    const float inv = dead ? 0.0f : static_cast<float>(1.0 / sum);
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const bool on = lane + 64 * m < groups;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[8 * m + i] = (on && !dead) ? v[8 * m + i] * inv : -INFINITY;
    }
}

// k rungs of "largest remaining probability, lowest index on ties" over the probabilities held as by
// softmax_probs; lane j keeps the j-th selected probability and id.
// For a row whose exponentials all vanished every probability is -inf, nothing ever beats the running best of
// -inf, and the reference keeps expert 0 with the value read back from the row.
template <int M>
WD_DEV void rungs_on_probs(float (&v)[8 * M], int k, int lane, float &top_mine, int &id_mine) {
    top_mine = 0.0f;
    id_mine = 0;
    for (int j = 0; j < k; ++j) {
        // this lane's largest remaining probability; lowest slot on ties
        float bv = v[0];
#pragma unroll
        for (int i = 1; i < 8 * M; ++i) bv = __builtin_fmaxf(bv, v[i]);
        int slot = 8 * M - 1;
#pragma unroll
        for (int i = 8 * M - 2; i >= 0; --i) slot = (v[i] == bv) ? i : slot;
        const float best = wave_max(bv);
        int win = 0;
        if (best > -INFINITY) {
            // lowest expert index among the lanes holding `best`: slots of group l come before the
            // slots of group l + 64, and lower lanes before higher ones inside a group row
            const bool mine = bv == best;
            unsigned long long mask = __builtin_amdgcn_ballot_w64(mine && slot < 8);
            if (M == 2 && mask == 0ull) mask = __builtin_amdgcn_ballot_w64(mine);
            const int wl = __builtin_ctzll(mask);
            const int ws = __builtin_amdgcn_readlane(slot, wl);
            win = (wl + 64 * (ws >> 3)) * 8 + (ws & 7);
#pragma unroll
            for (int i = 0; i < 8 * M; ++i) v[i] = (lane == wl && ws == i) ? -INFINITY : v[i];
        }
        if (lane == j) {
            top_mine = best;
            id_mine = win;
        }
    }
}

// Renormalisation: the selected probabilities summed in selection order in a double, clamp, divide, optional
// scale; lanes 0..k-1 write ids/weights through the given pointers (LDS or global).
WD_DEV void finish_weights(float top_mine, int id_mine, int k, float w_scale, int32_t *ids, float *weights,
                           const int32_t *__restrict__ override_ids, int lane) {
    double wsum = 0.0;
    for (int j = 0; j < k; ++j) wsum += static_cast<double>(readlane_f(top_mine, j));
    const float denom = __builtin_fmaxf(static_cast<float>(wsum), 6.103515625e-5f);
    if (lane < k) {
        float wj = top_mine / denom;
        if (w_scale != 0.0f && w_scale != 1.0f) wj = wj * w_scale;
        weights[lane] = wj;
        ids[lane] = override_ids ? override_ids[lane] : id_mine;
    }
}

template <int M>
WD_DEV void topk_wave_m(const float *logits, int n, int k, float w_scale, int32_t *ids, float *weights,
                        const int32_t *__restrict__ override_ids, int lane) {
    float v[8 * M];
    bool dead;
    softmax_probs<M>(logits, n, lane, v, dead);
    float top_mine;
    int id_mine;
    rungs_on_probs<M>(v, k, lane, top_mine, id_mine);
    finish_weights(top_mine, id_mine, k, w_scale, ids, weights, override_ids, lane);
}

// The ids held by lanes 0..k-1 (k <= 16) of every row of lanes into the kTagCopies replicas: four replicas
// per store instruction, so that the last replica goes out a quarter of the stores after the first.
WD_DEV void publish_ids_of_rows(int id, int k, uint32_t *tagged, int tag_side, int lane) {
    const int j = lane & 15, c4 = lane >> 4;
    if (j >= k) return;
#pragma unroll
    for (int c0 = 0; c0 < kTagCopies; c0 += 4)  // (the sides in turn)
        __hip_atomic_store(tagged + ((c0 & 4) ? tag_side : 0) + ((c0 >> 3) * 4 + c4) * 16 + j, static_cast<uint32_t>(id), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The ids held by lanes 0..k-1 only.
WD_DEV void publish_ids(int id_mine, int k, uint32_t *tagged, int tag_side, int lane) {
    const wd_uint2v t16 = __builtin_amdgcn_permlane16_swap(static_cast<uint32_t>(id_mine), static_cast<uint32_t>(id_mine), false, false);
    const wd_uint2v t32 = __builtin_amdgcn_permlane32_swap(t16.x, t16.x, false, false);
    publish_ids_of_rows(static_cast<int>(t32.x), k, tagged, tag_side, lane);
}

// The same selection by a workgroup of eight waves (every thread must call it; it contains barriers).
// Expert m * 512 + 64 * wave + lane belongs to (wave, lane): one or two logits per lane.  A wave instruction
// takes four cycles and a chain of k dependent arg-max steps costs about 0.2 us each, so the selection is made by
// thresholding and counting instead:
//   1. every row of 16 lanes publishes its largest logit (32 rows in the workgroup);
//   2. every wave finds T, the smallest of the row maxima that have fewer than k larger ones: at least k logits are
//      >= T, so the k largest are among the candidates {logit >= T} - a few dozen at most for any row that is not
//      nearly constant.  The candidates (logit, exponential, id) are compacted into one list in LDS (ballot, one
//      LDS atomic per wave); meanwhile the exponentials and the per-8 sums (a group is eight consecutive lanes)
//      are computed eight waves wide, and every wave notes its largest exponential outside the candidates;
//   3. wave 0 ranks the candidates by counting (one uniform read and a compare per candidate); rank r < k makes
//      a candidate the r-th selected.  exp is monotone only up to rounding and equal probabilities must go to the
//      lower id, so the result is checked: it is the reference's selection exactly when the probabilities are
//      strictly decreasing and the last one is strictly above every probability left.  The test is made on the
//      exponentials, with a margin that carries it over to the probabilities (see there), so that the ids go out
//      before the denominator is summed.  If it fails (ties - which also make the counted ranks collide -,
//      near-ties, rounding inversions, rows with -inf or NaN, a dead row, more than 64 candidates) wave 0 runs the
//      reference's rungs over the probabilities themselves.
// lds: 4 * (512 * M + 600) bytes of scratch.  The results are written by wave 0 (lanes 0..k-1).
// tagged != null: as soon as the ids are known - before the renormalisation, which only the weights need - id j
// goes to every replica with device-scope atomic stores (the readers poll them).
// Ids given by the caller (override_ids) are requested up front, so their round trip is not behind the selection.
// The three steps as functions of their own, so that a caller with the logits already in registers (or with waves
// that only keep the barriers company) can compose them.  LDS layout of the selection's scratch:
template <int M>
struct TopkLds {
    float *p, *gsum, *rmx, *cl, *ce, *rest, *selp;
    int *cid, *ncand, *sel;
    static constexpr int kRows = 32, kList = 64;
    static_assert(kRows + 2 * kList >= 2 * 64, "rmx, cl and ce as one: the one-wave form's 64 keys and their 64 experts");
    WD_DEV explicit TopkLds(uint8_t *lds) {
        p = reinterpret_cast<float *>(lds);        // [512 M] exponentials by expert id
        gsum = p + 512 * M;                        // [64 M] per-8 sums by group
        rmx = gsum + 64 * M;                       // [kRows] largest logit of every row of 16 lanes
        cl = rmx + kRows;                          // [kList] candidates: logit,
        ce = cl + kList;                           // [kList] exponential,
        cid = reinterpret_cast<int *>(ce + kList); // [kList] id
        ncand = cid + kList;                       // [4] their number
        sel = ncand + 4;                           // [16] the r-th selected id
        selp = reinterpret_cast<float *>(sel + 16);  // [16] its exponential
        rest = selp + 16;                          // [8] largest exponential outside the candidates, by wave
    }
};
constexpr int kTopkLdsBytes1 = 4 * (512 + 600), kTopkLdsBytes2 = 4 * (1024 + 600);

// Step 1 (waves 0..7, before the first barrier): the row maxima of the logits held in l[] (expert m * 512 + 64 * wave + lane).
template <int M>
WD_DEV void topk_block_step1(const float (&l)[M], const TopkLds<M> &s, int lane, int wave) {
    if (wave == 0 && lane == 0) s.ncand[0] = 0;
    float lm = l[0];
#pragma unroll
    for (int m = 1; m < M; ++m) lm = __builtin_fmaxf(lm, l[m]);
    lm = __builtin_fmaxf(lm, dpp_f<kDppXor1>(lm, lm));
    lm = __builtin_fmaxf(lm, dpp_f<kDppXor2>(lm, lm));
    lm = __builtin_fmaxf(lm, dpp_f<kDppRor4>(lm, lm));
    lm = __builtin_fmaxf(lm, dpp_f<kDppRor8>(lm, lm));
    if ((lane & 15) == 0) s.rmx[wave * 4 + (lane >> 4)] = lm;
}

// Step 2 (waves 0..7, between the barriers): threshold, exponentials and per-8 sums, candidate list.
template <int M>
WD_DEV void topk_block_step2(const float (&l)[M], int n, int k, const TopkLds<M> &s, int lane, int wave) {
    auto nan_is_large = [](float v) { return v != v ? INFINITY : v; };
    const float r = s.rmx[lane & 31];
    const float mx = wave_max(r);
    float thr;
    {
        int larger = 0;
#pragma unroll
        for (int t = 0; t < 8; ++t) {  // the same 16 bytes for every lane: broadcast reads
            const float4 q = *reinterpret_cast<const float4 *>(s.rmx + 4 * t);
            larger += (q.x > r ? 1 : 0) + (q.y > r ? 1 : 0) + (q.z > r ? 1 : 0) + (q.w > r ? 1 : 0);
        }
        thr = -wave_max(larger < k ? -r : -INFINITY);
    }
    float rme = 0.0f;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int id = m * 512 + wave * 64 + lane;
        const float e = (id < n) ? exp_ggml(l[m] - mx) : 0.0f;
        const float gs = close_lanes8(e);
        if ((lane & 7) == 0) s.gsum[m * 64 + wave * 8 + (lane >> 3)] = gs;
        s.p[id] = e;
        const bool c = l[m] >= thr && l[m] > -INFINITY;
        const unsigned long long cm = __builtin_amdgcn_ballot_w64(c);
        if (cm != 0ull) {
            int base = 0;
            if (lane == 0) base = atomicAdd(s.ncand, static_cast<int>(__builtin_popcountll(cm)));
            base = __builtin_amdgcn_readfirstlane(base);
            const int pos = base + static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(cm >> 32),
                                                        __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(cm), 0u)));
            if (c && pos < 64) {
                s.cl[pos] = l[m];
                s.ce[pos] = e;
                s.cid[pos] = id;
            }
        }
        rme = __builtin_fmaxf(rme, c ? 0.0f : nan_is_large(e));
    }
    rme = wave_max(rme);
    if (lane == 0) s.rest[wave] = rme;
}

// Step 3 (wave 0, after the second barrier): ranks, check, publication of the ids, denominator, weights.
// id_given: the caller's id for lane j < k when the ids are replaced (override), requested before step 1.
template <int M>
WD_DEV void topk_block_step3(int n, int k, float w_scale, int32_t *ids, float *weights, bool override_ids, int id_given,
                             const TopkLds<M> &s, int lane, unsigned long long *stamps, uint32_t *tagged, int tag_side) {
#define WD_STAMP(i) do { if (stamps && lane == 0) stamps[i] = wall_clock64(); } while (0)
    auto nan_is_large = [](float v) { return v != v ? INFINITY : v; };
    const int groups = n >> 3;
    // ranks of the candidates
    const int nc = s.ncand[0];
    const float got_l = s.cl[lane], got_e = s.ce[lane];  // requested together with the count, not behind it
    const int got_id = s.cid[lane];
    const bool fits = nc <= 64;
    const bool mine = fits && lane < nc;
    const float my_l = mine ? got_l : -INFINITY;
    const float my_e = mine ? got_e : 0.0f;
    const int my_id = mine ? got_id : -1;
    if (lane < 16) s.sel[lane] = -1;
    int rk = 0;
    const int steps = fits ? (nc + 3) & ~3 : 0;  // lanes past the list hold -inf, which is ahead of nothing
    for (int src = 0; src < steps; src += 4) {
#pragma unroll
        for (int u = 0; u < 4; ++u) rk += (readlane_f(my_l, src + u) > my_l) ? 1 : 0;
    }
    wave_lds_fence();
    if (mine && rk < k) {
        s.sel[rk] = my_id;  // equal logits collide here; the loser stays among the rest and fails the test below
        s.selp[rk] = my_e;
    }
    wave_lds_fence();
    const bool taken = mine && rk < k && s.sel[rk < k ? rk : 0] == my_id;
    float rest_all = wave_max((mine && !taken) ? nan_is_large(my_e) : 0.0f);
#pragma unroll
    for (int w = 0; w < 8; ++w) rest_all = __builtin_fmaxf(rest_all, s.rest[w]);
    if (!fits) rest_all = INFINITY;
    WD_STAMP(3);

    // The ids do not wait for the denominator: p = e * inv with one inv in [2^-10, 1] for the whole row is
    // monotone in e, and two exponentials that differ by more than a few units in the last place (and are not
    // tiny) cannot round to the same product, so this test on the exponentials implies the one on the
    // probabilities.  A NaN counts as larger than everything.
    const int idc = (lane < k) ? s.sel[lane] : -1;
    const bool have = idc >= 0 && idc < n;
    const float top_e = have ? s.selp[lane] : 0.0f;
    const float nxt = dpp_f<kDppShl1>(0.0f, top_e);  // k <= 16: the selected sit in one row of lanes
    const float below = (lane == k - 1 ? rest_all : nxt) * 1.000001f;
    const bool good = lane >= k || (have && top_e >= 0x1p-100f && top_e > below);
    const bool all_good = __builtin_amdgcn_ballot_w64(good) == ~0ull;
    int id_mine = override_ids ? id_given : idc;
    if (all_good && tagged) {
        publish_ids(id_mine, k, tagged, tag_side, lane);
    }
    WD_STAMP(6);

    // the denominator (only the weights and the slow path need it)
    float gs[M];
#pragma unroll
    for (int m = 0; m < M; ++m) gs[m] = (lane + 64 * m < groups) ? s.gsum[m * 64 + lane] : 0.0f;
    const double sum = sum_groups<M>(gs, groups, lane);
    const float inv = (sum == 0.0) ? 0.0f : static_cast<float>(1.0 / sum);
    const bool dead = sum == 0.0;
    float top_mine = top_e * inv;
    if (!all_good) {
        auto rungs = [&](auto rows) {
            constexpr int R = decltype(rows)::value;
            float v[8 * R];
#pragma unroll
            for (int m = 0; m < R; ++m)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int ix = (lane + 64 * m) * 8 + i;
                    v[8 * m + i] = (ix < n && !dead) ? s.p[ix] * inv : -INFINITY;
                }
            rungs_on_probs<R>(v, k, lane, top_mine, id_mine);
        };
        // (16 of 72..256 experts: with fewer rows of lanes than there are experts to select the threshold excludes nobody, and this
        // is the rule; by the rungs for 1024 dispatch AB took 19.7 us instead of 17.1, top-16 of 128)
        if (M == 1 || n <= 512) rungs(std::integral_constant<int, 1>{});
        else rungs(std::integral_constant<int, M>{});
        if (override_ids) id_mine = id_given;
        if (tagged) publish_ids(id_mine, k, tagged, tag_side, lane);
    }
    finish_weights(top_mine, id_mine, k, w_scale, ids, weights, nullptr, lane);
    WD_STAMP(7);
#undef WD_STAMP
}

template <int M>
WD_DEV void topk_block_m(const float *logits, int n, int k, float w_scale, int32_t *ids, float *weights,
                         const int32_t *__restrict__ override_ids, uint8_t *lds, int lane, int wave,
                         unsigned long long *stamps = nullptr, uint32_t *tagged = nullptr, int tag_side = 0) {
#define WD_STAMP(i) do { if (stamps && wave == 0 && lane == 0) stamps[i] = wall_clock64(); } while (0)
    const TopkLds<M> s(lds);
    WD_STAMP(0);
    int id_given = 0;
    if (override_ids && wave == 0 && lane < k) id_given = override_ids[lane];
    float l[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int id = m * 512 + wave * 64 + lane;
        l[m] = (id < n) ? __hip_atomic_load(logits + id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : -INFINITY;
    }
    topk_block_step1<M>(l, s, lane, wave);
    __syncthreads();
    WD_STAMP(1);
    topk_block_step2<M>(l, n, k, s, lane, wave);
    __syncthreads();
    WD_STAMP(2);
    if (wave == 0)
        topk_block_step3<M>(n, k, w_scale, ids, weights, override_ids != nullptr, id_given, s, lane, stamps, tagged, tag_side);
#undef WD_STAMP
}

WD_DEV void topk_wave(const float *logits, int n, int k, float w_scale, int32_t *ids, float *weights,
                      const int32_t *__restrict__ override_ids, int lane) {
    if (n <= 512)
        topk_wave_m<1>(logits, n, k, w_scale, ids, weights, override_ids, lane);
    else
        topk_wave_m<2>(logits, n, k, w_scale, ids, weights, override_ids, lane);
}

// ---- the same selection by ONE wave that holds M = 1, 2, 4 or 8 logits per lane --------------------------------------
// lv[j] is the logit of expert 64 j + lane (-inf at and beyond n; n <= 64 M, k <= 15).  Everybody behind the selection waits for it and a
// single wave's time is the length of its dependent steps, so step A counts instead of searching and keeps what is not needed for the
// ids out of the way:
//   * every logit becomes a 32-bit key, its bits mapped so that unsigned order is float order;
//   * the largest keys of the sixteen groups of lanes that are equal modulo 16 are ranked among themselves, four comparisons in each row of
//     lanes (the rows hold the same sixteen, each turned by four lanes more than the one before); T, the (k+1)-th of them, is a lower bound of the
//     (k+1)-th largest key.  From k = 12 on sixteen groups exclude too little: 32 groups of lanes equal modulo 32;
//   * the keys not below T - 18 or so of 512 - are compacted into LDS with their experts and ranked by counting, one half of the wave against the
//     first sixteen of the list and the other against the second; lists of 33 to 64 (one row in a thousand of random logits, ten of 512, and rows whose
//     favourites crowd into few groups), by uniform reads; longer ones are not accepted;
//   * rank r goes to slot r.  Equal keys collide there and leave the slot behind them empty.
// The slots are accepted as the selection only when the first k are filled, and the (k+1)-th too unless every expert is selected, and the
// differences d_j = l_j - l_0, as the reference takes them ahead of its exponentials, fall by kSelGap from one to the next and by kSelGapLast from the k-th to the
// (k+1)-th, and the k-th is not below kSelFloor.  exp_ggml is within two units in the last place of the true exponential (relative error below 2^-22) on
// normal results, so the exponentials then fall by a factor of more than 1 + 2^-19.5 (1 + 2^-17.2 at the end, where what was not taken may be anything up
// to the (k+1)-th): probabilities, products with one 1/sum in [2^-10, 1], stay strictly ordered, and exp itself is not needed before the ids are out.
// Rows the test does not accept (ties, near-ties, NaN, +inf, fewer than k + 1 finite logits, selected exponentials below
// 2^-100) take the reference's rungs over all probabilities in step B.
// Alone on the device, from the logits in registers until the ids are on their way: 512 experts of which 10 1,810 cycles (0.75 us), 64 of which 6 1,220; by uniform
// reads over keys of 23 bits, with the exponentials ahead of the ids, 3,770 and 2,130.
struct SelWaveState {
    float d;       // every row of lanes, lane j < k of it: the j-th largest logit minus the largest (accepted rows)
    int id;        // its expert
    bool fast;     // step A accepted the row (the same in every lane)
};
constexpr float kSelGap = 0x1p-19f, kSelGapLast = 0x1p-17f, kSelFloor = -69.0f;  // (e^-69 > 2^-100)
constexpr uint32_t kSelFinite = 0x00800000u;  // keys from here on are above -inf's

// Step A.  Returns with st.fast, and for accepted rows the ids of the selection in lanes 0..k-1 of every row of lanes of st.id.
// Of the scratch it uses the candidates' and the selection's places only (rmx, cl, ce; sel, selp).
// FEW (k < 12 only): fewer registers, for the resident stack.  (48 layers whose lists are of 33 to 64: 13.45 us each, left to step B 16.6; with a trace 10.3, 12.25.)
template <int M, bool FEW = false>
WD_DEV void sel_wave_ids(const float (&lv)[M], int n, int k, const TopkLds<1> &s, int lane, SelWaveState &st) {
    constexpr int kEq = 32, kUgt = 34, kUge = 35, kOge = 3;  // of the compares into scalar masks
    uint32_t *const ck = reinterpret_cast<uint32_t *>(s.rmx);  // [64] keys of the candidates,
    int *const cid = reinterpret_cast<int *>(s.rmx) + 64;      // [64] their experts
    ck[lane & 31] = 0u;  // (behind the end of the list nothing is ahead of anything)
    s.sel[lane & 15] = 0;
    const int j = lane & 15;
    const unsigned long long first_k = ((1ull << k) - 1ull) * 0x0001000100010001ull;  // lanes 0..k-1 of every row of lanes
    const float gap_needed = j == k - 1 ? kSelGapLast : kSelGap;
    uint32_t h[M], head = 0u, least = 0xffffffffu;
#pragma unroll
    for (int i = 0; i < M; ++i) {
        const uint32_t b = f_bits(lv[i]);
        h[i] = b ^ (static_cast<uint32_t>(static_cast<int>(b) >> 31) | 0x80000000u);
        head = max(head, h[i]), least = min(least, h[i]);
    }
    // (NaN with the sign set is below -inf; others are above +inf and fail as the largest)
    const unsigned long long below_inf = __builtin_amdgcn_uicmp(kSelFinite - 1u, least, kUgt);
    auto swap16 = [](uint32_t v) { return __builtin_amdgcn_permlane16_swap(v, v, false, false); };
    auto swap32 = [](uint32_t v) { return __builtin_amdgcn_permlane32_swap(v, v, false, false); };
    const wd_uint2v h32 = swap32(head);
    head = max(h32.x, h32.y);
    int larger = 0;
    if (FEW || M == 1 || __builtin_expect(k < 12, 1)) {
        const wd_uint2v h16 = swap16(head);
        head = max(h16.x, h16.y);
        int turned = dpp_i<kDppRor4, 0xa>(static_cast<int>(head), static_cast<int>(head));
        turned = dpp_i<kDppRor8, 0xc>(turned, turned);
        larger = static_cast<uint32_t>(turned) > head ? 1 : 0;
        larger += static_cast<uint32_t>(dpp_i<0x121, 0xf, 0xf, true>(0, turned)) > head ? 1 : 0;
        larger += static_cast<uint32_t>(dpp_i<0x122, 0xf, 0xf, true>(0, turned)) > head ? 1 : 0;
        larger += static_cast<uint32_t>(dpp_i<0x123, 0xf, 0xf, true>(0, turned)) > head ? 1 : 0;
        const wd_uint2v a = swap16(static_cast<uint32_t>(larger));
        const wd_uint2v b = swap32(a.x + a.y);
        larger = static_cast<int>(b.x + b.y);
    } else {
#pragma nounroll
        for (int g = 0; g < 32; g += 4) {
#pragma unroll
            for (int u = 0; u < 4; ++u) larger += static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(head), g + u)) > head ? 1 : 0;
        }
    }
    // (with k groups or fewer that hold experts - at most 64 of these then - every key is a candidate)
    const unsigned long long at = __builtin_amdgcn_uicmp(static_cast<uint32_t>(larger), static_cast<uint32_t>(k), kEq);
    const uint32_t kth = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(head), __builtin_ctzll(at | (1ull << 63))));
    const uint32_t thr = at ? max(kth, kSelFinite) : kSelFinite;
    unsigned long long m[M];
    int first[M + 1];
    first[0] = 0;
#pragma unroll
    for (int i = 0; i < M; ++i) m[i] = __builtin_amdgcn_uicmp(h[i], thr, kUge);
#pragma unroll
    for (int i = 0; i < M; ++i) first[i + 1] = first[i] + static_cast<int>(__builtin_popcountll(m[i]));
    const int count = first[M];
    // every lane writes each of its keys, no branch: what is no candidate, and what a list of more than 32 has too much, goes behind the 32 places
#pragma unroll
    for (int i = 0; i < M; ++i) {
        const int before = first[i] + static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(m[i] >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(m[i]), 0u)));
        const int place = min(h[i] >= thr ? before : 63, lane | 32);
        ck[place] = h[i], cid[place] = 64 * i + lane;
    }
    wave_lds_fence();
    uint32_t key = ck[lane & 31];
    int id = cid[lane & 31], rank = 0;
    uint4 q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = reinterpret_cast<const uint4 *>(ck)[4 * (lane >> 5) + i];
    asm volatile("" : "+v"(id));  // (asked for here and not where it is used)
    if (__builtin_expect(count <= 32, 1)) {
        unsigned long long ahead[16];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            ahead[4 * i] = __builtin_amdgcn_uicmp(q[i].x, key, kUgt), ahead[4 * i + 1] = __builtin_amdgcn_uicmp(q[i].y, key, kUgt),
            ahead[4 * i + 2] = __builtin_amdgcn_uicmp(q[i].z, key, kUgt), ahead[4 * i + 3] = __builtin_amdgcn_uicmp(q[i].w, key, kUgt);
#pragma unroll
        for (int i = 0; i < 16; ++i) rank += __builtin_amdgcn_inverse_ballot_w64(ahead[i]) ? 1 : 0;
        const wd_uint2v t = swap32(static_cast<uint32_t>(rank));
        rank = static_cast<int>(t.x + t.y);
    } else if (!FEW || count <= 64) {
        int base = 0;
        ck[lane] = 0u;
        wave_lds_fence();
#pragma unroll
        for (int i = 0; i < M; ++i) {
            uint32_t h_i = h[i];
            unsigned long long in = m[i];
            int before = first[i];
            if (FEW) {  // (worked out again: held until here they cost the resident stack its last registers)
                h_i = f_bits(lv[i]);
                asm volatile("" : "+v"(h_i));
                h_i ^= static_cast<uint32_t>(static_cast<int>(h_i) >> 31) | 0x80000000u;
                in = __builtin_amdgcn_uicmp(h_i, thr, kUge), before = base;
                base += static_cast<int>(__builtin_popcountll(in));
            }
            before += static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(in >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(in), 0u)));
            if (h_i >= thr) ck[min(before, 63)] = h_i, cid[min(before, 63)] = 64 * i + lane;  // (a list of more than 64 is not used)
        }
        wave_lds_fence();
        key = ck[lane], id = cid[lane];
#pragma nounroll
        for (int src = 0; src < 64; src += 4) {
#pragma unroll
            for (int u = 0; u < 4; ++u) rank += static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(key), src + u)) > key ? 1 : 0;
        }
    }
    if (key != 0u && rank <= k) s.sel[rank] = static_cast<int>(key), s.selp[rank] = bits_f(static_cast<uint32_t>(id));
    wave_lds_fence();
    const uint32_t mine = static_cast<uint32_t>(s.sel[j]);  // the j-th largest key of the row, 0 if there is none
    const int idc = static_cast<int>(f_bits(s.selp[j]));
    wave_lds_fence();
    const float l = mine ? bits_f(mine ^ (~static_cast<uint32_t>(static_cast<int>(mine) >> 31) | 0x80000000u)) : -INFINITY;
    const float d = l - readlane_f(l, 0);
    const float nxt = dpp_f<kDppShl1>(-INFINITY, d);  // k + 1 <= 16: a row of lanes holds them
    const unsigned long long apart = __builtin_amdgcn_fcmpf(d - nxt, gap_needed, kOge) & __builtin_amdgcn_fcmpf(d, kSelFloor, kOge);
    // (with every expert selected there is no (k+1)-th, and nothing left that could be above the last)
    const unsigned long long filled = __builtin_amdgcn_uicmp(mine, 0u, kUgt) | (n == k ? ~0ull : 0ull);
    st.d = d, st.id = idc;
    st.fast = (~apart & first_k) == 0ull && (filled >> k & 1ull) != 0ull && below_inf == 0ull && count <= 64;
}

// Step B, first half (any wave that holds the logits; it need not be the wave of step A): every exponential into s.p,
// the per-8 sums, and the row's 1/sum as the reference takes it (0 for a row whose exponentials all vanished: `dead`).
template <int M>
WD_DEV float sel_wave_denominator(const float (&lv)[M], int n, const TopkLds<1> &s, int lane, bool &dead) {
    const int groups = n >> 3;
    float lm = lv[0];
#pragma unroll
    for (int j = 1; j < M; ++j) lm = __builtin_fmaxf(lm, lv[j]);
    const float mx = wave_max(lm);
#pragma unroll
    for (int j = 0; j < M; ++j) {
        const int id = 64 * j + lane;
        const float e = (id < n) ? exp_ggml(lv[j] - mx) : 0.0f;
        const float gs = close_lanes8(e);
        if ((lane & 7) == 0) s.gsum[8 * j + (lane >> 3)] = gs;
        s.p[id] = e;
    }
    wave_lds_fence();
    const float g1[1] = {lane < groups ? s.gsum[lane] : 0.0f};
    const double sum = sum_groups<1>(g1, groups, lane);
    dead = sum == 0.0;
    return dead ? 0.0f : static_cast<float>(1.0 / sum);
}

// Step B, second half (the wave of step A; s.p and inv as the first half left them, which may have been another wave
// on the far side of a barrier): for rows step A did not accept the reference's rungs over the probabilities; then lanes
// 0..k-1 write the weights and the ids (ids_given: id_given instead).
WD_DEV void sel_wave_weights(int n, int k, float w_scale, const TopkLds<1> &s, int lane, SelWaveState &st, float inv, bool dead,
                             int32_t *ids, float *weights, bool ids_given, int id_given) {
    float top_mine = exp_ggml(st.d) * inv;
    int id_mine = st.id;
    if (!st.fast) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int ix = lane * 8 + i;
            v[i] = (ix < n && !dead) ? s.p[ix] * inv : -INFINITY;
        }
        rungs_on_probs<1>(v, k, lane, top_mine, id_mine);
        st.id = id_mine;
    }
    finish_weights(top_mine, ids_given ? id_given : id_mine, k, w_scale, ids, weights, nullptr, lane);
}

// ---- selection inside the dispatch that computes the logits ------------------------------------------------------------
// Every router wave hands its logit on as a word that cannot be kHandEmpty (hand[e], the shared expert's gate logit in
// hand[n_slot]; for either side); dispatch C sets the words back.  A workgroup of its own, behind the router's, selects: it polls the words
// until all are there.  It waits for workgroups with lower indices only, as every wait inside a dispatch does.  No router workgroup waits for its own word,
// counts itself or looks at the row.
// (Selected by the router workgroups that end last - each waits until its words are acknowledged and looks at the row, a ticket names the
// one to publish - the ids of 2048 / 512 are out 7.2 us after the dispatch's start, by a workgroup of its own 5.6; 64 experts of 1024 / 256 5.1, 3.9.
// us per layer: 2560 / 640 24.64, so 24.39; 2048 / 512 20.0, 19.65; 1024 / 256 11.75, 11.67.  Four tokens of 2048 / 512, whose router workgroups
// counted themselves and the last one polled, 39.95, 39.55.)
// (By the last router workgroup where nobody waits for the ids, whichever the others do: split 2048 / 512 24.8, by a workgroup of its own 23.4; split
// 2560 / 640 30.5, 28.3; dispatch A alone 8.8, 7.6 and 9.9, 8.9.)
struct HandRow {
    const uint32_t *hand;  // the copy of the reader's side
    int n, n_slot;
    bool gate;  // hand[n_slot] is one of the row's
    unsigned limit;  // polls before one that waits for the row gives up
};
WD_DEV const uint32_t *hand_copy(const uint32_t *hand, int hand_side) { return hand + (xcc_side() ? hand_side : 0); }
WD_DEV uint32_t hand_load(const uint32_t *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// `words` of them back to "not yet", in both copies (the count in the second one's place is as it was).
WD_DEV void hand_clear(uint32_t *hand, int hand_side, int words, int thread, int threads) {
    for (int i = thread; i < words; i += threads) {
        __hip_atomic_store(hand + i, kHandEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(hand + hand_side + i, kHandEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}
// Sets the words back where no dispatch C does: the one of the router workgroups and the selecting one that is done last, behind every other
// one's last use of them.  Every thread of each of the n_wgs must call it.  (A fill launched behind the dispatch instead, us per layer with the ids through the host: 2048 / 512
// 46.2, so 45.0; 1024 / 256 37.9, 36.9; 4096 / 1536 66.5, 65.5.)
WD_DEV void hand_close(uint32_t *hand, int hand_side, int n_slot, int n_wgs, int &last) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);  // what this wave has asked for of the words is there
    __syncthreads();
    if (threadIdx.x == 0) last = __hip_atomic_fetch_add(hand + n_slot + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u == static_cast<uint32_t>(n_wgs - 1);
    __syncthreads();
    if (!last) return;
    hand_clear(hand, hand_side, n_slot + 2, static_cast<int>(threadIdx.x), static_cast<int>(blockDim.x));
}
// lv[j]: logit 64 j + lane, once the row is complete (beyond the limit words that did not come are NaN, what is selected then are experts of
// the layer, and the status makes the results NaN).  Returns whether it was.
// Another stream's kernel may keep router workgroups from their places for a while.  Where workgroups of the dispatch wait for the ids, these give up
// after spin_limit polls, 25 ms by default, and the selection, which begins before them, must not do so ahead of them: beyond the tens of microseconds
// in which the words are due a poll takes 4 us, so the same number of polls is 0.25 s.  Where nobody waits for the ids (they are known before the launch, or the
// routed part is another one), nobody gives up, so the selection must not either: kHandPatient polls, a quarter of a minute, are there for a broken device.
constexpr unsigned kHandFastPolls = 64, kHandPatient = 1u << 22;
template <int M>
WD_DEV bool hand_gather(const HandRow &r, int lane, float (&lv)[M]) {
    for (unsigned polls = 0; polls < r.limit; ++polls) {
        if (polls > kHandFastPolls) __builtin_amdgcn_s_sleep(127);
        const uint32_t g = r.gate ? hand_load(r.hand + r.n_slot) : 0u;
        bool there = hand_arrived(g);
#pragma unroll
        for (int j = 0; j < M; ++j) {
            const uint32_t w = (64 * j + lane < r.n) ? hand_load(r.hand + 64 * j + lane) : f_bits(-INFINITY);
            there = there && hand_arrived(w), lv[j] = bits_f(w);
        }
        if (__builtin_amdgcn_ballot_w64(there) == ~0ull) return true;
    }
    return false;
}

// The selections below return whether the row's words came (a wave that does not wait for them: true; the caller sets the status otherwise).
// n <= 64 M logits, k <= 15: wave 0 ranks and publishes the ids, wave 1 takes the exponentials and the denominator meanwhile, and wave 0 forms
// the weights behind one barrier.  Every thread of the workgroup must call it.  ids, weights: LDS.
template <int M>
WD_DEV bool topk_two_waves(const HandRow &row, int k, float w_scale, int32_t *ids, float *weights, const int32_t *__restrict__ override_ids,
                           uint8_t *lds, int lane, int wave, unsigned long long *stamps, uint32_t *tagged, int tag_side) {
#define WD_STAMP(i) do { if (stamps && wave == 0 && lane == 0) stamps[i] = wall_clock64(); } while (0)
    const TopkLds<1> s(lds);
    const int n = row.n;
    SelWaveState st;
    int id_given = 0;
    bool there = true;
    float lv[M];
    if (wave <= 1) {
        if (override_ids && wave == 0 && lane < k) id_given = override_ids[lane];
        there = hand_gather<M>(row, lane, lv);
    }
    WD_STAMP(0);
    if (wave == 0) {
        sel_wave_ids(lv, n, k, s, lane, st);
        WD_STAMP(3);
        if (st.fast && tagged) {
            if (override_ids) publish_ids(id_given, k, tagged, tag_side, lane);
            else publish_ids_of_rows(st.id, k, tagged, tag_side, lane);
        }
        WD_STAMP(6);
    } else if (wave == 1) {
        bool dead;
        const float inv = sel_wave_denominator(lv, n, s, lane, dead);
        if (lane == 0) s.rest[0] = inv, s.rest[1] = dead ? 1.0f : 0.0f;
    }
    __syncthreads();
    if (wave == 0) {
        const bool fast = st.fast;
        sel_wave_weights(n, k, w_scale, s, lane, st, s.rest[0], s.rest[1] != 0.0f, ids, weights, override_ids != nullptr, id_given);
        if (!fast && tagged) publish_ids(override_ids ? id_given : st.id, k, tagged, tag_side, lane);
        WD_STAMP(7);
    }
#undef WD_STAMP
    return there;
}

// Every thread of the workgroup must call it.  Two waves select where one can hold the row (n <= 512, k <= 15); ids and weights are left in
// LDS by wave 0.
// (The block form takes 3.0 us from the logits to the ids for 6 of 64 experts - with fewer rows of lanes than there are experts to select its threshold
// excludes nobody - and 2.2 for 10 of 512.)
WD_DEV bool topk_block(const HandRow &row, int k, float w_scale, int32_t *ids, float *weights, const int32_t *__restrict__ override_ids,
                       uint8_t *lds, int lane, int wave, unsigned long long *stamps = nullptr, uint32_t *tagged = nullptr, int tag_side = 0) {
    const int n = row.n;
    if (n <= 512 && k <= 15) {
        if (n <= 64) return topk_two_waves<1>(row, k, w_scale, ids, weights, override_ids, lds, lane, wave, stamps, tagged, tag_side);
        if (n <= 128) return topk_two_waves<2>(row, k, w_scale, ids, weights, override_ids, lds, lane, wave, stamps, tagged, tag_side);
        if (n <= 256) return topk_two_waves<4>(row, k, w_scale, ids, weights, override_ids, lds, lane, wave, stamps, tagged, tag_side);
        return topk_two_waves<8>(row, k, w_scale, ids, weights, override_ids, lds, lane, wave, stamps, tagged, tag_side);
    }
    float lv[16];
    const bool there = hand_gather<16>(row, lane, lv);  // (every wave)
    topk_block_m<2>(reinterpret_cast<const float *>(row.hand), n, k, w_scale, ids, weights, override_ids, lds, lane, wave, stamps, tagged, tag_side);
    return there;
}

// Stand-alone softmax/top-k dispatch: one wave (src/qwen38_moe.cuh:711-818).
// If gate_logit != null, gate_logit[0] is replaced by sigmoid_ggml(gate_logit[0]) (shared expert gate).
// If override_ids != null the selected ids are replaced by override_ids[0..k) after the weights are formed.
__global__ __launch_bounds__(64) void k_topk_softmax(const float *__restrict__ logits, int n, int k, float w_scale,
                                                      int32_t *__restrict__ ids, float *__restrict__ weights,
                                                      float *__restrict__ gate_logit,
                                                      const int32_t *__restrict__ override_ids) {
    const int lane = threadIdx.x;
    if (gate_logit && lane == 0) gate_logit[0] = sigmoid_ggml(gate_logit[0]);
    if (n <= 512 && k <= 15) {  // threshold and ranks first, the reference's rungs for the rows that need them
        __shared__ __align__(16) uint8_t s_sel[kTopkLdsBytes1];
        const TopkLds<1> s(s_sel);
        float lv[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) lv[j] = (64 * j + lane < n) ? logits[64 * j + lane] : -INFINITY;
        SelWaveState st;
        sel_wave_ids(lv, n, k, s, lane, st);
        int id_given = 0;
        if (override_ids && lane < k) id_given = override_ids[lane];
        bool dead;
        const float inv = sel_wave_denominator(lv, n, s, lane, dead);
        sel_wave_weights(n, k, w_scale, s, lane, st, inv, dead, ids, weights, override_ids != nullptr, id_given);
        return;
    }
    topk_wave(logits, n, k, w_scale, ids, weights, override_ids, lane);
}

// ---- router rows -------------------------------------------------------------------------------------------
// ggml's closing tree over the 32 accumulators of a row, held one per lane by lanes 0..31 or 32..63: the upper sixteen
// onto the lower, then 8, 4, 1 and 2 further on (the order of src/qwen38_moe.cuh:198-245).  Lane moves inside the vector
// unit instead of five trips through the LDS crossbar.  Valid in lanes 0 and 32.
WD_DEV float router_close32(float s) {
    const wd_uint2v w = __builtin_amdgcn_permlane16_swap(f_bits(s), f_bits(s), false, false);
    s = bits_f(w.x) + bits_f(w.y);
    s = s + dpp_f<0x108>(0.0f, s);  // row_shl:8
    s = s + dpp_f<kDppShl4>(0.0f, s);
    s = s + dpp_f<kDppShl1>(0.0f, s);
    return s + dpp_f<kDppShl2>(0.0f, s);
}

// Rows come in spans of 2048 columns, the lower half of the wave's lanes taking the first 1024 and the upper half the rest; a
// half's part of a span is up to four groups of 256 columns, eight per lane (hidden is a multiple of 256).  The rows lie on the way to
// the ids; with a test, an address and a select for every column in the groups' place, us per layer from HBM, so / with groups:
// 1024 / 256 15.7 / 14.1, 1536 / 512 19.0 / 18.2, 2560 / 640 25.2 / 24.5, 3072 / 768 27.0 / 25.7; six variants of dispatch AB spilled.
struct RouterSpan {
    int lower, upper;  // groups of the halves
    WD_DEV explicit RouterSpan(int cols) : lower(min(cols, 1024) >> 8), upper(max(min(cols, 2048) - 1024, 0) >> 8) {}
};
// The lane's weights of the span at column c0 (groups that the row does not have: those of the first group, not used).
WD_DEV void router_span_load(const float *wr, int c0, const RouterSpan &sp, bool upper, int t, float (&wv)[32]) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const float *p = wr + (c0 + t + (upper ? (g < sp.upper ? 1024 + 256 * g : 0) : (g < sp.lower ? 256 * g : 0)));
#pragma unroll
        for (int u = 0; u < 8; ++u) wv[8 * g + u] = gld_f32(p + 32 * u);
    }
}
// The values of x that the lane's weights of the span meet, all at once.  x: the half's first column of the lane.
WD_DEV void router_span_x(const float *x, const RouterSpan &sp, bool upper, float (&xv)[32]) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const float *p = x + 256 * max(min(g, (upper ? sp.upper : sp.lower) - 1), 0);
#pragma unroll
        for (int u = 0; u < 8; ++u) xv[8 * g + u] = p[32 * u];
    }
}
// A half's multiply-adds of the span, continuing the chain from v.
WD_DEV float router_span_run(const float (&wv)[32], const float (&xv)[32], int groups, float v) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        if (g < groups) {
#pragma unroll
            for (int u = 0; u < 8; ++u) v = __builtin_fmaf(wv[8 * g + u], xv[8 * g + u], v);
        }
    }
    return v;
}
// The logit in lane 32 of the wave, to both copies of hand[slot] by one instruction.
WD_DEV void router_hand_on(float logit, uint32_t *hand, int hand_side, int slot, int lane) {
    const uint32_t word = hand_word_bits(f_bits(readlane_f(logit, 32)));
    if (lane < 2) __hip_atomic_store(hand + (lane == 0 ? 0 : hand_side) + slot, word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// x to LDS, by the whole workgroup of 512 threads.  The first 4096 columns are requested ahead of the row's weights: loads return in order, and so x is in LDS and in the
// lanes' registers (router_span_x) while the weights are on their way.  (Behind them, and x read from LDS
// between the multiply-adds, us per layer: 2048 / 512 18.7, so 18.4; 2560 / 640 22.9, 22.5; 1024 / 1024 17.6, 17.3; four tokens of 2048 / 512 38.2, 37.8.)
struct RouterX {
    float4 first, second = make_float4(0.f, 0.f, 0.f, 0.f);
    WD_DEV RouterX(const float *__restrict__ x, int cols) {
        const int i = static_cast<int>(threadIdx.x) * 4;
        first = *reinterpret_cast<const float4 *>(x + min(i, cols - 4));
        if (cols > 2048) second = *reinterpret_cast<const float4 *>(x + min(i + 2048, cols - 4));
        __builtin_amdgcn_sched_barrier(0);
    }
    WD_DEV void stage(const float *__restrict__ x, float *xs, int cols) const {
        const int i = static_cast<int>(threadIdx.x) * 4;
        if (i < cols) *reinterpret_cast<float4 *>(xs + i) = first;
        if (i + 2048 < cols) *reinterpret_cast<float4 *>(xs + i + 2048) = second;
        for (int j = i + 4096; j < cols; j += 2048) *reinterpret_cast<float4 *>(xs + j) = *reinterpret_cast<const float4 *>(x + j);
    }
};

// One row per wave, x staged once per workgroup in LDS (f32 [cols]).
// Accumulator t (of ggml's 4 x 8) of the row lives in lanes t and t + 32: for every span of 2048 columns lane t
// runs the multiply-adds of columns [span, span + 1024) and hands the value to lane t + 32, which continues with
// [span + 1024, span + 2048) and hands it back for the next span, so each chain still sees its columns in
// ascending order while a lane holds only 32 weights (half the registers of the 32-lanes-per-row version,
// which lets three workgroups of the merged dispatch share a compute unit).
// Every thread of the workgroup must call it (it contains a barrier).
// The row's result goes to hand[row], the extra row's to hand[extra_slot] (of both sides' copies); it is returned as well (lane 32), with the row in `done`
// (-1: this wave has none).
WD_DEV float router_rows_wave(const float *__restrict__ w, const float *__restrict__ x, float *xs, uint32_t *hand, int hand_side, int rows,
                              int cols, const float *__restrict__ extra_w, int extra_slot, int wg, int &done) {
    const int lane = threadIdx.x & 63, t = lane & 31;
    const bool upper = lane >= 32;
    const int row = wg * static_cast<int>(blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int total = rows + (extra_w ? 1 : 0);
    const bool on = row < total;
    const float *wr = on ? (row < rows ? w + static_cast<size_t>(row) * cols : extra_w) : x;
    wr = uniform_ptr(wr);  // the row is the same for the whole wave (two vector registers fewer)
    const RouterX rx(x, cols);
    float wv[32], xv[32];
    router_span_load(wr, 0, RouterSpan(cols), upper, t, wv);  // (a wave without a row: from x; behind a branch x would be waited for with everything else)
    rx.stage(x, xs, cols);
    __syncthreads();
    float s = 0.0f;  // the chain value; valid in the half that ran last
    if (on) {
        for (int i0 = 0; i0 < cols; i0 += 2048) {
            const RouterSpan sp(cols - i0);
            if (i0 > 0) router_span_load(wr, i0, sp, upper, t, wv);
            if (!upper || sp.upper > 0) router_span_x(xs + i0 + t + (upper ? 1024 : 0), sp, upper, xv);
            // the lower half advances the chain (from the upper half's value of the previous span) ...
            const wd_uint2v back = __builtin_amdgcn_permlane32_swap(f_bits(s), f_bits(s), false, false);
            if (!upper) s = router_span_run(wv, xv, sp.lower, i0 == 0 ? 0.0f : bits_f(back.y));
            // ... and the upper half continues from its result
            const wd_uint2v fwd = __builtin_amdgcn_permlane32_swap(f_bits(s), f_bits(s), false, false);
            if (upper) s = router_span_run(wv, xv, sp.upper, bits_f(fwd.x));
        }
    }
    // the 32 accumulators are final in the upper half (lanes 32..63): ggml's closing tree
    const float acc = router_close32(s);
    done = on ? (row < rows ? row : extra_slot) : -1;
    if (on) router_hand_on(acc, hand, hand_side, done, lane);
    return acc;
}

// The same for rows of 2049..4096 columns, two waves per row: wave 2 w takes the first 2048 columns of row (4 wg + w),
// wave 2 w + 1 the rest, both with every load of theirs in flight from the start - one trip to memory instead of one per
// span.  The chains still see their columns in ascending order: the second wave starts from the 32 accumulators the
// first one leaves in LDS (`over`: 4 x 32 floats).  Every thread of the (512-thread) workgroup must call it.
WD_DEV float router_rows_wave_pair(const float *__restrict__ w, const float *__restrict__ x, float *xs, float *over, uint32_t *hand, int hand_side,
                                   int rows, int cols, const float *__restrict__ extra_w, int extra_slot, int wg, int &done) {
    const int lane = threadIdx.x & 63, t = lane & 31, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const bool upper = lane >= 32, second = (wave & 1) != 0;
    const int row = wg * 4 + (wave >> 1);
    const int total = rows + (extra_w ? 1 : 0);
    const bool on = row < total;
    const float *wr = on ? (row < rows ? w + static_cast<size_t>(row) * cols : extra_w) : x;
    wr = uniform_ptr(wr);
    const int c0 = second ? 2048 : 0;
    const RouterSpan sp(cols - c0);
    const RouterX rx(x, cols);
    float wv[32], xv[32];
    router_span_load(wr, c0, sp, upper, t, wv);
    rx.stage(x, xs, cols);
    __syncthreads();
    if (!upper || sp.upper > 0) router_span_x(xs + c0 + t + (upper ? 1024 : 0), sp, upper, xv);
    // one copy of the chain code for both waves of a pair: turn 0 is the first wave's, turn 1 the second's
    float s = 0.0f;
#pragma unroll 1
    for (int turn = 0; turn < 2; ++turn) {
        if (second == (turn == 1)) {
            const float start = s;
            if (on && !upper) s = router_span_run(wv, xv, sp.lower, start);
            const wd_uint2v fwd = __builtin_amdgcn_permlane32_swap(f_bits(s), f_bits(s), false, false);
            if (upper) s = on ? router_span_run(wv, xv, sp.upper, bits_f(fwd.x)) : bits_f(fwd.x);
        }
        if (turn == 0) {
            if (!second && upper) over[(wave >> 1) * 32 + t] = s;
            __syncthreads();
            if (second) s = over[(wave >> 1) * 32 + t];
        }
    }
    done = -1;
    if (!second) return 0.0f;
    // the 32 accumulators are final in the upper half (lanes 32..63): ggml's closing tree
    const float acc = router_close32(s);
    done = on ? (row < rows ? row : extra_slot) : -1;
    if (on) router_hand_on(acc, hand, hand_side, done, lane);
    return acc;
}

// ---- dispatch AB ------------------------------------------------------------------------------------------
// n_router_wgs workgroups for the router rows, one that selects the experts and publishes the ids,
// then n_shared_wgs workgroups for the shared expert's gate/up; the rest for the routed gate/up, one (expert rung,
// group of eight rows) item each: a (gate, up) row pair per wave.  The routed workgroups are dispatched after the router
// ones (lower block index first), quantise x and stage the codebooks while the router runs, then poll the published ids;
// as soon as these appear they request their weights.  This removes a launch, a round trip for the ids and the serial
// activation set-up from the critical path of the layer.  Where the ids are known before the launch (ids_known: a routing
// trace, or a selection that is in the scratch) nothing is waited for and the weights are requested ahead of the set-up.
//
// Hand-off to the selecting workgroup: see hand_gather; no cache-wide release/acquire is needed for 2 KB of data.
//
// Publication: id j goes, as one 32-bit word, to ids_tagged[c][j] of every replica c with a device-scope atomic
// store; a word other than kTagInvalid is the id itself, so a reader needs no second flag.  The words are reset
// to kTagInvalid by dispatch C (or by the caller) before the next layer pass uses them.  The wait is bounded:
// when it runs out the workgroup sets status[0] and returns.
//
// TYPE: gate/up tensor type (21 IQ3_S, 22 IQ2_S, 8 Q8_0, 20 IQ4_NL).
// FETCH: how rows come in, and with it how the router's rows are taken:
//   8   IQ rows of eight super-blocks on 16-byte boundaries (hidden 2048): one aligned 16-byte load per lane (iq_rows8_coal)
//   10  IQ rows of ten (hidden 2560): iq_rows10_coal
//   1   other hidden up to 2048: IQ rows as the 16-byte words that cover them, one load per lane (iq_rows_cover)
//   2   hidden 2049..4096: the same with two loads per lane
//   0   anything else (hidden beyond 4096, IQ tensors that do not start on 16-byte boundaries): fields loaded one by one
//   Router rows of 2049..4096 columns take two waves each (10 and 2: at hidden 4096 a row by one wave, two dependent trips
//   to memory, took 8.7 us of the dispatch, by two 3.3), others one.
// dynamic LDS: the larger of 4 * H + 16 bytes (x of the router rows) and the quantised x (H bytes + scales, layer_ab_stage)
// with the per-wave staging area of the IQ rows behind it (layer_ab_stage_bytes).
// LOOP: the grid has fewer routed workgroups than there are items; they walk them with the stride of their number.
__host__ __device__ inline uint32_t layer_ab_stage(int H) { return static_cast<uint32_t>(H + H / 16 + 15) & ~15u; }
template <int TYPE, int FETCH>
constexpr bool kAbIq = (TYPE == 21 || TYPE == 22);
template <int TYPE, int FETCH>
__host__ __device__ inline uint32_t layer_ab_stage_bytes(int H) {  // per wave
    if (!kAbIq<TYPE, FETCH> || FETCH == 0) return 0;
    if (FETCH == 8) return 2 * kIqStageBytes;
    if (FETCH == 10) return 2 * kIqStage10Bytes;
    return 2 * iq_cover_bytes<TYPE>(H >> 8);
}

// Workgroups per compute unit: three.  (Two for the rows taken field by field: Q8_0, hidden 5120 / ffn 1024, top-8 and the shared
// expert 49.5 us against 40.6; IQ4_NL 43.7 against 36.4; IQ2_S 35.7 against 30.6.)  The loop over IQ3_S rows taken field by field
// does not fit 80 registers - 22 are spilled - and runs two (hidden 4096 / ffn 1536, top-8: 32.5 us against 44.9).
template <int TYPE, int FETCH, bool LOOP>
constexpr int kAbPerCu = TYPE == 21 && FETCH == 0 && LOOP ? 2 : 3;
template <int TYPE, int FETCH, bool LOOP = false, bool PART = false, bool TRACE = false>
__global__ __launch_bounds__(512, (2 * kAbPerCu<TYPE, FETCH, LOOP>)) void k_layer_ab(LayerArgs a) {
    constexpr bool kIq = kAbIq<TYPE, FETCH>, kWide = FETCH == 10 || FETCH == 2;
    constexpr bool kTwoPasses = kWide;  // Q8_0 rows of 65..128 blocks
    constexpr int kIqType = kIq ? TYPE : 21;
    extern __shared__ __align__(16) uint8_t lds_ab[];
    __shared__ __align__(16) uint8_t s_union[sizeof(Q8RowTile) * 8 > sizeof(IqTables) ? sizeof(Q8RowTile) * 8 : sizeof(IqTables)];
    __shared__ int s_last;  // (hand_close)
    const int blk = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (a.dry) return;
    const int groups = (a.F + 7) / 8;
    // (known where the fetch is made for it: 56 registers instead of 80 at 2048 without the loop, 73 and none spilled with it.  us per layer from
    // HBM, unknown / known: 2048 / 512 19.61 / 19.48, 2048 / 768 20.20 / 20.14, IQ2_S 19.05 / 18.97, 2560 / 640 24.72 / 24.61, IQ2_S 23.16 / 23.20)
    const int H = FETCH == 8 ? 2048 : (FETCH == 10 ? 2560 : a.H);

    mark<TRACE>(a, blk < a.n_select_wgs + a.n_router_wgs + a.n_shared_wgs ? 0 : 1, 0);
    if (blk < a.n_router_wgs) {
        const int rows = a.preselected ? 0 : a.E;
        int row;
        float logit;
        if (kWide)  // two waves per row, four rows per workgroup (the host sizes the grid for it)
            logit = router_rows_wave_pair(a.router, a.x, reinterpret_cast<float *>(lds_ab), reinterpret_cast<float *>(s_union), a.hand, a.hand_side, rows, H,
                                          a.sh_inp, a.E, blk, row);
        else
            logit = router_rows_wave(a.router, a.x, reinterpret_cast<float *>(lds_ab), a.hand, a.hand_side, rows, H, a.sh_inp, a.E, blk, row);
        mark<TRACE>(a, 0, 1);
        if (lane == 32 && row >= 0 && row < rows) a.logits[row] = logit;  // (the caller's view)
        // (no selection: the one wave with the shared gate's row)
        if (a.preselected && row == a.E && lane == 32) a.shared_gate[0] = sigmoid_ggml(bits_f(hand_word_bits(f_bits(logit))));
        mark<TRACE>(a, 0, 2);
        if (a.close_hand) hand_close(a.hand, a.hand_side, a.E, a.n_select_wgs + a.n_router_wgs, s_last);
        return;
    }
    if (blk < a.n_router_wgs + a.n_select_wgs) {
        // results land behind the selection's own scratch
        static_assert(sizeof(s_union) >= kTopkLdsBytes2 + 128, "selection scratch, ids and weights must fit the shared area");
        int32_t *lds_ids = reinterpret_cast<int32_t *>(s_union + kTopkLdsBytes2);
        float *lds_w = reinterpret_cast<float *>(s_union + kTopkLdsBytes2 + 64);
        if (wave == 0) __builtin_amdgcn_s_setprio(3);
        if (TRACE && a.trace && threadIdx.x == 0) a.trace[(0 * 16 + 8) * 8 + 0] = wall_clock64();
        // the selection itself publishes the replicas that the routed workgroups wait for, ahead of the weights
        const uint32_t *const hand = hand_copy(a.hand, a.hand_side);
        const bool there = topk_block(HandRow{hand, a.E, a.E, a.sh_inp != nullptr, a.hand_limit}, a.k, a.w_scale, lds_ids, lds_w, a.ids_override, s_union, lane, wave,
                                      (TRACE && a.trace) ? a.trace + (0 * 16 + 9) * 8 : nullptr, a.ids_known ? nullptr : a.ids_tagged, a.tag_side);
        if (!there && lane == 0) __hip_atomic_store(a.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // off the selection's path: the shared expert's gate
        if (a.sh_inp && wave == 5 && lane == 0) a.shared_gate[0] = sigmoid_ggml(bits_f(hand_load(hand + a.E)));
        if (wave == 0) {
            wave_lds_fence();
            // the plain copies for dispatch C
            if (lane < a.k) {
                a.ids[lane] = lds_ids[lane];
                a.weights[lane] = lds_w[lane];
                if (a.host_ids) __hip_atomic_store(a.host_ids + lane, static_cast<uint32_t>(lds_ids[lane]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
            if (TRACE && a.trace && lane == 0) a.trace[(0 * 16 + 8) * 8 + 1] = wall_clock64();
        }
        mark<TRACE>(a, 0, 2);
        if (a.close_hand) hand_close(a.hand, a.hand_side, a.E, a.n_select_wgs + a.n_router_wgs, s_last);
        return;
    }
    const int wg = blk - a.n_select_wgs;

    int8_t *xq = reinterpret_cast<int8_t *>(lds_ab);
    uint8_t *xscale = lds_ab + H;  // Q8_K: f32 [H/256]; Q8_0: f16 [H/32]
    if (wg < a.n_router_wgs + a.n_shared_wgs) {
        Q8RowTile *tiles = reinterpret_cast<Q8RowTile *>(s_union);
        const int r = (wg - a.n_router_wgs) * 8 + wave;
        const int nb = H >> 5;
        const size_t rb = static_cast<size_t>(nb) * 34;
        const size_t off = static_cast<size_t>(min(r, a.F - 1)) * rb;
        const uint8_t *const rows[2] = {uniform_ptr(a.sh_gate + off), uniform_ptr(a.sh_up + off)};  // one row pair per wave
        float gu[2];
        q8_row_pair<0, kTwoPasses>(rows, nb, xq, reinterpret_cast<const uint16_t *>(xscale), tiles[wave], lane, gu, [&]() {
            lds_quantize_q8_0(a.x, H, xq, reinterpret_cast<uint16_t *>(xscale), threadIdx.x, 512);
            __syncthreads();
        });
        if (lane == 0 && r < a.F) a.act[static_cast<size_t>(a.k) * a.F + r] = silu_ggml(gu[0]) * gu[1];
        return;
    }

    // routed gate/up
    const int bw = wg - a.n_router_wgs - a.n_shared_wgs;
    IqTables &tables = *reinterpret_cast<IqTables *>(s_union);
    auto set_up = [&]() {  // what does not need the ids
        if (kIq) {
            stage_tables<TYPE == 21, TYPE == 22>(tables, threadIdx.x, 512);
            for (int b = wave; b < (H >> 8); b += 8)
                wave_quantize_q8_k_block(a.x + b * 256, xq + b * 256, reinterpret_cast<float *>(xscale) + b, lane);
        } else {
            lds_quantize_q8_0(a.x, H, xq, reinterpret_cast<uint16_t *>(xscale), threadIdx.x, 512);
        }
        mark<TRACE>(a, 1, 1);
    };
    __shared__ int s_expert;
    const int n_routed_wgs = LOOP ? static_cast<int>(gridDim.x) - a.n_select_wgs - a.n_router_wgs - a.n_shared_wgs : 0;
    // With known ids the set-up is done behind the requests of the first item (the variants named here have no registers
    // to hold these meanwhile).
    constexpr bool kBehind = FETCH != 0 && !(TYPE == 8 && LOOP);
    bool pending = true;
    if (!kBehind || !a.ids_known) {
        set_up();
        pending = false;
    }
    auto wait_for_id = [&](int j) {
        const uint32_t *src = tag_copy(a.ids_tagged, a.tag_side, bw) + j;
        uint32_t id = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        unsigned polls = 0;
        while (id == kTagInvalid && ++polls < a.spin_limit) {
            __builtin_amdgcn_s_sleep(4);
            id = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (id == kTagInvalid) __hip_atomic_store(a.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return static_cast<int>(id);
    };
    // One item per workgroup unless the grid was capped (LOOP).  Behind the first one the waves go on by themselves: nothing of what they share is
    // written again, and the ids come together, so that each wave reads the next item's where it lies.  (Between two barriers an item begins when the slowest
    // wave of the one before is done: 4096 / 1536 IQ3_S, eight of 128 experts, 36.8 us per layer, so 36.0; 2560 / 640, where few workgroups have a second item, the same.)
    int item = bw;
    bool first = true;
    do {
        const int j = item / groups;
        const int rg = item - j * groups;
        int e;
        if (a.ids_known) {
            e = checked_expert(a.gate_up, sld_i32(a.ids_known + j));
            if (!kBehind && first) __syncthreads();
        } else if (LOOP && !first) {
            e = __builtin_amdgcn_readfirstlane(wait_for_id(j));
            if (e < 0 || e >= a.E) return;  // (as below)
        } else {
            if (threadIdx.x == 0) s_expert = wait_for_id(j);
            __syncthreads();
            e = s_expert;
            if (e < 0 || e >= a.E) return;  // the wait ran out (status is set): leave without touching memory
        }
        mark<TRACE>(a, 1, 2);
        const uint8_t *gate = mat_ptr_expert<0>(a.gate_up, e);
        const uint8_t *up = mat_ptr_expert<1>(a.gate_up, e);
        float *act = a.act + static_cast<size_t>(j) * a.F;
        const int r = rg * 8 + wave;
        auto pre = [&]() {
            if (kBehind && pending) {
                set_up();
                __syncthreads();
                pending = false;
            }
        };
        float gu[2];
        if (kIq) {
            const int nb = H >> 8;
            const size_t rb = static_cast<size_t>(nb) * (TYPE == 21 ? 110 : 82);
            const size_t off = static_cast<size_t>(min(r, a.F - 1)) * rb;
            const uint8_t *const rows[2] = {uniform_ptr(gate + off), uniform_ptr(up + off)};  // one row pair per wave
            // (PART) the chunk sums of the pair: gate row r of rung j, the up row F rows further on
            const size_t pg = static_cast<size_t>(nb) * 8;
            int32_t *pp = PART ? a.gup_part + (static_cast<size_t>(j) * 2 * a.F + min(r, a.F - 1)) * pg : nullptr;
            uint8_t *const stage = lds_ab + layer_ab_stage(H) + wave * layer_ab_stage_bytes<TYPE, FETCH>(H);
            const float *xd = reinterpret_cast<const float *>(xscale);
            if (FETCH == 10)
                iq_rows10_coal<kIqType, 2, PART>(rows, tables, xq, xd, lane, gu, stage, pp, a.F * pg, pre);
            else if (FETCH == 8)
                iq_rows8_coal<kIqType, 2, PART>(rows, tables, xq, xd, lane, gu, stage, pp, a.F * pg, pre);
            else if (FETCH != 0)
                iq_rows_cover<kIqType, 2, FETCH == 0 ? 1 : (FETCH > 2 ? 2 : FETCH), PART>(rows, nb, tables, xq, xd, lane, gu, stage, pp, a.F * pg, pre);
            else
                iq_rows_q8k<kIqType, 2, PART>(rows, nb, tables, xq, xd, lane, gu, pp, a.F * pg, pre);
        } else {
            Q8RowTile *tiles = reinterpret_cast<Q8RowTile *>(s_union);
            const int nb = H >> 5;
            const size_t rb = static_cast<size_t>(nb) * (TYPE == 8 ? 34 : 18);
            const size_t off = static_cast<size_t>(min(r, a.F - 1)) * rb;
            const uint8_t *const rows[2] = {uniform_ptr(gate + off), uniform_ptr(up + off)};
            q8_row_pair<(TYPE == 8 ? 0 : 1), kTwoPasses>(rows, nb, xq, reinterpret_cast<const uint16_t *>(xscale), tiles[wave], lane, gu, pre);
        }
        if (lane == 0 && r < a.F) act[r] = silu_ggml(gu[0]) * gu[1];
        mark<TRACE>(a, 1, 3);
        if (LOOP) {
            item += n_routed_wgs;
            first = false;
            wave_lds_fence();  // (the wave's staging is written again)
        }
    } while (LOOP && item < a.n_routed_items);
}

// (workgroup 0 of dispatch C) The words of this layer pass are done with: ids published, logits handed on.
WD_DEV void layer_clear_handed(const LayerArgs &a, int threads) {
    if (!a.clear_tagged || blockIdx.x != 0) return;
    for (int i = threadIdx.x; i < kTagCopies * 8; i += threads) {
        __hip_atomic_store(a.ids_tagged + i, kTagInvalid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(a.ids_tagged + a.tag_side + i, kTagInvalid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    hand_clear(a.hand, a.hand_side, a.E + 1, static_cast<int>(threadIdx.x), threads);
}

// ---- the combine at the end of dispatch C ---------------------------------------------------------------------
// The operands of one wave's four rows, requested when the dispatch begins: lane m keeps router weight m, lane 16 the shared
// gate; the residual values that the rows' owner updates at its end (nothing else writes them meanwhile): lane 4c + r
// holds stream c of row r0 + r.
struct FoldOps {
    float w = 0.0f, res = 0.0f, stream_w = 0.0f;
    unsigned bad = 0u;  // a bounded wait of this layer pass ran out: the results below are replaced by NaN
};
// What the weight of the lane's residual stream is made of, asked for ahead of the dispatch's weights so that it can be
// worked out (layer_c_stream_weight) while these are on their way and not behind the last barrier.  (2560 / 640, ten Q8_0 experts and the shared one, four streams:
// 23.9 us per layer behind it, so 23.0.)
struct StreamOps {
    float inject = 0.0f;
    uint64_t entry = 0u;
};
WD_DEV StreamOps layer_c_stream_request(const LayerArgs &a, bool folds, int lane) {
    StreamOps s;
    if (folds && a.hc > 0) s.inject = a.hc_inject[min(lane >> 2, a.hc - 1)], s.entry = exp2f_entry(lane);
    return s;
}
WD_DEV float layer_c_stream_weight(const LayerArgs &a, const StreamOps &s, bool folds) {
    float w = 0.0f;
    if (folds && a.hc > 0) {
        w = hc_weight_of_wave(s.inject, a.hc, s.entry);
        asm volatile("" : "+v"(w));  // (here and not where it is used)
    }
    return w;
}
WD_DEV FoldOps layer_c_fold_request(const LayerArgs &a, int r0, int nrows, int lane) {
    FoldOps o;
    o.bad = __hip_atomic_load(a.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (lane < a.k) o.w = a.weights[lane];
    if (lane == 16 && a.sh_inp) o.w = a.shared_gate[0];
    if (a.residual) {
        const int c = a.hc > 0 ? min(lane >> 2, a.hc - 1) : 0;
        o.res = a.residual[static_cast<size_t>(c) * a.H + r0 + min(lane & 3, nrows - 1)];
    }
    return o;
}
// The weighted sum in order over k <= 16 matrices: y[m * STRIDE] is matrix m's result (memory up to y[15 * STRIDE]), lane m of w its weight.  Behind the
// last barrier of a dispatch a single wave runs it: results are requested from LDS eight at once, weights are lane reads, and in the
// last four terms what has no matrix adds -0.0, which leaves every sum as it is.  (A loop that reads term and weight through LDS when it
// needs them: a layer of 1024 / 256, six of 64 experts and the shared one, 11.09 us, so 10.87.)
template <int STRIDE>
WD_DEV float fold_in_order(const float *y, float w, int k) {
    float acc = 0.0f;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        if (half == 1 && k <= 8) break;
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = y[(8 * half + u) * STRIDE];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int m = 8 * half + 4 * q;
            if (m + 4 <= k) {
#pragma unroll
                for (int u = 0; u < 4; ++u) acc = acc + v[4 * q + u] * readlane_f(w, m + u);
            } else if (m < k) {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float prod = v[4 * q + u] * readlane_f(w, m + u);
                    acc = acc + (m + u < k ? prod : -0.0f);
                }
            }
        }
    }
    return acc;
}
// A dispatch C's dynamic LDS: the results ([n_act][stride] floats) and behind them what its waves own; at least as much as fold_in_order
// reads, which is up to fifteen matrices past the last one's.
constexpr size_t layer_c_lds(size_t n_act, size_t stride, size_t of_waves) {
    const size_t results = 4 * n_act * stride, read = 4 * (n_act + 15) * stride;
    return results + of_waves > read ? results + of_waves : read;
}
// Rows r0 .. r0 + nrows - 1 (at most four): matrix m's result for row r0 + q at ybuf[m * STRIDE + q].  One wave.
template <int STRIDE>
WD_DEV void layer_c_fold(const LayerArgs &a, const FoldOps &ops, const float *ybuf, int r0, int nrows, int lane) {
    const bool shared = a.sh_inp != nullptr;
    // every lane folds row r0 + (lane & 3); lanes 0..3 store it
    const int row = r0 + lane;
    const bool on = lane < nrows;
    const float *const mine = ybuf + (lane & 3);
    const float y_shared = shared ? mine[a.k * STRIDE] : 0.0f;
    float acc = fold_in_order<STRIDE>(mine, ops.w, a.k);
    float o = acc;
    if (shared) {
        const float prod = y_shared * readlane_f(ops.w, 16);
        o = acc + prod;
    }
    if (ops.bad) acc = o = __builtin_nanf("");  // the caller sees the failure in its data, without a synchronisation
    // (The order counts where a caller passed one buffer twice: the output over any view of the scratch, the residual over the output.)
    if (on) {
        if (a.expert_out)
            for (int m = 0; m < a.k; ++m) a.expert_out[static_cast<size_t>(m) * a.H + row] = mine[m * STRIDE];
        if (shared) a.down_f32[row] = y_shared;
        a.accum[row] = acc;
        a.out[row] = o;
    }
    if (a.residual) {
        if (a.hc > 0) {
            const int c = lane >> 2;
            if (c < a.hc && (lane & 3) < nrows) {
                const float weighted = o * ops.stream_w;
                const float v = ops.res + weighted;
                a.residual[static_cast<size_t>(c) * a.H + r0 + (lane & 3)] = a.hc_round_half ? round_half(v) : v;
            }
        } else if (on) {
            const float scaled = o * a.residual_scale;
            a.residual[row] = ops.res + scaled;
        }
    }
}
// What a wave's matrix gives: NaN for an expert that has no slot (reported through the status word), so that every sum it goes into is one.
WD_DEV float or_nan(float y, bool missing) { return missing ? __builtin_nanf("") : y; }

// ---- dispatch C -----------------------------------------------------------------------------------------
// All down projections of a few output rows per workgroup, a wave per matrix (the k routed down tensors, then the shared
// one); each wave re-quantises the activation of its own matrix while its weights are in flight, and the first waves then
// fold the results in the reference order (layer_c_fold).
// KIND: down tensor kind (0 Q8_0, 1 IQ4_NL); the shared expert's is always Q8_0.
//
// k_layer_c: four rows, pass by pass: rows of any length, any number of matrices (waves take the matrices in turn).
// grid = ceil(H / 4), block = 64 * min(n_act, 16) with n_act = k + 1 matrices (k without the shared expert).
// dynamic LDS (layer_c_lds): [n_act][4] floats, then per wave F bytes + F/32 halves (+ pad).
template <int KIND, bool PART = false, bool TRACE = false>
__global__ __launch_bounds__(1024) void k_layer_c(LayerArgs a) {
    extern __shared__ __align__(16) uint8_t lds_c[];
    __shared__ Q8Tile tiles[16];
    const int n_act = a.k + (a.sh_inp ? 1 : 0);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nwaves = blockDim.x >> 6;
    const size_t per_wave = (static_cast<size_t>(a.F) + a.F / 16 + 15) & ~static_cast<size_t>(15);
    float *ybuf = reinterpret_cast<float *>(lds_c);  // [n_act][4]
    int8_t *aq = reinterpret_cast<int8_t *>(lds_c + 16 * n_act + wave * per_wave);
    uint16_t *ad = reinterpret_cast<uint16_t *>(aq + a.F);
    const int r0 = blockIdx.x * 4;
    const int nrows = min(4, a.H - r0);
    const int nb = a.F >> 5;
    if (a.dry) return;
    // every routed workgroup of this layer pass finished with the previous dispatch: make the ids published
    // for them invalid again (this dispatch reads the plain copy)
    layer_clear_handed(a, blockDim.x);
    mark<TRACE>(a, 2, 0);
    const StreamOps stream = layer_c_stream_request(a, wave == 0, lane);
    FoldOps ops;
    if (wave == 0) ops = layer_c_fold_request(a, r0, nrows, lane);
    ops.stream_w = layer_c_stream_weight(a, stream, wave == 0);
    for (int m = wave; m < n_act; m += nwaves) {
        const bool is_shared = m == a.k;
        // m is the same for the whole wave: the id comes through the scalar path
        bool missing = false;
        const uint8_t *const w = is_shared ? a.sh_down : mat_ptr_expert_uniform<0>(a.down, checked_expert(a.down, sld_i32(a.ids + m)), missing);
        const bool q8 = KIND == 0 || is_shared;  // the same in every lane
        const uint8_t *const rows = w + static_cast<size_t>(r0) * nb * (q8 ? 34 : 18);
        auto quantise = [&]() {
            wave_lds_fence();
            lds_quantize_q8_0(a.act + static_cast<size_t>(m) * a.F, a.F, aq, ad, lane, 64);
            wave_lds_fence();
            mark<TRACE>(a, 2, 1);
        };
        int32_t *pp = (PART && !is_shared) ? a.down_part + (static_cast<size_t>(m) * a.H + r0) * (static_cast<size_t>(nb) * 8) : nullptr;
        float y;
        if (PART && !is_shared) y = q8_rows4<KIND, true>(rows, nrows, nb, aq, ad, tiles[wave], lane, pp, quantise);
        else if (q8) y = q8_rows4<0, false>(rows, nrows, nb, aq, ad, tiles[wave], lane, nullptr, quantise);
        else y = q8_rows4<KIND, false>(rows, nrows, nb, aq, ad, tiles[wave], lane, nullptr, quantise);
        if ((lane & 15) == 0) ybuf[m * 4 + (lane >> 4)] = or_nan(y, missing);
        mark<TRACE>(a, 2, 2);
    }
    __syncthreads();
    mark<TRACE>(a, 2, 3);
    if (wave == 0) layer_c_fold<4>(a, ops, ybuf, r0, nrows, lane);
    mark<TRACE>(a, 2, 4);
}

// k_layer_c8: eight rows per workgroup and wave: half the waves to launch, half the activations to quantise and, per 64
// blocks, half the chain steps of the four-row form; all bytes of the eight rows are requested at once, behind the activation.
// PASSES: of eight blocks per row (F <= 256 PASSES).  grid = H / 8, block = 64 max(n_act, 2) with at most 16 matrices; waves 0
// and 1 fold four rows each.  (Hidden 4096, eight experts with rows of 48 Q8_0 blocks, 53.5 MB: 25.7 us in the four-row form
// with two matrices per wave, 16.1 so, 14.7 with WORDS - the bytes alone take 9 -; hidden 2560, ten IQ4_NL experts of 20
// blocks and the shared one: 11.8, 10.1; hidden 2048, eight Q8_0 experts of 24: 8.9, 6.8; hidden 2048, ten of 16 and the shared one:
// 6.7, 6.4 with part of the weights in the last-level cache, 6.7, 6.9 with all of them from HBM.)
// TWO: seventeen matrices (top-16 and the shared expert), nine waves with two each, one after the other: rows of 9..24 blocks.
// (Hidden 2560, rows of 20 Q8_0 blocks: 13.2 us, in the four-row form with sixteen waves 20.5, here with sixteen 14.8; hidden 2048,
// 16 blocks: 7.8, 9.7, 7.9; hidden 1024, eight blocks: 6.1, 5.6.)
// WORDS: the rows come through LDS as aligned words (Q8Rows8Fetch), otherwise a lane loads its own blocks (Q8Rows8Blocks).
// dynamic LDS (layer_c_lds): [n_act][8] floats, then per wave the tile (WORDS: the staging area, which it lies in) and the quantised
// activation (F bytes + F/32 halves, padded).
template <bool WORDS>
__host__ __device__ inline uint32_t layer_c8_wave_bytes(int F) {
    static_assert(sizeof(Q8Tile8) <= kQ8Rows8StageBytes, "the tile lies in the staging area");
    return (WORDS ? kQ8Rows8StageBytes : static_cast<uint32_t>(sizeof(Q8Tile8))) + (static_cast<uint32_t>(F + F / 16 + 15) & ~15u);
}
// Registers: grids of more than 256 workgroups (hidden beyond 2048) want two on a compute unit, which with nine to twelve waves each takes six waves per SIMD, so
// at most 80 registers.  Rows of 25..32 blocks that a lane loads itself stay below by asking for what the fold needs behind the quantisation
// (kLate; eleven IQ4_NL matrices, 5120 / 1024: 46.2 us per layer with 83 registers, 42.8 with 78); two matrices per wave of 17..24 blocks by the
// general quantisation (ORDINARY false: 5120 / 768 IQ4_NL 53.2 with 87, 50.7 with 79; where one workgroup per compute unit is all there is, 2048 / 768, the
// ordinary one is the faster, 22.3 against 23.1).  Thirteen to sixteen matrices of 17..24 blocks need eight waves per SIMD, 64 registers: the general quantisation, and
// what the fold needs asked for behind the chains (kLast; us of the dispatch at 5120 / 768 with 73 registers, asked for behind the quantisation with 70, so: thirteen IQ4_NL
// 14.3, 15.5, 12.0, sixteen 16.2, 17.4, 13.8; Q8_0, 73, 60 and 60 registers, 15.5, 13.7, 13.7 and 18.8, 17.0, 17.1).
template <int KIND, int PASSES, bool WORDS, bool PART = false, bool TRACE = false, bool TWO = false, bool ORDINARY = true>
__global__ __launch_bounds__(TWO ? 576 : 1024, TWO ? (ORDINARY ? 1 : 6) : !ORDINARY ? 8 : PASSES == 4 && !WORDS && !PART && !TRACE ? 6 : 1) void k_layer_c8(LayerArgs a) {
    constexpr int STEPS = (PASSES + 1) / 2;  // of sixteen blocks
    constexpr bool kLast = !TWO && !ORDINARY, kLate = (PASSES == 4 && !WORDS) || kLast;
    extern __shared__ __align__(16) uint8_t lds_c8[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int n_act = a.k + (a.sh_inp ? 1 : 0);
    const uint32_t per_wave = layer_c8_wave_bytes<WORDS>(a.F);
    float *ybuf = reinterpret_cast<float *>(lds_c8);
    uint8_t *stage = lds_c8 + 32 * n_act + wave * per_wave;
    Q8Tile8 &tile = *reinterpret_cast<Q8Tile8 *>(stage);
    int8_t *aq = reinterpret_cast<int8_t *>(stage + (WORDS ? kQ8Rows8StageBytes : sizeof(Q8Tile8)));
    uint16_t *ad = reinterpret_cast<uint16_t *>(aq + a.F);
    const int r0 = blockIdx.x * 8, nb = a.F >> 5;
    if (a.dry) return;
    layer_clear_handed(a, 64 * (TWO ? 9 : n_act));
    mark<TRACE>(a, 2, 0);
    StreamOps stream;
    if (!kLast) stream = layer_c_stream_request(a, wave < 2, lane);
    FoldOps ops;
    float stream_w = 0.0f;
    int m = TWO ? wave : min(wave, n_act - 1);  // (a second wave without a matrix of its own repeats the first's)
    do {
        int lane = threadIdx.x & 63;
        if constexpr (TWO || kLast) asm volatile("" : "+v"(lane));  // (nothing per lane is kept from one matrix to the next: it would take 30 registers)
        const bool is_shared = m == a.k, q8 = KIND == 0 || is_shared;
        // the activation first: its address needs no expert id, and loads return in order - it is quantised while the weights are
        // still on their way
        float4 v[2 * STEPS];
#pragma unroll
        for (int i = 0; i < STEPS; ++i) {
            const float *p = a.act + static_cast<size_t>(m) * a.F + min(512 * i + lane * 8, a.F - 8);
            v[2 * i] = *reinterpret_cast<const float4 *>(p), v[2 * i + 1] = *reinterpret_cast<const float4 *>(p + 4);
        }
        bool missing = false;
        const uint8_t *const rows = uniform_ptr((is_shared ? a.sh_down : mat_ptr_expert_uniform<0>(a.down, checked_expert(a.down, sld_i32(a.ids + m)), missing)) +
                                                static_cast<size_t>(r0) * nb * (q8 ? 34 : 18));
        auto run = [&](auto kind, auto part) {
            constexpr int K = decltype(kind)::value;
            constexpr bool P = decltype(part)::value;
            typename std::conditional<WORDS, Q8Rows8Fetch<K, STEPS>, Q8Rows8Blocks<K, PASSES>>::type fetch;
            fetch.request(rows, nb, lane);
            if (!kLate && wave < 2 && (!TWO || m < 9)) ops = layer_c_fold_request(a, r0 + 4 * wave, 4, lane);
            if (kLate && !kLast) stream_w = layer_c_stream_weight(a, stream, wave < 2);
#pragma unroll
            for (int i = 0; i < STEPS; ++i)
                lds_quantize_q8_0_step<ORDINARY>(v[2 * i], v[2 * i + 1], 512 * i + lane * 8 < a.F, 512 * i + lane * 8, aq, ad, lane);
            if (kLate && !kLast && wave < 2) ops = layer_c_fold_request(a, r0 + 4 * wave, 4, lane);
            if (!kLate && (!TWO || m < 9)) stream_w = layer_c_stream_weight(a, stream, wave < 2);
            mark<TRACE>(a, 2, 1);
            Q8Chain ch;
            int32_t *pp = P ? a.down_part + (static_cast<size_t>(m) * a.H + r0) * (static_cast<size_t>(nb) * 8) : nullptr;
#pragma unroll
            for (int q = 0; q < STEPS; ++q) {
                Q8Block w0, w1;
                if constexpr (WORDS) {
                    wave_lds_fence();  // the step before has been read
                    fetch.park(q, stage, lane);
                    wave_lds_fence();
                    // (both blocks of the step before the first pass: its tile takes the parked words' place)
                    w0 = q8_rows8_block<K>(stage, nb, lane >> 3, lane & 7), w1 = q8_rows8_block<K>(stage, nb, lane >> 3, 8 + (lane & 7));
                } else {
                    if (q == 0) wave_lds_fence();
                    w0 = fetch.w[2 * q], w1 = fetch.w[min(2 * q + 1, PASSES - 1)];
                }
                q8_rows8_pass<K, P>(w0, 16 * q, nb, aq, ad, tile, lane, ch, pp);
                if (2 * q + 1 < PASSES && 16 * q + 8 < nb) q8_rows8_pass<K, P>(w1, 16 * q + 8, nb, aq, ad, tile, lane, ch, pp);
            }
            return q8_rows8_close<K>(ch, nb, tile, lane);
        };
        float y;
        if (PART && !is_shared) y = run(std::integral_constant<int, KIND>{}, std::integral_constant<bool, PART>{});
        else if (q8) y = run(std::integral_constant<int, 0>{}, std::false_type{});
        else y = run(std::integral_constant<int, KIND>{}, std::false_type{});
        if (wave < n_act && (lane & 7) == 0) ybuf[m * 8 + (lane >> 3)] = or_nan(y, missing);
        m += 9;
    } while (TWO && m < n_act);
    if (kLast) {
        stream = layer_c_stream_request(a, wave < 2, lane);
        if (wave < 2) ops = layer_c_fold_request(a, r0 + 4 * wave, 4, lane);
        stream_w = layer_c_stream_weight(a, stream, wave < 2);
    }
    mark<TRACE>(a, 2, 2);
    __syncthreads();
    mark<TRACE>(a, 2, 3);
    ops.stream_w = stream_w;
    if (wave < 2) layer_c_fold<8>(a, ops, ybuf + 4 * wave, r0 + 4 * wave, 4, lane);
    mark<TRACE>(a, 2, 4);
}

// k_layer_c_even: one workgroup for every compute unit, hidden / 256 rows each.  Eight rows per workgroup spread other hidden sizes
// than 2048 and 4096 unevenly: 2560 is 320 workgroups, two of them on 64 of the 256 compute units, and the dispatch takes as long
// as those (the second one of a compute unit has its activations quantised 4.3 us after its start, the others 1.9); 1024 leaves
// half of the compute units without work.  A wave takes its matrix's rows, up to 64 / LPR of them by lanes that hold one block
// each, or (GROUPS 2) two such groups one after the other: the second one's blocks are requested pass by pass, as the registers of
// the first one's are free (all of both at once: 2560 / 640 IQ4_NL 8.9 us, so 8.4; 3072 / 768 Q8_0 13.0, 12.4).  As two workgroups per
// compute unit the groups take 0.3 us more at 2560 and 2.5 more at 3072 / 1024.  (Figures: layer_c_evenly.)
// grid = 256, block = 64 max(n_act, 2 GROUPS) with at most 16 matrices; waves 0 .. 2 GROUPS - 1 fold up to four rows each.
// dynamic LDS (layer_c_lds): [n_act][16] floats, then per wave the tile and the quantised activation (layer_c_even_wave_bytes).
template <int LPR>
__host__ __device__ inline uint32_t layer_c_even_wave_bytes(int F) {
    return ((static_cast<uint32_t>(sizeof(Q8TileN<LPR>)) + 15) & ~15u) + (static_cast<uint32_t>(F + F / 16 + 15) & ~15u);
}
template <int KIND, int LPR, int GROUPS, int PASSES>
__global__ __launch_bounds__(1024) void k_layer_c_even(LayerArgs a) {
    constexpr int STEPS = LPR * PASSES <= 48 ? (LPR * PASSES + 15) / 16 : 3;  // of the activation
    constexpr bool kBoth = GROUPS == 2 && PASSES == 1, kThen = GROUPS == 2 && PASSES > 1;
    extern __shared__ __align__(16) uint8_t lds_ce[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int n_act = a.k + (a.sh_inp ? 1 : 0), n_waves = max(n_act, 2 * GROUPS);
    const uint32_t per_wave = layer_c_even_wave_bytes<LPR>(a.F);
    float *ybuf = reinterpret_cast<float *>(lds_ce);
    uint8_t *const mine = lds_ce + 64 * n_act + wave * per_wave;
    Q8TileN<LPR> &tile = *reinterpret_cast<Q8TileN<LPR> *>(mine);
    int8_t *aq = reinterpret_cast<int8_t *>(mine + ((sizeof(Q8TileN<LPR>) + 15) & ~15u));
    uint16_t *ad = reinterpret_cast<uint16_t *>(aq + a.F);
    const int R = a.H >> 8, r0 = blockIdx.x * R, nb = a.F >> 5;
    const int rows0 = GROUPS == 1 ? R : (R + 1) >> 1;
    if (a.dry) return;
    layer_clear_handed(a, 64 * n_waves);
    const StreamOps stream = layer_c_stream_request(a, 4 * wave < R, lane);
    FoldOps ops;
    float stream_w = 0.0f;
    const int m = min(wave, n_act - 1);  // (a wave without a matrix of its own repeats the last one's)
    const bool is_shared = m == a.k, q8 = KIND == 0 || is_shared;
    // (the activation first, as in k_layer_c8)
    float4 v[2 * STEPS];
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
        const float *p = a.act + static_cast<size_t>(m) * a.F + min(512 * i + lane * 8, a.F - 8);
        v[2 * i] = *reinterpret_cast<const float4 *>(p), v[2 * i + 1] = *reinterpret_cast<const float4 *>(p + 4);
    }
    bool missing = false;
    const uint8_t *const rows = uniform_ptr((is_shared ? a.sh_down : mat_ptr_expert_uniform<0>(a.down, checked_expert(a.down, sld_i32(a.ids + m)), missing)) +
                                            static_cast<size_t>(r0) * nb * (q8 ? 34 : 18));
    auto run = [&](auto kind) {
        constexpr int K = decltype(kind)::value;
        const uint8_t *const rows1 = rows + static_cast<uint32_t>(rows0 * nb * (K == 0 ? 34 : 18));
        const Q8RowsNAt<K, LPR> at0(lane, rows0), at1(lane, R - rows0);
        Q8Block w[kBoth ? 2 * PASSES : PASSES];
#pragma unroll
        for (int q = 0; q < PASSES; ++q) w[q] = q8_rowsn_load<K, LPR>(rows, q * LPR, nb, rows0, at0);
        if (kBoth) {
#pragma unroll
            for (int q = 0; q < PASSES; ++q) w[PASSES + q] = q8_rowsn_load<K, LPR>(rows1, q * LPR, nb, R - rows0, at1);
        }
        if (4 * wave < R) ops = layer_c_fold_request(a, r0 + 4 * wave, min(4, R - 4 * wave), lane);
#pragma unroll
        for (int i = 0; i < STEPS; ++i)
            lds_quantize_q8_0_step(v[2 * i], v[2 * i + 1], 512 * i + lane * 8 < a.F, 512 * i + lane * 8, aq, ad, lane);
        stream_w = layer_c_stream_weight(a, stream, 4 * wave < R);
        wave_lds_fence();
        Q8Chain ch;
#pragma unroll
        for (int q = 0; q < PASSES; ++q) {
            if (q > 0 && q * LPR >= nb) break;
            q8_rowsn_pass<K, LPR>(w[q], q * LPR, nb, aq, ad, tile, at0, ch);
            if (kThen) w[q] = q8_rowsn_load<K, LPR>(rows1, q * LPR, nb, R - rows0, at1);
        }
        const float y0 = q8_rowsn_close<K, LPR>(ch, nb, tile, at0);
        if (wave < n_act && (lane & 7) == 0 && (lane >> 3) < rows0) ybuf[m * 16 + (lane >> 3)] = or_nan(y0, missing);
        if constexpr (GROUPS == 1) return;
        ch = Q8Chain();
#pragma unroll
        for (int q = 0; q < PASSES; ++q) {
            if (q > 0 && q * LPR >= nb) break;
            q8_rowsn_pass<K, LPR>(w[kBoth ? PASSES + q : q], q * LPR, nb, aq, ad, tile, at1, ch);
        }
        const float y1 = q8_rowsn_close<K, LPR>(ch, nb, tile, at1);
        if (wave < n_act && (lane & 7) == 0 && (lane >> 3) < R - rows0) ybuf[m * 16 + rows0 + (lane >> 3)] = or_nan(y1, missing);
    };
    if (q8) run(std::integral_constant<int, 0>{});
    else run(std::integral_constant<int, KIND>{});
    __syncthreads();
    ops.stream_w = stream_w;
    if (4 * wave < R) layer_c_fold<16>(a, ops, ybuf + 4 * wave, r0 + 4 * wave, min(4, R - 4 * wave), lane);
}

}  // namespace wd
