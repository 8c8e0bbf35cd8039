// Whole-layer entry points: scratch object and the staged layer pass (one launch per stage,
// every stage a stand-alone operator of wd_ops.hip resolved against the device-side ids).
#include "wd_profile.hpp"
#include "wd_common.h"
#include "wd_tokens.cuh"
#include "wd_resident.cuh"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

using namespace wd;

namespace {
constexpr int kTagRecords = 64;  // one record per layer of a stack (modulo), so that a chain of layers needs no reset in between
constexpr int kTagRecordsPerPiece = kSidePiece / (kTagCopies * 8 * 4);
constexpr int kTagUnits = kTagRecords / kTagRecordsPerPiece;  // of two pieces
constexpr int kHostWords = 48 + 8 * 2 * kHandChunks;
}  // namespace

struct wd_moe_scratch {
    int hidden = 0, ffn = 0, n_experts = 0, max_k = 0;
    uint8_t *block = nullptr;
    float *logits = nullptr;
    int32_t *ids = nullptr;
    float *weights = nullptr;
    int8_t *xk_qs = nullptr;
    float *xk_d = nullptr;
    int16_t *xk_bs = nullptr;
    int8_t *x0_qs = nullptr;
    uint16_t *x0_d = nullptr;
    float *gate_up = nullptr;
    float *act = nullptr;
    int8_t *act_qs = nullptr;
    uint16_t *act_d = nullptr;
    float *expert_out = nullptr;
    float *accum = nullptr;
    float *down_f32 = nullptr;
    float *shared_gate = nullptr;
    int32_t *gup = nullptr;
    int32_t *dp = nullptr;
    int gup_type = -1, dp_type = -1;
    uint32_t *hand = nullptr;             // [n_experts + 2] logits on their way to the selection inside dispatch AB,
    int hand_side = 0;                    // and those of side 1 (LayerArgs)
    unsigned long long *trace = nullptr;  // device [3][16][8] time stamps, see wd_moe_scratch_trace
    int trace_wg = 0;
    int32_t *h_ids = nullptr;             // pinned [kHostWords]: [0..15] routed ids for callers that must see them on the host,
                                          // [16] mirror of the status word, written by the resident launch when a wait runs out,
                                          // [32..47] the selection as dispatch AB reports it (cached_routed_reported), [48..] votes (side_vote)
    // ids published inside the merged dispatch, kTagRecords records.  sided: kTagRecordsPerPiece records' copies of side 0 and those of side 1 in two
    // pieces of kSidePiece bytes, flip: side 1's first; otherwise [record][kTagCopies][16].
    uint32_t *tagged = nullptr;
    bool sided = false;
    int flip = 0;
    uint32_t *tags(int rec) const {
        if (!sided) return tagged + static_cast<size_t>(rec) * kTagCopies * 16;
        return tagged + (2 * (rec / kTagRecordsPerPiece) + flip) * (kSidePiece / 4) + (rec % kTagRecordsPerPiece) * (kTagCopies * 8);
    }
    int tag_side() const { return !sided ? kTagCopies * 8 : (flip ? -kSidePiece / 4 : kSidePiece / 4); }
    unsigned *status = nullptr;           // [0] != 0: a bounded wait inside a dispatch ran out
    unsigned spin_limit = kSpinLimit;
    int compute_units = 256;              // of the device the scratch lives on
    // the resident stack kernel (wd_resident.cuh): hand-off buffers, device copy of the layer descriptors
    uint8_t *res_block = nullptr, *res_alloc = nullptr;  // (the block begins on a boundary of kSideChunk inside the allocation)
    unsigned res_flips = 0;
    // Device copies of the layer descriptors of the stacks this scratch has run ([kResMaxLayers], then one ResidentViews
    // each).  A copy is never overwritten: a captured graph keeps the address of the copy it was recorded with.
    struct ResDescSet {
        std::vector<ResidentLayer> shadow;
        ResidentLayer *dev = nullptr;
    };
    std::vector<ResDescSet> res_sets;
    int res_fits = -1;                            // -1 not asked yet; 1: the device holds the whole grid at once
    int trace_layer = 0;
    bool trace_all = false;                       // the trace buffer has the resident kernel's size
    // wd_moe_layer_tokens_pairs_f32: a ring of pointer tables (pinned staging + device copy), kPairRing x [kPairEntries][3]
    const uint8_t **pair_host = nullptr, **pair_dev = nullptr;
    hipEvent_t pair_done[4] = {nullptr, nullptr, nullptr, nullptr};
    bool pair_used[4] = {false, false, false, false};
    int pair_next = 0;
};
constexpr int kPairRing = 4;

namespace {

struct Carver {
    size_t off = 0;
    size_t take(size_t bytes) {
        const size_t at = off;
        off += (bytes + 255) & ~static_cast<size_t>(255);
        return at;
    }
};

}  // namespace

namespace {

// One thread of a workgroup: whether the second of two pieces of kSidePiece bytes is nearer to side 0 than the first (> 0).  Times round trips of
// device-scope accesses whose loads and stores leave the words as they are (all ones; every workgroup has a line of its own).
WD_DEV int side_vote(uint32_t *pieces) {
    long long sum = 0;
    for (int turn = 0; turn < 10; ++turn) {
        uint32_t *p = pieces + (turn & 1) * (kSidePiece / 4) + (blockIdx.x & 7) * 64;
        const long long t0 = clock64();
        __hip_atomic_store(p, kHandEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        uint32_t v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(v)::"memory");
        const long long t = clock64() - t0;
        if (turn >= 2) sum += (turn & 1) ? -t : t;
    }
    return static_cast<int>(xcc_side() ? -sum : sum);
}
// (host) From the votes of workgroups 0..7: 1 where the first piece is side 1's.
int side_flip_of(const int *votes) {
    int second = 0;  // workgroups that say that the second piece is side 0's
    for (int g = 0; g < 8; ++g) second += votes[g] > 0 ? 1 : 0;
    return second > 4 ? 1 : 0;
}
// A scratch's block: zeros, but for the words that are handed on, which are "not yet" (ones_at .. ones_end, in words).  Workgroups 0..7 vote on
// the first two pieces at `sided`.
__global__ __launch_bounds__(256) void k_scratch_init(uint32_t *block, unsigned words, unsigned ones_at, unsigned ones_end, uint32_t *sided, int *votes) {
    for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < words; i += gridDim.x * 256) block[i] = i >= ones_at && i < ones_end ? kHandEmpty : 0u;
    if (blockIdx.x < 8 && threadIdx.x == 0) votes[blockIdx.x] = side_vote(sided);
}
// The resident stack's hand-off block: every word of both sets "not yet written", no launch finished.
__global__ __launch_bounds__(256) void k_hand_block_init(uint4 *block) {
    for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < kHandBytes / 16; i += gridDim.x * 256) {
        const uint32_t v = i < kHandEpoch / 16 ? kHandEmpty : 0u;
        block[i] = make_uint4(v, v, v, v);
    }
}
// Workgroups 8 q .. 8 q + 7 vote on the first two pieces of chunk q.
__global__ __launch_bounds__(64) void k_side_votes(uint32_t *base, int *votes) {
    if (threadIdx.x == 0) votes[blockIdx.x] = side_vote(base + static_cast<size_t>(blockIdx.x >> 3) * (kSideChunk / 4));
}

}  // namespace

extern "C" {

int wd_moe_scratch_create(wd_moe_scratch **out, int hidden, int expert_ffn, int n_experts, int max_k) {
    WD_REQUIRE(out != nullptr, "wd_moe_scratch_create: null output pointer");
    WD_REQUIRE(hidden > 0 && hidden % 256 == 0, "MoE scratch: hidden must be a positive multiple of 256 (got %d)", hidden);
    WD_REQUIRE(expert_ffn > 0 && expert_ffn % 32 == 0, "MoE scratch: expert_ffn must be a positive multiple of 32 (got %d)",
               expert_ffn);
    WD_REQUIRE(n_experts > 0 && max_k > 0 && max_k <= 16, "MoE scratch: invalid expert counts (%d experts, k=%d)",
               n_experts, max_k);
    wd_moe_scratch *s = new (std::nothrow) wd_moe_scratch;
    WD_REQUIRE(s != nullptr, "MoE scratch: out of host memory");
    s->hidden = hidden, s->ffn = expert_ffn, s->n_experts = n_experts, s->max_k = max_k;
    const size_t H = hidden, F = expert_ffn, K1 = max_k + 1;
    Carver c;
    const size_t o_logits = c.take(sizeof(float) * n_experts), o_ids = c.take(sizeof(int32_t) * 16),
                 o_w = c.take(sizeof(float) * 16), o_xkq = c.take(H), o_xkd = c.take(sizeof(float) * (H / 256)),
                 o_xkb = c.take(sizeof(int16_t) * (H / 16)), o_x0q = c.take(H),
                 o_x0d = c.take(sizeof(uint16_t) * (H / 32)), o_gu = c.take(sizeof(float) * K1 * 2 * F),
                 o_act = c.take(sizeof(float) * K1 * F), o_aq = c.take(K1 * F),
                 o_ad = c.take(sizeof(uint16_t) * K1 * (F / 32)), o_eo = c.take(sizeof(float) * K1 * H),
                 o_acc = c.take(sizeof(float) * H), o_dn = c.take(sizeof(float) * H), o_sg = c.take(256),
                 o_status = c.take(256);
    // the words that are handed on: the logits where they do not fit a piece, then (from a boundary of two pieces, within 2 MB, in which the
    // halves keep their order) two pieces for them and those of the published ids
    const size_t side_bytes = 2 * static_cast<size_t>(kSidePiece) * (1 + kTagUnits);
    const size_t o_hand = c.take(sizeof(uint32_t) * (n_experts + 2)), o_side = c.take(2 * side_bytes + 2 * kSidePiece);
    const hipError_t e = hipMalloc(reinterpret_cast<void **>(&s->block), c.off);
    if (e != hipSuccess) {
        delete s;
        return fail(WD_ERR_HIP, "hipMalloc MoE scratch (%zu bytes) failed: %s", c.off, hipGetErrorString(e));
    }
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0)
        s->compute_units = cus;
    uint8_t *b = s->block;
    s->logits = reinterpret_cast<float *>(b + o_logits);
    s->ids = reinterpret_cast<int32_t *>(b + o_ids);
    s->weights = reinterpret_cast<float *>(b + o_w);
    s->xk_qs = reinterpret_cast<int8_t *>(b + o_xkq);
    s->xk_d = reinterpret_cast<float *>(b + o_xkd);
    s->xk_bs = reinterpret_cast<int16_t *>(b + o_xkb);
    s->x0_qs = reinterpret_cast<int8_t *>(b + o_x0q);
    s->x0_d = reinterpret_cast<uint16_t *>(b + o_x0d);
    s->gate_up = reinterpret_cast<float *>(b + o_gu);
    s->act = reinterpret_cast<float *>(b + o_act);
    s->act_qs = reinterpret_cast<int8_t *>(b + o_aq);
    s->act_d = reinterpret_cast<uint16_t *>(b + o_ad);
    s->expert_out = reinterpret_cast<float *>(b + o_eo);
    s->accum = reinterpret_cast<float *>(b + o_acc);
    s->down_f32 = reinterpret_cast<float *>(b + o_dn);
    s->shared_gate = reinterpret_cast<float *>(b + o_sg);
    s->hand = reinterpret_cast<uint32_t *>(b + o_hand);
    uintptr_t side = (reinterpret_cast<uintptr_t>(b + o_side) + 2 * kSidePiece - 1) & ~static_cast<uintptr_t>(2 * kSidePiece - 1);
    if (side / kSideChunk != (side + side_bytes - 1) / kSideChunk) side = (side / kSideChunk + 1) * kSideChunk;
    uint32_t *const units = reinterpret_cast<uint32_t *>(side);
    s->tagged = units + 2 * kSidePiece / 4, s->sided = true;
    s->status = reinterpret_cast<unsigned *>(b + o_status);
    if (hipHostMalloc(reinterpret_cast<void **>(&s->h_ids), sizeof(int32_t) * kHostWords, hipHostMallocDefault) != hipSuccess) {
        (void)hipFree(s->block);
        delete s;
        return fail(WD_ERR_HIP, "hipHostMalloc MoE scratch ids failed");
    }
    std::memset(s->h_ids, 0, sizeof(int32_t) * kHostWords);
    // (its own code and not the thread's last error, which may be of an older call of the caller's)
    hipError_t init = enqueue_reported(k_scratch_init, dim3(64), dim3(256), 0, nullptr, reinterpret_cast<uint32_t *>(b), static_cast<unsigned>(c.off / 4),
                                       static_cast<unsigned>(o_hand / 4), static_cast<unsigned>(c.off / 4), units, s->h_ids);
    if (init == hipSuccess) init = hipStreamSynchronize(nullptr);
    if (init != hipSuccess) {
        (void)hipHostFree(s->h_ids);
        (void)hipFree(s->block);
        delete s;
        return fail(WD_ERR_HIP, "MoE scratch: the first launch failed: %s", hipGetErrorString(init));
    }
    s->flip = side_flip_of(s->h_ids);
    if (sizeof(uint32_t) * (static_cast<size_t>(n_experts) + 2) <= kSidePiece)
        s->hand = units + s->flip * (kSidePiece / 4), s->hand_side = s->flip ? -kSidePiece / 4 : kSidePiece / 4;
    std::memset(s->h_ids, 0, sizeof(int32_t) * kHostWords);
    *out = s;
    return WD_OK;
}

int wd_moe_scratch_destroy(wd_moe_scratch *s) {
    if (!s) return WD_OK;
    (void)hipFree(s->block);
    (void)hipFree(s->gup);
    (void)hipFree(s->dp);
    (void)hipFree(s->trace);
    (void)hipFree(s->res_alloc);
    for (wd_moe_scratch::ResDescSet &d : s->res_sets) (void)hipFree(d.dev);
    (void)hipHostFree(s->h_ids);
    (void)hipFree(s->pair_dev);
    (void)hipHostFree(s->pair_host);
    for (hipEvent_t ev : s->pair_done)
        if (ev) (void)hipEventDestroy(ev);
    delete s;
    return WD_OK;
}

int wd_moe_scratch_status(wd_moe_scratch *s) {
    if (!s) return -1;
    unsigned v = 0;
    if (hipMemcpy(&v, s->status, sizeof(v), hipMemcpyDeviceToHost) != hipSuccess) return -1;
    return static_cast<int>(v);
}
const unsigned *wd_moe_scratch_status_word(wd_moe_scratch *s) { return s ? s->status : nullptr; }
int wd_moe_scratch_set_wait_limit(wd_moe_scratch *s, unsigned polls) {
    WD_REQUIRE(s != nullptr, "wd_moe_scratch_set_wait_limit: null scratch");
    s->spin_limit = polls ? polls : kSpinLimit;
    // a fresh start: clear the status word and make the published ids invalid again
    WD_HIP(hipDeviceSynchronize());  // (a launch that gave up may still be running and would set the words again)
    WD_HIP(hipMemset(s->status, 0, sizeof(unsigned)));
    reinterpret_cast<volatile int32_t *>(s->h_ids)[16] = 0;
    WD_HIP(hipMemset(s->tagged, 0xff, 2 * static_cast<size_t>(kSidePiece) * kTagUnits));
    for (uint32_t *hand : {s->hand, s->hand + s->hand_side}) WD_HIP(hipMemset(hand, 0xff, sizeof(uint32_t) * (s->n_experts + 2)));
    if (s->res_block) WD_HIP(hipMemset(s->res_block, 0xff, kHandEpoch));
    return WD_OK;
}
float *wd_moe_scratch_logits(wd_moe_scratch *s) { return s->logits; }
int32_t *wd_moe_scratch_ids(wd_moe_scratch *s) { return s->ids; }
float *wd_moe_scratch_weights(wd_moe_scratch *s) { return s->weights; }
float *wd_moe_scratch_gate_up(wd_moe_scratch *s) { return s->gate_up; }
float *wd_moe_scratch_act(wd_moe_scratch *s) { return s->act; }
int8_t *wd_moe_scratch_act_qs(wd_moe_scratch *s) { return s->act_qs; }
uint16_t *wd_moe_scratch_act_scales(wd_moe_scratch *s) { return s->act_d; }
float *wd_moe_scratch_expert_out(wd_moe_scratch *s) { return s->expert_out; }
float *wd_moe_scratch_accum(wd_moe_scratch *s) { return s->accum; }
float *wd_moe_scratch_down_f32(wd_moe_scratch *s) { return s->down_f32; }
float *wd_moe_scratch_shared_gate(wd_moe_scratch *s) { return s->shared_gate; }
int32_t *wd_moe_scratch_gate_up_partials(wd_moe_scratch *s) { return s->gup; }
int32_t *wd_moe_scratch_down_partials(wd_moe_scratch *s) { return s->dp; }

// Profiling aid: allocates (once) a buffer of 3 x 16 x 8 time stamps (100 MHz counter) that the fused
// dispatches A, B, C fill for workgroup `wg` (per wave, per marked point); returns its device address.
unsigned long long *wd_moe_scratch_trace(wd_moe_scratch *s, int wg) {
    if (!s) return nullptr;
    if (!s->trace) {
        if (hipMalloc(reinterpret_cast<void **>(&s->trace), sizeof(unsigned long long) * 3 * 16 * 8) != hipSuccess) return nullptr;
        (void)hipMemset(s->trace, 0, sizeof(unsigned long long) * 3 * 16 * 8);
    }
    for (int d = 0; d < 3; ++d) {  // earliest-start cells start at the maximum
        const unsigned long long big = ~0ull;
        (void)hipMemcpy(s->trace + (d * 16 + 15) * 8, &big, sizeof(big), hipMemcpyHostToDevice);
        (void)hipMemset(s->trace + (d * 16 + 15) * 8 + 1, 0, sizeof(big));
    }
    s->trace_wg = wg;
    return s->trace;
}

// Profiling aid of the resident stack kernel: 12 x 16 time stamps (100 MHz counter; per wave, per marked point) of
// workgroup `wg` in layer `layer`; returns the device address of the buffer (shared with wd_moe_scratch_trace).
unsigned long long *wd_moe_scratch_trace_resident(wd_moe_scratch *s, int wg, int layer) {
    if (!s) return nullptr;
    const size_t bytes = sizeof(unsigned long long) * kResWgs * 4 * 16;  // also covers the per-layer kernels' 3 x 16 x 8
    if (s->trace && !s->trace_all) {
        (void)hipFree(s->trace);
        s->trace = nullptr;
    }
    if (!s->trace) {
        if (hipMalloc(reinterpret_cast<void **>(&s->trace), bytes) != hipSuccess) return nullptr;
        s->trace_all = true;
    }
    (void)hipMemset(s->trace, 0, bytes);
    s->trace_wg = wg, s->trace_layer = layer;
    return s->trace;
}

int wd_moe_scratch_enable_partials(wd_moe_scratch *s, int gate_type, int down_type) {
    WD_REQUIRE(s != nullptr, "enable partials: null scratch");
    const int pg = partials_per_row(gate_type, s->hidden), pd = partials_per_row(down_type, s->ffn);
    WD_REQUIRE(pg > 0 && pd > 0, "enable partials: unsupported tensor types %d / %d", gate_type, down_type);
    (void)hipFree(s->gup);
    (void)hipFree(s->dp);
    s->gup = s->dp = nullptr;
    WD_HIP(hipMalloc(reinterpret_cast<void **>(&s->gup), sizeof(int32_t) * s->max_k * 2 * s->ffn * pg));
    WD_HIP(hipMalloc(reinterpret_cast<void **>(&s->dp), sizeof(int32_t) * s->max_k * s->hidden * pd));
    s->gup_type = gate_type, s->dp_type = down_type;
    return WD_OK;
}

}  // extern "C"

namespace {

int check_layer(const wd_moe_layer *L, const wd_moe_scratch *s, unsigned flags) {
    WD_REQUIRE(L && s, "MoE layer: null layer or scratch");
    WD_REQUIRE(L->hidden == s->hidden && L->expert_ffn == s->ffn, "MoE layer geometry mismatch: layer %d/%d, scratch %d/%d",
               L->hidden, L->expert_ffn, s->hidden, s->ffn);
    WD_REQUIRE(L->n_experts > 0 && L->n_experts <= s->n_experts, "MoE layer: %d experts exceed the scratch (%d)",
               L->n_experts, s->n_experts);
    WD_REQUIRE(L->top_k > 0 && L->top_k <= s->max_k && L->top_k <= L->n_experts, "MoE layer: top_k %d out of range",
               L->top_k);
    WD_REQUIRE(L->gate_type == L->up_type, "MoE layer: gate and up tensors must share a type (%d vs %d)", L->gate_type,
               L->up_type);
    WD_REQUIRE(consumes_q8k(L->gate_type) || L->gate_type == WD_TYPE_Q8_0 || L->gate_type == WD_TYPE_IQ4_NL,
               "MoE layer: unsupported gate/up type %d", L->gate_type);
    WD_REQUIRE(L->down_type == WD_TYPE_Q8_0 || L->down_type == WD_TYPE_IQ4_NL, "MoE layer: unsupported down type %d",
               L->down_type);
    WD_REQUIRE(L->router != nullptr, "MoE layer: null router");
    // the selection sums the probabilities in groups of eight experts and holds at most 1024 of them (src/qwen38_moe.cuh:686-688)
    if (!(flags & WD_MOE_PRESELECTED))
        WD_REQUIRE(L->n_experts % 8 == 0 && L->n_experts <= 1024,
                   "MoE layer: the router's selection needs n_experts (%d) to be a multiple of 8, at most 1024", L->n_experts);
    if (L->slot_of_expert) {
        WD_REQUIRE(L->slot_pool != nullptr && L->slot_bytes > 0, "MoE layer: slot table without a slot pool");
    } else {
        WD_REQUIRE(L->gate && L->up && L->down, "MoE layer: null expert tensors");
    }
    if (L->shared_gate_inp) WD_REQUIRE(L->shared_gate && L->shared_up && L->shared_down, "MoE layer: incomplete shared expert");
    return WD_OK;
}

MatSrc routed_src(const wd_moe_layer *L, const wd_moe_scratch *s, const int32_t *ids, bool down) {
    MatSrc m{};
    m.ids = ids;
    m.slot_status = s->status;
    m.n_experts = static_cast<unsigned>(L->n_experts);
    m.per_expert = down ? 1 : 2;
    if (L->slot_of_expert) {
        m.slot_of_expert = L->slot_of_expert;
        m.pool = L->slot_pool;
        m.slot_bytes = L->slot_bytes;
        if (down) {
            m.slot_off[0] = L->slot_gate_bytes + L->slot_up_bytes;
        } else {
            m.slot_off[0] = 0;
            m.slot_off[1] = L->slot_gate_bytes;
        }
    } else if (down) {
        m.base[0] = L->down;
        m.stride[0] = L->down_stride;
    } else {
        m.base[0] = L->gate, m.base[1] = L->up;
        m.stride[0] = L->gate_stride, m.stride[1] = L->up_stride;
    }
    return m;
}

template <int TYPE>
void launch_iq(bool part, dim3 grid, hipStream_t st, MatSrc src, int rows, int cols, const int8_t *qs, const float *d,
               float *out, int32_t *partials, int ppr) {
    if (part)
        enqueue(k_gemv_iq<TYPE, true>, grid, dim3(256), 0, st, src, rows, cols, qs, d, out, partials, ppr);
    else
        enqueue(k_gemv_iq<TYPE, false>, grid, dim3(256), 0, st, src, rows, cols, qs, d, out, nullptr, 0);
}

template <int KIND>
void launch_q8(bool part, dim3 grid, hipStream_t st, MatSrc src, int rows, int cols, const int8_t *qs,
               const uint16_t *d, int act_stride, float *out, int32_t *partials, int ppr) {
    if (part)
        enqueue(k_gemv_q8<KIND, true>, grid, dim3(256), 0, st, src, rows, cols, qs, d, act_stride, out, partials, ppr);
    else
        enqueue(k_gemv_q8<KIND, false>, grid, dim3(256), 0, st, src, rows, cols, qs, d, act_stride, out, nullptr, 0);
}

// One grouped GEMV of `mats` matrices of `type` ([rows][cols]) against the layer's quantised input
// (shared activation) or against per-matrix Q8_0 activations (act_stride != 0).
int grouped_gemv(int type, MatSrc src, int mats, int rows, int cols, const wd_moe_scratch *s, const int8_t *q0,
                 const uint16_t *d0, int act_stride, float *out, int32_t *partials, hipStream_t st) {
    const dim3 grid((rows + 15) / 16, mats);
    const int ppr = partials_per_row(type, cols);
    const bool part = partials != nullptr;
    switch (type) {
        case WD_TYPE_IQ3_S: launch_iq<21>(part, grid, st, src, rows, cols, s->xk_qs, s->xk_d, out, partials, ppr); break;
        case WD_TYPE_IQ2_S: launch_iq<22>(part, grid, st, src, rows, cols, s->xk_qs, s->xk_d, out, partials, ppr); break;
        case WD_TYPE_Q8_0: launch_q8<0>(part, grid, st, src, rows, cols, q0, d0, act_stride, out, partials, ppr); break;
        case WD_TYPE_IQ4_NL: launch_q8<1>(part, grid, st, src, rows, cols, q0, d0, act_stride, out, partials, ppr); break;
        default: return fail(WD_ERR_UNSUPPORTED, "grouped GEMV: unsupported type %d", type);
    }
    WD_LAUNCH_CHECK();
    return WD_OK;
}

}  // namespace

namespace {

// The hyper-connection form of the residual update: residual is [hc][hidden] and stream c receives
// out * 2 sigmoid(inject[c] / hc) (src/qwen38_hc.cuh:2530-2547).
struct HcSpec {
    const float *inject;
    int hc, round_half;
};

// One layer, one launch per stage.  ids_override (device, k ids) replaces the router's ids while
// keeping its weights; residual (device f32[hidden]) receives residual += layer output.
int layer_staged(const wd_moe_layer *L, const float *d_x, float *d_out, wd_moe_scratch *s, unsigned flags,
                 const int32_t *ids_override, float *residual, float residual_scale, hipStream_t st,
                 const HcSpec *hc = nullptr) {
    const int H = L->hidden, F = L->expert_ffn, E = L->n_experts, k = L->top_k;
    const bool shared = L->shared_gate_inp != nullptr;
    const bool pre = (flags & WD_MOE_PRESELECTED) != 0;

    // 1. router logits (+ the shared expert's gate logit as one more row), softmax/top-k, sigmoid
    if (!pre) {
        {
            SiteScope site(WD_SITE_ROUTER_GEMV, st);
            enqueue(k_router_gemv, dim3((E + (shared ? 1 : 0) + 7) / 8), dim3(256), 0, st,
                L->router, d_x, s->logits, E, H, shared ? L->shared_gate_inp : nullptr, s->shared_gate);
            WD_LAUNCH_CHECK();
        }
        SiteScope site(WD_SITE_ROUTER_TOPK, st);
        enqueue(k_topk_softmax, dim3(1), dim3(64), 0, st, s->logits, E, k, L->expert_scale, s->ids, s->weights,
                                                     shared ? s->shared_gate : nullptr, ids_override);
        WD_LAUNCH_CHECK();
    } else if (shared) {
        SiteScope site(WD_SITE_SHARED_GATE, st);
        enqueue(k_router_gemv, dim3(1), dim3(256), 0, st, L->router, d_x, s->logits, 0, H, L->shared_gate_inp, s->shared_gate);
        WD_LAUNCH_CHECK();
        enqueue(k_sigmoid1, dim3(1), dim3(64), 0, st, s->shared_gate);
        WD_LAUNCH_CHECK();
    }

    // 2. quantise the layer input for the consumers that need it
    {
        SiteScope site(WD_SITE_RX_QUANT, st);
        if (consumes_q8k(L->gate_type)) {
            enqueue(k_q8_k_quantize, dim3((H / 256 + 3) / 4), dim3(256), 0, st, d_x, H / 256, s->xk_qs, s->xk_d, s->xk_bs);
            WD_LAUNCH_CHECK();
        }
        if (!consumes_q8k(L->gate_type) || shared) {
            enqueue(k_q8_0_quantize, dim3((H / 32 + 31) / 32), dim3(256), 0, st, d_x, H / 32, s->x0_qs, s->x0_d);
            WD_LAUNCH_CHECK();
        }
    }

    // 3. gate/up of the k selected experts in one dispatch (2k matrices), then the shared expert's
    const bool part = s->gup != nullptr && s->gup_type == L->gate_type && s->dp_type == L->down_type;
    {
        SiteScope site(WD_SITE_GATE_UP_GEMV, st);
        if (const int rc = grouped_gemv(L->gate_type, routed_src(L, s, s->ids, false), 2 * k, F, H, s, s->x0_qs, s->x0_d, 0,
                                        s->gate_up, part ? s->gup : nullptr, st))
            return rc;
    }
    if (shared) {
        SiteScope site(WD_SITE_SHARED, st);
        MatSrc g{}, u{};
        g.single = L->shared_gate, u.single = L->shared_up;
        float *gu = s->gate_up + static_cast<size_t>(2) * k * F;
        if (const int rc = grouped_gemv(WD_TYPE_Q8_0, g, 1, F, H, s, s->x0_qs, s->x0_d, 0, gu, nullptr, st)) return rc;
        if (const int rc = grouped_gemv(WD_TYPE_Q8_0, u, 1, F, H, s, s->x0_qs, s->x0_d, 0, gu + F, nullptr, st)) return rc;
    }

    // 4. SwiGLU in f32, 5. Q8_0 re-quantisation, for k (+1) experts at once
    const int n_act = k + (shared ? 1 : 0);
    {
        SiteScope site(WD_SITE_SILU, st);
        enqueue(k_silu_mul_experts, dim3((F + 255) / 256, n_act), dim3(256), 0, st, s->gate_up, s->act, F);
        WD_LAUNCH_CHECK();
    }
    {
        SiteScope site(WD_SITE_Q8_QUANT, st);
        enqueue(k_q8_0_quantize, dim3((n_act * F / 32 + 31) / 32), dim3(256), 0, st, s->act, n_act * F / 32, s->act_qs, s->act_d);
        WD_LAUNCH_CHECK();
    }

    // 6. down projections: k routed matrices with their own activations, then the shared expert
    {
        SiteScope site(WD_SITE_DOWN_GEMV, st);
        if (const int rc = grouped_gemv(L->down_type, routed_src(L, s, s->ids, true), k, H, F, s, s->act_qs, s->act_d, F,
                                        s->expert_out, part ? s->dp : nullptr, st))
            return rc;
    }
    if (shared) {
        SiteScope site(WD_SITE_SHARED, st);
        MatSrc d{};
        d.single = L->shared_down;
        if (const int rc = grouped_gemv(WD_TYPE_Q8_0, d, 1, H, F, s, s->act_qs + static_cast<size_t>(k) * F,
                                        s->act_d + static_cast<size_t>(k) * (F / 32), 0, s->down_f32, nullptr, st))
            return rc;
    }

    // 7. ordered weighted sum and the shared branch
    {
        SiteScope site(WD_SITE_ACCUM, st);
        enqueue(k_combine, dim3((H + 255) / 256), dim3(256), 0, st, s->expert_out, s->weights, k, shared ? s->down_f32 : nullptr,
                                                                s->shared_gate, s->accum, d_out, hc ? nullptr : residual,
                                                                residual_scale, H);
        WD_LAUNCH_CHECK();
    }
    if (hc && residual) {
        SiteScope site(WD_SITE_HC_COMBINE, st);
        enqueue(k_hc_combine<0>, dim3((H * hc->hc + 255) / 256), dim3(256), 0, st, residual, d_out, nullptr, nullptr, hc->inject, H,
                                                                             hc->hc, hc->round_half);
        WD_LAUNCH_CHECK();
    }
    return WD_OK;
}

LayerArgs fused_args(const wd_moe_layer *L, const float *d_x, float *d_out, wd_moe_scratch *s, unsigned flags,
                     const int32_t *ids_override, float *residual, float residual_scale, int rec = 0,
                     const HcSpec *hc = nullptr) {
    LayerArgs a{};
    a.H = L->hidden, a.F = L->expert_ffn, a.E = L->n_experts, a.k = L->top_k;
    a.w_scale = L->expert_scale;
    a.x = d_x;
    a.router = L->router;
    a.gate_up = routed_src(L, s, s->ids, false);
    a.down = routed_src(L, s, s->ids, true);
    a.sh_inp = L->shared_gate_inp;
    a.sh_gate = L->shared_gate, a.sh_up = L->shared_up, a.sh_down = L->shared_down;
    a.logits = s->logits, a.ids = s->ids, a.weights = s->weights;
    a.ids_override = ids_override;
    a.act = s->act;
    a.shared_gate = s->shared_gate;
    a.expert_out = (flags & WD_MOE_KEEP_EXPERT_OUT) ? s->expert_out : nullptr;
    a.accum = s->accum, a.down_f32 = s->down_f32, a.out = d_out;
    a.residual = residual, a.residual_scale = residual_scale;
    if (hc) a.hc_inject = hc->inject, a.hc = hc->hc, a.hc_round_half = hc->round_half;
    a.preselected = (flags & WD_MOE_PRESELECTED) ? 1 : 0;
    a.dry = (flags & WD_MOE_DRY) ? 1 : 0;
    a.ids_known = ids_override;  // a routing trace: the ids do not depend on the router
    a.trace = s->trace, a.trace_wg = s->trace_wg;
    a.hand = s->hand, a.hand_side = s->hand_side;
    a.ids_tagged = s->tags(rec % kTagRecords), a.tag_side = s->tag_side();
    a.clear_tagged = 1;
    a.status = s->status;
    a.spin_limit = s->spin_limit;
    // the chunk sums go out of the fused dispatches when the scratch was asked to keep them and the gate/up rows are of
    // the kinds whose fused kernels export them (other layers take the staged dispatches for that)
    if (s->gup && !(flags & WD_MOE_STAGED) && consumes_q8k(L->gate_type) && s->gup_type == L->gate_type && s->dp_type == L->down_type)
        a.gup_part = s->gup, a.down_part = s->dp;
    return a;
}

// Dispatch AB (or the part of it that `m` describes) of one row fetch.
template <int TYPE, int FETCH>
void launch_layer_ab_fetch(bool loop, int grid, hipStream_t st, const LayerArgs &m) {
    const size_t routed = layer_ab_stage(m.H) + 8 * static_cast<size_t>(layer_ab_stage_bytes<TYPE, FETCH>(m.H));
    const size_t lds = std::max(sizeof(float) * static_cast<size_t>(m.H) + 16, routed);
    const dim3 block(512);
    const bool part = m.gup_part != nullptr;  // the variants that also store the int32 chunk sums
    // (the time stamps are a variant of their own, so that the others run without their tests; no stamps are taken
    // while the chunk sums are exported)
    const bool trace = m.trace != nullptr && !part;
    if constexpr (TYPE == 21 || TYPE == 22) {
        if (loop && part) return enqueue(k_layer_ab<TYPE, FETCH, true, true>, grid, block, lds, st, m);
        if (part) return enqueue(k_layer_ab<TYPE, FETCH, false, true>, grid, block, lds, st, m);
    }
    if (loop && trace)
        enqueue(k_layer_ab<TYPE, FETCH, true, false, true>, grid, block, lds, st, m);
    else if (loop)
        enqueue(k_layer_ab<TYPE, FETCH, true>, grid, block, lds, st, m);
    else if (trace)
        enqueue(k_layer_ab<TYPE, FETCH, false, false, true>, grid, block, lds, st, m);
    else
        enqueue(k_layer_ab<TYPE, FETCH, false>, grid, block, lds, st, m);
}
template <int TYPE>
void launch_layer_ab(int fetch, bool loop, int grid, hipStream_t st, const LayerArgs &m) {
    switch (fetch) {
        case 8:
            if constexpr (TYPE == 21 || TYPE == 22) return launch_layer_ab_fetch<TYPE, 8>(loop, grid, st, m);
            [[fallthrough]];
        case 10:
            if constexpr (TYPE == 21 || TYPE == 22) return launch_layer_ab_fetch<TYPE, 10>(loop, grid, st, m);
            [[fallthrough]];
        case 1: return launch_layer_ab_fetch<TYPE, 1>(loop, grid, st, m);
        case 2: return launch_layer_ab_fetch<TYPE, 2>(loop, grid, st, m);
        default: return launch_layer_ab_fetch<TYPE, 0>(loop, grid, st, m);
    }
}
// Dispatch AB: with `front` the router, the selection and the shared expert's gate/up, with `routed` the routed gate/up.
int launch_ab(const LayerArgs &a, const wd_moe_layer *L, const wd_moe_scratch *s, bool front, bool routed, hipStream_t st) {
    const int H = a.H, F = a.F, groups = (F + 7) / 8;
    const bool iq = consumes_q8k(L->gate_type), shared = a.sh_inp != nullptr;
    auto al16 = [](const void *p, size_t v) { return reinterpret_cast<uintptr_t>(p) % 16 == 0 && v % 16 == 0; };
    // IQ tensors that start on 16-byte boundaries (F rows are whole 16-byte words, F being a multiple of 32)
    const bool words = !iq || (L->slot_of_expert ? al16(L->slot_pool, L->slot_bytes) && L->slot_gate_bytes % 16 == 0
                                                 : al16(L->gate, L->gate_stride) && al16(L->up, L->up_stride));
    int fetch = !words || H > 4096 ? 0 : (H > 2048 ? 2 : 1);
    if (iq && words && H == 2048) fetch = 8;
    if (iq && words && H == 2560) fetch = 10;
    const bool wide = fetch == 2 || fetch == 10;
    LayerArgs m = a;
    const int router_rows_n = front ? (a.preselected ? 0 : a.E) + (shared ? 1 : 0) : 0;
    m.n_router_wgs = wide ? (router_rows_n + 3) / 4 : (router_rows_n + 7) / 8;  // two waves or one per row
    m.n_select_wgs = front && !a.preselected ? 1 : 0;
    m.n_shared_wgs = front && shared ? groups : 0;
    m.n_routed_items = routed ? a.k * groups : 0;
    if (!routed) m.ids_tagged = nullptr;  // nobody waits for them inside this launch
    if (!front || a.preselected) m.ids_known = s->ids;
    m.hand_limit = routed && !m.ids_known ? a.spin_limit : kHandPatient;
    // A compute unit holds three of these workgroups.  The router and shared ones leave well before the ids are
    // published, so a few routed ones that have to wait for their places still start in time.  But when the routed
    // ones alone are more than the device holds at once (hidden 2560: 800 against 768), the surplus would start -
    // quantise x, stage the codebooks - only after others have finished: the grid is then cut and the routed workgroups walk the items in a
    // loop.  Cut by the places of the router's workgroups, which are the last to leave, and not by the shared expert's; by neither
    // where that saves a round of the loop.  us per layer, cut by both / by the router's / by neither: 2560 / 640 IQ2_S with a shared expert, 800 items, 24.3 /
    // 23.8 / 24.0 (a workgroup for every item 26.0); 3328 / 864 Q8_0 with one, 972, 31.6 / 28.7 / 28.8; 2048 / 992 Q8_0 with one, 1240, 24.5 / 22.7 /
    // 23.1; without one 1536 / 832 IQ2_S, 936, 18.0 / 18.0 / 18.4, and 4096 / 1536, 1536 items in three rounds / three / two, 40.0 / 40.0 / 39.3.
    // (Rows of two waves, beyond 2048 columns, count as one: the figures above are with that.)
    const int capacity = 3 * s->compute_units, router_places = (router_rows_n + 7) / 8;
    auto rounds = [&](int wgs) { return (m.n_routed_items + wgs - 1) / wgs; };
    // (The loop that runs two per compute unit, kAbPerCu, takes all of its places: with the shared expert's workgroups counted among
    // them hidden 7168 / ffn 2048, top-8, has 256 routed workgroups left and takes 106 us, so 68; 5120 / 1024 40.7, 34.2.)
    const bool two = fetch == 0 && L->gate_type == WD_TYPE_IQ3_S;
    const int cut = std::max(capacity - router_places, 1);
    const int looping = two ? kAbPerCu<21, 0, true> * s->compute_units : (rounds(cut) > rounds(capacity) ? capacity : cut);
    const int routed_wgs = m.n_routed_items <= capacity - 8 ? m.n_routed_items : std::min(m.n_routed_items, looping);
    const int grid = m.n_select_wgs + m.n_router_wgs + m.n_shared_wgs + routed_wgs;
    if (grid == 0) return WD_OK;
    const bool loop = routed_wgs < m.n_routed_items;
    switch (L->gate_type) {
        case WD_TYPE_IQ3_S: launch_layer_ab<21>(fetch, loop, grid, st, m); break;
        case WD_TYPE_IQ2_S: launch_layer_ab<22>(fetch, loop, grid, st, m); break;
        case WD_TYPE_Q8_0: launch_layer_ab<8>(fetch, loop, grid, st, m); break;
        case WD_TYPE_IQ4_NL: launch_layer_ab<20>(fetch, loop, grid, st, m); break;
        default: return fail(WD_ERR_UNSUPPORTED, "fused layer: unsupported gate/up type %d", L->gate_type);
    }
    WD_LAUNCH_CHECK();
    return WD_OK;
}
template <int KIND>
void launch_layer_c(hipStream_t st, const LayerArgs &a) {
    const int n_act = a.k + (a.sh_inp ? 1 : 0), waves = std::min(n_act, 16);
    const size_t per_wave = (static_cast<size_t>(a.F) + a.F / 16 + 15) & ~static_cast<size_t>(15);
    const size_t lds = layer_c_lds(n_act, 4, waves * per_wave);
    const dim3 grid((a.H + 3) / 4), block(64 * waves);
    if (a.down_part)
        enqueue(k_layer_c<KIND, true>, grid, block, lds, st, a);
    else if (a.trace)
        enqueue(k_layer_c<KIND, false, true>, grid, block, lds, st, a);
    else
        enqueue(k_layer_c<KIND>, grid, block, lds, st, a);
}
template <int KIND, int PASSES, bool WORDS>
void launch_layer_c8(hipStream_t st, const LayerArgs &a) {
    const int n_act = a.k + (a.sh_inp ? 1 : 0), waves = std::max(n_act, 2);
    const size_t lds = layer_c_lds(n_act, 8, waves * static_cast<size_t>(layer_c8_wave_bytes<WORDS>(a.F)));
    const dim3 grid(a.H / 8), block(64 * waves);
    if (a.down_part)
        enqueue(k_layer_c8<KIND, PASSES, WORDS, true>, grid, block, lds, st, a);
    else if (a.trace)
        enqueue(k_layer_c8<KIND, PASSES, WORDS, false, true>, grid, block, lds, st, a);
    else if (PASSES == 3 && n_act > 12 && a.H > 2048)  // more workgroups than compute units: the form of which two fit one
        enqueue(k_layer_c8<KIND, PASSES, WORDS, false, false, false, PASSES != 3>, grid, block, lds, st, a);
    else
        enqueue(k_layer_c8<KIND, PASSES, WORDS>, grid, block, lds, st, a);
}
template <int KIND>
void launch_layer_c8_two(hipStream_t st, const LayerArgs &a) {
    const size_t lds = layer_c_lds(a.k + 1, 8, 9 * static_cast<size_t>(layer_c8_wave_bytes<false>(a.F)));
    const dim3 grid(a.H / 8), block(64 * 9);
    if (a.F <= 512)
        enqueue(k_layer_c8<KIND, 2, false, false, false, true>, grid, block, lds, st, a);
    else if (a.H <= 2048)
        enqueue(k_layer_c8<KIND, 3, false, false, false, true>, grid, block, lds, st, a);
    else  // more workgroups than compute units: the form of which two fit one
        enqueue(k_layer_c8<KIND, 3, false, false, false, true, false>, grid, block, lds, st, a);
}
template <int KIND>
void launch_layer_c8(bool words, hipStream_t st, const LayerArgs &a) {
    if (a.F <= 512) launch_layer_c8<KIND, 2, false>(st, a);
    else if (a.F <= 768) launch_layer_c8<KIND, 3, false>(st, a);
    else if (a.F <= 1024) KIND == 0 && words ? launch_layer_c8<0, 4, true>(st, a) : launch_layer_c8<KIND, 4, false>(st, a);
    else words ? launch_layer_c8<KIND, 6, true>(st, a) : launch_layer_c8<KIND, 6, false>(st, a);
}

template <int KIND, int LPR, int GROUPS, int PASSES = 1>
void launch_layer_c_even(hipStream_t st, const LayerArgs &a) {
    // (rows of 48 blocks at most; four passes, then six)
    if constexpr (PASSES * LPR < 48) {
        if (a.F > 32 * PASSES * LPR) return launch_layer_c_even<KIND, LPR, GROUPS, (PASSES < 4 ? PASSES + 1 : 6)>(st, a);
    }
    const int n_act = a.k + (a.sh_inp ? 1 : 0), waves = std::max(n_act, 2 * GROUPS);
    const size_t lds = layer_c_lds(n_act, 16, waves * static_cast<size_t>(layer_c_even_wave_bytes<LPR>(a.F)));
    enqueue(k_layer_c_even<KIND, LPR, GROUPS, PASSES>, dim3(256), dim3(64 * waves), lds, st, a);
}
template <int KIND>
void launch_layer_c_even(hipStream_t st, const LayerArgs &a) {
    const int R = a.H / 256;
    if (R <= 4) launch_layer_c_even<KIND, 16, 1>(st, a);
    else if (R == 5) launch_layer_c_even<KIND, 12, 1>(st, a);
    else if (R == 6) launch_layer_c_even<KIND, 10, 1>(st, a);
    else if (R <= 10) launch_layer_c_even<KIND, 12, 2>(st, a);  // (9 and 10: layer_c_evenly takes neither 7 nor 8)
    else if (R <= 12) launch_layer_c_even<KIND, 10, 2>(st, a);
    else if (R <= 14) launch_layer_c_even<KIND, 9, 2>(st, a);
    else launch_layer_c_even<KIND, 8, 2>(st, a);
}
// Whether dispatch C takes the form with one workgroup of hidden / 256 rows per compute unit (k_layer_c_even) where the eight-row
// form would do: us of the dispatch, weights from HBM, eight-row / even.
//   hidden 512 to 1280, always (256: rows of one workgroup in eight's place, 256 3.3 / 3.5, 1280 8.3 / 7.0): 1024 / 512, ten and the shared expert 6.30 / 5.16; 1024 / 256, eight 4.23 / 4.07; 1280 / 1248, eight 9.83 / 8.69;
//   1536, where ten lanes a row need fewer passes than eight: 1248 10.2 / 9.1, IQ4_NL 640 6.2 / 5.8, but 512 5.8 / 5.9;
//   not 1792 (768, eight: 7.0 / 7.2) and 2048 (two groups of four rows, 640 IQ4_NL, ten and the shared one: 7.7 / 8.1);
//   beyond, where there are waves enough: 2560 / 640 IQ4_NL, ten and the shared one 10.2 / 8.4, 1280 17.9 / 13.1, three matrices of 768 6.1 / 5.8; 3072 /
//   768, ten and the shared one 13.0 / 12.4, four and the shared one 7.8 / 7.4, but three 6.2 / 6.7; 3328 / 640 IQ4_NL, eight 8.4 / 8.1, four and
//   the shared one 7.0 / 7.3; 4096 / 256, eight 6.6 / 6.0;
//   and beyond 3072 not for the bytes that the aligned words are for: 3584 / 1536, eight: 15.1 / 17.4 (2560, ten and the shared one: 19.7 / 16.8).
bool layer_c_evenly(int H, int F, int n_act, bool words) {
    const int R = H / 256, nb = F / 32;
    if (R <= 5) return R > 1 || nb > 16;
    if (R == 6) return (nb + 9) / 10 < (nb + 7) / 8;
    return R > 8 && R <= 16 && n_act >= (R <= 12 ? 5 : 6) && !(words && R > 12);
}

// What dispatches A and AB hand on - the ids published in the scratch's records, and the logits - is set back by dispatch C,
// and where C does not follow by the dispatch itself (the logits, close_hand) and by these: a pass that finds what another one left
// takes that one's ids.
__global__ __launch_bounds__(kTagCopies * 8) void k_reset_tags(uint32_t *tags, int tag_side) {
    tags[threadIdx.x] = kTagInvalid, tags[tag_side + static_cast<int>(threadIdx.x)] = kTagInvalid;
}
void reset_tags(const wd_moe_scratch *s, int rec, hipStream_t st) {
    enqueue(k_reset_tags, dim3(1), dim3(kTagCopies * 8), 0, st, s->tags(rec % kTagRecords), s->tag_side());
}
// (of a scratch made by wd_moe_scratch_create)
int reset_all_published(const wd_moe_scratch *s, hipStream_t st) {
    const size_t n = 2 * static_cast<size_t>(kSidePiece / 4) * kTagUnits;
    enqueue(k_fill_u32, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, st, s->tagged, kTagInvalid, n);
    WD_LAUNCH_CHECK();
    return WD_OK;
}
int reset_published(const wd_moe_scratch *s, int rec, hipStream_t st) {
    reset_tags(s, rec, st);
    WD_LAUNCH_CHECK();
    return WD_OK;
}
// Both, behind an error after which no dispatch C comes.  (The error stays the one to report.)
void reset_handed(const wd_moe_scratch *s, int rec, hipStream_t st) {
    const size_t n = static_cast<size_t>(s->n_experts) + 2;
    reset_tags(s, rec, st);
    for (uint32_t *hand : {s->hand, s->hand + s->hand_side}) enqueue(k_fill_u32, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, st, hand, kHandEmpty, n);
    (void)hipGetLastError();
}

// report: null, or the host words that dispatch AB reports its selection to.  An expert without a slot is then no error: its
// rows are computed again once it has one.
// rec: which of the scratch's records of published ids the pass uses; chain: the caller sets it back.
int layer_fused_queue(const wd_moe_layer *L, const float *d_x, float *d_out, wd_moe_scratch *s, unsigned flags,
                      const int32_t *ids_override, float *residual, float residual_scale, hipStream_t st, int rec,
                      const HcSpec *hc, uint32_t *report, bool chain) {
    const int H = L->hidden, F = L->expert_ffn, k = L->top_k;
    const bool shared = L->shared_gate_inp != nullptr;
    LayerArgs a = fused_args(L, d_x, d_out, s, flags, ids_override, residual, residual_scale, rec, hc);
    if (report) a.host_ids = report, a.gate_up.slot_status = nullptr;
    const unsigned only = flags & (WD_MOE_ONLY_A | WD_MOE_ONLY_B | WD_MOE_ONLY_C);
    const bool run_a = !only || (only & WD_MOE_ONLY_A), run_b = !only || (only & WD_MOE_ONLY_B);
    a.close_hand = only && !(only & WD_MOE_ONLY_C) && !report;
    // router + selection + shared gate/up + routed gate/up in one launch (the routed workgroups wait for the ids
    // inside the dispatch) unless the caller asked for the two parts apart
    const bool merged = run_a && run_b && !(flags & WD_MOE_SPLIT_AB);
    if (merged) {
        SiteScope site(WD_SITE_FUSED_AB, st);
        if (const int rc = launch_ab(a, L, s, true, true, st)) return rc;
    } else {
        if (run_a) {
            SiteScope site(WD_SITE_FUSED_A, st);
            if (const int rc = launch_ab(a, L, s, true, false, st)) return rc;
        }
        if (run_b) {
            SiteScope site(WD_SITE_FUSED_B, st);
            if (const int rc = launch_ab(a, L, s, false, true, st)) return rc;
        }
    }
    if (only && !(only & WD_MOE_ONLY_C)) {
        // dispatch C, which sets the handed words back, is not part of this call (with a report it follows in the same one)
        return merged && !chain && !report && !a.dry ? reset_published(s, rec, st) : static_cast<int>(WD_OK);
    }
    SiteScope site(WD_SITE_FUSED_C, st);
    const int n_act = k + (shared ? 1 : 0);
    const bool q8 = L->down_type == WD_TYPE_Q8_0;
    if (n_act > 16 && F > 256 && F <= 768 && !a.down_part && !a.trace) {  // (chunk sums and time stamps: the four-row form has them)
        q8 ? launch_layer_c8_two<0>(st, a) : launch_layer_c8_two<1>(st, a);
    } else if (F <= 1536 && n_act <= 16) {
        // The aligned fetch where every down tensor starts on a 16-byte boundary and the rows' bytes are what the dispatch
        // waits for: 32 MB and more (Q8_0 rows of 48 blocks, 53.5 MB: 14.7 us against 16.1; 40: 12.6, 13.3; 33: 11.4, 11.7; 26.7: 10.0,
        // 10.1; 32 blocks, 44.6 MB: 12.5, 13.9; 35.7: 10.7, 11.5; 26.7: 9.2, 9.5; at 21 MB it loses, 9.5 against 9.0).  IQ4_NL rows,
        // half as long, only beyond 32 blocks (48 blocks, 42.5 MB: 20.0, 20.4; 35.4: 19.1, 19.3; 32 blocks, 37.7 MB: 18.6, 17.2).
        auto al16 = [](const void *p, size_t v) { return reinterpret_cast<uintptr_t>(p) % 16 == 0 && v % 16 == 0; };
        const bool words = static_cast<size_t>(n_act) * wd_tensor_bytes(L->down_type, H, F) >= 32000000 && (q8 || F > 1024) && al16(L->shared_down, 0) &&
                           (L->slot_of_expert ? al16(L->slot_pool, L->slot_bytes) && (L->slot_gate_bytes + L->slot_up_bytes) % 16 == 0
                                              : al16(L->down, L->down_stride));
        // (chunk sums and time stamps: the eight-row form has them)
        if (!a.down_part && !a.trace && layer_c_evenly(H, F, n_act, words)) q8 ? launch_layer_c_even<0>(st, a) : launch_layer_c_even<1>(st, a);
        else q8 ? launch_layer_c8<0>(words, st, a) : launch_layer_c8<1>(words, st, a);
    } else {
        q8 ? launch_layer_c<0>(st, a) : launch_layer_c<1>(st, a);
    }
    WD_LAUNCH_CHECK();
    return WD_OK;
}

int layer_fused(const wd_moe_layer *L, const float *d_x, float *d_out, wd_moe_scratch *s, unsigned flags,
                const int32_t *ids_override, float *residual, float residual_scale, hipStream_t st, int rec = 0,
                const HcSpec *hc = nullptr, uint32_t *report = nullptr, bool chain = false) {
    const int rc = layer_fused_queue(L, d_x, d_out, s, flags, ids_override, residual, residual_scale, st, rec, hc, report, chain);
    if (rc != WD_OK) reset_handed(s, rec, st);
    return rc;
}

int layer_dispatch(const wd_moe_layer *L, const float *d_x, float *d_out, wd_moe_scratch *s, unsigned flags,
                   const int32_t *ids_override, float *residual, float residual_scale, hipStream_t st, int rec = 0,
                   const HcSpec *hc = nullptr, bool chain = false) {
    const bool want_partials = s->gup != nullptr;
    const bool fused_exports = consumes_q8k(L->gate_type) && s->gup_type == L->gate_type && s->dp_type == L->down_type;
    if ((flags & WD_MOE_STAGED) || (want_partials && !fused_exports))
        return layer_staged(L, d_x, d_out, s, flags, ids_override, residual, residual_scale, st, hc);
    return layer_fused(L, d_x, d_out, s, flags, ids_override, residual, residual_scale, st, rec, hc, nullptr, chain);
}

}  // namespace

extern "C" int wd_moe_layer_f32(const wd_moe_layer *L, const float *d_x, float *d_out, wd_moe_scratch *s,
                                unsigned flags, void *stream) {
    if (const int rc = check_layer(L, s, flags)) return rc;
    WD_REQUIRE(d_x && d_out, "MoE layer: null activation or output pointer");
    SiteScope site(WD_SITE_ROUTED_TOTAL, as_stream(stream));
    return layer_dispatch(L, d_x, d_out, s, flags, nullptr, nullptr, 0.0f, as_stream(stream));
}

extern "C" int wd_moe_layer_hc_f32(const wd_moe_layer *L, const float *d_x, float *d_out, float *d_residual,
                                   const float *d_inject, int hc, int round_half, wd_moe_scratch *s, unsigned flags,
                                   void *stream) {
    if (const int rc = check_layer(L, s, flags)) return rc;
    WD_REQUIRE(d_x && d_out && d_residual && d_inject, "MoE layer with combine: null activation, output, residual or inject pointer");
    WD_REQUIRE(hc >= 1 && hc <= 16, "MoE layer with combine: 1..16 residual streams (got %d)", hc);
    WD_REQUIRE(!(flags & (WD_MOE_ONLY_A | WD_MOE_ONLY_B | WD_MOE_ONLY_C | WD_MOE_DRY)), "MoE layer with combine: measurement flags are not supported");
    const HcSpec spec{d_inject, hc, round_half ? 1 : 0};
    SiteScope site(WD_SITE_ROUTED_TOTAL, as_stream(stream));
    return layer_dispatch(L, d_x, d_out, s, flags, nullptr, d_residual, 0.0f, as_stream(stream), 0, &spec);
}

extern "C" int wd_hc_combine_f32(float *d_residual, const float *d_block_out, const float *d_inject, int hidden, int hc,
                                 int round_half, void *stream) {
    WD_REQUIRE(d_residual && d_block_out && d_inject, "combine: null pointer");
    WD_REQUIRE(hidden > 0 && hc > 0 && static_cast<long long>(hidden) * hc < (1LL << 31), "combine: bad geometry %d x %d", hc, hidden);
    SiteScope site(WD_SITE_HC_COMBINE, as_stream(stream));
    enqueue(k_hc_combine<0>, dim3((hidden * hc + 255) / 256), dim3(256), 0, as_stream(stream), d_residual, d_block_out, nullptr, nullptr,
                                                                                          d_inject, hidden, hc, round_half ? 1 : 0);
    WD_LAUNCH_CHECK();
    return WD_OK;
}

extern "C" int wd_hc_combine_moe_f32(float *d_residual, const float *d_routed, const void *d_shared, int shared_is_half,
                                     const float *d_shared_gate, const float *d_inject, int hidden, int hc, int round_half,
                                     void *stream) {
    WD_REQUIRE(d_residual && d_routed && d_shared && d_shared_gate && d_inject, "combine: null pointer");
    WD_REQUIRE(hidden > 0 && hc > 0 && static_cast<long long>(hidden) * hc < (1LL << 31), "combine: bad geometry %d x %d", hc, hidden);
    SiteScope site(WD_SITE_HC_COMBINE, as_stream(stream));
    const dim3 grid((hidden * hc + 255) / 256), block(256);
    if (shared_is_half)
        enqueue(k_hc_combine<2>, grid, block, 0, as_stream(stream), d_residual, d_routed, d_shared, d_shared_gate, d_inject, hidden, hc, round_half ? 1 : 0);
    else
        enqueue(k_hc_combine<1>, grid, block, 0, as_stream(stream), d_residual, d_routed, d_shared, d_shared_gate, d_inject, hidden, hc, round_half ? 1 : 0);
    WD_LAUNCH_CHECK();
    return WD_OK;
}

extern "C" int wd_shared_expert_f32(const wd_moe_layer *L, const float *d_x, wd_moe_scratch *s, void *stream) {
    WD_REQUIRE(L && s && d_x, "shared expert: null layer, scratch or activation");
    WD_REQUIRE(L->hidden == s->hidden && L->expert_ffn == s->ffn, "shared expert geometry mismatch: layer %d/%d, scratch %d/%d",
               L->hidden, L->expert_ffn, s->hidden, s->ffn);
    WD_REQUIRE(L->shared_gate_inp && L->shared_gate && L->shared_up && L->shared_down, "shared expert: incomplete weights");
    const int H = L->hidden, F = L->expert_ffn, slot = s->max_k;
    const hipStream_t st = as_stream(stream);
    SiteScope site(WD_SITE_SHARED, st);
    enqueue(k_router_gemv, dim3(1), dim3(256), 0, st, L->router, d_x, s->logits, 0, H, L->shared_gate_inp, s->shared_gate);
    WD_LAUNCH_CHECK();
    enqueue(k_sigmoid1, dim3(1), dim3(64), 0, st, s->shared_gate);
    WD_LAUNCH_CHECK();
    enqueue(k_q8_0_quantize, dim3((H / 32 + 31) / 32), dim3(256), 0, st, d_x, H / 32, s->x0_qs, s->x0_d);
    WD_LAUNCH_CHECK();
    MatSrc g{}, u{}, d{};
    g.single = L->shared_gate, u.single = L->shared_up, d.single = L->shared_down;
    float *gu = s->gate_up + static_cast<size_t>(2) * slot * F;
    float *act = s->act + static_cast<size_t>(slot) * F;
    int8_t *aq = s->act_qs + static_cast<size_t>(slot) * F;
    uint16_t *ad = s->act_d + static_cast<size_t>(slot) * (F / 32);
    if (const int rc = grouped_gemv(WD_TYPE_Q8_0, g, 1, F, H, s, s->x0_qs, s->x0_d, 0, gu, nullptr, st)) return rc;
    if (const int rc = grouped_gemv(WD_TYPE_Q8_0, u, 1, F, H, s, s->x0_qs, s->x0_d, 0, gu + F, nullptr, st)) return rc;
    enqueue(k_silu_mul_experts, dim3((F + 255) / 256, 1), dim3(256), 0, st, gu, act, F);
    WD_LAUNCH_CHECK();
    enqueue(k_q8_0_quantize, dim3((F / 32 + 31) / 32), dim3(256), 0, st, act, F / 32, aq, ad);
    WD_LAUNCH_CHECK();
    return grouped_gemv(WD_TYPE_Q8_0, d, 1, H, F, s, aq, ad, 0, s->down_f32, nullptr, st);
}

namespace {

// The hand-off buffers of the resident stack kernel, allocated on first use.
int resident_prepare(wd_moe_scratch *s) {
    if (s->res_block) return WD_OK;
    uint8_t *alloc = nullptr;
    WD_HIP(hipMalloc(reinterpret_cast<void **>(&alloc), kHandBytes + kSideChunk));
    uint8_t *const b = reinterpret_cast<uint8_t *>((reinterpret_cast<uintptr_t>(alloc) + kSideChunk - 1) & ~static_cast<uintptr_t>(kSideChunk - 1));
    int *const votes = s->h_ids + 48;
    std::memset(votes, 0, sizeof(int) * 8 * 2 * kHandChunks);
    hipError_t e = enqueue_reported(k_hand_block_init, dim3(kHandBytes / 16 / 256 / 4 + 1), dim3(256), 0, nullptr, reinterpret_cast<uint4 *>(b));
    if (e == hipSuccess) e = enqueue_reported(k_side_votes, dim3(8 * 2 * kHandChunks), dim3(64), 0, nullptr, reinterpret_cast<uint32_t *>(b), votes);
    if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
    if (e != hipSuccess) {
        (void)hipFree(alloc);
        return fail(WD_ERR_HIP, "MoE stack: the hand-off block's first launch failed: %s", hipGetErrorString(e));
    }
    s->res_flips = 0;
    for (int q = 0; q < 2 * kHandChunks; ++q) s->res_flips |= static_cast<unsigned>(side_flip_of(votes + 8 * q)) << q;
    s->res_alloc = alloc;
    s->res_block = b;
    return WD_OK;
}

// The device copy of these layer descriptors: the one made for an equal stack before, or a new one (null: none may be
// made now - a graph is being recorded, or the scratch already holds kResMaxDescSets different stacks).
constexpr size_t kResMaxDescSets = 32;
ResidentLayer *resident_descriptors(wd_moe_scratch *s, const std::vector<ResidentLayer> &want, bool capturing) {
    for (const wd_moe_scratch::ResDescSet &d : s->res_sets)
        if (d.shadow.size() == want.size() && std::memcmp(d.shadow.data(), want.data(), sizeof(ResidentLayer) * want.size()) == 0) return d.dev;
    if (capturing || s->res_sets.size() >= kResMaxDescSets) return nullptr;
    wd_moe_scratch::ResDescSet d;
    const size_t desc_bytes = sizeof(ResidentLayer) * kResMaxLayers + sizeof(ResidentViews);
    if (hipMalloc(reinterpret_cast<void **>(&d.dev), desc_bytes) != hipSuccess) return nullptr;
    const ResidentViews v{s->logits, s->weights, s->accum, s->down_f32, s->shared_gate, s->ids};
    if (hipMemcpy(d.dev, want.data(), sizeof(ResidentLayer) * want.size(), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(d.dev + kResMaxLayers, &v, sizeof(v), hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipFree(d.dev);
        return nullptr;
    }
    d.shadow = want;
    s->res_sets.push_back(d);
    return d.dev;
}

bool aligned16(const void *p, size_t stride) { return reinterpret_cast<uintptr_t>(p) % 16 == 0 && stride % 16 == 0; }

// Whether the stack can run as one resident launch (see wd_resident.cuh for the geometry it is written for).
bool resident_shape(const wd_moe_layer *layers, int n_layers, const wd_moe_scratch *s, unsigned flags) {
    if (flags != 0 || n_layers > kResMaxLayers || s->gup != nullptr) return false;
    const wd_moe_layer &f = layers[0];
    if (f.hidden != kResH || f.expert_ffn != kResF || f.n_experts > 512 || f.n_experts % 8 != 0 || f.top_k > kResMaxK) return false;
    if (!consumes_q8k(f.gate_type) && f.gate_type != WD_TYPE_Q8_0) return false;
    for (int l = 0; l < n_layers; ++l) {
        const wd_moe_layer &L = layers[l];
        if (L.hidden != f.hidden || L.expert_ffn != f.expert_ffn || L.n_experts != f.n_experts || L.top_k != f.top_k) return false;
        if (L.gate_type != f.gate_type || L.up_type != f.gate_type || L.down_type != WD_TYPE_Q8_0 || L.slot_of_expert) return false;
        if (L.gate_stride != f.gate_stride || L.up_stride != f.up_stride || L.down_stride != f.down_stride) return false;
        if ((L.shared_gate_inp != nullptr) != (f.shared_gate_inp != nullptr)) return false;
        if (!aligned16(L.gate, L.gate_stride) || !aligned16(L.up, L.up_stride) || !aligned16(L.down, L.down_stride)) return false;
        if (reinterpret_cast<uintptr_t>(L.router) % 16 != 0) return false;
        if (L.shared_gate_inp && (!aligned16(L.shared_down, 0) || reinterpret_cast<uintptr_t>(L.shared_gate_inp) % 4 != 0)) return false;
    }
    return true;
}

constexpr int kTakePerLayer = 1;  // (not an error code) the stack cannot run as one resident launch

template <int TYPE>
int resident_launch(const ResidentArgs &a, wd_moe_scratch *s, hipStream_t st) {
    if (s->res_fits < 0) {  // both variants of the kernel (with and without the time stamps) must fit
        int plain = 0, stamped = 0;
        // (more dynamic LDS than a kernel may have without asking)
        const hipError_t a0 = hipFuncSetAttribute(reinterpret_cast<const void *>(k_stack_resident<TYPE, false>), hipFuncAttributeMaxDynamicSharedMemorySize, kResLdsBytes);
        const hipError_t a1 = hipFuncSetAttribute(reinterpret_cast<const void *>(k_stack_resident<TYPE, true>), hipFuncAttributeMaxDynamicSharedMemorySize, kResLdsBytes);
        const hipError_t e0 = hipOccupancyMaxActiveBlocksPerMultiprocessor(&plain, k_stack_resident<TYPE, false>, kResThreads, kResLdsBytes);
        const hipError_t e1 = hipOccupancyMaxActiveBlocksPerMultiprocessor(&stamped, k_stack_resident<TYPE, true>, kResThreads, kResLdsBytes);
        s->res_fits = (a0 == hipSuccess && a1 == hipSuccess && e0 == hipSuccess && e1 == hipSuccess && std::min(plain, stamped) * s->compute_units >= kResWgs) ? 1 : 0;
    }
    if (!s->res_fits) return kTakePerLayer;  // the workgroups would wait for each other without all being on the device
    SiteScope site(WD_SITE_STACK_RESIDENT, st);
    if (a.trace)  // (the variant with the time stamps only when they are asked for)
        enqueue(k_stack_resident<TYPE, true>, dim3(kResWgs), dim3(kResThreads), kResLdsBytes, st, a);
    else
        enqueue(k_stack_resident<TYPE, false>, dim3(kResWgs), dim3(kResThreads), kResLdsBytes, st, a);
    WD_LAUNCH_CHECK();
    return WD_OK;
}

// Routed experts in a slot pool (see ResidentArgs): the layers' gate/up/down point into the pool, their strides are a slot.
struct ResidentSlots {
    const int32_t *rows_trace;   // device [n_layers][k] slot numbers
    const uint32_t *fill_need;   // device [n_layers]
    const uint32_t *fill_done;   // device [n_layers]
    unsigned n_slots;
};

// Returns kTakePerLayer when the stack has to take the per-layer dispatches instead.
int stack_resident(const wd_moe_layer *layers, int n_layers, float *d_x, float *d_layer_out, wd_moe_scratch *s,
                   const int32_t *d_ids_trace, float residual_scale, hipStream_t st, const ResidentSlots *slots = nullptr) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cap) != hipSuccess) return kTakePerLayer;
    const bool capturing = cap != hipStreamCaptureStatusNone;
    if (!s->res_block) {
        if (capturing) return kTakePerLayer;  // nothing may be allocated while a graph is recorded
        if (const int rc = resident_prepare(s)) return rc;
    }
    std::vector<ResidentLayer> want(n_layers);
    for (int l = 0; l < n_layers; ++l) {
        const wd_moe_layer &L = layers[l];
        ResidentLayer &d = want[l];
        std::memset(&d, 0, sizeof(d));
        d.router = L.router, d.sh_inp = L.shared_gate_inp;
        d.sh_gate = L.shared_gate, d.sh_up = L.shared_up, d.sh_down = L.shared_down;
        d.gate = L.gate, d.up = L.up, d.down = L.down;
        d.w_scale = L.expert_scale;
    }
    ResidentLayer *const descriptors = resident_descriptors(s, want, capturing);
    if (!descriptors) return kTakePerLayer;
    // a wait of an earlier launch on this scratch ran out: its results were NaN, and so would this launch's be
    if (reinterpret_cast<const volatile int32_t *>(s->h_ids)[16] != 0)
        return fail(WD_ERR_STATE, "MoE stack: a wait inside an earlier resident launch on this scratch ran out (is other work resident on the device?); "
                                  "wd_moe_scratch_set_wait_limit resets the scratch");
    ResidentArgs a{};
    a.layers = descriptors, a.n_layers = n_layers, a.E = layers[0].n_experts, a.k = layers[0].top_k;
    a.shared = layers[0].shared_gate_inp != nullptr;
    a.gate_stride = layers[0].gate_stride, a.up_stride = layers[0].up_stride, a.down_stride = layers[0].down_stride;
    a.x = d_x, a.out = d_layer_out, a.residual_scale = residual_scale, a.ids_trace = d_ids_trace;
    a.row_limit = static_cast<unsigned>(a.E);
    if (slots) {
        if (!d_ids_trace) return kTakePerLayer;  // (the slots of a layer are known before the launch only with a routing trace)
        a.rows_trace = slots->rows_trace, a.fill_need = slots->fill_need, a.fill_done = slots->fill_done, a.row_limit = slots->n_slots;
    }
    a.views = reinterpret_cast<const ResidentViews *>(descriptors + kResMaxLayers);
    a.hand = s->res_block, a.side_flips = s->res_flips, a.status = s->status, a.spin_limit = s->spin_limit;
    a.status_host = reinterpret_cast<unsigned *>(s->h_ids + 16);
    a.trace = s->trace, a.trace_wg = s->trace_wg, a.trace_layer = s->trace_layer;
    switch (layers[0].gate_type) {
        case WD_TYPE_IQ3_S: return resident_launch<21>(a, s, st);
        case WD_TYPE_IQ2_S: return resident_launch<22>(a, s, st);
        default: return resident_launch<8>(a, s, st);  // Q8_0 gate/up rows
    }
}

}  // namespace

extern "C" int wd_moe_stack_f32(const wd_moe_layer *layers, int n_layers, float *d_x, float *d_layer_out,
                                wd_moe_scratch *s, const int32_t *d_ids_trace, float residual_scale, unsigned flags,
                                void *stream) {
    WD_REQUIRE(layers && n_layers > 0, "MoE stack: no layers");
    WD_REQUIRE(d_x && d_layer_out, "MoE stack: null activation or output pointer");
    for (int l = 0; l < n_layers; ++l) {
        if (const int rc = check_layer(&layers[l], s, flags)) return rc;
    }
    SiteScope site(WD_SITE_STACK_TOTAL, as_stream(stream));
    if (resident_shape(layers, n_layers, s, flags)) {
        const int rc = stack_resident(layers, n_layers, d_x, d_layer_out, s, d_ids_trace, residual_scale, as_stream(stream));
        if (rc != kTakePerLayer) return rc;
    }
    flags &= ~WD_MOE_PER_LAYER;
    const hipStream_t st = as_stream(stream);
    // (layers without dispatch C leave their ids in a record each: all are set back when they have been used, and at the end)
    const bool chain = (flags & (WD_MOE_ONLY_A | WD_MOE_ONLY_B)) && !(flags & WD_MOE_ONLY_C);
    for (int l = 0; l < n_layers; ++l) {
        const int32_t *trace = d_ids_trace ? d_ids_trace + static_cast<size_t>(l) * layers[l].top_k : nullptr;
        int rc = WD_OK;
        {
            SiteScope layer_site(WD_SITE_ROUTED_TOTAL, st);
            rc = layer_dispatch(&layers[l], d_x, d_layer_out, s, flags, trace, d_x, residual_scale, st, l, nullptr, chain);
        }
        if (chain && (rc || l + 1 == n_layers || (l + 1) % kTagRecords == 0)) {
            const int rc_reset = reset_all_published(s, st);
            if (rc == WD_OK) rc = rc_reset;
        }
        if (rc) return rc;
    }
    return WD_OK;
}

namespace {
// Dispatch AB of a token batch: ta.front_wgs workgroups of the first part, and with `routed` those of the second.
template <int TYPE, int FETCH>
void launch_tokens_ab_fetch(const TokenArgs &ta, bool routed, int items, int cus, hipStream_t st) {
    const int H = ta.common.H;
    size_t lds = static_cast<size_t>(ta.T) * (H + sizeof(float) * (H / 256));
    if (FETCH != 0) lds = ((lds + 15) & ~static_cast<size_t>(15)) + 8 * 2 * static_cast<size_t>(iq_cover_bytes<TYPE>(H / 256));
    lds = tokens_ab_lds(H, lds);
    // persistent: as many workgroups as a compute unit holds walk the items
    auto grid = [&](int per_cu) { return dim3(ta.front_wgs + (routed ? std::min(items, per_cu * cus) : 0)); };
    if (ta.T <= 4) enqueue(k_tokens_ab<TYPE, 4, FETCH>, grid(kTokensBPerCu<TYPE, 4, FETCH>), dim3(512), lds, st, ta);
    else enqueue(k_tokens_ab<TYPE, kMaxTokens, FETCH>, grid(kTokensBPerCu<TYPE, kMaxTokens, FETCH>), dim3(512), lds, st, ta);
}
template <int TYPE>
void launch_tokens_ab(const wd_moe_layer *L, const TokenArgs &ta, bool routed, int items, int cus, bool table, bool tables_aligned, hipStream_t st) {
    const int H = L->hidden;
    // rows of tensors that start on 16-byte boundaries: the aligned fetch, one item ahead
    auto al16 = [](const void *p, size_t v) { return reinterpret_cast<uintptr_t>(p) % 16 == 0 && v % 16 == 0; };
    const bool words = table ? tables_aligned
                             : (L->slot_of_expert ? al16(L->slot_pool, L->slot_bytes) && L->slot_gate_bytes % 16 == 0
                                                  : al16(L->gate, L->gate_stride) && al16(L->up, L->up_stride));
    if (!words || H > 4096) launch_tokens_ab_fetch<TYPE, 0>(ta, routed, items, cus, st);
    else if (H == 2048) launch_tokens_ab_fetch<TYPE, 8>(ta, routed, items, cus, st);
    else if (H == 2560) launch_tokens_ab_fetch<TYPE, 10>(ta, routed, items, cus, st);
    else if (H <= 2304) launch_tokens_ab_fetch<TYPE, 1>(ta, routed, items, cus, st);
    else launch_tokens_ab_fetch<TYPE, 2>(ta, routed, items, cus, st);
}
template <int KIND, int LPR, int PASSES = (LPR == 16 ? 1 : 2)>  // (tokens_c_even_lanes: more than 16 blocks for the others)
void launch_tokens_c_even(const TokenArgs &ta, hipStream_t st) {
    if constexpr (PASSES * LPR < 48) {  // (as in launch_layer_c_even)
        if (ta.common.F > 32 * PASSES * LPR) return launch_tokens_c_even<KIND, LPR, (PASSES < 4 ? PASSES + 1 : 6)>(ta, st);
    }
    const size_t lds = layer_c_lds(static_cast<size_t>(ta.T) * (ta.common.k + 1), 16, kTokensCEvenWaves * static_cast<size_t>(layer_c_even_wave_bytes<LPR>(ta.common.F)));
    enqueue(k_tokens_c_even<KIND, LPR, PASSES>, dim3(256), dim3(64 * kTokensCEvenWaves), lds, st, ta);
}
// Lanes per row of the form with hidden / 256 rows per workgroup (k_tokens_c_even), 0 where the eight-row form stays: it pays where
// the rows take fewer passes than with eight lanes each, for more than 16 blocks (up to hidden 1024: for all).  us per layer of the
// whole pass, weights from HBM, eight-row / even: four tokens, top-8 and the shared expert, 736: hidden 512 44.3 / 40.8, 1280 47.3 / 44.6, 2304 69.7 /
// 64.9, but (three passes either way) 1536 47.4 / 47.3, 3072 71.9 / 73.4; seven tokens, top-5, IQ4_NL of 1184: 1024 70.8 / 57.9, 1536
// 73.7 / 64.6, 2560 96.1 / 86.8, 3072 111 / 104; five, top-4, IQ4_NL of 480: 1024 30.0 / 29.3, but (two passes either way) 2304
// 40.2 / 41.1.  Beyond hidden 3072, where the groups are of seven and eight rows, nothing is left: 3584 / 1184 113.5 / 113.1, 736 73.9 / 75.3.
int tokens_c_even_lanes(int H, int F) {
    const int R = H / 256, nb = F / 32;
    const int lanes = R <= 4 ? 16 : (R == 5 || R == 9 || R == 10 ? 12 : (R == 6 || R == 11 || R == 12 ? 10 : 8));
    return (nb > 16 || R <= 4) && (nb + lanes - 1) / lanes < (nb + 7) / 8 ? lanes : 0;
}
template <int KIND>
void launch_tokens_c_even(int lanes, const TokenArgs &ta, hipStream_t st) {
    if (lanes == 16) launch_tokens_c_even<KIND, 16>(ta, st);
    else if (lanes == 12) launch_tokens_c_even<KIND, 12>(ta, st);
    else launch_tokens_c_even<KIND, 10>(ta, st);
}
template <int KIND, int PASSES>
void launch_tokens_c(const TokenArgs &ta, hipStream_t st) {
    constexpr int kWaves = kTokensCWaves<PASSES>;
    const size_t lds = layer_c_lds(static_cast<size_t>(ta.T) * (ta.common.k + 1), 8, kWaves * static_cast<size_t>(layer_c8_wave_bytes<false>(ta.common.F)));
    enqueue(k_tokens_c<KIND, PASSES>, ta.common.H / 8, 64 * kWaves, lds, st, ta);
}
template <int KIND>
void launch_tokens_c(const TokenArgs &ta, hipStream_t st) {
    const int F = ta.common.F;
    if (F <= 512) launch_tokens_c<KIND, 2>(ta, st);
    else if (F <= 768) launch_tokens_c<KIND, 3>(ta, st);
    else if (F <= 1024) launch_tokens_c<KIND, 4>(ta, st);
    else launch_tokens_c<KIND, 6>(ta, st);
}
// gu_table / down_table: null, or device tables of pointers ([entry][2] gate and up, [entry] down) that take the place of
// the layer's routed tensors, the ids of the pass being entry numbers; tables_aligned: every pointer in them is 16-byte aligned.
int tokens_pass(const wd_moe_layer *L, const float *d_x, float *d_out, int tokens, wd_moe_scratch *const *scratch_per_token,
                unsigned flags, void *stream, const uint8_t *const *gu_table, const uint8_t *const *down_table, bool tables_aligned) {
    WD_REQUIRE(tokens > 0 && tokens <= kMaxTokens, "multi-token pass: 1..%d tokens (got %d)", kMaxTokens, tokens);
    WD_REQUIRE(scratch_per_token != nullptr && d_x && d_out, "multi-token pass: null pointer");
    for (int t = 0; t < tokens; ++t) {
        WD_REQUIRE(scratch_per_token[t] != nullptr, "multi-token pass: null scratch for token %d", t);
        for (int q = 0; q < t; ++q)
            WD_REQUIRE(scratch_per_token[q] != scratch_per_token[t], "multi-token pass: tokens %d and %d share a scratch", q, t);
        if (const int rc = check_layer(L, scratch_per_token[t], flags)) return rc;
    }
    hipStream_t st = as_stream(stream);
    const int H = L->hidden, F = L->expert_ffn, k = L->top_k;
    SiteScope total_site(WD_SITE_TOKENS_TOTAL, st);
    // the union pass takes every gate/up type (Q8_0 and IQ4_NL rows up to hidden 4096); down rows of more than 48 blocks take the
    // one-token dispatch per token, on the activations the union pass left
    const bool iq = consumes_q8k(L->gate_type);
    const bool union_path = !(flags & WD_MOE_STAGED) && (iq || H <= 4096) && tokens * k <= 128 &&
                            scratch_per_token[0]->gup == nullptr &&
                            !(flags & (WD_MOE_ONLY_A | WD_MOE_ONLY_B | WD_MOE_ONLY_C | WD_MOE_DRY));
    const bool down_tokens = F <= 1536;
    if (gu_table) WD_REQUIRE(union_path && iq, "multi-token pass on a pointer table: IQ3_S / IQ2_S gate and up tensors, at most 128 (token, expert) pairs, no staging flags");
    // (before anything is launched: what the dispatches hand on is set back by a dispatch C)
    WD_REQUIRE(!down_table || down_tokens, "multi-token pass on a pointer table: this down tensor (type %d, %d columns) has no multi-token dispatch", L->down_type, F);
    if (!union_path) {
        // same results, one pass per token (every pass reads its own experts)
        for (int t = 0; t < tokens; ++t)
            if (const int rc = layer_dispatch(L, d_x + static_cast<size_t>(t) * H, d_out + static_cast<size_t>(t) * H,
                                              scratch_per_token[t], flags, nullptr, nullptr, 0.0f, st))
                return rc;
        return WD_OK;
    }
    TokenArgs ta{};
    ta.T = tokens;
    ta.common = fused_args(L, d_x, d_out, scratch_per_token[0], flags, nullptr, nullptr, 0.0f);
    ta.common.gate_up = routed_src(L, scratch_per_token[0], nullptr, false);  // the kernels pass the expert id themselves
    ta.common.down = routed_src(L, scratch_per_token[0], nullptr, true);
    if (gu_table) {
        ta.common.gate_up.table = gu_table, ta.common.gate_up.per_expert = 2;
        ta.common.down.table = down_table, ta.common.down.per_expert = 1;
    }
    for (int t = 0; t < tokens; ++t) {
        wd_moe_scratch *s = scratch_per_token[t];
        TokenSlots &k_ = ta.tok[t];
        k_.x = d_x + static_cast<size_t>(t) * H, k_.out = d_out + static_cast<size_t>(t) * H;
        k_.logits = s->logits, k_.ids = s->ids, k_.weights = s->weights, k_.act = s->act;
        k_.shared_gate = s->shared_gate, k_.hand = s->hand, k_.hand_side = s->hand_side;
        k_.expert_out = (flags & WD_MOE_KEEP_EXPERT_OUT) ? s->expert_out : nullptr;
        k_.accum = s->accum, k_.down_f32 = s->down_f32;
        k_.tagged = s->tags(0), k_.tag_side = s->tag_side(), k_.status = s->status;
    }
    LayerArgs &a = ta.common;
    const bool wide = H > 2048 && H <= 4096;  // two waves per router row
    const int router_rows_n = (a.preselected ? 0 : a.E) + (a.sh_inp ? 1 : 0);
    a.n_router_wgs = wide ? (router_rows_n + 3) / 4 : (router_rows_n + 7) / 8;
    const int grid_a = tokens_a_grid(a.n_router_wgs, a.sh_inp ? (F + 7) / 8 : 0).total(tokens, !a.preselected);
    const int items_b = tokens * k * ((F + 7) / 8);
    const int cus = scratch_per_token[0]->compute_units;
    // The parts that `front` and `routed` name
    auto launch_ab = [&](bool front, bool routed) {
        ta.front_wgs = front ? grid_a : 0, ta.wait_ids = front && routed ? 1 : 0;  // (the ids are not in the scratches then)
        a.hand_limit = ta.wait_ids ? a.spin_limit : kHandPatient;
        const size_t lds_q8 = std::max(static_cast<size_t>(tokens) * (H + H / 16), sizeof(float) * static_cast<size_t>(H) + 16);
        const dim3 grid_q8(ta.front_wgs + (routed ? std::min(items_b, 2 * cus) : 0));
        switch (L->gate_type) {
            case WD_TYPE_IQ3_S: launch_tokens_ab<21>(L, ta, routed, items_b, cus, gu_table != nullptr, tables_aligned, st); break;
            case WD_TYPE_IQ2_S: launch_tokens_ab<22>(L, ta, routed, items_b, cus, gu_table != nullptr, tables_aligned, st); break;
            case WD_TYPE_Q8_0: enqueue(k_tokens_ab_q8<0>, grid_q8, dim3(512), lds_q8, st, ta); break;
            default: enqueue(k_tokens_ab_q8<1>, grid_q8, dim3(512), lds_q8, st, ta); break;
        }
        WD_LAUNCH_CHECK();
        return static_cast<int>(WD_OK);
    };
    auto queue = [&]() {
        // One launch where the ids come out of it; ids that are there already need no wait, and the site profiler brackets the parts
        if (!a.preselected && !(flags & WD_MOE_SPLIT_AB) && !SiteProfiler::instance().enabled()) {
            if (const int rc = launch_ab(true, true)) return rc;
        } else {
            if (grid_a > 0) {  // router, selection and shared gate/up of every token
                SiteScope site(WD_SITE_TOKENS_A, st);
                if (const int rc = launch_ab(true, false)) return rc;
            }
            SiteScope site(WD_SITE_TOKENS_B, st);
            if (const int rc = launch_ab(false, true)) return rc;
        }
        SiteScope c_site(WD_SITE_TOKENS_C, st);
        if (!down_tokens) {
            for (int t = 0; t < tokens; ++t)
                if (const int rc = layer_fused(L, d_x + static_cast<size_t>(t) * H, d_out + static_cast<size_t>(t) * H, scratch_per_token[t],
                                               flags | WD_MOE_ONLY_C, nullptr, nullptr, 0.0f, st))
                    return rc;
            return static_cast<int>(WD_OK);
        }
        if (const int lanes = tokens_c_even_lanes(H, F)) L->down_type == WD_TYPE_Q8_0 ? launch_tokens_c_even<0>(lanes, ta, st) : launch_tokens_c_even<1>(lanes, ta, st);
        else L->down_type == WD_TYPE_Q8_0 ? launch_tokens_c<0>(ta, st) : launch_tokens_c<1>(ta, st);
        WD_LAUNCH_CHECK();
        return static_cast<int>(WD_OK);
    };
    const int rc = queue();
    if (rc != WD_OK)  // (as in layer_fused)
        for (int t = 0; t < tokens; ++t) reset_handed(scratch_per_token[t], 0, st);
    return rc;
}
}  // namespace

extern "C" int wd_moe_layer_tokens_f32(const wd_moe_layer *L, const float *d_x, float *d_out, int tokens,
                                       wd_moe_scratch *const *scratch_per_token, unsigned flags, void *stream) {
    return tokens_pass(L, d_x, d_out, tokens, scratch_per_token, flags, stream, nullptr, nullptr, false);
}

extern "C" int wd_moe_layer_tokens_pairs_f32(const wd_moe_layer *L, const uint8_t *const *h_gate, const uint8_t *const *h_up,
                                             const uint8_t *const *h_down, int n_entries, const float *d_x, float *d_out, int tokens,
                                             wd_moe_scratch *const *scratch_per_token, unsigned flags, void *stream) {
    WD_REQUIRE(L && h_gate && h_up && h_down && scratch_per_token && scratch_per_token[0], "multi-token pass on a pointer table: null argument");
    WD_REQUIRE(n_entries > 0 && n_entries <= kPairEntries, "multi-token pass on a pointer table: 1..%d entries (got %d)", kPairEntries, n_entries);
    WD_REQUIRE(flags & WD_MOE_PRESELECTED, "multi-token pass on a pointer table: the selection (entry numbers) must be in the scratches");
    bool aligned = true;
    for (int i = 0; i < n_entries; ++i) {
        WD_REQUIRE(h_gate[i] && h_up[i] && h_down[i], "multi-token pass on a pointer table: entry %d has a null pointer", i);
        WD_REQUIRE((reinterpret_cast<uintptr_t>(h_gate[i]) | reinterpret_cast<uintptr_t>(h_up[i]) | reinterpret_cast<uintptr_t>(h_down[i])) % 2 == 0,
                   "multi-token pass on a pointer table: entry %d is not 2-byte aligned", i);
        aligned = aligned && (reinterpret_cast<uintptr_t>(h_gate[i]) | reinterpret_cast<uintptr_t>(h_up[i]) | reinterpret_cast<uintptr_t>(h_down[i])) % 16 == 0;
    }
    wd_moe_layer Lt = *L;  // the routed tensors come from the table: the descriptor's own are placeholders for the checks
    Lt.slot_of_expert = nullptr;
    Lt.gate = h_gate[0], Lt.up = h_up[0], Lt.down = h_down[0];
    Lt.n_experts = n_entries < Lt.top_k ? Lt.top_k : n_entries;
    wd_moe_scratch *s = scratch_per_token[0];
    hipStream_t st = as_stream(stream);
    // the table goes up through a ring of pinned entries that this call may have to wait for: not something a graph
    // can record
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    WD_HIP(hipStreamIsCapturing(st, &cap));
    WD_REQUIRE(cap == hipStreamCaptureStatusNone, "multi-token pass on a pointer table: the stream is being captured (the table upload cannot be recorded)");
    if (!s->pair_host)  // once per scratch
        WD_HIP(hipHostMalloc(reinterpret_cast<void **>(&s->pair_host), sizeof(void *) * 3 * kPairEntries * kPairRing, hipHostMallocDefault));
    if (!s->pair_dev) WD_HIP(hipMalloc(reinterpret_cast<void **>(&s->pair_dev), sizeof(void *) * 3 * kPairEntries * kPairRing));
    for (hipEvent_t &ev : s->pair_done)
        if (!ev) WD_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    const int slot = s->pair_next;
    s->pair_next = (slot + 1) % kPairRing;
    if (s->pair_used[slot]) WD_HIP(hipEventSynchronize(s->pair_done[slot]));  // the pass that read this entry of the ring has run
    const uint8_t **h = s->pair_host + static_cast<size_t>(slot) * 3 * kPairEntries, **d = s->pair_dev + static_cast<size_t>(slot) * 3 * kPairEntries;
    for (int i = 0; i < kPairEntries; ++i) {  // entries the caller did not give point at entry 0
        const int from = i < n_entries ? i : 0;
        h[2 * i] = h_gate[from], h[2 * i + 1] = h_up[from], h[2 * kPairEntries + i] = h_down[from];
    }
    WD_HIP(hipMemcpyAsync(d, h, sizeof(void *) * 3 * kPairEntries, hipMemcpyHostToDevice, st));
    const int rc = tokens_pass(&Lt, d_x, d_out, tokens, scratch_per_token, flags, stream, d, d + 2 * kPairEntries, aligned);
    WD_HIP(hipEventRecord(s->pair_done[slot], st));
    s->pair_used[slot] = true;
    return rc;
}
