// __global__ kernels of the stand-alone operators (64-wide wavefronts, 256-thread workgroups).
#pragma once

#include "wd_rows.cuh"

namespace wd {

// Where the weight matrices of a grouped dispatch live.
//   table != null      matrix m = table[m]                       (expert pointer table)
//   ids   != null      matrix m belongs to expert ids[m / per_expert], tensor m % per_expert:
//                        resident:  base[t] + expert * stride[t]
//                        slot pool: pool + slot_of_expert[expert] * slot_bytes + slot_off[t]
//   otherwise          the single matrix `single`
struct MatSrc {
    const uint8_t *single;
    const uint8_t *const *table;
    const int32_t *ids;
    int per_expert;
    const uint8_t *base[2];
    size_t stride[2];
    const int32_t *slot_of_expert;
    const uint8_t *pool;
    size_t slot_bytes;
    size_t slot_off[2];
    unsigned *slot_status;  // set to 2 when an expert without a slot is asked for, to 3 for one that the layer does not have (may be null)
    unsigned n_experts;     // experts of the tensors (0: not known, ids are taken as they are)
};

// An id that the caller gave (a routing trace, a selection left in the scratch) may lie outside the layer's experts: such
// a request is reported through the status word and reads expert 0 instead of an address outside the tensors.
WD_DEV int checked_expert(const MatSrc &s, int e) {
    if (s.n_experts != 0u && static_cast<unsigned>(e) >= s.n_experts) {
        if (s.slot_status) __hip_atomic_store(s.slot_status, 3u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        e = 0;
    }
    return e;
}

// The slot of an expert that is not in the pool is -1: such a request is reported through the status word and reads
// slot 0 (memory that exists, values that mean nothing) instead of an address before the pool.
WD_DEV size_t checked_slot(const MatSrc &s, int slot) {
    if (slot < 0) {
        if (s.slot_status) __hip_atomic_store(s.slot_status, 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        slot = 0;
    }
    return static_cast<size_t>(slot);
}

WD_DEV const uint8_t *mat_ptr(const MatSrc &s, int m) {
    if (s.table) return s.table[m];
    if (s.ids) {
        const int j = m / s.per_expert, t = m - j * s.per_expert;
        const int e = checked_expert(s, s.ids[j]);
        if (s.slot_of_expert) return s.pool + checked_slot(s, s.slot_of_expert[e]) * s.slot_bytes + s.slot_off[t];
        return s.base[t] + static_cast<size_t>(e) * s.stride[t];
    }
    return s.single;
}

// Tensor T (0 = the first, 1 = the second of an expert's tensors in this source) of expert e.  T is a template
// argument so that base, stride and slot offset are fixed members of the argument block (scalar registers, loaded
// without waiting for e) instead of a lookup by a computed index.
template <int T>
WD_DEV const uint8_t *mat_ptr_expert(const MatSrc &s, int e) {
    if (s.slot_of_expert) return s.pool + checked_slot(s, s.slot_of_expert[e]) * s.slot_bytes + s.slot_off[T];
    return s.base[T] + static_cast<size_t>(e) * s.stride[T];
}

// The same for an e that is the same in every lane: the slot comes through the scalar path, so the lookup neither
// waits for nor is counted among the wave's vector loads.
// `missing` is set when it has none.
template <int T>
WD_DEV const uint8_t *mat_ptr_expert_uniform(const MatSrc &s, int e, bool &missing) {
    if (s.slot_of_expert) {
        const int slot = sld_i32(s.slot_of_expert + e);
        missing = slot < 0;
        return s.pool + checked_slot(s, slot) * s.slot_bytes + s.slot_off[T];
    }
    return s.base[T] + static_cast<size_t>(e) * s.stride[T];
}
template <int T>
WD_DEV const uint8_t *mat_ptr_expert_uniform(const MatSrc &s, int e) {
    bool missing;
    return mat_ptr_expert_uniform<T>(s, e, missing);
}

__global__ void k_fill_u32(uint32_t *dst, uint32_t v, size_t n) {
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = v;
}

// ---- Q8_K quantiser: one wave per 256-value block, four values per lane -------------------
__global__ __launch_bounds__(256) void k_q8_k_quantize(const float *__restrict__ x, int blocks,
                                                        int8_t *__restrict__ qs, float *__restrict__ scales,
                                                        int16_t *__restrict__ bsums) {
    const int lane = threadIdx.x & 63;
    const int blk = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (blk >= blocks) return;
    const float4 v = reinterpret_cast<const float4 *>(x + static_cast<size_t>(blk) * 256)[lane];
    float amax = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(v.x), __builtin_fabsf(v.y)),
                                 __builtin_fmaxf(__builtin_fabsf(v.z), __builtin_fabsf(v.w)));
    amax = wave_max_nonneg(amax);
    uint32_t packed = 0;
    int part = 0;
    float d = 0.0f;
    if (amax != 0.0f) {
        // always-negative inverse scale (reference convention): quants carry the sign of -x
        const float iscale = -127.0f / amax;
        const int q0 = min(127, static_cast<int>(__builtin_rintf(v.x * iscale)));
        const int q1 = min(127, static_cast<int>(__builtin_rintf(v.y * iscale)));
        const int q2 = min(127, static_cast<int>(__builtin_rintf(v.z * iscale)));
        const int q3 = min(127, static_cast<int>(__builtin_rintf(v.w * iscale)));
        packed = (q0 & 0xff) | ((q1 & 0xff) << 8) | ((q2 & 0xff) << 16) | (static_cast<uint32_t>(q3 & 0xff) << 24);
        part = q0 + q1 + q2 + q3;
        d = 1.0f / iscale;
    }
    reinterpret_cast<uint32_t *>(qs + static_cast<size_t>(blk) * 256)[lane] = packed;
    part = quad_sum_i(part);
    if ((lane & 3) == 0) bsums[static_cast<size_t>(blk) * 16 + (lane >> 2)] = static_cast<int16_t>(part);
    if (lane == 0) scales[blk] = d;
}

// ---- Q8_0 quantiser: eight lanes per 32-value block, four values per lane -----------------
// (inv: 127 / amax, for a caller that packs more than four values of a block)
WD_DEV uint32_t q8_0_pack4_scaled(float4 v, float inv) {
    const int q0 = max(-128, min(127, static_cast<int>(__builtin_rintf(v.x * inv))));
    const int q1 = max(-128, min(127, static_cast<int>(__builtin_rintf(v.y * inv))));
    const int q2 = max(-128, min(127, static_cast<int>(__builtin_rintf(v.z * inv))));
    const int q3 = max(-128, min(127, static_cast<int>(__builtin_rintf(v.w * inv))));
    return (q0 & 0xff) | ((q1 & 0xff) << 8) | ((q2 & 0xff) << 16) | (static_cast<uint32_t>(q3 & 0xff) << 24);
}
WD_DEV uint32_t q8_0_pack4(float4 v, float amax) {
    if (amax == 0.0f) return 0u;
    const float inv = 127.0f / amax;
    const int q0 = max(-128, min(127, static_cast<int>(__builtin_rintf(v.x * inv))));
    const int q1 = max(-128, min(127, static_cast<int>(__builtin_rintf(v.y * inv))));
    const int q2 = max(-128, min(127, static_cast<int>(__builtin_rintf(v.z * inv))));
    const int q3 = max(-128, min(127, static_cast<int>(__builtin_rintf(v.w * inv))));
    return (q0 & 0xff) | ((q1 & 0xff) << 8) | ((q2 & 0xff) << 16) | (static_cast<uint32_t>(q3 & 0xff) << 24);
}

// ---- the quantisers' arithmetic on ordinary blocks ----------------------------------------------------------------
// In dispatch C the quantisation of 512 values by a wave was 100 vector instructions, of 164 with the down rows behind it.  On blocks whose largest
// magnitude is between 2^-100 and 2^100 and which hold no NaN it takes 55, with the same bits:
//   * a quotient by one step of Newton's iteration on the reciprocal and one correction of the quotient: what remains of an IEEE division without the scaling
//     and the special cases (equal to it for every float of the range, 1,677,721,601 of them, for 127 / a and for a / 127: test_gpu_quantiser);
//   * a value times the inverse scale rounded to an integer by adding 1.5 * 2^23: the sum's low byte is the quant, and anything that is not a number
//     of the range shows in the upper bits, of eight values at once.
// A wave with any other block takes the general form for all of its blocks.  (us per layer: 2560 / 640, IQ4_NL down 21.7, so 21.4; 4096 / 1536 37.6, 37.2.  The
// resident stack, 48 layers: the same within noise; the token batches' dispatch has no registers for it.)
constexpr float kQuantAdd = 0x1.8p23f;
constexpr uint32_t kQuantTop = 0x4b400000u + 127u;   // bits of the sum for 127; smaller ones down to -128 are below
constexpr uint32_t kQuantLo = (127u - 100u) << 23, kQuantSpan = 200u << 23;  // bits of 2^-100, up to 2^100
WD_DEV float quot_ordinary(float n, float a) {
    float y = __builtin_amdgcn_rcpf(a);
    y = __builtin_fmaf(__builtin_fmaf(-a, y, 1.0f), y, y);
    const float q = n * y;
    return __builtin_fmaf(__builtin_fmaf(-a, q, n), y, q);
}
WD_DEV float over_127(float a) {
    constexpr float c = 1.0f / 127.0f;
    const float q = a * c;
    return __builtin_fmaf(__builtin_fmaf(-127.0f, q, a), c, q);
}
// max(|a|, |b|, |c|).  (fmaxf of values from memory takes an instruction more per value, which quiets signalling NaN; here a NaN shows in the quants.)
WD_DEV float max3_abs(float a, float b, float c) {
    float m;
    asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(m) : "v"(a), "v"(b), "v"(c));
    return m;
}
WD_DEV uint32_t quants_ordinary(const float4 &v, float inv, uint32_t &worst) {
    const uint32_t t0 = f_bits(v.x * inv + kQuantAdd), t1 = f_bits(v.y * inv + kQuantAdd), t2 = f_bits(v.z * inv + kQuantAdd), t3 = f_bits(v.w * inv + kQuantAdd);
    worst = max(max(worst, t0), t1), worst = max(max(worst, t2), t3);
    const uint32_t lo = __builtin_amdgcn_perm(t1, t0, 0x0c0c0400u), hi = __builtin_amdgcn_perm(t3, t2, 0x0c0c0400u);
    return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}
// any lane's (the same in every lane)
WD_DEV bool quants_not_ordinary(uint32_t worst, uint32_t amax_bits, bool on = true) {
    return __builtin_amdgcn_ballot_w64(on && (worst > kQuantTop || amax_bits - kQuantLo > kQuantSpan)) != 0ull;
}
// f2h_ref of a number that is not NaN
WD_DEV uint16_t f2h_number(float v) {
    const uint16_t h = __builtin_bit_cast(uint16_t, static_cast<_Float16>(v));
    return __builtin_fabsf(v) < 0x1p-24f ? static_cast<uint16_t>(h & 0x8000u) : h;
}


__global__ __launch_bounds__(256) void k_q8_0_quantize(const float *__restrict__ x, int blocks,
                                                        int8_t *__restrict__ qs, uint16_t *__restrict__ scales) {
    const int sub = threadIdx.x & 7;
    const int blk = blockIdx.x * 32 + (threadIdx.x >> 3);
    const bool on = blk < blocks;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (on) v = reinterpret_cast<const float4 *>(x + static_cast<size_t>(blk) * 32)[sub];
    float amax = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(v.x), __builtin_fabsf(v.y)),
                                 __builtin_fmaxf(__builtin_fabsf(v.z), __builtin_fabsf(v.w)));
    amax = oct_max_nonneg(amax);
    if (!on) return;
    reinterpret_cast<uint32_t *>(qs + static_cast<size_t>(blk) * 32)[sub] = q8_0_pack4(v, amax);
    if (sub == 0) scales[blk] = f2h_ref(amax / 127.0f);
}

// ---- the reference's plain Q8_0 x Q8_1 path and its half-input quantiser ----------------------------------------
// IEEE float -> half bits (the reference's __float2half), unlike f2h_ref.
WD_DEV uint16_t f2h_rn(float v) {
    const _Float16 f = static_cast<_Float16>(v);
    uint16_t h;
    __builtin_memcpy(&h, &f, 2);
    return h;
}
// The largest |v| of the block of 32 values held four per lane by eight consecutive lanes.
WD_DEV float block32_amax(const float4 &v) {
    float amax = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(v.x), __builtin_fabsf(v.y)),
                                 __builtin_fmaxf(__builtin_fabsf(v.z), __builtin_fabsf(v.w)));
    return oct_max_nonneg(amax);
}
// q8_1_quantize_f32_kernel, src/lowbit.cuh:287-308: d = amax / 127, q = roundf(x / d) (a division; halves away from
// zero), scale = half(d).  Eight lanes per block, four values per lane.
__global__ __launch_bounds__(256) void k_q8_1_quantize(const float *__restrict__ x, int blocks, int8_t *__restrict__ qs,
                                                        uint16_t *__restrict__ scales) {
    const int sub = threadIdx.x & 7;
    const int blk = blockIdx.x * 32 + (threadIdx.x >> 3);
    const bool on = blk < blocks;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (on) v = reinterpret_cast<const float4 *>(x + static_cast<size_t>(blk) * 32)[sub];
    const float amax = block32_amax(v);
    if (!on) return;
    const float d = amax / 127.0f;
    auto q = [&](float t) { return amax == 0.0f ? 0 : static_cast<int>(__builtin_roundf(t / d)); };
    const int q0 = q(v.x), q1 = q(v.y), q2 = q(v.z), q3 = q(v.w);
    reinterpret_cast<uint32_t *>(qs + static_cast<size_t>(blk) * 32)[sub] =
        (q0 & 0xff) | ((q1 & 0xff) << 8) | ((q2 & 0xff) << 16) | (static_cast<uint32_t>(q3 & 0xff) << 24);
    if (sub == 0) scales[blk] = f2h_rn(d);
}
// q8_0_quantize_half_kernel, src/warodecode.cu:1504-1520: half input, inv = 127 / amax, q = lrintf(v * inv) clamped to
// +-127, scale = half(amax / 127).
__global__ __launch_bounds__(256) void k_q8_0_quantize_f16(const uint16_t *__restrict__ x, int blocks, int8_t *__restrict__ qs,
                                                            uint16_t *__restrict__ scales) {
    const int sub = threadIdx.x & 7;
    const int blk = blockIdx.x * 32 + (threadIdx.x >> 3);
    const bool on = blk < blocks;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (on) {
        const uint2 h = reinterpret_cast<const uint2 *>(x + static_cast<size_t>(blk) * 32)[sub];
        v = make_float4(h2f(static_cast<uint16_t>(h.x)), h2f(static_cast<uint16_t>(h.x >> 16)), h2f(static_cast<uint16_t>(h.y)),
                        h2f(static_cast<uint16_t>(h.y >> 16)));
    }
    const float amax = block32_amax(v);
    if (!on) return;
    const float inv = amax == 0.0f ? 0.0f : 127.0f / amax;
    auto q = [&](float t) { return max(-127, min(127, static_cast<int>(__builtin_rintf(t * inv)))); };
    const int q0 = q(v.x), q1 = q(v.y), q2 = q(v.z), q3 = q(v.w);
    reinterpret_cast<uint32_t *>(qs + static_cast<size_t>(blk) * 32)[sub] =
        (q0 & 0xff) | ((q1 & 0xff) << 8) | ((q2 & 0xff) << 16) | (static_cast<uint32_t>(q3 & 0xff) << 24);
    if (sub == 0) scales[blk] = f2h_rn(amax / 127.0f);
}
// q8_0_q8_1_gemv_f32_kernel, src/lowbit.cuh:310-341: one wave per row, lane = block (64 blocks a pass); the row's sum
// runs over the blocks in ascending order, one rounded multiply of the two scales, one with the integer sum, one add.
// block_sums (optional): int32 [rows][cols / 32].
__global__ __launch_bounds__(256) void k_gemv_q8_0_q8_1(const uint8_t *__restrict__ w, int rows, int cols,
                                                         const int8_t *__restrict__ qs, const uint16_t *__restrict__ scales,
                                                         float *__restrict__ y, int32_t *__restrict__ block_sums) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int nb = cols >> 5;
    const uint8_t *wr = w + static_cast<size_t>(row) * nb * 34;
    float sum = 0.0f;
    for (int base = 0; base < nb; base += 64) {
        const int b = base + lane;
        float prod = 0.0f;
        if (b < nb) {
            const uint8_t *blk = wr + static_cast<size_t>(b) * 34;
            int dot = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t wq = static_cast<uint32_t>(ldu<uint16_t>(blk + 2 + 4 * i)) | (static_cast<uint32_t>(ldu<uint16_t>(blk + 4 + 4 * i)) << 16);
                dot = sdot4(wq, *reinterpret_cast<const uint32_t *>(qs + b * 32 + 4 * i), dot);
            }
            if (block_sums) block_sums[static_cast<size_t>(row) * nb + b] = dot;
            const float scale = h2f(ldu<uint16_t>(blk)) * h2f(scales[b]);
            prod = scale * static_cast<float>(dot);
        }
        const int n = min(64, nb - base);
        for (int i = 0; i < n; ++i) sum = sum + readlane_f(prod, i);
    }
    if (lane == 0) y[row] = sum;
}
// Element-wise half <-> float (IEEE rounding on the way down).
__global__ void k_f16_to_f32(const uint16_t *__restrict__ src, float *__restrict__ dst, size_t n) {
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = h2f(src[i]);
}
__global__ void k_f32_to_f16(const float *__restrict__ src, uint16_t *__restrict__ dst, size_t n) {
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = f2h_rn(src[i]);
}

// ---- router GEMV: 32 lanes per row, lane t owns accumulator t of the 4x8 scheme --------------
// (src/qwen38_moe.cuh:198-245).  Optional extra row (the shared expert's gate vector).
__global__ __launch_bounds__(256) void k_router_gemv(const float *__restrict__ w, const float *__restrict__ x,
                                                      float *__restrict__ logits, int rows, int cols,
                                                      const float *__restrict__ extra_w,
                                                      float *__restrict__ extra_out) {
    const int t = threadIdx.x & 31;
    const int row = blockIdx.x * 8 + (threadIdx.x >> 5);
    const int total = rows + (extra_w ? 1 : 0);
    const bool on = row < total;
    const float *wr = on ? (row < rows ? w + static_cast<size_t>(row) * cols : extra_w) : w;
    const int np = cols & ~31;
    float s = 0.0f;
    if (on) {
#pragma unroll 16
        for (int i = 0; i < np; i += 32) s = __builtin_fmaf(wr[i + t], x[i + t], s);
    }
    float o = __shfl_down(s, 16, 32);
    if (t < 16) s = s + o;
    o = __shfl_down(s, 8, 32);
    if (t < 8) s = s + o;
    o = __shfl_down(s, 4, 32);
    if (t < 4) s = s + o;
    o = __shfl_down(s, 1, 32);
    if (t == 0 || t == 2) s = s + o;
    o = __shfl_down(s, 2, 32);
    float acc = s + o;
    if (on && t == 0) {
        for (int c = np; c < cols; ++c) acc = acc + wr[c] * x[c];
        if (row < rows)
            logits[row] = acc;
        else
            extra_out[0] = acc;
    }
}

// ---- IQ3_S / IQ2_S x Q8_K GEMV: 16 rows per workgroup, 4 per wave, grid.y = matrix -----------
template <int TYPE, bool PART>
__global__ __launch_bounds__(256) void k_gemv_iq(MatSrc src, int rows, int cols, const int8_t *__restrict__ act_qs,
                                                  const float *__restrict__ act_d, float *__restrict__ out,
                                                  int32_t *__restrict__ partials, int ppr) {
    __shared__ IqTables tables;
    stage_tables<TYPE == 21, TYPE == 22>(tables, threadIdx.x, 256);
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = blockIdx.y;
    const uint8_t *w = mat_ptr(src, m);
    const int nb = cols >> 8;
    const size_t rb = static_cast<size_t>(nb) * (TYPE == 21 ? 110 : 82);
    const int r0 = blockIdx.x * 16 + wave * 4;
    for (int r = r0; r < min(rows, r0 + 4); ++r) {
        int32_t *pp = PART ? partials + (static_cast<size_t>(m) * rows + r) * ppr : nullptr;
        const float y = iq_row_q8k<TYPE, PART>(w + static_cast<size_t>(r) * rb, nb, tables, act_qs, act_d, lane, pp);
        if (lane == 0) out[static_cast<size_t>(m) * rows + r] = y;
    }
}

// ---- IQ3_S / IQ2_S x Q8_K, one matrix: eight rows at a time, one lane per (row, super-block) ------------------------
// A lane decodes all eight 32-value blocks of one super-block and keeps the eight chunk sums over them in its registers
// (integers: any order), which takes the exchange between the lanes of a super-block away that k_gemv_iq pays per row (seven
// lane swaps and as many additions for eight super-blocks); the sums then go through LDS once, and lane (row, chunk) runs the
// chain of its chunk over the super-blocks in order, eight rows at a time (the other form: sixteen instructions per row).
// Eight rows are 8 nb blocks in a row, a whole number of 16-byte words; the words are fetched lane by lane (two-byte aligned
// where the rows are) and the fields are picked out of LDS.  The activation is staged with a stride of 272 bytes per
// super-block (eight of them at once fall on different banks).
// us, k_gemv_iq -> here: IQ3_S 2048 x 2048 6.0 -> 4.1, 5000 x 2560 11.4 -> 6.7, 500 x 16384 29.5 -> 8.5 (split); 20000 x 4096
// 21.8 -> 17.7, 40000 x 5120 55.5 -> 35.2 = 2.5 TB/s (many rows); IQ2_S 6.2 -> 4.2, 11.1 -> 6.0, 30.1 -> 7.3; 19.8 -> 14.7,
// 52.8 -> 29.0.  The many-row form is bound by vector instructions and codebook look-ups: a fourth workgroup per compute unit
// changes nothing (36.2).
template <int TYPE>
constexpr int kIqBlk = TYPE == 21 ? 110 : 82;
constexpr int kIqActStride = 272;
WD_DEV void iq_stage_activation(int8_t *aq, float *ad, const int8_t *act_qs, const float *act_d, int nb, int threads) {
    for (int i = threadIdx.x; i < nb * 16; i += threads)
        *reinterpret_cast<uint4 *>(aq + (i >> 4) * kIqActStride + (i & 15) * 16) = reinterpret_cast<const uint4 *>(act_qs)[i];
    for (int i = threadIdx.x; i < nb; i += threads) ad[i] = act_d[i];
}
WD_DEV void iq_load_act(uint32_t (&a)[8], const int8_t *aq) {
    const uint4 a0 = *reinterpret_cast<const uint4 *>(aq), a1 = *reinterpret_cast<const uint4 *>(aq + 16);
    a[0] = a0.x, a[1] = a0.y, a[2] = a0.z, a[3] = a0.w, a[4] = a1.x, a[5] = a1.y, a[6] = a1.z, a[7] = a1.w;
}
// A super-block in registers: the dwords behind its scale, so that the fields of block ib are picked at compile time.
template <int TYPE>
struct IqBlockRegs {
    static constexpr int kWords = (kIqBlk<TYPE> - 2) / 4;
    uint32_t v[kWords];
    float d;
    // off: the block's (even) offset in the stage; up to four bytes behind the block are read
    WD_DEV void load(const uint8_t *stage, uint32_t off) {
        const uint32_t sh = (off + 2) & 2u;
        const uint32_t *r = reinterpret_cast<const uint32_t *>(stage + (off + 2 - sh));
        d = h2f(*reinterpret_cast<const uint16_t *>(stage + off));
        uint32_t lo = r[0];
#pragma unroll
        for (int j = 0; j < kWords; ++j) {
            const uint32_t hi = r[j + 1];
            v[j] = __builtin_amdgcn_alignbyte(hi, lo, sh);
            lo = hi;
        }
    }
    WD_DEV IqFields fields(int ib) const {
        IqFields f;
        f.d = 0;
        f.qh = v[16 + (ib >> 2)] >> (8 * (ib & 3));  // (of its bits above the eighth none is used)
        if (TYPE == 21) {
            f.qs = make_uint2(v[2 * ib], v[2 * ib + 1]);
            f.sg = v[18 + ib];
            f.sc = v[TYPE == 21 ? 26 : 0] >> (8 * (ib >> 1));
        } else {
            f.qs = make_uint2(v[ib], v[8 + ib]);
            f.sg = 0;
            f.sc = (v[18 + (ib >> 2)] >> (8 * (ib & 3))) & 0xffu;
        }
        return f;
    }
};
constexpr int kIqTileRow = 72;                              // [row][super-block][chunk], rows padded (bank spread)
constexpr int kIqTileWords = 8 * kIqTileRow;

// Many rows: the waves of the grid take the groups of eight rows in turn, eight super-blocks at a time, one such chunk ahead in
// registers.  Rows that are no whole number of chunks end with a chunk of their last eight super-blocks, of which the first
// have been there already and get the scale zero; rows of fewer than eight are one chunk with idle lanes.  rows >= 8.
// dynamic LDS: nb * kIqActStride, nb floats (rounded to 16 bytes), then per wave the stage, later the tile in the same place.
template <int TYPE>
constexpr int kIqWaveStage = 64 * kIqBlk<TYPE> + 16;
template <int TYPE, bool PART>
__global__ __launch_bounds__(256) void k_gemv_iq_rows8(const uint8_t *__restrict__ w, int rows, int nb, const int8_t *__restrict__ act_qs,
                                                        const float *__restrict__ act_d, float *__restrict__ out, int32_t *__restrict__ partials) {
    constexpr int kBlk = kIqBlk<TYPE>, kRowWords = 8 * kBlk / 16, kLoads = (8 * kRowWords + 63) / 64;
    static_assert(kIqWaveStage<TYPE> >= (kIqTileWords + 64) * 4, "the tile lies where the stage was");
    __shared__ IqTables tables;
    extern __shared__ __align__(16) uint8_t iq_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int8_t *aq = reinterpret_cast<int8_t *>(iq_lds);
    float *ad = reinterpret_cast<float *>(iq_lds + nb * kIqActStride);
    uint8_t *stage = iq_lds + nb * kIqActStride + ((nb * 4 + 15) & ~15) + wave * kIqWaveStage<TYPE>;
    float *tile = reinterpret_cast<float *>(stage), *tile_d = tile + kIqTileWords;
    const size_t rb = static_cast<size_t>(nb) * kBlk;
    const int n_groups = (rows + 7) >> 3, n_waves = gridDim.x * 4, first = blockIdx.x * 4 + wave;
    const int my_groups = first < n_groups ? (n_groups - first + n_waves - 1) / n_waves : 0;
    const int nchunks = (nb + 7) >> 3, skipped = nb < 8 ? 0 : 8 * nchunks - nb;
    const int row = lane >> 3, pos = lane & 7;
    // (fewer than eight super-blocks: the eight rows are one run of words)
    const int words = nb < 8 ? nb * kBlk / 2 : 8 * kRowWords;
    uint32_t goff[kLoads], loff[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int u = min(i * 64 + lane, words - 1), r = u / kRowWords;
        goff[i] = nb < 8 ? 16u * u : static_cast<uint32_t>(r * rb + 16 * (u - r * kRowWords));
        loff[i] = 16u * u;
    }
    const uint32_t my_block = static_cast<uint32_t>((nb < 8 ? row * nb + min(pos, nb - 1) : 8 * row + pos) * kBlk);
    int f_group = min(first, n_groups - 1), f_chunk = 0, fetched = 0;
    const int items = my_groups * nchunks;
    auto chunk_start = [&](int chunk) { return nb < 8 ? 0 : min(8 * chunk, nb - 8); };
    uint4 f[kLoads];
    auto fetch = [&]() {
        // (a last group of fewer than eight rows is moved up to end with the matrix)
        const uint8_t *p = uniform_ptr(w + static_cast<size_t>(min(8 * f_group, rows - 8)) * rb + static_cast<size_t>(chunk_start(f_chunk)) * kBlk);
#pragma unroll
        for (int i = 0; i < kLoads; ++i) f[i] = gld_u128(p + goff[i]);
        if (++fetched < items) {  // (past the wave's last chunk the same one again, not used)
            if (++f_chunk == nchunks) f_chunk = 0, f_group += n_waves;
        }
    };
    fetch();
    stage_tables<TYPE == 21, TYPE == 22>(tables, threadIdx.x, 256);
    iq_stage_activation(aq, ad, act_qs, act_d, nb, 256);
    __syncthreads();
    if (my_groups == 0) return;  // wave-uniform
    float acc = 0.0f;
    int group = first, chunk = 0;
    for (int t = 0; t < items; ++t) {
        wave_lds_fence();  // the previous chunk's tile has been read
#pragma unroll
        for (int i = 0; i < kLoads; ++i) *reinterpret_cast<uint4 *>(stage + loff[i]) = f[i];
        wave_lds_fence();
        fetch();
        const int b0 = chunk_start(chunk), sb = min(b0 + pos, nb - 1);
        const bool on = b0 + pos < nb && (chunk < nchunks - 1 || pos >= skipped);
        const int out_row = min(8 * group, rows - 8) + row;
        IqBlockRegs<TYPE> blk;
        blk.load(stage, my_block);
        int sum[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int ib = 0; ib < 8; ++ib) {
            uint32_t a[8];
            iq_load_act(a, aq + sb * kIqActStride + ib * 32);
            int p[8];
            iq_chunks<TYPE>(blk.fields(ib), ib, tables, a, p);
#pragma unroll
            for (int c = 0; c < 8; ++c) sum[c] += p[c];
        }
        if (PART && on) {
#pragma unroll
            for (int c = 0; c < 8; ++c) partials[(static_cast<size_t>(out_row) * nb + sb) * 8 + c] = sum[c];
        }
        wave_lds_fence();  // every lane has its block in registers
        float4 *dst = reinterpret_cast<float4 *>(tile + row * kIqTileRow + pos * 8);
        dst[0] = make_float4(static_cast<float>(sum[0]), static_cast<float>(sum[1]), static_cast<float>(sum[2]), static_cast<float>(sum[3]));
        dst[1] = make_float4(static_cast<float>(sum[4]), static_cast<float>(sum[5]), static_cast<float>(sum[6]), static_cast<float>(sum[7]));
        tile_d[lane] = on ? blk.d * ad[sb] : 0.0f;
        wave_lds_fence();
#pragma unroll
        for (int s = 0; s < 8; ++s) acc = __builtin_fmaf(tile_d[row * 8 + s], tile[row * kIqTileRow + s * 8 + pos], acc);
        if (++chunk == nchunks) {
            const float y = close_lanes8(acc);
            if (pos == 0) out[out_row] = TYPE == 22 ? 0.125f * y : y;
            acc = 0.0f, chunk = 0, group += n_waves;
        }
    }
}

// Few rows: one workgroup per group of eight rows, `parts` waves for every eight super-blocks, of which wave `part` takes the
// 32-value blocks part, part + parts, ...; their chunk sums are added (integers) by the wave that runs the chains.
// 64 * parts * ceil(nb / 8) threads, rows >= 8.  dynamic LDS: the activation as above, the rows (8 nb blocks and 16 bytes),
// then a tile per wave.
template <int TYPE>
static size_t iq_split_lds(int nb, int parts) {
    const int nchunks = (nb + 7) / 8;
    return static_cast<size_t>(nb) * kIqActStride + ((nb * 4 + 15) & ~15) + ((static_cast<size_t>(8) * nb * kIqBlk<TYPE> + 31) & ~size_t(15)) +
           static_cast<size_t>(nchunks) * (parts * kIqTileWords + 64) * 4;
}
template <int TYPE, bool PART>
__global__ __launch_bounds__(512) void k_gemv_iq_split(const uint8_t *__restrict__ w, int rows, int nb, int parts, const int8_t *__restrict__ act_qs,
                                                        const float *__restrict__ act_d, float *__restrict__ out, int32_t *__restrict__ partials) {
    constexpr int kBlk = kIqBlk<TYPE>;
    __shared__ IqTables tables;
    extern __shared__ __align__(16) uint8_t iq_lds[];
    const int threads = blockDim.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nchunks = (nb + 7) >> 3, chunk = wave / parts, part = wave - chunk * parts;
    int8_t *aq = reinterpret_cast<int8_t *>(iq_lds);
    float *ad = reinterpret_cast<float *>(iq_lds + nb * kIqActStride);
    uint8_t *stage = iq_lds + nb * kIqActStride + ((nb * 4 + 15) & ~15);
    int32_t *tiles = reinterpret_cast<int32_t *>(stage + ((8 * nb * kBlk + 31) & ~15));
    float *scales = reinterpret_cast<float *>(tiles + nchunks * parts * kIqTileWords);
    const int base_row = min(8 * static_cast<int>(blockIdx.x), rows - 8);
    const uint8_t *src = uniform_ptr(w + static_cast<size_t>(base_row) * nb * kBlk);
    const int words = nb * kBlk / 2;
    // at most eight words per thread: nb 55 words over 64 ceil(nb / 8) threads or more
    uint4 f[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if (i * threads < words) f[i] = gld_u128(src + 16 * min(i * threads + static_cast<int>(threadIdx.x), words - 1));
    stage_tables<TYPE == 21, TYPE == 22>(tables, threadIdx.x, threads);
    iq_stage_activation(aq, ad, act_qs, act_d, nb, threads);
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if (i * threads < words) reinterpret_cast<uint4 *>(stage)[min(i * threads + static_cast<int>(threadIdx.x), words - 1)] = f[i];
    __syncthreads();
    const int row = lane >> 3, pos = lane & 7;
    {
        const bool on = 8 * chunk + pos < nb;
        const int sb = min(8 * chunk + pos, nb - 1);
        const uint32_t off = static_cast<uint32_t>((row * nb + sb) * kBlk);
        int sum[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        for (int ib = part; ib < 8; ib += parts) {
            const IqFields f_ib = iq_fields_shifted<TYPE>(stage + off, ib, (off + 2) & 2u);
            uint32_t a[8];
            iq_load_act(a, aq + sb * kIqActStride + ib * 32);
            int p[8];
            iq_chunks<TYPE>(f_ib, ib, tables, a, p);
#pragma unroll
            for (int c = 0; c < 8; ++c) sum[c] += p[c];
        }
        int4 *dst = reinterpret_cast<int4 *>(tiles + wave * kIqTileWords + row * kIqTileRow + pos * 8);
        dst[0] = make_int4(sum[0], sum[1], sum[2], sum[3]);
        dst[1] = make_int4(sum[4], sum[5], sum[6], sum[7]);
        if (part == 0) scales[64 * chunk + lane] = on ? h2f(*reinterpret_cast<const uint16_t *>(stage + off)) * ad[sb] : 0.0f;
    }
    __syncthreads();
    if (wave != 0) return;
    float acc = 0.0f;
    for (int ch = 0; ch < nchunks; ++ch) {
        const int32_t *tile = tiles + ch * parts * kIqTileWords + row * kIqTileRow + pos;
        float dv[8];
        int pv[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) dv[s] = scales[64 * ch + 8 * row + s], pv[s] = tile[8 * s];
        for (int q = 1; q < parts; ++q) {
#pragma unroll
            for (int s = 0; s < 8; ++s) pv[s] += tile[q * kIqTileWords + 8 * s];
        }
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            if (PART && 8 * ch + s < nb) partials[(static_cast<size_t>(base_row + row) * nb + 8 * ch + s) * 8 + pos] = pv[s];
            acc = __builtin_fmaf(dv[s], static_cast<float>(pv[s]), acc);
        }
    }
    const float y = close_lanes8(acc);
    if (pos == 0) out[base_row + row] = TYPE == 22 ? 0.125f * y : y;
}

// ---- Q8_0 / IQ4_NL / Q4_0 x Q8_0 GEMV: 16 rows per workgroup, 4 per wave ----------------------
// act_stride: elements between the activations of consecutive matrices (0 = one shared activation).
template <int KIND, bool PART>
__global__ __launch_bounds__(256) void k_gemv_q8(MatSrc src, int rows, int cols, const int8_t *__restrict__ act_qs,
                                                  const uint16_t *__restrict__ act_d, int act_stride,
                                                  float *__restrict__ out, int32_t *__restrict__ partials, int ppr) {
    __shared__ Q8Tile tiles[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = blockIdx.y;
    const uint8_t *w = mat_ptr(src, m);
    const int nb = cols >> 5;
    const int8_t *aq = act_qs + static_cast<size_t>(m) * act_stride;
    const uint16_t *ad = act_d + static_cast<size_t>(m) * (act_stride >> 5);
    const int r0 = blockIdx.x * 16 + wave * 4;
    if (r0 >= rows) return;
    const int nrows = min(4, rows - r0);
    const size_t rb = static_cast<size_t>(nb) * (KIND == 0 ? 34 : 18);
    int32_t *pp = PART ? partials + (static_cast<size_t>(m) * rows + r0) * ppr : nullptr;
    float y;
    if (KIND == 2)
        y = q4_0_rows4<PART>(w + r0 * rb, nrows, nb, aq, ad, lane, pp);
    else
        y = q8_rows4<(KIND == 1 ? 1 : 0), PART>(w + r0 * rb, nrows, nb, aq, ad, tiles[wave], lane, pp);
    const int r4 = lane >> 4;
    if ((lane & 15) == 0 && r4 < nrows) out[static_cast<size_t>(m) * rows + r0 + r4] = y;
}

// ---- Q4_0 x Q8_0 GEMV, streaming form ---------------------------------------------------------------------
// For matrices whose rows are a whole number of 8-block groups (144 bytes = nine 16-byte words) and whose group
// count per row (lpr) divides 64.  A wave owns 64 consecutive groups per pass (64 * 144 = 9216 contiguous bytes,
// 64 / lpr rows): nine fully coalesced 16-byte loads per lane bring them in, LDS turns the lane-interleaved words
// into one group per lane (both sides conflict-free: stride 16 in, stride 144 out), and the 18-byte blocks are cut
// out of the 36 dwords in registers (even blocks with four byte-align ops, odd blocks are dword aligned).  Lane l
// always works on column group l % lpr.  The workgroup keeps the activation in LDS (each group's 256 bytes padded
// to 272 so that the 16-byte reads of neighbouring groups fall on different banks), with the per-block scale as a
// float and 8 * sum(a) beside it; Block sums are exact; the float side adds a lane's
// eight blocks in order and folds the row's lanes with an xor tree (Q4_0 has no canonical float order).
// A wave takes NP consecutive passes and requests all of them before it touches the first.
// RAGGED: any row of eight blocks or more and 64 groups or fewer, on any two-byte boundary.  A row is lpr = ceil(nb / 8) groups
// of which the last holds the row's LAST eight blocks (those that the group before has as well get the scale zero), a pass is
// floor(64 / lpr) rows, and the words are fetched group by group.  The sum of a row's lanes is the same tree over any lpr.
// (us, general kernel -> here: 2048 x 12288 16.7 -> 7.2, 5000 x 5120 9.6 -> 7.1, 100000 x 1056 22.5 -> 16.1.)
// grid.x * WPB waves * NP passes cover ceil(rows / floor(64 / lpr)) passes.
// dynamic LDS: lpr * 272 bytes of quants, then 8 lpr floats, then 8 lpr ints.
// (the body: `block` is the workgroup's number among those of its matrix)
template <bool PART, int NP, int WPB, bool RAGGED>
WD_DEV void gemv_q4_stream_body(const uint8_t *__restrict__ w, int rows, int nb, const int8_t *__restrict__ act_qs,
                                const uint16_t *__restrict__ act_d, float *__restrict__ out, int32_t *__restrict__ partials,
                                int block) {
    __shared__ uint4 stage[WPB][9 * 64];
    extern __shared__ __align__(16) uint8_t q4_act[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lpr = (nb + 7) >> 3, lpr_shift = __builtin_ctz(lpr), rpp = RAGGED ? 64 / lpr : 64 >> lpr_shift;
    const int inv = (65535 + lpr) / lpr;  // n / lpr = n inv / 65536 for the n below 64 that are divided here
    const int rsub = RAGGED ? (lane * inv) >> 16 : lane >> lpr_shift, col = RAGGED ? lane - rsub * lpr : lane & (lpr - 1);
    const bool last_group = RAGGED && col == lpr - 1;
    const int skip = last_group ? 8 * lpr - nb : 0, first_block = last_group ? nb - 8 : 8 * col;
    float *ad = reinterpret_cast<float *>(q4_act + lpr * 272);
    int *corr = reinterpret_cast<int *>(ad + 8 * lpr);
    const size_t rb = static_cast<size_t>(nb) * 18;
    const long long pass0 = (static_cast<long long>(block) * WPB + wave) * NP;
    uint4 v[NP][9];
    auto fetch = [&](long long pass, int slot) {
        const long long row0 = pass * rpp;
        const long long left = static_cast<long long>(rows) - row0;
        const size_t valid = left <= 0 ? 0 : static_cast<size_t>(left < rpp ? left : rpp) * rb;
        const uint8_t *base = w + static_cast<size_t>(row0) * rb;
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            if constexpr (RAGGED) {
                const int word = k * 64 + lane, group = word / 9, r = (group * inv) >> 16, g = group - r * lpr;
                const size_t off = r * rb + (g == lpr - 1 ? rb - 144 : static_cast<size_t>(g) * 144) + 16 * (word - 9 * group);
                v[slot][k] = r < rpp && off < valid ? gld_u128(base + off) : make_uint4(0, 0, 0, 0);
            } else {
                const size_t off = static_cast<size_t>(k) * 1024 + static_cast<size_t>(lane) * 16;
                v[slot][k] = off < valid ? gld_u128_aligned(base + off) : make_uint4(0, 0, 0, 0);
            }
        }
    };
    // activation into LDS: thread t takes 16-byte pieces t, t + blockDim.x, ...; a block's two pieces give its sum.  The
    // first piece is requested before the weights so that it can be consumed while they are still in flight.
    const int n_pieces = lpr * 16;
    auto block_of = [&](int i) { return RAGGED && (i >> 4) == lpr - 1 ? nb - 8 + ((i & 15) >> 1) : i >> 1; };  // of piece i
    uint4 q0 = make_uint4(0, 0, 0, 0);
    uint16_t d0 = 0;
    if (static_cast<int>(threadIdx.x) < n_pieces) {
        q0 = *reinterpret_cast<const uint4 *>(act_qs + block_of(threadIdx.x) * 32 + (threadIdx.x & 1) * 16);
        d0 = act_d[block_of(threadIdx.x)];
    }
#pragma unroll
    for (int p = 0; p < NP; ++p) fetch(pass0 + p, p);
    for (int i = threadIdx.x; i < n_pieces; i += WPB * 64) {
        const bool first = i == static_cast<int>(threadIdx.x);
        const uint4 q = first ? q0 : *reinterpret_cast<const uint4 *>(act_qs + block_of(i) * 32 + (i & 1) * 16);
        *reinterpret_cast<uint4 *>(q4_act + (i >> 4) * 272 + (i & 15) * 16) = q;
        int s = sdot4(0x01010101u, q.x, 0);
        s = sdot4(0x01010101u, q.y, s);
        s = sdot4(0x01010101u, q.z, s);
        s = sdot4(0x01010101u, q.w, s);
        s += lane_xor(s, 1);
        if ((i & 1) == 0) {
            corr[i >> 1] = 8 * s;
            ad[i >> 1] = h2f(first ? d0 : act_d[block_of(i)]);
        }
    }
    __syncthreads();
    const uint8_t *my_act = q4_act + col * 272;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const long long row0 = (pass0 + p) * rpp;
        if (row0 >= rows) break;  // wave-uniform
#pragma unroll
        for (int k = 0; k < 9; ++k) stage[wave][k * 64 + lane] = v[p][k];
        wave_lds_fence();
        uint32_t d[36];
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            const uint4 u = stage[wave][lane * 9 + k];
            d[4 * k] = u.x, d[4 * k + 1] = u.y, d[4 * k + 2] = u.z, d[4 * k + 3] = u.w;
        }
        wave_lds_fence();
        const int row = static_cast<int>(row0) + rsub;
        const bool on = row < rows && (!RAGGED || rsub < rpp);
        float sumf = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int m = j >> 1;
            uint32_t n[4], dw;
            if ((j & 1) == 0) {
                dw = d[9 * m] & 0xffffu;
#pragma unroll
                for (int l = 0; l < 4; ++l) n[l] = __builtin_amdgcn_alignbyte(d[9 * m + l + 1], d[9 * m + l], 2);
            } else {
                dw = d[9 * m + 4] >> 16;
#pragma unroll
                for (int l = 0; l < 4; ++l) n[l] = d[9 * m + 5 + l];
            }
            const uint4 lo = *reinterpret_cast<const uint4 *>(my_act + j * 32), hi = *reinterpret_cast<const uint4 *>(my_act + j * 32 + 16);
            const uint32_t al[4] = {lo.x, lo.y, lo.z, lo.w}, ah[4] = {hi.x, hi.y, hi.z, hi.w};
            int sumi = -corr[col * 8 + j];  // sum (nibble - 8) * a = sum nibble * a - 8 * sum a
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                sumi = sdot4(n[l] & 0x0f0f0f0fu, al[l], sumi);
                sumi = sdot4((n[l] >> 4) & 0x0f0f0f0fu, ah[l], sumi);
            }
            if (PART && on && j >= skip) partials[static_cast<size_t>(row) * nb + first_block + j] = sumi;
            const float term = h2f(static_cast<uint16_t>(dw)) * ad[col * 8 + j] * static_cast<float>(sumi);
            sumf += RAGGED && j < skip ? 0.0f : term;
        }
        if constexpr (RAGGED) {
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) {
                const float other = __shfl_down(sumf, off, 64);
                if (col + off < lpr && col < off) sumf += other;
            }
        } else {
            for (int mask = lpr >> 1; mask >= 1; mask >>= 1) sumf += lane_xor(sumf, mask);
        }
        if (col == 0 && on) out[row] = sumf;
    }
}
template <bool PART, int NP, int WPB, bool RAGGED>
__global__ __launch_bounds__(WPB * 64) void k_gemv_q4_stream(const uint8_t *__restrict__ w, int rows, int nb,
                                                         const int8_t *__restrict__ act_qs,
                                                         const uint16_t *__restrict__ act_d, float *__restrict__ out,
                                                         int32_t *__restrict__ partials) {
    gemv_q4_stream_body<PART, NP, WPB, RAGGED>(w, rows, nb, act_qs, act_d, out, partials, static_cast<int>(blockIdx.x));
}
// Several matrices of one row length in one launch (see k_gemv_q8_rows8_split_batch): workgroup b belongs to the item
// whose range of workgroups holds b and does there what k_gemv_q4_stream does for that item alone.
// The table travels with the launch, whose host time grows with it (184 bytes 2.2 to 2.3 us, 648 2.35 to 2.4; 2.7 and 3.0 to 3.4 in
// another process): one for few items (184 bytes) beside one for many (648).
constexpr int kGemvBatchMax = 16, kGemvBatchFew = 4;
template <int MAX>
struct GemvBatch {
    const uint8_t *w[MAX];
    const int8_t *act_qs[MAX];
    const uint16_t *act_d[MAX];
    float *out[MAX];
    int rows[MAX];
    int first_group[MAX + 1];  // the item's first workgroup; first_group[n]: all workgroups
    int n;
};
template <int MAX>
WD_DEV int gemv_batch_item(const GemvBatch<MAX> &b) {
    int item = 0;
    for (int i = 1; i < b.n; ++i)
        if (static_cast<int>(blockIdx.x) >= b.first_group[i]) item = i;
    return __builtin_amdgcn_readfirstlane(item);
}
template <int WPB, bool RAGGED, int MAX>
__global__ __launch_bounds__(WPB * 64) void k_gemv_q4_stream_batch(GemvBatch<MAX> b, int nb) {
    const int item = gemv_batch_item(b);
    gemv_q4_stream_body<false, 1, WPB, RAGGED>(b.w[item], b.rows[item], nb, b.act_qs[item], b.act_d[item], b.out[item], nullptr,
                                       static_cast<int>(blockIdx.x) - b.first_group[item]);
}

// ---- dense Q8_0 / IQ4_NL x Q8_0 GEMV, streaming: one lane per (row, chain) --------------------------------------
// The reference order of a Q8_0 row (src/qwen38_cpu_moe.cuh:690-722) is eight chains, chain c over bytes 4c..4c+3 of
// every block, each one fma(d_w d_a, float(dot4), acc) per block in block order: the chains of a row are as long as
// the row, and nothing shortens them.  IQ4_NL (:377-422) has the same eight chains - c < 4: the low nibbles of bytes
// 4c..4c+3, c >= 4: the high ones of bytes 4(c-4).. -, each kept twice, over the even and over the odd blocks, and an
// unpaired last block apart.  A wave therefore takes eight rows and gives every (row, chain) pair a lane
// (lane = 8 row + chain): each fma instruction then advances 64 chains, no value crosses lanes until the closing tree,
// and the cost per block and row is under one vector instruction (IQ4_NL: two).
// The eight rows are fetched KB blocks at a time (whole 16-byte words because KB is a multiple of 8) with lane-contiguous
// 16-byte loads, one chunk ahead in a second register set, and copied to LDS with a row stride that spreads the eight rows
// over the banks.  Blocks are 34 or 18 bytes, so the four bytes of a lane are dword aligned in the odd blocks of a chunk and
// two bytes off in the even ones (two dwords and a v_alignbyte); the parity is the same for every lane, so the unrolled loop
// knows it at compile time.
// Rows that are no whole number of chunks end with a chunk of their LAST KB blocks, whose first blocks have been there
// already and get the scale zero: every chunk is KB blocks long, starts at offset zero of its stage and reads nothing outside
// its row.  RAGGED: such rows, and rows that do not start on 16-byte boundaries (loads are then two-byte aligned).
// The activation's quants and its scales (as floats, in the order of the chunks) are staged in LDS once per workgroup.
// us, general kernel -> here: IQ4_NL 30000 x 4096 31.0 -> 21.0 (3.3 TB/s: vector instructions), 20000 x 1024 7.9 -> 6.7; Q8_0
// 100000 x 1056 35.0 -> 31.9; whole Q8_0 chunks stream at 4.9 TB/s (30000 x 4096, 26.7).
// dynamic LDS: cols bytes, a float per block of every chunk, then one stage of 8 * kQ8sRowStride<KIND, KB> bytes per wave.
template <int KIND>
constexpr int kQ8sBlk = KIND == 0 ? 34 : 18;
template <int KIND, int KB>
constexpr int kQ8sRowStride = KIND == 0 ? (KB == 32 ? 1184 : 544) : (KB == 32 ? 672 : 288);  // a chunk + padding, 8 (mod 32) dwords

template <int KIND, int KB>
struct Q8sFetch {
    static constexpr int kWordsPerRow = kQ8sBlk<KIND> * KB / 16;      // 16-byte words of a row's chunk
    static constexpr int kWords = 8 * kWordsPerRow;                    // of the eight rows
    static constexpr int kLoads = (kWords + 63) / 64;
    uint4 u[kLoads];
};
template <bool RAGGED>
WD_DEV uint4 q8s_load(const uint8_t *p) {
    return RAGGED ? gld_u128(p) : gld_u128_aligned(p);
}

// Eight blocks of a lane's row (lane = 8 row + chain) out of a staged chunk: the lane's four bytes of every block, the
// blocks' scales, the activation's four bytes and scales.  The LDS reads are issued as one group, so that a caller can put
// the next group's before the arithmetic of this one.
template <int KIND>
struct Q8sBatch {
    uint32_t w[12];  // blocks 0 2 4 6 of the batch: two dwords each (w[3i], w[3i+1]); blocks 1 3 5 7: w[3i+2]
    uint32_t dw[8], a[8];
    float4 da[2];
    // my: the lane's bytes of the chunk's first block; row_blocks: the row's first block in the stage; my_a / ad: the
    // activation's quants at the lane's chain and its scales, of the chunk's first block; s: batch in the chunk.
    WD_DEV void load(const uint8_t *my, const uint8_t *row_blocks, const int8_t *my_a, const float *ad, int s) {
        constexpr int kBlk = kQ8sBlk<KIND>;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint8_t *blk = my + kBlk * (8 * s + 2 * i);
            w[3 * i] = *reinterpret_cast<const uint32_t *>(blk);
            w[3 * i + 1] = *reinterpret_cast<const uint32_t *>(blk + 4);
            w[3 * i + 2] = *reinterpret_cast<const uint32_t *>(blk + kBlk + 2);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            dw[i] = *reinterpret_cast<const uint16_t *>(row_blocks + kBlk * (8 * s + i));
            a[i] = *reinterpret_cast<const uint32_t *>(my_a + 32 * (8 * s + i));
        }
        da[0] = *reinterpret_cast<const float4 *>(ad + 8 * s);
        da[1] = *reinterpret_cast<const float4 *>(ad + 8 * s + 4);
    }
    // block i of the batch: its scale product and its chunk sum (nibble: 0 or 4, the lane's half of the bytes)
    WD_DEV float scale(int i) const {
        const float d[8] = {da[0].x, da[0].y, da[0].z, da[0].w, da[1].x, da[1].y, da[1].z, da[1].w};
        return h2f(static_cast<uint16_t>(dw[i])) * d[i];
    }
    WD_DEV int dot(int i, int nibble) const {
        const uint32_t q = (i & 1) ? w[3 * (i >> 1) + 2] : __builtin_amdgcn_alignbyte(w[3 * (i >> 1) + 1], w[3 * (i >> 1)], 2);
        return sdot4(KIND == 0 ? q : iq4nl_low(q >> nibble), a[i], 0);
    }
};
// use(batch, s) for the batches s of a chunk in order.  AHEAD: the next eight blocks are requested from LDS before the
// arithmetic of these, where the registers reach for two batches (72 of them); elsewhere they would be spilled.
template <int KIND, int KB, bool AHEAD, typename Use>
WD_DEV void q8s_batches(const uint8_t *my, const uint8_t *row_blocks, const int8_t *my_a, const float *ad, Use &&use) {
    Q8sBatch<KIND> t0, t1;
    if (!AHEAD) {
#pragma unroll
        for (int s = 0; s < KB / 8; ++s) {
            t0.load(my, row_blocks, my_a, ad, s);
            use(t0, s);
            __builtin_amdgcn_sched_barrier(0);
        }
        return;
    }
    t0.load(my, row_blocks, my_a, ad, 0);
#pragma unroll
    for (int s = 0; s < KB / 8; s += 2) {
        t1.load(my, row_blocks, my_a, ad, s + 1);
        __builtin_amdgcn_sched_barrier(0);
        use(t0, s);
        if (s + 2 < KB / 8) t0.load(my, row_blocks, my_a, ad, s + 2);
        __builtin_amdgcn_sched_barrier(0);
        use(t1, s + 1);
    }
}
// The unpaired last block of an IQ4_NL row: its scale times the whole-block integer sum (exact below 2^24).
WD_DEV float q8s_tail(float scale, int p) {
    p += lane_xor(p, 1);
    p += lane_xor(p, 2);
    p += lane_xor(p, 4);
    return scale * static_cast<float>(p);
}
// The activation into LDS: its quants, and its scales in the order of chunks of `chunk` blocks (the last one: the row's last
// `chunk` blocks).
WD_DEV void q8s_stage_activation(int8_t *aq, float *ad, const int8_t *act_qs, const uint16_t *act_d, int nb, int chunk, int threads) {
    const int whole = (nb + chunk - 1) / chunk * chunk, last = whole - chunk;
    for (int i = threadIdx.x; i < nb * 2; i += threads) reinterpret_cast<uint4 *>(aq)[i] = reinterpret_cast<const uint4 *>(act_qs)[i];
    for (int i = threadIdx.x; i < whole; i += threads) ad[i] = h2f(act_d[i < last ? i : i - whole + nb]);
}

template <int KIND, int KB, bool RAGGED, bool PART>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_gemv_q8_rows8(const uint8_t *__restrict__ w, int rows, int nb,
                                                              const int8_t *__restrict__ act_qs, const uint16_t *__restrict__ act_d,
                                                              float *__restrict__ out, int32_t *__restrict__ partials) {
    constexpr int WAVES = 4, kBlk = kQ8sBlk<KIND>;
    using Fetch = Q8sFetch<KIND, KB>;
    constexpr int RS = kQ8sRowStride<KIND, KB>;
    extern __shared__ __align__(16) uint8_t q8s_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cols = nb * 32, nchunks = (nb + KB - 1) / KB, skipped = nchunks * KB - nb;
    int8_t *aq = reinterpret_cast<int8_t *>(q8s_lds);
    float *ad = reinterpret_cast<float *>(q8s_lds + cols);
    uint8_t *stage = q8s_lds + cols + nchunks * KB * 4 + wave * (8 * RS);
    const size_t rb = static_cast<size_t>(nb) * kBlk;
    // the waves of the grid take the groups of eight rows in turn (rows >= 8)
    const int n_groups = (rows + 7) >> 3, n_waves = gridDim.x * WAVES, first = blockIdx.x * WAVES + wave;
    const int my_groups = first < n_groups ? (n_groups - first + n_waves - 1) / n_waves : 0;
    // where the lane's words of a chunk lie: in memory (relative to the chunk of the group's first row) and in the stage
    const int row = lane >> 3, c = lane & 7, nibble = c & 4;
    uint32_t goff[Fetch::kLoads], loff[Fetch::kLoads];
#pragma unroll
    for (int i = 0; i < Fetch::kLoads; ++i) {
        const int u = min(i * 64 + lane, Fetch::kWords - 1);
        const int r = u / Fetch::kWordsPerRow, within = u - r * Fetch::kWordsPerRow;
        goff[i] = static_cast<uint32_t>(r * rb + 16 * within);
        loff[i] = static_cast<uint32_t>(r * RS + 16 * within);
    }
    // a chunk's first block in its row
    auto first_block = [&](int chunk) { return RAGGED && chunk == nchunks - 1 ? nb - KB : chunk * KB; };
    // the fetch runs one chunk ahead of the arithmetic, over the group boundaries
    int f_group = min(first, n_groups - 1), f_chunk = 0, fetched = 0;
    const int items = my_groups * nchunks;
    Fetch f;
    auto fetch = [&]() {
        // a last group of fewer than eight rows is moved up to end with the matrix: it then repeats rows of the group
        // before it, which come out the same
        const uint8_t *p = uniform_ptr(w + static_cast<size_t>(min(8 * f_group, rows - 8)) * rb + static_cast<size_t>(first_block(f_chunk)) * kBlk);
#pragma unroll
        for (int i = 0; i < Fetch::kLoads; ++i) f.u[i] = q8s_load<RAGGED>(p + goff[i]);
        // past the wave's last chunk the same chunk is requested again (and not used), so that every turn issues the
        // same number of requests
        if (++fetched < items) {
            if (++f_chunk == nchunks) f_chunk = 0, f_group += n_waves;
        }
    };
    fetch();
    q8s_stage_activation(aq, ad, act_qs, act_d, nb, KB, 64 * WAVES);
    __syncthreads();
    if (my_groups == 0) return;  // wave-uniform
    const uint8_t *row_blocks = stage + row * RS, *my = row_blocks + 4 * (KIND == 0 ? c : c & 3);
    float acc = 0.0f, odd = 0.0f, tail = 0.0f;
    int group = first, chunk = 0;
    for (int t = 0; t < items; ++t) {
        wave_lds_fence();  // the previous chunk has been read
#pragma unroll
        for (int i = 0; i < Fetch::kLoads; ++i) *reinterpret_cast<uint4 *>(stage + loff[i]) = f.u[i];
        wave_lds_fence();
        fetch();  // a later chunk, into the registers just written out
        const bool last = chunk == nchunks - 1;
        const int b0 = first_block(chunk), skip = RAGGED && last ? skipped : 0;
        const bool unpaired = KIND == 1 && RAGGED && last && (nb & 1);
        if (unpaired) {  // (the chunk then starts with an odd block; the closing sum takes the two in either order)
            const float swap = acc;
            acc = odd, odd = swap;
        }
        const int out_row = min(8 * group, rows - 8) + row;
        int32_t *pp = PART ? partials + (static_cast<size_t>(out_row) * nb + b0) * 8 + c : nullptr;
        const int8_t *my_a = aq + 4 * c + 32 * b0;
        const float *my_d = ad + chunk * KB;
        auto compute_batch = [&](const Q8sBatch<KIND> &bt, int s) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int at = 8 * s + i, p = bt.dot(i, nibble);
                float scale = bt.scale(i);
                if (PART && at >= skip) pp[at * 8] = p;
                if (RAGGED && at < skip) scale = 0.0f;
                if (RAGGED && KIND == 1 && at == KB - 1 && unpaired) {
                    tail = q8s_tail(scale, p);
                    scale = 0.0f;
                }
                float &chain = KIND == 1 && (i & 1) ? odd : acc;
                chain = __builtin_fmaf(scale, static_cast<float>(p), chain);
            }
            asm volatile("" : "+v"(acc), "+v"(odd));  // (batch by batch: the products are not kept for later)
        };
        q8s_batches<KIND, KB, KB == 16>(my, row_blocks, my_a, my_d, compute_batch);
        if (++chunk == nchunks) {
            float y = close_lanes8(KIND == 1 ? acc + odd : acc);
            if (RAGGED && KIND == 1 && (nb & 1)) y = y + tail;
            if (c == 0) out[out_row] = y;
            acc = 0.0f, odd = 0.0f, chunk = 0, group += n_waves;
        }
    }
}

// ---- the same, few rows: the waves of a workgroup share the eight rows of a group ----------------------------------
// With few row groups a group's wave runs alone on its SIMD and the time is the length of its chains (about 40 cycles
// per block: one wave issues an instruction every four cycles and a block is ten of them).  Only the fma itself has to
// run in block order.  So wave v of a workgroup takes blocks [v NCH*KB, (v+1) NCH*KB) of the eight rows (the last one the
// last NCH*KB), requests all of them at once, turns them into (d_w d_a, float(dot4)) pairs in registers at its own pace, and
// then the waves run their parts of the chains one after the other, handing the 64 accumulators on through LDS: NCH*KB
// dependent fma per wave, nothing else.  Lane = 8 row + chain and RAGGED as in k_gemv_q8_rows8; up to eight waves (WAVES, or any
// number when that is 0), nb > their blocks but those of the last, and nb >= NCH*KB.
// dynamic LDS: cols bytes, a float per block of every wave, 512 bytes of accumulators, then one stage of
// 8 * kQ8sRowStride<KIND, KB> per wave.
// us, general kernel or single waves -> here: IQ4_NL 2048 x 2048 7.3 -> 3.8, 1500 x 16384 45.6 -> 10.7; Q8_0 3000 x 2592 8.4 -> 6.1,
// 2048 x 12288 15.2 -> 11.0, 520 x 1600 5.2 -> 3.3.
// (the body: `group` is the workgroup's group of eight rows)
template <int KIND, int KB, int NCH, int WAVES, bool RAGGED, bool PART>
WD_DEV void gemv_q8_rows8_split_body(const uint8_t *__restrict__ w, int rows, int nb, const int8_t *__restrict__ act_qs,
                                     const uint16_t *__restrict__ act_d, float *__restrict__ out, int32_t *__restrict__ partials,
                                     int group) {
    constexpr int SEG = NCH * KB, kBlk = kQ8sBlk<KIND>;
    using Fetch = Q8sFetch<KIND, KB>;
    constexpr int RS = kQ8sRowStride<KIND, KB>;
    extern __shared__ __align__(16) uint8_t q8p_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cols = nb * 32, waves = WAVES ? WAVES : (nb + SEG - 1) / SEG;
    const bool last = wave == waves - 1;
    int8_t *aq = reinterpret_cast<int8_t *>(q8p_lds);
    float *ad = reinterpret_cast<float *>(q8p_lds + cols);
    float *carry = reinterpret_cast<float *>(q8p_lds + cols + waves * SEG * 4);
    uint8_t *stage = q8p_lds + cols + waves * SEG * 4 + 512 + wave * (8 * RS);
    const size_t rb = static_cast<size_t>(nb) * kBlk;
    const int row = lane >> 3, c = lane & 7, nibble = c & 4;
    // a last group of fewer than eight rows is moved up to end with the matrix (rows >= 8)
    const int base_row = min(8 * group, rows - 8);
    const int first_block = RAGGED && last ? nb - SEG : wave * SEG, skip = RAGGED && last ? waves * SEG - nb : 0;
    const bool unpaired = KIND == 1 && RAGGED && last && (nb & 1);
    const uint8_t *src = uniform_ptr(w + static_cast<size_t>(base_row) * rb + static_cast<size_t>(first_block) * kBlk);
    uint32_t loff[Fetch::kLoads];
    Fetch f[NCH];
#pragma unroll
    for (int i = 0; i < Fetch::kLoads; ++i) {
        const int u = min(i * 64 + lane, Fetch::kWords - 1);
        const int r = u / Fetch::kWordsPerRow, within = u - r * Fetch::kWordsPerRow;
        loff[i] = static_cast<uint32_t>(r * RS + 16 * within);
        const uint32_t goff = static_cast<uint32_t>(r * rb + 16 * within);
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) f[ch].u[i] = q8s_load<RAGGED>(src + goff + ch * (kBlk * KB));
    }
    q8s_stage_activation(aq, ad, act_qs, act_d, nb, SEG, 64 * waves);
    __syncthreads();
    const uint8_t *row_blocks = stage + row * RS, *my = row_blocks + 4 * (KIND == 0 ? c : c & 3);
    int32_t *pp = PART ? partials + (static_cast<size_t>(base_row + row) * nb + first_block) * 8 + c : nullptr;
    float dv[SEG], pv[SEG], acc = 0.0f, odd = 0.0f, tail = 0.0f;
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
        wave_lds_fence();  // the previous chunk has been read
#pragma unroll
        for (int i = 0; i < Fetch::kLoads; ++i) *reinterpret_cast<uint4 *>(stage + loff[i]) = f[ch].u[i];
        wave_lds_fence();
        const int8_t *my_a = aq + 4 * c + 32 * (first_block + ch * KB);
        const float *my_d = ad + wave * SEG + ch * KB;
        auto pairs = [&](const Q8sBatch<KIND> &bt, int s) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int at = ch * KB + 8 * s + i, p = bt.dot(i, nibble);
                float scale = bt.scale(i);
                if (PART && at >= skip) pp[at * 8] = p;
                if (RAGGED && at < skip) scale = 0.0f;
                if (RAGGED && KIND == 1 && at == SEG - 1 && unpaired) {
                    tail = q8s_tail(scale, p);
                    scale = 0.0f;
                }
                dv[at] = scale;
                pv[at] = static_cast<float>(p);
                // Made here: left to itself the compiler moves the products into the wave's turn, and the turns are serial
                // (five waves, 5000 x 5120: 13.7 us instead of 11.6).  Where the number of waves is known it does better.
                if (WAVES == 0) asm volatile("" : "+v"(dv[at]), "+v"(pv[at]));
            }
        };
        q8s_batches<KIND, KB, true>(my, row_blocks, my_a, my_d, pairs);
    }
    // the chains, one wave after the other in block order
    auto take_turn = [&](int turn) {
        if (wave == turn) {
            if (turn > 0) {
                acc = carry[lane];
                if (KIND == 1) odd = carry[64 + lane];
            }
            if (unpaired) {  // (the part starts with an odd block; the closing sum takes the two in either order)
                const float swap = acc;
                acc = odd, odd = swap;
            }
#pragma unroll
            for (int i = 0; i < SEG; ++i) {
                float &chain = KIND == 1 && (i & 1) ? odd : acc;
                chain = __builtin_fmaf(dv[i], pv[i], chain);
            }
            if (turn < waves - 1) {
                carry[lane] = acc;
                if (KIND == 1) carry[64 + lane] = odd;
            }
        }
        if (turn < waves - 1) __syncthreads();
    };
    if constexpr (WAVES != 0) {
#pragma unroll
        for (int turn = 0; turn < WAVES; ++turn) take_turn(turn);
    } else {
        for (int turn = 0; turn < waves; ++turn) take_turn(turn);
    }
    if (last) {
        float y = close_lanes8(KIND == 1 ? acc + odd : acc);
        if (KIND == 1 && unpaired) y = y + tail;
        if (c == 0) out[base_row + row] = y;
    }
}
template <int KIND, int KB, int NCH, int WAVES, bool RAGGED, bool PART>
__global__ __launch_bounds__(WAVES ? 64 * WAVES : 512) void k_gemv_q8_rows8_split(const uint8_t *__restrict__ w, int rows, int nb,
                                                              const int8_t *__restrict__ act_qs, const uint16_t *__restrict__ act_d,
                                                              float *__restrict__ out, int32_t *__restrict__ partials) {
    gemv_q8_rows8_split_body<KIND, KB, NCH, WAVES, RAGGED, PART>(w, rows, nb, act_qs, act_d, out, partials, static_cast<int>(blockIdx.x));
}
// Several matrices of the same row length in ONE launch (the projections a block applies to one or a few activations:
// each of them alone is bound by its launch, not by its bytes).  Workgroup b belongs to the item whose range of row
// groups holds b; what it computes is what k_gemv_q8_rows8_split computes for that item alone.
template <int KB, int NCH, int WAVES, bool RAGGED, int MAX>
__global__ __launch_bounds__(WAVES ? 64 * WAVES : 512) void k_gemv_q8_rows8_split_batch(GemvBatch<MAX> b, int nb) {
    const int item = gemv_batch_item(b);
    gemv_q8_rows8_split_body<0, KB, NCH, WAVES, RAGGED, false>(b.w[item], b.rows[item], nb, b.act_qs[item], b.act_d[item], b.out[item], nullptr,
                                                       static_cast<int>(blockIdx.x) - b.first_group[item]);
}

// ---- Q6_K x Q8_K GEMV: the waves of the grid take the rows in turn, pass by pass, one pass fetched ahead -------
// The activation (quants, scales, 16-value sums) is staged in LDS once per workgroup.
// dynamic LDS: kQ6ActStride bytes per super-block, then cols/256 floats, then cols/16 int16 (each part 16-byte
// aligned), then four wave stages of kQ6StageBytes.
// FULL: rows are a whole number of passes.
template <bool FULL>
struct Q6Walk {  // the passes of a wave's rows, in memory order
    const uint8_t *src;
    size_t row_skip;  // bytes from the end of one of the wave's rows to the start of its next
    int pass, npass, last_bytes;
    Q6Pieces full, last;
    WD_DEV bool is_last() const { return pass == npass - 1; }
    WD_DEV const Q6Pieces &pieces() const { return (FULL || !is_last()) ? full : last; }
    WD_DEV void advance() {
        src = uniform_ptr(src + ((FULL || !is_last()) ? 1680 : last_bytes) + (is_last() ? row_skip : 0));
        pass = is_last() ? 0 : pass + 1;
    }
};

template <bool PART, bool ALIGNED, bool FULL>
__global__ __launch_bounds__(256) void k_gemv_q6k(const uint8_t *__restrict__ w, int rows, int cols,
                                                   const int8_t *__restrict__ act_qs, const float *__restrict__ act_d,
                                                   const int16_t *__restrict__ act_bsums, float *__restrict__ out,
                                                   int32_t *__restrict__ partials) {
    extern __shared__ __align__(16) uint8_t q6_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nb = cols >> 8, npass = (nb + 7) >> 3;
    const int aq_bytes = nb * kQ6ActStride;
    int8_t *aq = reinterpret_cast<int8_t *>(q6_lds);
    float *ad = reinterpret_cast<float *>(q6_lds + aq_bytes);
    int16_t *ab = reinterpret_cast<int16_t *>(q6_lds + aq_bytes + ((nb * 4 + 15) & ~15));
    uint8_t *stage = q6_lds + aq_bytes + ((nb * 4 + 15) & ~15) + nb * 32 + wave * kQ6StageBytes;
    const size_t rb = static_cast<size_t>(nb) * 210;
    // the waves of the grid take the rows in turn, so that the waves running together read neighbouring rows
    const int n_waves = gridDim.x * 4;
    const int r0 = blockIdx.x * 4 + wave;
    const int n_rows = r0 < rows ? (rows - r0 + n_waves - 1) / n_waves : 0;
    Q6Walk<FULL> fetch;  // runs one pass ahead of `work`
    fetch.src = uniform_ptr(w + static_cast<size_t>(min(r0, rows - 1)) * rb);  // a wave without rows asks for the last one
    fetch.row_skip = static_cast<size_t>(n_waves - 1) * rb;
    fetch.pass = 0, fetch.npass = npass, fetch.last_bytes = (nb - 8 * (npass - 1)) * 210;
    fetch.full = q6k_pieces(1680, lane), fetch.last = q6k_pieces(fetch.last_bytes, lane);
    Q6Walk<FULL> work = fetch;
    Q6Fetch fa = q6k_fetch<ALIGNED>(fetch.src, fetch.pieces()), fb;
    for (int i = threadIdx.x; i < cols / 16; i += 256)  // 16 words of 16 bytes per super-block
        reinterpret_cast<uint4 *>(aq + (i >> 4) * kQ6ActStride)[i & 15] = reinterpret_cast<const uint4 *>(act_qs)[i];
    for (int i = threadIdx.x; i < nb; i += 256) ad[i] = act_d[i];
    for (int i = threadIdx.x; i < nb * 8; i += 256) reinterpret_cast<uint32_t *>(ab)[i] = reinterpret_cast<const uint32_t *>(act_bsums)[i];
    __syncthreads();
    if (n_rows <= 0) return;  // wave-uniform
    const int items = n_rows * npass;
    long long r = r0;
    float acc = 0.0f;
    auto step = [&](const Q6Fetch &cur) {
        wave_lds_fence();  // the previous pass has been read
        q6k_stage(stage, cur, work.pieces());
        wave_lds_fence();
        acc = q6k_pass<PART, FULL>(stage, 8 * work.pass, nb, aq, ad, ab, lane, acc, PART ? partials + static_cast<size_t>(r) * nb * 8 : nullptr);
        if (work.is_last()) {
            const float y = q6k_close(acc);
            if (lane == 15) out[r] = y;
            r += n_waves;
        }
        work.advance();
    };
    // Two register sets take turns, so that the request for the next pass stays in flight while this one is worked on.
    // Every turn issues its three requests (after the wave's last pass: the same pass again, not used), so that the
    // count of requests in flight does not depend on the path taken.
    for (int t = 0; t < items; t += 2) {
        if (t + 1 < items) fetch.advance();
        fb = q6k_fetch<ALIGNED>(fetch.src, fetch.pieces());
        step(fa);
        if (t + 1 >= items) break;
        if (t + 2 < items) fetch.advance();
        fa = q6k_fetch<ALIGNED>(fetch.src, fetch.pieces());
        step(fb);
    }
}

// ---- elementwise ---------------------------------------------------------------------------------
__global__ void k_silu_mul_experts(const float *__restrict__ gate_up, float *__restrict__ act, int ffn) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ffn) return;
    const float *g = gate_up + static_cast<size_t>(2) * blockIdx.y * ffn;
    act[static_cast<size_t>(blockIdx.y) * ffn + i] = silu_ggml(g[i]) * g[ffn + i];
}

__global__ void k_weighted_accum(const float *__restrict__ experts, const float *__restrict__ weights,
                                 float *__restrict__ accum, int n, int k) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float a = accum[i];
    for (int j = 0; j < k; ++j) {
        const float prod = experts[static_cast<size_t>(j) * n + i] * weights[j];
        a = a + prod;
    }
    accum[i] = a;
}

// out may alias routed
__global__ void k_add_shared(const float *routed, const float *__restrict__ shared,
                             const float *__restrict__ gate, float *out, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float prod = shared[i] * gate[0];
    out[i] = routed[i] + prod;
}

// gate[0] = sigmoid_ggml(gate[0])
__global__ void k_sigmoid1(float *gate) {
    if (threadIdx.x == 0 && blockIdx.x == 0) gate[0] = sigmoid_ggml(gate[0]);
}

// accum[i] = ordered weighted sum of the k expert outputs (product rounded, then sum rounded);
// out[i] = accum[i] + shared[i] * gate[0] when a shared expert is present, else accum[i].
// residual (optional): residual[i] += out[i] * residual_scale.
__global__ void k_combine(const float *__restrict__ experts, const float *__restrict__ weights, int k,
                          const float *__restrict__ shared, const float *__restrict__ gate,
                          float *__restrict__ accum, float *__restrict__ out, float *__restrict__ residual,
                          float residual_scale, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float a = 0.0f;
    for (int j = 0; j < k; ++j) {
        const float prod = experts[static_cast<size_t>(j) * n + i] * weights[j];
        a = a + prod;
    }
    accum[i] = a;
    if (shared) {
        const float prod = shared[i] * gate[0];
        a = a + prod;
    }
    out[i] = a;
    if (residual) {  // next layer's input in a layer stack
        const float scaled = a * residual_scale;
        residual[i] = residual[i] + scaled;
    }
}

// Hyper-connection combine of the FFN branch: residual[c][h] += branch[h] * (2 sigmoid(inject[c] / hc)) for the hc
// residual streams, product rounded, then sum rounded (src/qwen38_hc.cuh:2530-2547).  SHARED: 0 = branch is block_out,
// 1 / 2 = branch = routed + shared * gate[0] with the shared expert's output as float / as half bits (:2241-2263).
template <int SHARED>
__global__ void k_hc_combine(float *__restrict__ residual, const float *__restrict__ block_out, const void *__restrict__ shared,
                             const float *__restrict__ gate, const float *__restrict__ inject, int hidden, int hc, int round) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= hidden * hc) return;
    const int c = i / hidden, h = i - c * hidden;
    float branch = block_out[h];
    if (SHARED != 0) {
        const float sh = SHARED == 1 ? static_cast<const float *>(shared)[h] : h2f(static_cast<const uint16_t *>(shared)[h]);
        const float weighted = sh * gate[0];
        branch = branch + weighted;
    }
    const float weighted = branch * hc_weight(inject[c], hc);
    const float v = residual[i] + weighted;
    residual[i] = round ? round_half(v) : v;
}

}  // namespace wd
