// Stand-alone operators of the MoE decode path: activation quantisers, router GEMV,
// softmax/top-k, low-bit GEMVs (one matrix or one dispatch over several expert matrices)
// and the elementwise stages.  Each extern "C" entry point mirrors one launcher of the
// reference operator surface (see include/warpdecode_amd.h for the citations).
#include <cstring>

#include "wd_common.h"
#include "wd_fused.cuh"
#include "wd_profile.hpp"

namespace wd {

thread_local std::string g_last_error;
std::string &last_error_slot() { return g_last_error; }

int fail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return code;
}

}  // namespace wd

using namespace wd;

extern "C" {

const char *wd_last_error(void) { return last_error_slot().c_str(); }

int wd_init(int device) {
    int count = 0;
    WD_HIP(hipGetDeviceCount(&count));
    WD_REQUIRE(device >= 0 && device < count, "wd_init: device %d out of range (%d devices)", device, count);
    WD_HIP(hipSetDevice(device));
    hipDeviceProp_t prop;
    WD_HIP(hipGetDeviceProperties(&prop, device));
    WD_REQUIRE(prop.warpSize == 64, "wd_init: device %s has %d-wide waves; this library is built for gfx950",
               prop.name, prop.warpSize);
    return noalloc_setup_current_device();
}

size_t wd_row_bytes(int type, int cols) { return row_bytes(type, cols); }
size_t wd_tensor_bytes(int type, int rows, int cols) {
    return rows > 0 ? static_cast<size_t>(rows) * row_bytes(type, cols) : 0;
}

// ---- runtime helpers ------------------------------------------------------------------
int wd_malloc(void **d_ptr, size_t bytes) {
    WD_REQUIRE(d_ptr != nullptr, "wd_malloc: null output pointer");
    WD_HIP(hipMalloc(d_ptr, bytes));
    return WD_OK;
}
int wd_free(void *d_ptr) {
    WD_HIP(hipFree(d_ptr));
    return WD_OK;
}
int wd_malloc_host(void **h_ptr, size_t bytes) {
    WD_REQUIRE(h_ptr != nullptr, "wd_malloc_host: null output pointer");
    WD_HIP(hipHostMalloc(h_ptr, bytes, hipHostMallocDefault));
    return WD_OK;
}
int wd_free_host(void *h_ptr) {
    WD_HIP(hipHostFree(h_ptr));
    return WD_OK;
}
int wd_memcpy_h2d(void *d_dst, const void *h_src, size_t bytes, void *stream) {
    if (stream)
        WD_HIP(hipMemcpyAsync(d_dst, h_src, bytes, hipMemcpyHostToDevice, as_stream(stream)));
    else
        WD_HIP(hipMemcpy(d_dst, h_src, bytes, hipMemcpyHostToDevice));
    return WD_OK;
}
int wd_memcpy_d2h(void *h_dst, const void *d_src, size_t bytes, void *stream) {
    if (stream)
        WD_HIP(hipMemcpyAsync(h_dst, d_src, bytes, hipMemcpyDeviceToHost, as_stream(stream)));
    else
        WD_HIP(hipMemcpy(h_dst, d_src, bytes, hipMemcpyDeviceToHost));
    return WD_OK;
}
int wd_memcpy_d2d(void *d_dst, const void *d_src, size_t bytes, void *stream) {
    WD_HIP(hipMemcpyAsync(d_dst, d_src, bytes, hipMemcpyDeviceToDevice, as_stream(stream)));
    return WD_OK;
}
int wd_memset(void *d_dst, int value, size_t bytes, void *stream) {
    WD_REQUIRE(bytes % 4 == 0, "wd_memset: size must be a multiple of 4 bytes");
    const uint32_t b = static_cast<uint32_t>(value) & 0xffu;
    const size_t n = bytes / 4;
    if (n == 0) return WD_OK;
    // a fill kernel rather than hipMemsetAsync, so the call may sit inside a captured graph
    enqueue(k_fill_u32, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, as_stream(stream),
        static_cast<uint32_t *>(d_dst), b * 0x01010101u, n);
    WD_LAUNCH_CHECK();
    return WD_OK;
}
int wd_stream_create(void **stream) {
    WD_REQUIRE(stream != nullptr, "wd_stream_create: null output pointer");
    hipStream_t s;
    WD_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    *stream = s;
    return WD_OK;
}
int wd_stream_destroy(void *stream) {
    WD_HIP(hipStreamDestroy(as_stream(stream)));
    return WD_OK;
}
int wd_stream_sync(void *stream) {
    WD_HIP(hipStreamSynchronize(as_stream(stream)));
    return WD_OK;
}
int wd_device_sync(void) {
    WD_HIP(hipDeviceSynchronize());
    return WD_OK;
}

// ---- quantisers -------------------------------------------------------------------------
int wd_q8_k_quantize_f32(const float *d_x, int elements, int8_t *d_qs, float *d_scales, int16_t *d_bsums,
                         void *stream) {
    WD_REQUIRE(elements > 0 && elements % 256 == 0,
               "Q8_K quantisation requires a positive multiple of 256 elements (got %d)", elements);
    WD_REQUIRE(d_x && d_qs && d_scales && d_bsums, "wd_q8_k_quantize_f32: null pointer");
    const int blocks = elements / 256;
    enqueue(k_q8_k_quantize, dim3((blocks + 3) / 4), dim3(256), 0, as_stream(stream), d_x, blocks, d_qs, d_scales, d_bsums);
    WD_LAUNCH_CHECK();
    return WD_OK;
}

int wd_q8_0_quantize_f32(const float *d_x, int elements, int8_t *d_qs, uint16_t *d_scales, void *stream) {
    WD_REQUIRE(elements > 0 && elements % 32 == 0,
               "Q8_0 quantisation requires a positive multiple of 32 elements (got %d)", elements);
    WD_REQUIRE(d_x && d_qs && d_scales, "wd_q8_0_quantize_f32: null pointer");
    const int blocks = elements / 32;
    enqueue(k_q8_0_quantize, dim3((blocks + 31) / 32), dim3(256), 0, as_stream(stream), d_x, blocks, d_qs, d_scales);
    WD_LAUNCH_CHECK();
    return WD_OK;
}

int wd_q8_1_quantize_f32(const float *d_x, int elements, int8_t *d_qs, uint16_t *d_scales, void *stream) {
    WD_REQUIRE(elements > 0 && elements % 32 == 0, "Q8_1 input must be a positive multiple of 32 (got %d)", elements);
    WD_REQUIRE(d_x && d_qs && d_scales, "wd_q8_1_quantize_f32: null pointer");
    const int blocks = elements / 32;
    enqueue(k_q8_1_quantize, dim3((blocks + 31) / 32), dim3(256), 0, as_stream(stream), d_x, blocks, d_qs, d_scales);
    WD_LAUNCH_CHECK();
    return WD_OK;
}
int wd_q8_0_quantize_f16(const uint16_t *d_x, int elements, int8_t *d_qs, uint16_t *d_scales, void *stream) {
    WD_REQUIRE(elements > 0 && elements % 32 == 0, "Q8_0 quantisation requires a positive multiple of 32 elements (got %d)", elements);
    WD_REQUIRE(d_x && d_qs && d_scales, "wd_q8_0_quantize_f16: null pointer");
    WD_REQUIRE(reinterpret_cast<uintptr_t>(d_x) % 8 == 0, "wd_q8_0_quantize_f16: the input must be 8-byte aligned");
    const int blocks = elements / 32;
    enqueue(k_q8_0_quantize_f16, dim3((blocks + 31) / 32), dim3(256), 0, as_stream(stream), d_x, blocks, d_qs, d_scales);
    WD_LAUNCH_CHECK();
    return WD_OK;
}
int wd_gemv_q8_0_q8_1_f32(const uint8_t *d_w, int rows, int cols, const int8_t *d_qs, const uint16_t *d_scales, float *d_y,
                          int32_t *d_block_sums, void *stream) {
    WD_REQUIRE(rows > 0 && cols > 0 && cols % 32 == 0, "Q8_0 x Q8_1 GEMV geometry mismatch (%d x %d)", rows, cols);
    WD_REQUIRE(d_w && d_qs && d_scales && d_y, "wd_gemv_q8_0_q8_1_f32: null pointer");
    WD_REQUIRE(reinterpret_cast<uintptr_t>(d_qs) % 4 == 0, "wd_gemv_q8_0_q8_1_f32: the quantised input must be 4-byte aligned");
    enqueue(k_gemv_q8_0_q8_1, dim3((rows + 3) / 4), dim3(256), 0, as_stream(stream), d_w, rows, cols, d_qs, d_scales, d_y, d_block_sums);
    WD_LAUNCH_CHECK();
    return WD_OK;
}
int wd_convert_f16_to_f32(const uint16_t *d_src, float *d_dst, size_t n, void *stream) {
    WD_REQUIRE(d_src && d_dst && n > 0, "wd_convert_f16_to_f32: invalid arguments");
    enqueue(k_f16_to_f32, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, as_stream(stream), d_src, d_dst, n);
    WD_LAUNCH_CHECK();
    return WD_OK;
}
int wd_convert_f32_to_f16(const float *d_src, uint16_t *d_dst, size_t n, void *stream) {
    WD_REQUIRE(d_src && d_dst && n > 0, "wd_convert_f32_to_f16: invalid arguments");
    enqueue(k_f32_to_f16, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, as_stream(stream), d_src, d_dst, n);
    WD_LAUNCH_CHECK();
    return WD_OK;
}

// ---- router -------------------------------------------------------------------------------
int wd_router_gemv_f32(const float *d_w, const float *d_x, float *d_logits, int rows, int cols, void *stream) {
    WD_REQUIRE(rows > 0 && cols > 0, "router GEMV: invalid shape %d x %d", rows, cols);
    WD_REQUIRE(d_w && d_x && d_logits, "wd_router_gemv_f32: null pointer");
    enqueue(k_router_gemv, dim3((rows + 7) / 8), dim3(256), 0, as_stream(stream), d_w, d_x, d_logits, rows, cols, nullptr,
                                                                             nullptr);
    WD_LAUNCH_CHECK();
    return WD_OK;
}

int wd_topk_softmax(const float *d_logits, int n_experts, int k, float expert_scale, int32_t *d_ids,
                    float *d_weights, void *stream) {
    WD_REQUIRE(n_experts > 0 && n_experts <= 1024 && n_experts % 8 == 0,
               "top-k softmax: n_experts must be a multiple of 8 in (0, 1024] (got %d)", n_experts);
    WD_REQUIRE(k > 0 && k <= 16 && k <= n_experts, "top-k softmax: k must be in (0, 16] (got %d)", k);
    WD_REQUIRE(d_logits && d_ids && d_weights, "wd_topk_softmax: null pointer");
    enqueue(k_topk_softmax, dim3(1), dim3(64), 0, as_stream(stream), d_logits, n_experts, k, expert_scale, d_ids, d_weights,
                                                                nullptr, nullptr);
    WD_LAUNCH_CHECK();
    return WD_OK;
}

}  // extern "C" (a template)
// One IQ matrix of eight rows or more, whose rows fit LDS eight at a time; the activation 16-byte aligned.
static bool iq_streams(int rows, int nb, const int8_t *qs) { return rows >= 8 && nb <= 64 && reinterpret_cast<uintptr_t>(qs) % 16 == 0; }
template <int TYPE>
static void launch_iq_stream(const uint8_t *w, int rows, int nb, const int8_t *qs, const float *d, float *out, int32_t *partials,
                             hipStream_t stream) {
    const int groups = (rows + 7) / 8, nchunks = (nb + 7) / 8;
    if (groups < 1024) {
        // fewer groups than SIMDs: up to eight waves share one
        const int parts = nchunks <= 2 ? 4 : (nchunks <= 4 ? 2 : 1);
        const size_t lds = iq_split_lds<TYPE>(nb, parts);
        auto launch = [&](auto kernel) { enqueue(kernel, groups, 64 * parts * nchunks, lds, stream, w, rows, nb, parts, qs, d, out, partials); };
        if (partials) launch(k_gemv_iq_split<TYPE, true>);
        else launch(k_gemv_iq_split<TYPE, false>);
        return;
    }
    // three workgroups of four waves are what LDS holds per compute unit
    const unsigned wgs = static_cast<unsigned>(std::min((groups + 3) / 4, 768));
    const size_t lds = static_cast<size_t>(nb) * kIqActStride + ((nb * 4 + 15) & ~15) + 4 * kIqWaveStage<TYPE>;
    auto launch = [&](auto kernel) { enqueue(kernel, wgs, 256, lds, stream, w, rows, nb, qs, d, out, partials); };
    if (partials) launch(k_gemv_iq_rows8<TYPE, true>);
    else launch(k_gemv_iq_rows8<TYPE, false>);
}
extern "C" {

// ---- GEMVs --------------------------------------------------------------------------------
static int launch_gemv_q8k(int type, MatSrc src, int mats, int rows, int cols, const int8_t *qs, const float *d,
                           float *out, int32_t *partials, hipStream_t stream) {
    WD_REQUIRE(type == WD_TYPE_IQ3_S || type == WD_TYPE_IQ2_S, "Q8_K-activation GEMV supports IQ3_S and IQ2_S (type %d)",
               type);
    WD_REQUIRE(rows > 0 && cols > 0 && cols % 256 == 0, "invalid low-bit matrix shape %d x %d", rows, cols);
    WD_REQUIRE(mats > 0 && mats <= 64, "expert batch must be in (0, 64] (got %d)", mats);
    WD_REQUIRE(qs && d && out, "low-bit GEMV: null pointer");
    if (mats == 1 && src.single && iq_streams(rows, cols / 256, qs)) {
        if (type == WD_TYPE_IQ3_S) launch_iq_stream<21>(src.single, rows, cols / 256, qs, d, out, partials, stream);
        else launch_iq_stream<22>(src.single, rows, cols / 256, qs, d, out, partials, stream);
        WD_LAUNCH_CHECK();
        return WD_OK;
    }
    const dim3 grid((rows + 15) / 16, mats), block(256);
    const int ppr = partials_per_row(type, cols);
    if (type == WD_TYPE_IQ3_S) {
        if (partials)
            enqueue(k_gemv_iq<21, true>, grid, block, 0, stream, src, rows, cols, qs, d, out, partials, ppr);
        else
            enqueue(k_gemv_iq<21, false>, grid, block, 0, stream, src, rows, cols, qs, d, out, nullptr, 0);
    } else {
        if (partials)
            enqueue(k_gemv_iq<22, true>, grid, block, 0, stream, src, rows, cols, qs, d, out, partials, ppr);
        else
            enqueue(k_gemv_iq<22, false>, grid, block, 0, stream, src, rows, cols, qs, d, out, nullptr, 0);
    }
    WD_LAUNCH_CHECK();
    return WD_OK;
}

// ---- the streaming kernels of Q8_0 and IQ4_NL rows (k_gemv_q8_rows8 and its split form) ---------------------------
// Rows of at least one chunk, up to what the activation may take of LDS; aligned activations; eight rows or more.  Many rows
// (no split) of 17 to 21 blocks stay with the general kernel: more than half of them would be repeated to fill the second chunk
// (9000 x 544 Q8_0: 5.4 us against 4.7).
static bool q8_streams(int rows, int nb, const int8_t *qs) {
    if (rows >= 8 * 1023 + 1 && nb > 16 && nb < 22) return false;
    return rows >= 8 && nb >= 16 && nb <= 512 && reinterpret_cast<uintptr_t>(qs) % 16 == 0;
}
// How the waves of a workgroup share rows of nb blocks, given `groups` groups of eight rows: kb * nch blocks per wave, as few
// repeated ones as the choice allows; kb == 0: rows enough to give every SIMD a group of its own (the kernel without split).
struct Q8Split {
    int kb, nch, waves;
    bool operator==(const Q8Split &o) const { return kb == o.kb && nch == o.nch && waves == o.waves; }
};
static Q8Split q8_split_for(int nb, int groups) {
    const int w16 = (nb + 15) / 16, w32 = (nb + 31) / 32, w64 = (nb + 63) / 64;
    if (groups >= 1024) return {0, 0, 0};
    if (nb < 32 || (16 * w16 < 32 * w32 && w16 <= 8)) return {16, 1, w16};
    // beyond five waves of 32 blocks: that many when a compute unit gets one workgroup, half (two chunks each) when it gets more
    if (w32 <= 5 || (w32 <= 8 && groups <= 256)) return {32, 1, w32};
    return {32, 2, w64};
}
static size_t q8_split_lds(int kind, const Q8Split &sp, int nb) {
    const int stride = kind == 0 ? (sp.kb == 32 ? kQ8sRowStride<0, 32> : kQ8sRowStride<0, 16>)
                                 : (sp.kb == 32 ? kQ8sRowStride<1, 32> : kQ8sRowStride<1, 16>);
    return static_cast<size_t>(nb) * 32 + static_cast<size_t>(sp.waves) * (sp.kb * sp.nch * 4 + 8 * stride) + 512;
}
// Rows of other lengths than whole chunks, or off 16-byte boundaries.
static bool q8_ragged(const uint8_t *w, int nb, int chunk) { return nb % chunk != 0 || reinterpret_cast<uintptr_t>(w) % 16 != 0; }

#define WD_Q8_FIXED_SPLITS \
    WD_Q8_SPLIT(32, 1, 2) WD_Q8_SPLIT(16, 1, 5) WD_Q8_SPLIT(32, 1, 4) WD_Q8_SPLIT(32, 1, 5) WD_Q8_SPLIT(32, 1, 8) \
    WD_Q8_SPLIT(32, 2, 4) WD_Q8_SPLIT(32, 2, 5) WD_Q8_SPLIT(32, 2, 8)

}  // extern "C" (a template)
template <int KIND>
static void launch_q8_stream(const uint8_t *w, int rows, int nb, const int8_t *qs, const uint16_t *d, float *out, int32_t *partials,
                             hipStream_t stream) {
    const int groups = (rows + 7) / 8;
    const Q8Split sp = q8_split_for(nb, groups);
    if (sp.kb) {
        const size_t lds = q8_split_lds(KIND, sp, nb);
        auto launch = [&](auto kernel) { enqueue(kernel, groups, 64 * sp.waves, lds, stream, w, rows, nb, qs, d, out, partials); };
        if constexpr (KIND == 0) {
            // whole chunks on 16-byte boundaries, the usual row lengths (2048, 2560, 4096, 5120, 8192, 10240, 16384 columns):
            // kernels that know their number of waves (2560 x 2560: 4.97 us, 5.16 with the number taken from nb)
            if (!partials && !q8_ragged(w, nb, sp.kb * sp.nch)) {
#define WD_Q8_SPLIT(KB_, NCH_, WAVES_)                                                 \
    if (sp == Q8Split{KB_, NCH_, WAVES_}) {                                             \
        launch(k_gemv_q8_rows8_split<0, KB_, NCH_, WAVES_, false, false>);               \
        return;                                                                          \
    }
                WD_Q8_FIXED_SPLITS
#undef WD_Q8_SPLIT
            }
        }
#define WD_Q8_SPLIT(KB_, NCH_)                                                           \
    if (sp.kb == KB_ && sp.nch == NCH_) {                                                 \
        if (partials) launch(k_gemv_q8_rows8_split<KIND, KB_, NCH_, 0, true, true>);       \
        else launch(k_gemv_q8_rows8_split<KIND, KB_, NCH_, 0, true, false>);               \
    }
        WD_Q8_SPLIT(16, 1)
        WD_Q8_SPLIT(32, 1)
        WD_Q8_SPLIT(32, 2)
#undef WD_Q8_SPLIT
        return;
    }
    // Workgroups of four waves, each taking several row groups beyond 1024 workgroups; chunks of about the same bytes for
    // both kinds
    const int kb = KIND == 1 && nb >= 64 ? 32 : 16, nchunks = (nb + kb - 1) / kb;
    const unsigned wgs = static_cast<unsigned>(std::min((groups + 3) / 4, 1024));
    const size_t lds = static_cast<size_t>(nb) * 32 + static_cast<size_t>(nchunks) * kb * 4 +
                       4 * 8 * (kb == 32 ? kQ8sRowStride<KIND, 32> : kQ8sRowStride<KIND, 16>);
    auto launch = [&](auto kernel) { enqueue(kernel, wgs, 256, lds, stream, w, rows, nb, qs, d, out, partials); };
    const bool ragged = q8_ragged(w, nb, kb);
    if (KIND == 1 && kb == 32) {
        if (partials) launch(k_gemv_q8_rows8<1, 32, true, true>);
        else if (ragged) launch(k_gemv_q8_rows8<1, 32, true, false>);
        else launch(k_gemv_q8_rows8<1, 32, false, false>);
    } else {
        if (partials) launch(k_gemv_q8_rows8<KIND, 16, true, true>);
        else if (ragged) launch(k_gemv_q8_rows8<KIND, 16, true, false>);
        else launch(k_gemv_q8_rows8<KIND, 16, false, false>);
    }
}

extern "C" {

// ---- Q4_0: the streaming kernel takes rows of 8 to 512 blocks, aligned activations -------------------------------------
// Rows that are no whole groups of eight blocks, groups that do not divide a wave, or a matrix off 16-byte boundaries.
static bool q4_ragged(const uint8_t *w, int nb) { return nb % 8 != 0 || 64 % (nb / 8) != 0 || reinterpret_cast<uintptr_t>(w) % 16 != 0; }
// Ragged ones only where the rows are long or the matrix is large: below, the general kernel, which stages nothing, ends sooner
// (us, general / streaming: 640 x 800 2.3 / 3.5, 520 x 1600 3.3 / 3.7, 9000 x 544 3.7 / 4.2; 2560 x 2560 4.5 / 4.1, 3000 x 2592
// 4.9 / 4.2, 5000 x 5120 9.6 / 7.1, 2048 x 12288 16.7 / 7.2, 100000 x 1056 22.5 / 16.0).
static bool q4_streams(const uint8_t *w, int rows, int nb, const int8_t *qs) {
    if (q4_ragged(w, nb < 8 ? 8 : nb) && nb < 64 && static_cast<long long>(rows) * nb < 200000) return false;
    return nb >= 8 && nb <= 512 && reinterpret_cast<uintptr_t>(qs) % 16 == 0;
}
// Its workgroups (waves per workgroup in *wpb): four waves stream best; two when the whole matrix is only a few hundred passes.
static long long q4_stream_wgs(int rows, int nb, int *wpb) {
    const int rpp = 64 / ((nb + 7) / 8);
    const long long passes = (static_cast<long long>(rows) + rpp - 1) / rpp;
    *wpb = passes <= 256 ? 2 : 4;
    return (passes + *wpb - 1) / *wpb;
}

static int launch_gemv_q8_0(int type, MatSrc src, int mats, int rows, int cols, const int8_t *qs, const uint16_t *d,
                            int act_per_mat, float *out, int32_t *partials, hipStream_t stream) {
    WD_REQUIRE(type == WD_TYPE_Q8_0 || type == WD_TYPE_IQ4_NL || type == WD_TYPE_Q4_0,
               "Q8_0-activation GEMV supports Q8_0, IQ4_NL and Q4_0 (type %d)", type);
    WD_REQUIRE(rows > 0 && cols > 0 && cols % 32 == 0, "invalid low-bit matrix shape %d x %d", rows, cols);
    WD_REQUIRE(mats > 0 && mats <= 64, "expert batch must be in (0, 64] (got %d)", mats);
    WD_REQUIRE(qs && d && out, "low-bit GEMV: null pointer");
    const dim3 grid((rows + 15) / 16, mats), block(256);
    const int ppr = partials_per_row(type, cols);
    const int act_stride = act_per_mat ? cols : 0;
    const int nb = cols / 32;
    if (type == WD_TYPE_Q4_0 && mats == 1 && src.single && q4_streams(src.single, rows, nb, qs)) {
        const int lpr = (nb + 7) / 8;
        const bool ragged = q4_ragged(src.single, nb);
        int wpb = 0;
        const unsigned wgs = static_cast<unsigned>(q4_stream_wgs(rows, nb, &wpb));
        const size_t lds = static_cast<size_t>(lpr) * (272 + 64);
        auto launch = [&](auto kernel) { enqueue(kernel, wgs, wpb * 64, lds, stream, src.single, rows, nb, qs, d, out, partials); };
        if (partials) {
            if (wpb == 2) ragged ? launch(k_gemv_q4_stream<true, 1, 2, true>) : launch(k_gemv_q4_stream<true, 1, 2, false>);
            else ragged ? launch(k_gemv_q4_stream<true, 1, 4, true>) : launch(k_gemv_q4_stream<true, 1, 4, false>);
        } else {
            if (wpb == 2) ragged ? launch(k_gemv_q4_stream<false, 1, 2, true>) : launch(k_gemv_q4_stream<false, 1, 2, false>);
            else ragged ? launch(k_gemv_q4_stream<false, 1, 4, true>) : launch(k_gemv_q4_stream<false, 1, 4, false>);
        }
        WD_LAUNCH_CHECK();
        return WD_OK;
    }
    if (type != WD_TYPE_Q4_0 && mats == 1 && src.single && q8_streams(rows, nb, qs)) {
        if (type == WD_TYPE_Q8_0) launch_q8_stream<0>(src.single, rows, nb, qs, d, out, partials, stream);
        else launch_q8_stream<1>(src.single, rows, nb, qs, d, out, partials, stream);
        WD_LAUNCH_CHECK();
        return WD_OK;
    }
#define WD_Q8_LAUNCH(KIND)                                                                                          \
    do {                                                                                                            \
        if (partials)                                                                                               \
            enqueue(k_gemv_q8<KIND, true>, grid, block, 0, stream, src, rows, cols, qs, d, act_stride, out, partials, ppr); \
        else                                                                                                        \
            enqueue(k_gemv_q8<KIND, false>, grid, block, 0, stream, src, rows, cols, qs, d, act_stride, out, nullptr, 0); \
    } while (0)
    if (type == WD_TYPE_Q8_0)
        WD_Q8_LAUNCH(0);
    else if (type == WD_TYPE_IQ4_NL)
        WD_Q8_LAUNCH(1);
    else
        WD_Q8_LAUNCH(2);
#undef WD_Q8_LAUNCH
    WD_LAUNCH_CHECK();
    return WD_OK;
}

int wd_gemv_q6_k_q8_k_f32(const uint8_t *d_w, int rows, int cols, const int8_t *d_act_qs, const float *d_act_scales,
                          const int16_t *d_act_bsums, float *d_out, int32_t *d_partials, void *stream) {
    WD_REQUIRE(d_w && d_act_qs && d_act_scales && d_act_bsums && d_out, "Q6_K GEMV: null pointer");
    WD_REQUIRE(rows > 0 && cols > 0 && cols % 256 == 0, "Q6_K x Q8_K GEMV geometry mismatch (%d x %d)", rows, cols);
    WD_REQUIRE(cols <= 32768, "Q6_K GEMV: at most 32768 columns (got %d)", cols);
    WD_REQUIRE(reinterpret_cast<uintptr_t>(d_act_qs) % 16 == 0 && reinterpret_cast<uintptr_t>(d_act_bsums) % 4 == 0,
               "Q6_K GEMV: the activation quants must be 16-byte aligned, the sums 4-byte aligned");
    const int nb = cols / 256;
    // rows are 210 * nb bytes: they all start on 16-byte boundaries when the matrix does and nb is a multiple of 8
    const bool aligned = reinterpret_cast<uintptr_t>(d_w) % 16 == 0 && nb % 8 == 0;
    // enough rows per wave to pay for staging the activation, few enough to keep every compute unit busy
    int rpw = rows / (4 * 2048);
    rpw = rpw < 1 ? 1 : (rpw > 10 ? 10 : rpw);
    const unsigned wgs = static_cast<unsigned>((static_cast<long long>(rows) + 4LL * rpw - 1) / (4LL * rpw));
    const size_t lds = static_cast<size_t>(nb) * kQ6ActStride + ((nb * 4 + 15) & ~15) + static_cast<size_t>(nb) * 32 + 4 * kQ6StageBytes;
    hipStream_t st = as_stream(stream);
    const bool full = nb % 8 == 0;
    auto launch = [&](auto kernel) { enqueue(kernel, wgs, 256, lds, st, d_w, rows, cols, d_act_qs, d_act_scales, d_act_bsums, d_out, d_partials); };
    if (d_partials) {
        if (aligned) launch(k_gemv_q6k<true, true, true>);  // aligned implies whole passes
        else if (full) launch(k_gemv_q6k<true, false, true>);
        else launch(k_gemv_q6k<true, false, false>);
    } else {
        if (aligned) launch(k_gemv_q6k<false, true, true>);
        else if (full) launch(k_gemv_q6k<false, false, true>);
        else launch(k_gemv_q6k<false, false, false>);
    }
    WD_LAUNCH_CHECK();
    return WD_OK;
}

int wd_gemv_q8_k_f32(int type, const uint8_t *d_w, int rows, int cols, const int8_t *d_act_qs,
                     const float *d_act_scales, float *d_out, int32_t *d_partials, void *stream) {
    WD_REQUIRE(d_w != nullptr, "low-bit GEMV: null weight pointer");
    MatSrc src{};
    src.single = d_w;
    return launch_gemv_q8k(type, src, 1, rows, cols, d_act_qs, d_act_scales, d_out, d_partials, as_stream(stream));
}

int wd_gemv_q8_0_f32(int type, const uint8_t *d_w, int rows, int cols, const int8_t *d_act_qs,
                     const uint16_t *d_act_scales, float *d_out, int32_t *d_partials, void *stream) {
    WD_REQUIRE(d_w != nullptr, "low-bit GEMV: null weight pointer");
    MatSrc src{};
    src.single = d_w;
    return launch_gemv_q8_0(type, src, 1, rows, cols, d_act_qs, d_act_scales, 0, d_out, d_partials, as_stream(stream));
}

// The workgroups of an item of a Q4_0 batch, 0 when the item is launched by itself.
static int q4_batch_wgs(const wd_gemv_item &it, int nb, int *wpb) {
    if (!q4_streams(it.d_w, it.rows, nb, it.d_act_qs)) return 0;
    const long long wgs = q4_stream_wgs(it.rows, nb, wpb);
    return wgs <= 4096 ? static_cast<int>(wgs) : 0;  // (large matrices are not bound by their launch)
}
static int gemv_q4_0_batch(const wd_gemv_item *items, int n_items, int cols, void *stream) {
    const int nb = cols / 32;
    int i = 0;
    while (i < n_items) {
        int wpb = 0, other = 0;
        const int wgs0 = q4_batch_wgs(items[i], nb, &wpb);
        int j = i + 1;
        if (wgs0)
            while (j < n_items && j - i < kGemvBatchMax && q4_batch_wgs(items[j], nb, &other) && other == wpb) ++j;
        if (!wgs0 || j - i == 1) {
            if (const int rc = wd_gemv_q8_0_f32(WD_TYPE_Q4_0, items[i].d_w, items[i].rows, cols, items[i].d_act_qs, items[i].d_act_scales,
                                                items[i].d_out, nullptr, stream))
                return rc;
            ++i;
            continue;
        }
        auto run = [&](auto max) {
            GemvBatch<decltype(max)::value> b{};
            b.n = j - i;
            int wgs = 0;
            bool ragged = false;
            for (int q = 0; q < b.n; ++q) {
                const wd_gemv_item &it = items[i + q];
                b.w[q] = it.d_w, b.act_qs[q] = it.d_act_qs, b.act_d[q] = it.d_act_scales, b.out[q] = it.d_out, b.rows[q] = it.rows;
                b.first_group[q] = wgs;
                ragged = ragged || q4_ragged(it.d_w, nb);
                wgs += q4_batch_wgs(it, nb, &other);
            }
            for (int q = b.n; q <= max; ++q) b.first_group[q] = wgs;
            const size_t lds = static_cast<size_t>((nb + 7) / 8) * (272 + 64);
            auto launch = [&](auto kernel) { enqueue(kernel, wgs, wpb * 64, lds, as_stream(stream), b, nb); };
            if (wpb == 2) ragged ? launch(k_gemv_q4_stream_batch<2, true, max>) : launch(k_gemv_q4_stream_batch<2, false, max>);
            else ragged ? launch(k_gemv_q4_stream_batch<4, true, max>) : launch(k_gemv_q4_stream_batch<4, false, max>);
        };
        if (j - i <= kGemvBatchFew) run(std::integral_constant<int, kGemvBatchFew>{});
        else run(std::integral_constant<int, kGemvBatchMax>{});
        WD_LAUNCH_CHECK();
        i = j;
    }
    return WD_OK;
}

int wd_gemv_q8_0_batch_f32(int type, const wd_gemv_item *items, int n_items, int cols, void *stream) {
    WD_REQUIRE(type == WD_TYPE_Q8_0 || type == WD_TYPE_Q4_0, "batched GEMV: Q8_0 (exact order) or Q4_0 matrices (type %d)", type);
    WD_REQUIRE(items != nullptr && n_items > 0, "batched GEMV: no items");
    WD_REQUIRE(cols > 0 && cols % 32 == 0, "batched GEMV: invalid row length %d", cols);
    for (int i = 0; i < n_items; ++i)
        WD_REQUIRE(items[i].d_w && items[i].d_act_qs && items[i].d_act_scales && items[i].d_out && items[i].rows > 0,
                   "batched GEMV: item %d has a null pointer or no rows", i);
    if (type == WD_TYPE_Q4_0) return gemv_q4_0_batch(items, n_items, cols, stream);
    const int nb = cols / 32;
    // One launch for as many items in a row as take the same split kernel: a workgroup does here exactly what it does for its
    // item alone; anything else is launched by itself.
    auto split_of = [&](const wd_gemv_item &it) {
        return q8_streams(it.rows, nb, it.d_act_qs) ? q8_split_for(nb, (it.rows + 7) / 8) : Q8Split{0, 0, 0};
    };
    int i = 0;
    while (i < n_items) {
        const Q8Split sp = split_of(items[i]);
        int j = i + 1;
        if (sp.kb)
            while (j < n_items && j - i < kGemvBatchMax && split_of(items[j]) == sp) ++j;
        if (!sp.kb || j - i == 1) {
            if (const int rc = wd_gemv_q8_0_f32(type, items[i].d_w, items[i].rows, cols, items[i].d_act_qs, items[i].d_act_scales,
                                                items[i].d_out, nullptr, stream))
                return rc;
            ++i;
            continue;
        }
        auto run = [&](auto max) {
            GemvBatch<decltype(max)::value> b{};
            b.n = j - i;
            int groups = 0;
            bool ragged = false;
            for (int q = 0; q < b.n; ++q) {
                const wd_gemv_item &it = items[i + q];
                b.w[q] = it.d_w, b.act_qs[q] = it.d_act_qs, b.act_d[q] = it.d_act_scales, b.out[q] = it.d_out, b.rows[q] = it.rows;
                b.first_group[q] = groups;
                groups += (it.rows + 7) / 8;
                ragged = ragged || q8_ragged(it.d_w, nb, sp.kb * sp.nch);
            }
            for (int q = b.n; q <= max; ++q) b.first_group[q] = groups;
            const size_t lds = q8_split_lds(0, sp, nb);
            auto launch = [&](auto kernel) { enqueue(kernel, groups, 64 * sp.waves, lds, as_stream(stream), b, nb); };
            bool fixed = false;
#define WD_Q8_SPLIT(KB_, NCH_, WAVES_)                                                                                       \
    if (!ragged && sp == Q8Split{KB_, NCH_, WAVES_}) launch(k_gemv_q8_rows8_split_batch<KB_, NCH_, WAVES_, false, max>), fixed = true;
            WD_Q8_FIXED_SPLITS
#undef WD_Q8_SPLIT
            if (fixed) {
            } else if (sp.kb == 16) launch(k_gemv_q8_rows8_split_batch<16, 1, 0, true, max>);
            else if (sp.nch == 1) launch(k_gemv_q8_rows8_split_batch<32, 1, 0, true, max>);
            else launch(k_gemv_q8_rows8_split_batch<32, 2, 0, true, max>);
        };
        if (j - i <= kGemvBatchFew) run(std::integral_constant<int, kGemvBatchFew>{});
        else run(std::integral_constant<int, kGemvBatchMax>{});
        WD_LAUNCH_CHECK();
        i = j;
    }
    return WD_OK;
}

int wd_gemv_q8_k_experts_f32(int type, const uint8_t *const *d_w_experts, int experts, int rows, int cols,
                             const int8_t *d_act_qs, const float *d_act_scales, float *d_out,
                             int32_t *d_partials, void *stream) {
    WD_REQUIRE(d_w_experts != nullptr, "expert GEMV: null pointer table");
    MatSrc src{};
    src.table = d_w_experts;
    return launch_gemv_q8k(type, src, experts, rows, cols, d_act_qs, d_act_scales, d_out, d_partials,
                           as_stream(stream));
}

int wd_gemv_q8_0_experts_f32(int type, const uint8_t *const *d_w_experts, int experts, int rows, int cols,
                             const int8_t *d_act_qs, const uint16_t *d_act_scales, float *d_out,
                             int32_t *d_partials, void *stream) {
    WD_REQUIRE(d_w_experts != nullptr, "expert GEMV: null pointer table");
    MatSrc src{};
    src.table = d_w_experts;
    return launch_gemv_q8_0(type, src, experts, rows, cols, d_act_qs, d_act_scales, 1, d_out, d_partials,
                            as_stream(stream));
}

// ---- elementwise ------------------------------------------------------------------------------
int wd_silu_mul_experts_f32(const float *d_gate_up, float *d_act, int ffn, int experts, void *stream) {
    WD_REQUIRE(ffn > 0 && experts > 0 && d_gate_up && d_act, "silu*up: invalid arguments");
    enqueue(k_silu_mul_experts, dim3((ffn + 255) / 256, experts), dim3(256), 0, as_stream(stream), d_gate_up, d_act, ffn);
    WD_LAUNCH_CHECK();
    return WD_OK;
}

int wd_weighted_accum_experts_f32(const float *d_experts, const float *d_weights, float *d_accum, int n, int k,
                                  void *stream) {
    WD_REQUIRE(n > 0 && k > 0 && d_experts && d_weights && d_accum, "weighted accumulate: invalid arguments");
    enqueue(k_weighted_accum, dim3((n + 255) / 256), dim3(256), 0, as_stream(stream), d_experts, d_weights, d_accum, n, k);
    WD_LAUNCH_CHECK();
    return WD_OK;
}

int wd_add_shared_f32(float *d_routed, const float *d_shared, const float *d_gate, int n, void *stream) {
    WD_REQUIRE(n > 0 && d_routed && d_shared && d_gate, "add shared: invalid arguments");
    SiteScope site(WD_SITE_FINISH, as_stream(stream));
    enqueue(k_add_shared, dim3((n + 255) / 256), dim3(256), 0, as_stream(stream), d_routed, d_shared, d_gate, d_routed, n);
    WD_LAUNCH_CHECK();
    return WD_OK;
}

// ---- site profiler -----------------------------------------------------------------------
int wd_profile_enable(int on) { return SiteProfiler::instance().enable(on != 0); }
int wd_profile_enabled(void) { return SiteProfiler::instance().enabled() ? 1 : 0; }
int wd_profile_begin(int site, void *stream) {
    WD_REQUIRE(site >= 0 && site < WD_PROFILE_SITE_COUNT, "profiler: site %d out of range", site);
    SiteProfiler::instance().begin(site, as_stream(stream));
    return WD_OK;
}
int wd_profile_end(int site, void *stream) {
    WD_REQUIRE(site >= 0 && site < WD_PROFILE_SITE_COUNT, "profiler: site %d out of range", site);
    SiteProfiler::instance().end(site, as_stream(stream));
    return WD_OK;
}
int wd_profile_flush_token(void) { return SiteProfiler::instance().flush_token(); }
int wd_profile_site(int site, wd_profile_site_stat *out, unsigned long long *tokens) {
    WD_REQUIRE(site >= 0 && site < WD_PROFILE_SITE_COUNT && out, "profiler: site %d out of range, or a null output", site);
    *out = SiteProfiler::instance().stat(site);
    if (tokens) *tokens = SiteProfiler::instance().tokens();
    return WD_OK;
}
const char *wd_profile_site_name(int site) { return profile_site_name(site); }
size_t wd_profile_report(char *buf, size_t cap) {
    const std::string r = SiteProfiler::instance().report();
    if (buf && cap) {
        const size_t n = r.size() < cap - 1 ? r.size() : cap - 1;
        std::memcpy(buf, r.data(), n);
        buf[n] = 0;
    }
    return r.size();
}
int wd_profile_reset(void) {
    SiteProfiler::instance().reset();
    return WD_OK;
}

}  // extern "C"
