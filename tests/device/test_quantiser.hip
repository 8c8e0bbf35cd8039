// The short forms of the activations' Q8_0 quantiser beside the general ones, for test_gpu_quantiser.py: every quotient of the range that they
// serve, and whole steps of 512 values.
#include "wd_common.h"
#include "wd_fused.cuh"

namespace wd {

// floats of bits first .. first + count - 1; wrong[i]: how many quotients i differ, wrong[2 + i]: bits of one of them.
__global__ __launch_bounds__(256) void k_quotients(uint32_t first, uint32_t count, uint32_t *wrong) {
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < count; i += gridDim.x * 256u) {
        const float a = bits_f(first + i);
        const float inverse = 127.0f / a, scale = a / 127.0f;
        if (f_bits(quot_ordinary(127.0f, a)) != f_bits(inverse)) atomicAdd(wrong, 1u), wrong[2] = first + i;
        if (f_bits(over_127(a)) != f_bits(scale)) atomicAdd(wrong + 1, 1u), wrong[3] = first + i;
    }
}

// Step s (values 512 s .. 512 s + 511) by wave s: quants and scales by the form that dispatch C takes and by the general one; general[s]: the former had
// to go over to the latter.
__global__ __launch_bounds__(64) void k_steps(const float *x, int8_t *qs, uint16_t *d, int8_t *qs_general, uint16_t *d_general, int *general) {
    const int lane = threadIdx.x, s = blockIdx.x, base = 512 * s + 8 * lane;
    const float4 v0 = *reinterpret_cast<const float4 *>(x + base), v1 = *reinterpret_cast<const float4 *>(x + base + 4);
    lds_quantize_q8_0_step<true>(v0, v1, true, base, qs, d, lane);
    lds_quantize_q8_0_step<false>(v0, v1, true, base, qs_general, d_general, lane);
    uint32_t m = umax_step<kDppXor1>(f_bits(max3_abs(max3_abs(max3_abs(v0.x, v0.y, v0.z), v0.w, v1.x), max3_abs(v1.y, v1.z, v1.w), 0.0f)));
    m = umax_step<kDppXor2>(m);
    uint32_t worst = 0u;
    const float inverse = quot_ordinary(127.0f, bits_f(m));
    (void)quants_ordinary(v0, inverse, worst), (void)quants_ordinary(v1, inverse, worst);
    const bool g = quants_not_ordinary(worst, m);
    if (lane == 0) general[s] = g;
}

}  // namespace wd

extern "C" int test_quotients(uint32_t first, uint32_t count, uint32_t *d_wrong) {
    wd::k_quotients<<<4096, 256>>>(first, count, d_wrong);
    return static_cast<int>(hipGetLastError());
}
extern "C" int test_steps(const float *x, int steps, int8_t *qs, uint16_t *d, int8_t *qs_general, uint16_t *d_general, int *general) {
    wd::k_steps<<<steps, 64>>>(x, qs, d, qs_general, d_general, general);
    return static_cast<int>(hipGetLastError());
}
extern "C" void test_range(uint32_t *lo, uint32_t *span) { *lo = wd::kQuantLo, *span = wd::kQuantSpan; }
