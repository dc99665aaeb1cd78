// Three chained v_mfma_f32_16x16x32_f16 from a given accumulator, as a row of the screened search computes a.b - n_b/2: the
// test compares them with 64-bit sums.
#include <hip/hip_runtime.h>

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

// One wave per item: a [16][96] and b [16][96] halves (b by columns of the product), c [16] by column, d [16][16].
__global__ __launch_bounds__(64) void k_products(const _Float16 *__restrict__ a, const _Float16 *__restrict__ b,
                                                 const float *__restrict__ c, float *__restrict__ d) {
    const int i = threadIdx.x & 15, g = threadIdx.x >> 4;
    const long long item = blockIdx.x;
    f4 acc;
    for (int q = 0; q < 4; ++q) acc[q] = c[item * 16 + i];
    for (int p = 0; p < 3; ++p) {
        const long long at = (item * 16 + i) * 96 + 32 * p + 8 * g;
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const h8 *>(a + at), *reinterpret_cast<const h8 *>(b + at), acc, 0, 0, 0);
    }
    for (int q = 0; q < 4; ++q) d[(item * 16 + 4 * g + q) * 16 + i] = acc[q];
}

extern "C" int mfma_error_run(const void *a, const void *b, const float *c, float *d, int items, void *stream) {
    if (!a || !b || !c || !d || items < 1) return 1;
    hipLaunchKernelGGL(k_products, dim3((unsigned)items), dim3(64), 0, (hipStream_t)stream, (const _Float16 *)a, (const _Float16 *)b, c, d);
    return hipGetLastError() == hipSuccess ? 0 : 2;
}
