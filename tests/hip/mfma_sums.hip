// Dot products of the two f16 matrix instructions that the inlier screens use
// (csrc/screen.hpp: 16x16x32, csrc/rmf.hip: 16x16x16), for the test of the FP32
// accumulation error that their bounds assume. One wavefront per batch of 16 x 16
// dot products of K terms.
#include <hip/hip_runtime.h>
#include <cstdint>

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

template <int K>
__global__ __launch_bounds__(64) void sums_kernel(const _Float16* __restrict__ a, const _Float16* __restrict__ b,
                                                  float* __restrict__ d)
{
    const uint32_t lane = threadIdx.x, r = lane & 15, q = lane >> 4;
    const size_t at = (size_t)blockIdx.x * 16 * K + r * K + q * (K / 4);
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    v4f s;
    if constexpr (K == 32)
        s = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const v8h*>(a + at), *reinterpret_cast<const v8h*>(b + at),
                                                   zero, 0, 0, 0);
    else
        s = __builtin_amdgcn_mfma_f32_16x16x16f16(*reinterpret_cast<const v4h*>(a + at), *reinterpret_cast<const v4h*>(b + at),
                                                  zero, 0, 0, 0);
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) d[(size_t)blockIdx.x * 256 + (4 * q + j) * 16 + r] = s[j];
}

// a, b: (batches, 16, k) f16, 16-byte aligned; d: (batches, 16, 16) FP32,
// d[i][j] = a[i] . b[j]; k is 16 or 32
extern "C" int mfma_sums(int k, const void* a, const void* b, float* d, uint32_t batches, hipStream_t stream)
{
    if ((k != 16 && k != 32) || a == nullptr || b == nullptr || d == nullptr || batches == 0) return -1;
    const _Float16 *x = static_cast<const _Float16*>(a), *y = static_cast<const _Float16*>(b);
    if (k == 32) sums_kernel<32><<<batches, 64, 0, stream>>>(x, y, d);
    else sums_kernel<16><<<batches, 64, 0, stream>>>(x, y, d);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
