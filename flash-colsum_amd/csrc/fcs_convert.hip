// fp32 operands rounded to fp16 on the way to the column-mean kernels, with the range test in the same pass.
//
// Bound by memory: 4 bytes read and 2 written per element.  One launch takes both operands, a thread keeps eight 16-byte loads
// in flight, and a value beyond fp16's range (or a NaN) is reported through a flag that only such a value touches, so there is
// nothing to clear and nothing to reduce.  Before, the library underneath made |x| of each operand (a copy), took its maximum
// (one pass, one number read back) and converted it (another pass): B 16, H 16, S 577, D 64 (2 x 37.8 MB) 12 + 16 + 9 us and a wait
// per operand; the call 138 us.  Now the call takes 54 us, and a small one (H 4, S 50) 25 us instead of 65.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fcs_device.h"
#include "flash_colsum.h"

namespace fcs {

constexpr int kConvThreads = 256;
constexpr int kConvDepth = 4;                            // 8-element pieces per thread and step
constexpr int kConvStep = kConvThreads * kConvDepth;     // pieces per workgroup and step
constexpr uint32_t kHalfMaxBits = 0x477fe000u;           // 65504.0f

// Pieces [0, p0) are those of the first operand, [p0, p0 + p1) those of the second; the last piece of an operand may be short.
__global__ __launch_bounds__(kConvThreads) void fcs_round_f16_kernel(const float *s0, _Float16 *d0, int64_t n0, int64_t p0,
                                                                      const float *s1, _Float16 *d1, int64_t n1, int64_t p1,
                                                                      uint32_t *flag)
{
    uint32_t worst = 0;  // largest |x| as a bit pattern: a NaN's is above every number's
    for (int64_t base = (int64_t)blockIdx.x * kConvStep; base < p0 + p1; base += (int64_t)gridDim.x * kConvStep) {
        floatx4 v[kConvDepth][2];
#pragma unroll
        for (int j = 0; j < kConvDepth; ++j) {
            v[j][0] = v[j][1] = floatx4{0.f, 0.f, 0.f, 0.f};
            const int64_t p = base + j * kConvThreads + (int)threadIdx.x;
            const bool second = p >= p0;
            const int64_t e = (second ? p - p0 : p) * 8, n = second ? n1 : n0;
            const float *s = (second ? s1 : s0) + e;
            if (p < p0 + p1 && e + 8 <= n) {
                v[j][0] = *reinterpret_cast<const floatx4 *>(s);
                v[j][1] = *reinterpret_cast<const floatx4 *>(s + 4);
            }
        }
#pragma unroll
        for (int j = 0; j < kConvDepth; ++j) {
            const int64_t p = base + j * kConvThreads + (int)threadIdx.x;
            if (p >= p0 + p1) continue;
            const bool second = p >= p0;
            const int64_t e = (second ? p - p0 : p) * 8, n = second ? n1 : n0;
            const float *s = (second ? s1 : s0) + e;
            _Float16 *d = (second ? d1 : d0) + e;
            if (e + 8 <= n) {
                half8 h;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float x = v[j][i >> 2][i & 3];
                    worst = max(worst, __builtin_bit_cast(uint32_t, x) & 0x7fffffffu);
                    h[i] = (_Float16)x;  // to nearest, ties to even
                }
                *reinterpret_cast<half8 *>(d) = h;
            } else {
                for (int i = 0; e + i < n; ++i) {
                    worst = max(worst, __builtin_bit_cast(uint32_t, s[i]) & 0x7fffffffu);
                    d[i] = (_Float16)s[i];
                }
            }
        }
    }
    if (worst > kHalfMaxBits) __hip_atomic_store(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace fcs

extern "C" int fcs_round_f16(const float *src0, void *dst0, int64_t n0, const float *src1, void *dst1, int64_t n1, uint32_t *flag,
                             void *hip_stream)
{
    if (!src0 || !dst0 || !src1 || !dst1 || !flag) return FCS_E_NULL;
    if (n0 < 1 || n1 < 1) return FCS_E_DIMS;
    for (const void *p : {(const void *)src0, (const void *)dst0, (const void *)src1, (const void *)dst1})
        if (reinterpret_cast<uintptr_t>(p) & 15u) return FCS_E_STRIDE;
    const int64_t p0 = (n0 + 7) / 8, p1 = (n1 + 7) / 8;
    const int64_t steps = (p0 + p1 + fcs::kConvStep - 1) / fcs::kConvStep;
    // 16 workgroups per compute unit at most: beyond that they walk
    const unsigned grid = (unsigned)(steps < 4096 ? steps : 4096);
    hipLaunchKernelGGL(fcs::fcs_round_f16_kernel, dim3(grid), dim3(fcs::kConvThreads), 0, reinterpret_cast<hipStream_t>(hip_stream),
                       src0, static_cast<_Float16 *>(dst0), n0, p0, src1, static_cast<_Float16 *>(dst1), n1, p1, flag);
    return (int)hipGetLastError();
}
