// Exhaustive check of vz::sqrt_rn (venusaur_amd/csrc/vz_device.h), the
// hardware reciprocal square root refined by one fma Newton-Raphson step,
// against the IEEE root sqrtf(x) for every float in [2^-64, 2^64): 128
// exponents, all 2^23 significands.  The root is also compared with
// (float)sqrt((double)x), which rounds once correctly (53 >= 2 * 24 + 2), and
// the unrefined x * v_rsq_f32(x) is counted as a control that the comparison
// can fail.  Values outside the range, where sqrt_rn takes the IEEE root, are
// checked at a few thousand places.  Test infrastructure: loaded only by
// tests/test_gpu_sqrt.py.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../venusaur_amd/csrc/vz_device.h"

namespace {

constexpr unsigned long long kExps = 128ull;  // biased exponents 63 .. 190: 2^-64 .. 2^63
constexpr unsigned long long kValues = kExps << 23;
constexpr unsigned long long kOutside = 1ull << 16;  // every 65536th of all floats

// out: [0] root != double reference, [1] sqrt_rn != root, [2] unrefined !=
// root, [3] values visited, [4] slots of bad taken; bad: the first mismatches
// of [1]
__global__ void k_sqrt(unsigned long long* out, uint32_t* bad)
{
    unsigned long long d_ref = 0, d_rn = 0, d_raw = 0, seen = 0;
    for (unsigned long long i = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x; i < kValues + kOutside;
         i += (unsigned long long)gridDim.x * blockDim.x) {
        const bool range = i < kValues;
        const uint32_t bits = range ? (uint32_t)i + (63u << 23) : (uint32_t)(i - kValues) << 16;
        const float x = __uint_as_float(bits);
        const float q = sqrtf(x), g = vz::sqrt_rn(x);
        if (range) {
            d_ref += __float_as_uint(q) != __float_as_uint((float)sqrt((double)x)) ? 1ull : 0ull;
            d_raw += __float_as_uint(x * __builtin_amdgcn_rsqf(x)) != __float_as_uint(q) ? 1ull : 0ull;
        }
        if (__float_as_uint(g) != __float_as_uint(q) && !(g != g && q != q)) {
            const unsigned long long k = atomicAdd(&out[4], 1ull);
            if (k < 4ull) bad[k] = bits;
            d_rn++;
        }
        seen++;
    }
    atomicAdd(&out[0], d_ref);
    atomicAdd(&out[1], d_rn);
    atomicAdd(&out[2], d_raw);
    atomicAdd(&out[3], seen);
}

}  // namespace

// Runs the check; out receives {root != double, sqrt_rn != root, unrefined !=
// root, values visited, values expected} and bad up to four mismatching
// inputs.  Returns 0, or a HIP error code.
extern "C" int vz_check_sqrt_rn(unsigned long long* out, uint32_t* bad)
{
    unsigned long long* d_out = nullptr;
    uint32_t* d_bad = nullptr;
    hipError_t err = hipMalloc(&d_out, 5 * sizeof(unsigned long long));
    if (err == hipSuccess) err = hipMalloc(&d_bad, 4 * sizeof(uint32_t));
    if (err == hipSuccess) err = hipMemset(d_out, 0, 5 * sizeof(unsigned long long));
    if (err == hipSuccess) err = hipMemset(d_bad, 0, 4 * sizeof(uint32_t));
    if (err == hipSuccess) {
        hipLaunchKernelGGL(k_sqrt, dim3(8192), dim3(256), 0, 0, d_out, d_bad);
        err = hipGetLastError();
    }
    if (err == hipSuccess) err = hipDeviceSynchronize();
    if (err == hipSuccess) err = hipMemcpy(out, d_out, 4 * sizeof(unsigned long long), hipMemcpyDeviceToHost);
    if (err == hipSuccess) err = hipMemcpy(bad, d_bad, 4 * sizeof(uint32_t), hipMemcpyDeviceToHost);
    out[4] = kValues + kOutside;
    if (d_out) (void)hipFree(d_out);
    if (d_bad) (void)hipFree(d_bad);
    return (int)err;
}
