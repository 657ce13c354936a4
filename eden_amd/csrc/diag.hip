// diag.hip -- self-test of device arithmetic the kernels rely on for bit-exactness: div_rn and
// the divisions by a known reciprocal (div_c, div_c2) against the compiler's division, over hashed
// operand pairs and a list of special values. Reached through include/edenhip_diag.h; not used by the simulation path.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/edenhip_diag.h"
#include "device_model.hpp"

using namespace edenhip;

namespace {

__device__ __forceinline__ uint64_t mix64(uint64_t x) {
    x ^= x >> 33;
    x *= 0xff51afd7ed558ccdull;
    x ^= x >> 33;
    x *= 0xc4ceb9fe1a85ec53ull;
    x ^= x >> 33;
    return x;
}

// operand i of pair k: raw random bits, or (every other pair) a random significand and sign
// with an exponent drawn from [80, 175], inside div_rn's fast range [67, 187]
__device__ __forceinline__ float operand(uint64_t seed, uint64_t k, int i) {
    const uint64_t h = mix64(seed ^ mix64(2 * k + (uint64_t)i));
    uint32_t bits = (uint32_t)h;
    if (k & 1) {
        const uint32_t e = 80u + (uint32_t)((h >> 32) % 96u);
        bits = (bits & 0x807FFFFFu) | (e << 23);
    }
    return __uint_as_float(bits);
}

__device__ __forceinline__ bool same(float a, float b) {
    const bool na = a != a, nb = b != b;
    return (na && nb) || __float_as_uint(a) == __float_as_uint(b);
}

__global__ void divide_check(uint64_t seed, int64_t count, const float *__restrict__ special, int32_t n_special,
                             unsigned long long *__restrict__ out) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    unsigned long long bad = 0;
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < count; k += stride) {
        const float n = operand(seed, (uint64_t)k, 0), d = operand(seed, (uint64_t)k, 1);
        if (!same(div_rn(n, d), n / d)) bad++;
    }
    const int64_t ns = (int64_t)n_special * n_special;
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < ns; k += stride) {
        const float n = special[k / n_special], d = special[k % n_special];
        if (!same(div_rn(n, d), n / d)) bad++;
    }
    if (bad) atomicAdd(out, bad);
}

// Mismatches of the divisions by a known reciprocal, each over the operands it is meant for:
// 0 div_c with 1 / d rounded to double, where n / d is zero, infinite, NaN or above the least
//   normal float; 1 the same with the reciprocal of a float refined from the double it was rounded
//   from (gate_next_fast's time constant), for moderate d; 2 div_c2, finite n and d
__device__ __forceinline__ void reciprocal_mismatches(float n, float d, unsigned long long (&bad)[3]) {
    auto in_range = [](float a, float q) { return a == 0.0f || !(fabsf(q) <= 0x1p-126f); };
    const float q = n / d;
    if (in_range(n, q) && !same(div_c(n, 1.0 / (double)d), q)) bad[0]++;
    const float ad = fabsf(d);
    if (ad >= 0x1p-60f && ad <= 0x1p60f) {
        const float tau = (float)recip64(d), qt = n / tau;
        if (in_range(n, qt) && !same(div_c(n, recip_refine((double)tau, (double)d)), qt)) bad[1]++;
    }
    if (fabsf(n) <= 0x1.fffffep127f && ad <= 0x1.fffffep127f && d != 0.0f) {
        const float q2 = div_c2(n, recip2(d));
        if (!same(q2, q) && !(q2 == 0.0f && q == 0.0f)) bad[2]++;
    }
}

__global__ void reciprocal_check(uint64_t seed, int64_t count, const float *__restrict__ special, int32_t n_special,
                                 unsigned long long *__restrict__ out) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x, first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long bad[3] = {0, 0, 0};
    for (int64_t k = first; k < count; k += stride)
        reciprocal_mismatches(operand(seed, (uint64_t)k, 0), operand(seed, (uint64_t)k, 1), bad);
    const int64_t ns = (int64_t)n_special * n_special;
    for (int64_t k = first; k < ns; k += stride) reciprocal_mismatches(special[k / n_special], special[k % n_special], bad);
    for (int i = 0; i < 3; i++)
        if (bad[i]) atomicAdd(out + i, bad[i]);
}

// One of the two checks above with its operands on the device, and its `n_out` counts.
template <class K>
int run_check(K kernel, uint64_t seed, int64_t count, const float *special, int32_t n_special, int64_t *mismatches, int n_out) {
    if (!mismatches || count < 0 || n_special < 0 || (n_special > 0 && !special)) return -1;
    float *d_special = nullptr;
    unsigned long long *d_out = nullptr;
    const size_t sb = sizeof(float) * (size_t)(n_special > 0 ? n_special : 1), ob = sizeof(unsigned long long) * (size_t)n_out;
    if (hipMalloc(&d_special, sb) != hipSuccess) return -2;
    if (hipMalloc(&d_out, ob) != hipSuccess) {
        (void)hipFree(d_special);
        return -2;
    }
    int rc = 0;
    unsigned long long h_out[3] = {};
    if ((n_special > 0 && hipMemcpy(d_special, special, sizeof(float) * (size_t)n_special, hipMemcpyHostToDevice) != hipSuccess) ||
        hipMemset(d_out, 0, ob) != hipSuccess)
        rc = -2;
    if (rc == 0) {
        hipLaunchKernelGGL(kernel, dim3(4096), dim3(256), 0, 0, seed, count, d_special, n_special, d_out);
        if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess ||
            hipMemcpy(h_out, d_out, ob, hipMemcpyDeviceToHost) != hipSuccess)
            rc = -2;
    }
    (void)hipFree(d_special);
    (void)hipFree(d_out);
    for (int i = 0; i < n_out; i++) mismatches[i] = (int64_t)h_out[i];
    return rc;
}

}  // namespace

extern "C" int edenhip_diag_divide(uint64_t seed, int64_t count, const float *special, int32_t n_special,
                                   int64_t *mismatches) {
    return run_check(divide_check, seed, count, special, n_special, mismatches, 1);
}

extern "C" int edenhip_diag_reciprocals(uint64_t seed, int64_t count, const float *special, int32_t n_special,
                                        int64_t mismatches[3]) {
    return run_check(reciprocal_check, seed, count, special, n_special, mismatches, 3);
}
