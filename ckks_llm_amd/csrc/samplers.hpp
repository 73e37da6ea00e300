// Step functions that turn random words into small signed integers (Sampler_impl.cuh:27-113).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ckks {

// Steps of the discrete Gaussian as thresholds on the 32-bit word: value >= k  <=>  u >= thr[k-1], k = 1..19; the negative side is
// the mirror image u -> ~u.  thr[k-1] = 2^32 - floor(2^32 * Q(k / 3.2) + 0.5) with Q the upper normal tail, i.e. the probability of a
// word is taken at the middle of its cell.  convert_gaussian_xq (Sampler_impl.cuh:27-70) evaluates the same step function in float
// arithmetic (trunc(3.2 * normcdfinvf(u / (2^32-1))), clamped to +-19.2); the two differ only for words within float rounding of a
// step, and an integer rule is the same on every machine.
struct GaussSteps {
    uint32_t thr[19];
};
const GaussSteps& gauss_steps();
// every threshold lies above 2^31, so only the larger of u and ~u can pass any
__device__ __forceinline__ int gauss_value(uint32_t u, const GaussSteps& g) {
    const uint32_t w = u > ~u ? u : ~u;
    int v = 0;
#pragma unroll
    for (int k = 0; k < 19; k++) v += (w >= g.thr[k]);
    return u >> 31 ? v : -v;
}

}  // namespace ckks
