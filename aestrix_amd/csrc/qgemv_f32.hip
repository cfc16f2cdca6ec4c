// qgemv_f32.hip -- the qGEMV (qgemv_kernel.hpp) for T = f32.
#include "qgemv_kernel.hpp"

namespace imq {

hipError_t launch_qgemv_f32(const uint32_t* w, const void* scales, const void* biases,
                            const void* x, void* y, int k, int n, int m, hipStream_t stream) {
  return launch_t<kF32>(w, scales, biases, x, y, k, n, m, nullptr, stream);
}

// The SiLU in the store: a launch of its own took about 2 us after each of the
// chain's first two projections (chain at four timesteps 56.2 -> 51.6 us).
hipError_t launch_qgemv_f32_silu(const uint32_t* w, const float* scales, const float* biases,
                                 const float* x, float* y, float* y_silu, int k, int n, int m,
                                 hipStream_t stream) {
  GvPair pr{0, 0, 0, 0, 1.0f, 1.0f};
  pr.silu = y_silu;
  return launch_t<kF32>(w, scales, biases, x, y, k, n, m, &pr, stream);
}

}  // namespace imq
