// qgemv_f32.hip -- the qGEMV (qgemv_kernel.hpp) for T = f32.
#include "qgemv_kernel.hpp"

namespace imq {

hipError_t launch_qgemv_f32(const uint32_t* w, const void* scales, const void* biases,
                            const void* x, void* y, int k, int n, int m, hipStream_t stream) {
  return launch_t<kF32>(w, scales, biases, x, y, k, n, m, nullptr, stream);
}

}  // namespace imq
