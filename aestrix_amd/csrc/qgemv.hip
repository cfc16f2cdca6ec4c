// qgemv.hip -- the qGEMV's launches (kernel: qgemv_kernel.hpp), 16-bit T.
#include "qgemv_kernel.hpp"

namespace imq {

hipError_t launch_qgemv(const uint32_t* w, const void* scales, const void* biases, const void* x,
                        void* y, int k, int n, int m, int dtype, hipStream_t stream) {
  switch (dtype) {
    case kBf16: return launch_t<kBf16>(w, scales, biases, x, y, k, n, m, nullptr, stream);
    case kF16: return launch_t<kF16>(w, scales, biases, x, y, k, n, m, nullptr, stream);
    case kF32: return launch_qgemv_f32(w, scales, biases, x, y, k, n, m, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_qgemv_resid_add(const uint32_t* w, const void* scales, const void* biases,
                                  const void* x, const void* resid, void* y, int k, int n, int m,
                                  int dtype, hipStream_t stream) {
  if (m > 4 || !resid) return hipErrorInvalidValue;
  GvPair pr{0, 0, 0, 0, 1.0f, 1.0f};
  pr.resid = resid;
  switch (dtype) {
    case kBf16: return launch_t<kBf16>(w, scales, biases, x, y, k, n, m, &pr, stream);
    case kF16: return launch_t<kF16>(w, scales, biases, x, y, k, n, m, &pr, stream);
    default: return hipErrorInvalidValue;
  }
}

bool qgemv_norm_fits(int k, int n, int m, int width, int dtype, const void* x, const float* nw) {
  if (m < 1 || m > kQgemvNormMaxM || (dtype != kBf16 && dtype != kF16)) return false;
  // The RMSNorm kernel's 16-byte form, at most two pieces per thread.
  if (k % 8 != 0 || k / 8 > 2 * kThreads) return false;
  if (((uintptr_t)x & 15u) != 0 || ((uintptr_t)nw & 15u) != 0) return false;
  // The x tile must be the whole row.
  const Plan p = width > 0 ? make_plan(k, 2 * width, m <= 1 ? 1 : 2, 2, 2)
                           : make_plan(k, n, m <= 1 ? 1 : 2, 2);
  return p.kt == k;
}

hipError_t launch_qgemv_norm(const uint32_t* w, const void* scales, const void* biases,
                             const void* x, const float* nw, float eps, void* y, int k, int n,
                             int m, int dtype, hipStream_t stream) {
  if (!qgemv_norm_fits(k, n, m, 0, dtype, x, nw)) return hipErrorInvalidValue;
  GvPair pr{0, 0, 0, 0, 1.0f, 1.0f};
  pr.norm_w = nw;
  pr.eps = eps;
  switch (dtype) {
    case kBf16: return launch_t<kBf16>(w, scales, biases, x, y, k, n, m, &pr, stream);
    default: return launch_t<kF16>(w, scales, biases, x, y, k, n, m, &pr, stream);
  }
}

hipError_t launch_qgemv_swiglu_norm(const uint32_t* w, const void* scales, const void* biases,
                                    const void* x, const float* nw, float eps, void* y, int ldy,
                                    int k, int n, int m, int width, int gate_row, int up_row,
                                    int dtype, hipStream_t stream) {
  if (!qgemv_norm_fits(k, n, m, width, dtype, x, nw)) return hipErrorInvalidValue;
  GvPair pr{gate_row, up_row, width, ldy, 1.0f, 1.0f};
  pr.norm_w = nw;
  pr.eps = eps;
  switch (dtype) {
    case kBf16: return launch_t<kBf16>(w, scales, biases, x, y, k, n, m, &pr, stream);
    default: return launch_t<kF16>(w, scales, biases, x, y, k, n, m, &pr, stream);
  }
}

hipError_t launch_qgemv_swiglu(const uint32_t* w, const void* scales, const void* biases,
                               const void* x, void* y, int ldy, int k, int n, int m, int width,
                               int gate_row, int up_row, float in_scale, float out_scale,
                               int dtype, hipStream_t stream) {
  if (m > kQgemvSwigluMaxM) return hipErrorInvalidValue;
  const GvPair pr{gate_row, up_row, width, ldy, in_scale, out_scale};
  switch (dtype) {
    case kBf16: return launch_t<kBf16>(w, scales, biases, x, y, k, n, m, &pr, stream);
    case kF16: return launch_t<kF16>(w, scales, biases, x, y, k, n, m, &pr, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace imq
