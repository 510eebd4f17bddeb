// lmx_digit_fmt.hip -- the digit kernels of one weight format (LMX_DIGIT_FMT,
// set by the build: one translation unit per format, compiled side by side).
#include "lmx_digit_kernels.hpp"

namespace lmx {

template <int FMT> int digit_gemv_fmt(const GemvArgs &a, int nv, void *stream);
template <int FMT> int digit_gemm_fmt(const GemvArgs &a, const DigitVectors &d, void *stream);
template <int FMT> int code_copy_fmt(const void *planes, size_t Npad, size_t Kp, void *codes, void *stream);

template <>
int digit_gemv_fmt<LMX_DIGIT_FMT>(const GemvArgs &a, int nv, void *stream) {
  return launch_digit_gemv_fmt<LMX_DIGIT_FMT>(a, nv, static_cast<hipStream_t>(stream));
}

template <>
int digit_gemm_fmt<LMX_DIGIT_FMT>(const GemvArgs &a, const DigitVectors &d, void *stream) {
  return launch_gemm_fmt<LMX_DIGIT_FMT>(a, d, static_cast<hipStream_t>(stream));
}

template <>
int code_copy_fmt<LMX_DIGIT_FMT>(const void *planes, size_t Npad, size_t Kp, void *codes, void *stream) {
  return launch_code_copy_fmt<LMX_DIGIT_FMT>(planes, Npad, Kp, codes, static_cast<hipStream_t>(stream));
}

}  // namespace lmx
