// The 16 x 16 x 4 matrix-core instruction of either data type.
#pragma once

namespace isvd {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Mfma;

template <>
struct Mfma<double> {
  using acc_t = d4;
  // v_mfma_f64_16x16x4f64: A lane holds A[lane%16][lane/16], B lane holds B[lane/16][lane%16];
  // D register g of a lane holds D[lane/16 + 4g][lane%16].
  static __device__ __forceinline__ acc_t run(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int g) { return (lane >> 4) + 4 * g; }
};

template <>
struct Mfma<float> {
  using acc_t = f4;
  // v_mfma_f32_16x16x4f32: same operand layout; D register g holds D[4*(lane/16) + g][lane%16].
  static __device__ __forceinline__ acc_t run(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int g) { return 4 * (lane >> 4) + g; }
};

}  // namespace isvd
