// The MFMA instruction of each operand type of the orbital contraction and the
// lane layout of its operands and results.
#pragma once
#include <hip/hip_bf16.h>
#include <hip/hip_runtime.h>

namespace qmcb {

typedef double d4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef __bf16 b8v __attribute__((ext_vector_type(8)));

template <typename TI>
struct Mfma;

template <>
struct Mfma<double> {
  typedef d4v acc_t;
  typedef double acc_s;
  static constexpr int KPL = 1;  // k values per lane per instruction
  __device__ static acc_t run(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // output row of accumulator element i in lane group lk = lane / 16
  __device__ static constexpr int row(int lk, int i) { return 4 * i + lk; }
};

template <>
struct Mfma<float> {
  typedef f4v acc_t;
  typedef float acc_s;
  static constexpr int KPL = 1;
  __device__ static acc_t run(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static constexpr int row(int lk, int i) { return 4 * lk + i; }
};

template <>
struct Mfma<__hip_bfloat16> {
  typedef f4v acc_t;
  typedef float acc_s;
  static constexpr int KPL = 8;
  __device__ static acc_t run(b8v a, b8v b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  __device__ static constexpr int row(int lk, int i) { return 4 * lk + i; }
};

}  // namespace qmcb
