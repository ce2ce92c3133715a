// Pieces shared by the matrix product kernels (gemm.hip, gemm_ksplit.hip): operand types, MFMA wrapper, LDS layout.
#pragma once

#include "h3hip_internal.h"

#include <string>
#include <type_traits>

namespace h3 {

// A product's operands as the host hands them to a kernel (strides in GemmParams, in elements).
struct GemmArgs {
  const char *a, *w;
  const float *sw, *sa;  // column and row scales (NULL where the format has none)
  char *out;             // C, or the residual X
  const float *bias;     // NULL: none
  const unsigned char *rtype;
  const float *gate;
  int ntypes;  // rows of the gate table
  bool vec;    // 16-byte accesses to the output and the column vectors are aligned
};

// gemm_ksplit.hip: the tile configurations (96 x 128 has no int8 form: its accumulators spill) and their launch.
enum { KSPLIT_32x32 = 0, KSPLIT_64x64 = 1, KSPLIT_96x64 = 2, KSPLIT_96x128 = 3 };
int launch_gemm_ksplit(int wfmt, int kcfg, int ot, int epi, const GemmArgs &g, const GemmParams &p, hipStream_t stream,
                       std::string *err);

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// operand types of a kernel: int8 (q8), half (f16, h8), bfloat (bf16)
enum { A_I8 = 0, A_F16 = 1, A_BF16 = 2 };
// epilogue scaling: sa[m] * sw[n] (q8), sw[n] (h8), none (f16, bf16)
enum { S_ROW_COL = 0, S_COL = 1, S_NONE = 2 };

enum { T_BF16 = 1, T_F16 = 2, T_F32 = 3 };

template <int AT>
using AccOf = typename std::conditional<AT == A_I8, i32x16, f32x16>::type;

// one 32 x 32 product over a 32-byte K slice per lane half (32 int8 or 16 16-bit values of K)
template <int AT>
__device__ __forceinline__ AccOf<AT> mma(i32x4 a, i32x4 b, AccOf<AT> c) {
  if constexpr (AT == A_I8) return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
  else if constexpr (AT == A_F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

}  // namespace

}  // namespace h3
