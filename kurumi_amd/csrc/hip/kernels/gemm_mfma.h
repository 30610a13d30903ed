// What the MFMA GEMM kernels share: operand types, the MFMA of each element type, the LDS stage's
// row length and the walk over tiles.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ku::hipbk {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((__vector_size__(4 * sizeof(short))));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
#define KU_LDS __attribute__((address_space(3)))

enum Elem : int { E_BF16 = 0, E_F16 = 1, E_FP8 = 2 };

constexpr int KB = 128;  // K bytes per stage (one row of an A/B^T stage)

template <int E>
struct Op;
template <>
struct Op<E_BF16> {
  static constexpr int KSTEP = 32;  // K bytes per MFMA (16 bf16)
  static constexpr int LV = 1;      // 16-byte pieces per lane per operand
  __device__ static void run(f32x16& c, const u32x4* a, const u32x4* b) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[0]), __builtin_bit_cast(bf16x8, b[0]), c,
                                                0, 0, 0);
  }
};
template <>
struct Op<E_F16> {
  static constexpr int KSTEP = 32;
  static constexpr int LV = 1;
  __device__ static void run(f32x16& c, const u32x4* a, const u32x4* b) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a[0]), __builtin_bit_cast(f16x8, b[0]), c, 0,
                                               0, 0);
  }
};
template <>
struct Op<E_FP8> {
  static constexpr int KSTEP = 64;  // 64 e4m3 per MFMA
  static constexpr int LV = 2;
  __device__ static void run(f32x16& c, const u32x4* a, const u32x4* b) {
    i32x8 av, bv;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      av[i] = (int)a[0][i];
      av[4 + i] = (int)a[1][i];
      bv[i] = (int)b[0][i];
      bv[4 + i] = (int)b[1][i];
    }
    // format 0 = e4m3 for both operands; zero scales select the unscaled instruction
    c = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, c, 0, 0, 0, 0, 0, 0);
  }
};

// consecutive ids go to XCD id % 8: regroup them into contiguous ranges per XCD, then walk tiles
// in groups of GM tile-rows so the tiles running together reuse A rows and B columns
__device__ __forceinline__ void tile_of(int pid, int tm, int tn, int* im, int* in) {
  const int total = tm * tn;
  const int per = total / 8;
  if (pid < per * 8) pid = (pid % 8) * per + pid / 8;
  constexpr int GM = 8;
  const int group = pid / (GM * tn);
  const int first = group * GM;
  const int gs = min(tm - first, GM);
  const int r = pid % (GM * tn);
  *im = first + r % gs;
  *in = r / gs;
}

}  // namespace

}  // namespace ku::hipbk
