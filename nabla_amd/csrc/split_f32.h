// float32 products on the bf16 matrix instruction.
//
// A float32 is three bf16 exactly, x = x1 + x2 + x3 (8 bits of the significand each, by two
// subtractions that are exact), and a product of two is
//   x1 y1 + (x1 y2 + x2 y1) + (x1 y3 + x2 y2 + x3 y1) + what is at most 2^-24 of it:
// (|x2| <= 2^-8 and |x3| <= 2^-17 of x, so x2 y3 + x3 y2 is up to 2^-24 together: 0.99 of that at x = y = 1 + 2^-8 - 2^-17.)
// Six bf16 products, each exact in the instruction's float32 sums.  The bf16 instruction has sixteen
// times the rate of the float32 one, so six of them take 0.38 of its time.
//   The first product is summed apart from the five small ones, whose roundings are then 2^-8 of its
// own, and one instruction adds 32 of a row's products where the float32 one adds two.  Error against
// float64, relative 2-norm, of a row of K normal / uniform positive numbers: K = 1024 2.0e-7 / 1.6e-7, K
// = 16384 8.2e-7 / 5.9e-7; the float32 instruction in one chain 5.9e-7 / 4.4e-7 and 2.2e-6 / 1.7e-6, in
// four 2.9e-7 / 1.2e-7 and 1.2e-6 / 4.4e-7.  (All six in one accumulator: as the one chain.)  K = 2 2.6e-8 against 3.1e-8;
// K = 1 is one product and one rounding, 2.53e-8, where the parts have 2.60e-8: the kernels multiply it as it is.
//   A number that is not finite, or rounds to infinity as a bf16, has no such parts and its sums come out
// as NaN: a wave with a sum that is not finite runs its tile again on the float32 instruction (SplitAcc::again)
// and stores those of it that the parts did not give.
//   What is cut is 2^16 x: a float32 is a multiple of 2^-149, and all that is left of 2^16 times it is one of 2^-133,
// the smallest bf16.  (Unscaled, numbers below 2^-109 lost digits: 1.5e-7 at 2^-112, 8.8e-6 at 2^-118.)  So numbers
// from 2^112 and sums from 2^96 on are those that are computed again.  The multiplication is one instruction a
// number on 5.5: us, products 4096 x 4096 x 1024 195 -> 195, 1024 x 2048 x 512 21.0 -> 21.9, input gradients
// of convolutions 3 %, odd channel counts up to 8 % (32 x 14 x 14, 20 -> 44 31.2 -> 34.2).
#pragma once
#include "nbk_common.h"

#include <type_traits>

typedef uint32_t sp_u4 __attribute__((ext_vector_type(4)));
typedef float sp_f2 __attribute__((ext_vector_type(2)));
typedef float sp_f4 __attribute__((ext_vector_type(4)));
typedef float sp_f4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef __bf16 sp_b2 __attribute__((ext_vector_type(2)));
typedef __bf16 sp_b8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint32_t split_pack(float a, float b) {
  const sp_f2 f = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, sp_b2));
}
constexpr float SPLIT_SCALE = 65536.f, SPLIT_UNSCALE = 1.f / (SPLIT_SCALE * SPLIT_SCALE);
// The three parts of eight numbers, as stored.
__device__ __forceinline__ void split8(const float* x, sp_u4 (&part)[3]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = x[2 * i] * SPLIT_SCALE, b = x[2 * i + 1] * SPLIT_SCALE;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const uint32_t u = split_pack(a, b);
      part[p][i] = u;
      a -= __uint_as_float(u << 16);
      b -= __uint_as_float(u & 0xffff0000u);
    }
  }
}

// An operand's K tile of 32 in LDS: [part][row][4 chunks of 8 k].  Chunk c of a row sits at c ^ -(row / 4):
// the sixteen rows (and two chunks) that a cycle of ds_read_b128 serves for a 16 x 16 x 32 fragment then lie
// in sixteen different slots of the 256-byte bank window.
constexpr int SPLIT_BK = 32;
__device__ __forceinline__ int split_slot(int row, int c) { return row * 4 + (c ^ (-(row >> 2) & 3)); }
template <int ROWS>
__device__ __forceinline__ void split_store(sp_u4* tile, int row, int c, const float* x) {
  sp_u4 part[3];
  split8(x, part);
#pragma unroll
  for (int p = 0; p < 3; ++p) tile[p * (ROWS * 4) + split_slot(row, c)] = part[p];
}

// A wave's TM x TN blocks of 16 x 16, NM accumulators for the first product (a tile of 32 k each in turn).
template <int TM, int TN, int NM>
struct SplitAcc {
  sp_f4 main[NM][TM][TN], small[TM][TN];
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        small[i][j] = (sp_f4)(0.f);
#pragma unroll
        for (int n = 0; n < NM; ++n) main[n][i][j] = (sp_f4)(0.f);
      }
  }
  // D register r of a lane is row (lane / 16) * 4 + r, column lane % 16 of the block.
  __device__ __forceinline__ float sum(int i, int j, int r) const {
    float s = main[0][i][j][r];
    if constexpr (NM == 2) s += main[1][i][j][r];
    return (s + small[i][j][r]) * SPLIT_UNSCALE;
  }
  // All of K on the float32 instruction, operands straight from memory: a(i, k, inside) and b(j, k, inside) are the
  // lane's row (lane % 16) of block i and its column of block j, zero past the end of K unless `inside` says
  // that k is not.  A step is 16 k, four consecutive ones a lane.
  template <class A, class B>
  __device__ __forceinline__ void again(int64_t k_begin, int64_t k_end, int lane, A a, B b) {
    zero();
    float fa[2][TM][4], fb[2][TN][4];  // (the next step's numbers are on their way)
    auto load = [&](auto set, int64_t k0) {
      const int64_t k = k0 + (lane >> 4) * 4;
      auto all = [&](auto inside) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
          for (int i = 0; i < TM; ++i) fa[set.value][i][e] = a(i, k + e, inside);
#pragma unroll
          for (int j = 0; j < TN; ++j) fb[set.value][j][e] = b(j, k + e, inside);
        }
      };
      if (k0 + 16 <= k_end) all(std::true_type{});
      else all(std::false_type{});
    };
    auto multiply = [&](auto set) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            main[e % NM][i][j] =
                __builtin_amdgcn_mfma_f32_16x16x4f32(fa[set.value][i][e], fb[set.value][j][e], main[e % NM][i][j], 0, 0, 0);
    };
    load(std::integral_constant<int, 0>{}, k_begin);
#pragma unroll 1
    for (int64_t k0 = k_begin; k0 < k_end; k0 += 32) {  // (past the end: zeros)
      load(std::integral_constant<int, 1>{}, k0 + 16);
      multiply(std::integral_constant<int, 0>{});
      load(std::integral_constant<int, 0>{}, k0 + 32);
      multiply(std::integral_constant<int, 1>{});
    }
  }
  __device__ __forceinline__ float sum_again(int i, int j, int r) const {
    float s = main[0][i][j][r];
    if constexpr (NM == 2) s += main[1][i][j][r];
    return s;
  }
  // One K tile; wm, wn: the wave's first row and column in the workgroup's tile.
  template <int BM, int BN, int SET>
  __device__ __forceinline__ void multiply(const sp_u4* a, const sp_u4* b, int wm, int wn, int lane) {
    const int row = lane & 15, c = lane >> 4;
    const sp_u4* pa = a + split_slot(wm + row, c);
    const sp_u4* pb = b + split_slot(wn + row, c);
    sp_b8 fa[3][TM], fb[3][TN];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[p][i] = __builtin_bit_cast(sp_b8, pa[p * (BM * 4) + i * 64]);
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[p][j] = __builtin_bit_cast(sp_b8, pb[p * (BN * 4) + j * 64]);
    }
    auto add = [&](sp_f4 (&acc)[TM][TN], int p, int q) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[p][i], fb[q][j], acc[i][j], 0, 0, 0);
    };
    add(main[SET % NM], 0, 0);
    add(small, 0, 1);
    add(small, 1, 0);
    add(small, 1, 1);
    add(small, 0, 2);
    add(small, 2, 0);
  }
};
