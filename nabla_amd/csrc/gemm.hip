// GEMM for gfx950: C[b] = alpha * A[b] @ B[b] (+bias) (act) (+residual).
//
// bf16 path (fp32 accumulate): v_mfma_f32_32x32x16_bf16.  A workgroup of four waves (2 x 2;
// 128 x 128 tile) or eight (2 x 4; 256 x 256 tile) owns a BM x BN tile of C; K advances in
// steps of 64 through two LDS buffers (64 x 64 tiles where the result is small).
//   * an operand that is contiguous along K sits in LDS as [row][64 k], 128-byte rows whose
//     eight 16-byte chunks are XOR-swizzled, so that the 16-byte fragment reads of the MFMA
//     (32 consecutive rows, one chunk) are conflict-free without padding;
//   * an operand that is contiguous along its row index (the transposed operand of the two
//     backward products, and B of the forward product) sits in LDS k-major, [64 k][rows], and
//     its MFMA fragments come out through the transposing read (ds_read_b64_tr_b16): the
//     swap_axes of the backward GEMMs never touches memory or the vector ALU.
// Two kernels share this layout idea: gemm_bf16_dl_kernel (aligned operands, K % 64 == 0 or
// both operands row-contiguous) copies global memory straight into LDS
// (global_load_lds_dwordx4); gemm_bf16_kernel takes every other shape through guarded loads and
// registers.
// fp32 path: out of bf16 parts (split_f32.h) on tiles of 128 x 128 or 64 x 64, small results on
// v_mfma_f32_32x32x2f32 with 32 x 32 a workgroup.
#include "nbk_common.h"
#include "split_f32.h"

#include <type_traits>
#include <utility>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
// 16-byte register / LDS unit.  A native vector (an SSA value), not the uint4 struct:
// arrays of structs that are filled by loads and drained by stores are turned into
// memcpy through a stack slot, which puts the staging registers in scratch.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Compile-time loop: accumulator tiles must be indexed with constants or they
// leave the register file.
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Part i of `total` items dealt as evenly as possible into `parts` consecutive shares.
constexpr int share(int total, int parts, int i) {
  return total * (i + 1) / parts - total * i / parts;
}

constexpr int GEMM_MAX_MEMBERS = 4;
struct GemmArgs {
  const void* A; const void* B; void* C; const void* bias; const void* residual;
  int64_t M, N, K;
  int64_t a_rs, a_cs, b_rs, b_cs, ldc;
  int64_t a_bs, b_bs, c_bs;
  int64_t batch_inner, a_bs2, b_bs2, c_bs2;  // batch_inner >= 1
  int32_t dtype_c, act;
  int32_t res_mul;  // the residual multiplies instead of adding
  float alpha;
  int32_t tiles_m, tiles_n;
  int32_t a_vec, b_vec;  // 16-byte accesses are legal for this operand
  void* C2;              // second result (derivative of the activation), or null
  const float* b_scales; // NF4-coded B only: one scale per `b_block` consecutive codes
  int32_t b_block;
  int32_t c_stream;      // C is larger than the last-level cache: store it with the non-temporal hint
  void* colsum;          // null, or [batch][N] in C's dtype: the column sums of B over K
  // More operand pairs whose products join the accumulator: C = A B + sum_i A_i B_i, all
  // oriented like A and B.  Direct-to-LDS kernels only.
  //   shallow pairs (n_shallow <= 2; K <= 64 each, own strides): one K tile each, the first tiles
  //   of the launch;
  //   deep pairs (n_deep <= 2; K % 64 == 0, the strides of A and B): their K tiles follow those
  //   of A and B.
  struct Shallow { const void* A; const void* B; int64_t K, a_rs, a_cs, b_rs, b_cs; } shallow[2];
  struct Deep { const void* A; const void* B; int64_t K; } deep[2];
  int32_t n_shallow, n_deep;
  int64_t k_last;        // contraction length of the last slice of a product split along K; 0: K
  // Products of one A in one launch, the outer batch index: their B, bias and, in elements from C, their results.
  struct Member { const void* B; const void* bias; int64_t c_off; } member[GEMM_MAX_MEMBERS];
  int32_t n_members;     // 0: none
};
// The right operand, bias and result of this workgroup's batch member.  (Chosen by comparisons: an index known only
// at run time keeps the compiler from loading the arguments once, at the start, and every use becomes a load of its own
// from the scalar cache: 140 instead of 11 in the 128 x 128 form with guarded loads, 128 x 512 x 4 with bias and residual
// 29.3 -> 31.8 us, and 0.2 to 0.4 us more on every launch of 64 x 64 tiles.)
struct GemmMember { const void* B; const void* bias; int64_t c_off; };
__device__ __forceinline__ GemmMember gemm_member(const GemmArgs& g, int64_t bo, int64_t bi, int elem) {
  GemmMember m = {(const char*)g.B + (bo * g.b_bs + bi * g.b_bs2) * elem, g.bias, bo * g.c_bs + bi * g.c_bs2};
#pragma unroll
  for (int i = 0; i < GEMM_MAX_MEMBERS; ++i)
    if (i < g.n_members && bo == i) m = {g.member[i].B, g.member[i].bias, g.member[i].c_off};
  return m;
}

// Contraction length of this workgroup's batch member (the slice is the inner batch index where there
// are two levels).
__device__ __forceinline__ int64_t gemm_slice_k(const GemmArgs& g, int64_t bo, int64_t bi, int batch) {
  const bool last = g.batch_inner > 1 ? bi == g.batch_inner - 1 : bo == (int64_t)batch - 1;
  return g.k_last > 0 && last ? g.k_last : g.K;
}

__device__ __forceinline__ float gemm_act(float v, int act) {
  if (act == NBK_ACT_RELU) return fmaxf(v, 0.f);
  if (act == NBK_ACT_GELU) return 0.5f * v * (1.f + erff(v * 0.70710678118654752440f));
  return v;
}

// Activation and its derivative at the same point (the second result of a launch).  LOWP: the
// results are stored as 16-bit floats, so hardware exp and a 1.5e-7 erf do.
template <bool LOWP>
__device__ __forceinline__ void gemm_act_pair(float x, int act, float& y, float& dy) {
  if (act == NBK_ACT_RELU) {
    y = fmaxf(x, 0.f);
    dy = x > 0.f ? 1.f : 0.f;
  } else if (act == NBK_ACT_GELU) {
    const float z = x * 0.70710678118654752440f;
    const float e = LOWP ? __expf(-z * z) : expf(-z * z);
    const float cdf = 0.5f * (1.f + (LOWP ? nbk_fast_erf_with(z, e) : erff(z)));
    y = x * cdf;
    dy = cdf + x * 0.39894228040143267794f * e;
  } else {
    y = x;
    dy = 1.f;
  }
}

// Workgroup ids are dealt round-robin to the 8 XCDs, each with its own L2.
// Re-number them so that every XCD works on one contiguous run of tiles, then
// walk that run in groups of 8 tile-rows per tile-column: workgroups that share
// an L2 also share the A and B panels they read.
__device__ __forceinline__ void gemm_tile_coords(int bid, int tiles_m, int tiles_n, int& tm,
                                                 int& tn) {
  {
    const int n = tiles_m * tiles_n;
    const int xcd = bid & 7, local = bid >> 3;
    const int per = n >> 3, rem = n & 7;
    bid = xcd < rem ? xcd * (per + 1) + local : rem * (per + 1) + (xcd - rem) * per + local;
  }
  const int group = 8;
  const int per_group = group * tiles_n;
  const int g = bid / per_group;
  const int first_m = g * group;
  const int gsize = min(group, tiles_m - first_m);
  const int r = bid - g * per_group;
  tm = first_m + r % gsize;
  tn = r / gsize;
}

// ---------------------------------------------------------------------------- bf16
__device__ __forceinline__ int swz(int row, int chunk) {
  return row * 8 + (chunk ^ (row & 7) ^ ((row >> 3) & 7));
}

// 16-byte guarded load of 8 consecutive bf16 along the unit-stride axis: one access, also where the
// rows start at an odd element (global memory takes any alignment; eight 2-byte loads and their
// packing bound every product with an odd row length, a vocabulary of no round size for one).
typedef u32x4 u32x4_any __attribute__((aligned(2)));
__device__ __forceinline__ u32x4 ld8_bf16(const uint16_t* p, int64_t valid) {
  u32x4 r = {0u, 0u, 0u, 0u};
  if (valid >= 8) return *(const u32x4_any*)p;
  if (valid <= 0) return r;
  uint16_t t[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) t[i] = i < valid ? p[i] : (uint16_t)0;
  r.x = t[0] | ((uint32_t)t[1] << 16);
  r.y = t[2] | ((uint32_t)t[3] << 16);
  r.z = t[4] | ((uint32_t)t[5] << 16);
  r.w = t[6] | ((uint32_t)t[7] << 16);
  return r;
}

// ---- NF4-coded B operand --------------------------------------------------------------------
// The sixteen levels (nabla/nn/finetune/qlora.py:18-38), copied to LDS by the kernels that
// dequantise: a lane looks up eight different entries per load.
__device__ const float nbk_nf4_levels[16] = {-1.0f,    -0.6962f, -0.5251f, -0.3949f, -0.2844f, -0.1848f,
                                             -0.0911f, 0.0f,     0.0796f,  0.1609f,  0.2461f,  0.3379f,
                                             0.4407f,  0.5626f,  0.7230f,  1.0f};
// Eight consecutive weights from their codes: level[code] * scale of the block the codes lie
// in (`flat` is the index of the first code in the flattened weight, a multiple of 8, and the
// block length is a multiple of 8, so the eight share a block); entries from `valid` on are 0.
__device__ __forceinline__ void nf4_load8(const uint8_t* codes, const float* scales, int block,
                                          const float* table, int64_t flat, int64_t valid, float* out) {
#pragma unroll
  for (int e = 0; e < 8; ++e) out[e] = 0.f;
  if (valid <= 0) return;
  const float s = scales[flat / block];
  uint64_t raw = 0;
  if (valid >= 8) {
    raw = *(const uint64_t*)(codes + flat);
  } else {
    for (int e = 0; e < valid; ++e) raw |= (uint64_t)codes[flat + e] << (8 * e);
  }
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (e < valid) out[e] = table[(raw >> (8 * e)) & 15] * s;
}

// ------------------------------------------------------- bf16, guarded register-staged loads
// The general form: any alignment, any K, ragged edges.  Every access is guarded element by
// element; it is kept out of the hot kernel because its code size alone would push the main
// loop out of the instruction cache.
// LDS geometry of one operand tile, in 16-byte chunks.  K-contiguous: [row][8 chunks],
// swizzled.  Row-contiguous: [64 k][ROWS / 8 + 4 chunks]; the pitch is 64 bytes past a
// multiple of 256, so the eight 32-byte row segments that half a wave touches in one
// transposing read (4 k-rows x 2 groups of 16 rows) fall on eight different bank groups.
template <int ROWS, bool KC>
struct TileGeom {
  static constexpr int PITCH = ROWS / 8 + 4;
  static constexpr int CHUNKS = KC ? ROWS * 8 : 64 * PITCH;
};

template <int ROWS, bool KC, int NT>
struct TileLoader {
  // NT lanes (256 or 512) share the tile: ROWS * 8 chunk tasks, ROWS * 8 / NT per lane.
  // KC : operand contiguous along K    -> task t is chunk t % 8 of row t / 8.
  // !KC: operand contiguous along rows -> task t is rows 8 * (t % (ROWS / 8)) .. + 8 of
  //      k-row t / (ROWS / 8): consecutive lanes read consecutive 16 bytes of one k-row.
  static constexpr int NREG = ROWS * 8 / NT;
  static constexpr int NC = ROWS / 8;
  static constexpr int PITCH = TileGeom<ROWS, KC>::PITCH;
  static_assert(ROWS == 256 || ROWS == 128, "tile rows");
  u32x4 reg[NREG];

  __device__ __forceinline__ void load(const uint16_t* base, int64_t rs, int64_t cs, int64_t row0,
                                       int64_t rows_total, int64_t k0, int64_t K) {
    const int tid = threadIdx.x;
    if (KC) {
#pragma unroll
      for (int s = 0; s < NREG; ++s) {
        const int t = tid + s * NT;
        const int row = t >> 3, c = t & 7;
        const int64_t gr = row0 + row, gk = k0 + c * 8;
        if (gr < rows_total) reg[s] = ld8_bf16(base + gr * rs + gk, K - gk);
        else reg[s] = (u32x4){0u, 0u, 0u, 0u};
      }
    } else {
#pragma unroll
      for (int s = 0; s < NREG; ++s) {
        const int t = tid + s * NT;
        const int k = t / NC, c = t % NC;
        const int64_t gr = row0 + c * 8, gk = k0 + k;
        if (gk < K) reg[s] = ld8_bf16(base + gk * cs + gr, rows_total - gr);
        else reg[s] = (u32x4){0u, 0u, 0u, 0u};
      }
    }
  }

  // The same tile from NF4 codes: `codes` addressed like `base` above, dequantised in registers
  // and rounded to bf16 once.
  __device__ __forceinline__ void load_nf4(const uint8_t* codes, const float* scales, int block,
                                           const float* table, int64_t rs, int64_t cs, int64_t row0,
                                           int64_t rows_total, int64_t k0, int64_t K) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int s = 0; s < NREG; ++s) {
      const int t = tid + s * NT;
      float w[8];
      if (KC) {
        const int row = t >> 3, c = t & 7;
        const int64_t gr = row0 + row, gk = k0 + c * 8;
        nf4_load8(codes, scales, block, table, gr * rs + gk, gr < rows_total ? K - gk : 0, w);
      } else {
        const int k = t / NC, c = t % NC;
        const int64_t gr = row0 + c * 8, gk = k0 + k;
        nf4_load8(codes, scales, block, table, gk * cs + gr, gk < K ? rows_total - gr : 0, w);
      }
      u32x4 r;
      r.x = (uint32_t)nbk_f32_to_bf16(w[0]) | ((uint32_t)nbk_f32_to_bf16(w[1]) << 16);
      r.y = (uint32_t)nbk_f32_to_bf16(w[2]) | ((uint32_t)nbk_f32_to_bf16(w[3]) << 16);
      r.z = (uint32_t)nbk_f32_to_bf16(w[4]) | ((uint32_t)nbk_f32_to_bf16(w[5]) << 16);
      r.w = (uint32_t)nbk_f32_to_bf16(w[6]) | ((uint32_t)nbk_f32_to_bf16(w[7]) << 16);
      reg[s] = r;
    }
  }

  // The tile goes to LDS in NPIECE independent pieces so that the K loop can place
  // them between its matrix instructions.
  static constexpr int NPIECE = NREG;
  template <int P>
  __device__ __forceinline__ void store_piece(u32x4* lds) {
    const int t = threadIdx.x + P * NT;
    if (KC) lds[swz(t >> 3, t & 7)] = reg[P];
    else lds[(t / NC) * PITCH + t % NC] = reg[P];
  }
  __device__ __forceinline__ void store(u32x4* lds) {
    static_for<NPIECE>([&](auto pc) { store_piece<decltype(pc)::value>(lds); });
  }
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// Transposing LDS read: the 16 lanes of a group hand in 16 addresses of 4 consecutive
// 16-bit values, In[p][e]; lane i of the group receives In[4 j + i / 4][i % 4], j = 0..3.
// With lane p pointing at (k-row p / 4, rows 4 * (p % 4) .. + 4) of a k-major tile, lane i
// ends up with 4 consecutive k of row i: half an MFMA operand fragment.
__device__ __forceinline__ s16x4 lds_read_tr(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
}

// The same read as inline assembly, for kernels that fill LDS with global_load_lds: the
// compiler puts a wait for every such copy in flight in front of the intrinsic form (it cannot
// tell that the two never touch the same buffer between two barriers).  It knows nothing about
// the result being asynchronous either: lds_wait_for() has to stand between these reads and
// the first use of their results.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}
__device__ __forceinline__ bf16x8 lds_read_tr_pair(uint32_t addr, int off_lo, int off_hi) {
  s16x4 lo, hi;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo) : "v"(addr), "n"(off_lo) : "memory");
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(addr), "n"(off_hi) : "memory");
  const s16x8 u = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return *(const bf16x8*)&u;
}
__device__ __forceinline__ bf16x8 lds_read_b128(uint32_t addr) {
  u32x4 u;
  asm volatile("ds_read_b128 %0, %1" : "=v"(u) : "v"(addr) : "memory");
  return *(const bf16x8*)&u;
}
template <int N>
__device__ __forceinline__ void lds_wait_for(bf16x8 (&f)[N]) {
  static_assert(N == 2 || N == 4 || N == 8, "fragments per set");
  if constexpr (N == 2)
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f[0]), "+v"(f[1])::"memory");
  else if constexpr (N == 4)
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3])::"memory");
  else
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]),
                   "+v"(f[7])::"memory");
}

extern __shared__ __align__(16) u32x4 gemm_lds[];

// Epilogue shared by the bf16 kernels (the caller has passed a workgroup barrier: the tile
// buffers are free).
// EPI: 0 plain, 1 bias only (as lean as the plain form), 2 bias / activation / residual (the
// residual requested for the whole wave tile up front), 3 bias and an added residual read pass by
// pass (for kernels whose occupancy hides that latency and must not lose it to registers), 4 bias
// and an added bf16 residual that the caller requested before its product (`pre`: the 16-byte
// piece of every pass of every band, in this function's lane layout -- gemm_residual_prefetch).
// Each wave passes its accumulators through a private LDS slab, a band of 32 rows of its tile
// at a time (`scatter(band, slab)` writes the band's accumulators there, row-major with a
// pitch of WN + 4 floats), so that C is written as whole 16-byte (bf16) / 32-byte (fp32)
// pieces of a row: 8 columns per lane.  The plain form (no bias / activation / residual)
// is a separate instantiation: the fused form carries erf() bodies, and an epilogue that does
// not fit the instruction cache costs more than the whole K loop of a short GEMM.
// The residual pieces this lane adds in an EPI 4 epilogue, requested up front (rows and columns
// past the edge read a valid address and are never used).  The caller has checked that C is
// bf16 and that residual, ldc and N allow 16-byte pieces.
template <int TM, int WN>
__device__ __forceinline__ void gemm_residual_prefetch(const GemmArgs& g, int64_t m0, int64_t n0, int wm,
                                                       int wn, int lane, uint4 (&pre)[TM * (WN / 16)]) {
  constexpr int LANES_PER_ROW = WN / 8, ROWS_PER_PASS = 64 / LANES_PER_ROW, NP = 32 / ROWS_PER_PASS;
  const int sub_r = lane / LANES_PER_ROW, sub_c = (lane % LANES_PER_ROW) * 8;
  int64_t col = n0 + wn + sub_c;
  col = col + 8 <= g.N ? col : 0;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int pass = 0; pass < NP; ++pass) {
      int64_t row = m0 + wm + i * 32 + pass * ROWS_PER_PASS + sub_r;
      row = row < g.M ? row : g.M - 1;
      pre[i * NP + pass] = *(const uint4*)((const uint16_t*)g.residual + row * g.ldc + col);
    }
}

template <int TM, int WN, bool FAST, int EPI, typename Scatter>
__device__ __forceinline__ void gemm_epilogue_bands(Scatter&& scatter, const GemmArgs& g, int64_t m0,
                                                    int64_t n0, int wm, int wn, int64_t c_off, const void* bias,
                                                    int wave, int lane, const uint4* pre = nullptr) {
  constexpr int SLAB_LD = WN + 4;  // floats per slab row (padding spreads the row groups)
  float* slab = (float*)gemm_lds + wave * (32 * SLAB_LD);
  const bool out_f32 = g.dtype_c == NBK_F32;
  constexpr int LANES_PER_ROW = WN / 8;        // each lane writes 8 consecutive columns
  constexpr int ROWS_PER_PASS = 64 / LANES_PER_ROW;
  const int sub_r = lane / LANES_PER_ROW, sub_c = (lane % LANES_PER_ROW) * 8;
  const int64_t col = n0 + wn + sub_c;
  const bool vec_store = FAST && (col + 8 <= g.N) && ((g.ldc & 7) == 0) && ((g.c_bs & 7) == 0) &&
                         ((g.c_bs2 & 7) == 0);
  float bias_v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) bias_v[e] = 0.f;
  // (the usual way in line: behind the other one, 6 KB of code further, it costs a trip for instructions, 0.5 us a launch)
  if (EPI != 0 && __builtin_expect(bias != nullptr, 1)) {
    if (__builtin_expect(!out_f32 && col + 8 <= g.N && (((uintptr_t)bias + 2 * (uintptr_t)col) & 15) == 0, 1)) {
      const uint4 bu = *(const uint4*)((const uint16_t*)bias + col);  // eight 16-bit values at once
      bias_v[0] = __uint_as_float(bu.x << 16); bias_v[1] = __uint_as_float(bu.x & 0xffff0000u);
      bias_v[2] = __uint_as_float(bu.y << 16); bias_v[3] = __uint_as_float(bu.y & 0xffff0000u);
      bias_v[4] = __uint_as_float(bu.z << 16); bias_v[5] = __uint_as_float(bu.z & 0xffff0000u);
      bias_v[6] = __uint_as_float(bu.w << 16); bias_v[7] = __uint_as_float(bu.w & 0xffff0000u);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (col + e < g.N) bias_v[e] = nbk_load_as_f32(bias, col + e, g.dtype_c);
    }
  }
  constexpr int NP = 32 / ROWS_PER_PASS;
  const bool res_vec = EPI == 2 && g.residual && vec_store && !out_f32;
  // the residual of the whole wave tile is requested before the first slab round trip, so that
  // its latency is paid once and not pass by pass (the K loop's registers are free by now)
  uint4 rpre[EPI == 2 ? TM : 1][NP];
  if constexpr (EPI == 2) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int pass = 0; pass < NP; ++pass) {
        const int64_t row = m0 + wm + i * 32 + pass * ROWS_PER_PASS + sub_r;
        rpre[i][pass] = make_uint4(0u, 0u, 0u, 0u);
        if (res_vec && row < g.M)
          rpre[i][pass] = *(const uint4*)((const uint16_t*)g.residual + c_off + row * g.ldc + col);
      }
  }
  static_for<TM>([&](auto ti) {
    constexpr int i = decltype(ti)::value;
    scatter(ti, slab);
    // the slab is private to the wave: no workgroup barrier, only LDS ordering
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    auto one_pass = [&](int pass, const uint4 u) {
      const int lr = pass * ROWS_PER_PASS + sub_r;
      const int64_t row = m0 + wm + i * 32 + lr;
      float v[8];
      const float4 p0 = *(const float4*)&slab[lr * SLAB_LD + sub_c];
      const float4 p1 = *(const float4*)&slab[lr * SLAB_LD + sub_c + 4];
      v[0] = p0.x; v[1] = p0.y; v[2] = p0.z; v[3] = p0.w;
      v[4] = p1.x; v[5] = p1.y; v[6] = p1.z; v[7] = p1.w;
      if (row < g.M && col < g.N) {
        const int64_t idx = c_off + row * g.ldc + col;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= g.alpha;
        if (EPI == 1 || EPI == 3 || EPI == 4) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += bias_v[e];
        }
        if (EPI == 4) {
          v[0] += __uint_as_float(u.x << 16); v[1] += __uint_as_float(u.x & 0xffff0000u);
          v[2] += __uint_as_float(u.y << 16); v[3] += __uint_as_float(u.y & 0xffff0000u);
          v[4] += __uint_as_float(u.z << 16); v[5] += __uint_as_float(u.z & 0xffff0000u);
          v[6] += __uint_as_float(u.w << 16); v[7] += __uint_as_float(u.w & 0xffff0000u);
        }
        if (EPI == 3 && g.residual) {
          if (vec_store && !out_f32) {
            const uint4 ru = *(const uint4*)((const uint16_t*)g.residual + idx);
            v[0] += __uint_as_float(ru.x << 16); v[1] += __uint_as_float(ru.x & 0xffff0000u);
            v[2] += __uint_as_float(ru.y << 16); v[3] += __uint_as_float(ru.y & 0xffff0000u);
            v[4] += __uint_as_float(ru.z << 16); v[5] += __uint_as_float(ru.z & 0xffff0000u);
            v[6] += __uint_as_float(ru.w << 16); v[7] += __uint_as_float(ru.w & 0xffff0000u);
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (col + e < g.N) v[e] += nbk_load_as_f32(g.residual, idx + e, g.dtype_c);
          }
        }
        if (EPI == 2) {
          float res[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) res[e] = 0.f;
          if (res_vec) {
            res[0] = __uint_as_float(u.x << 16); res[1] = __uint_as_float(u.x & 0xffff0000u);
            res[2] = __uint_as_float(u.y << 16); res[3] = __uint_as_float(u.y & 0xffff0000u);
            res[4] = __uint_as_float(u.z << 16); res[5] = __uint_as_float(u.z & 0xffff0000u);
            res[6] = __uint_as_float(u.w << 16); res[7] = __uint_as_float(u.w & 0xffff0000u);
          } else if (g.residual) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (col + e < g.N) res[e] = nbk_load_as_f32(g.residual, idx + e, g.dtype_c);
          }
          if (g.C2) {
            // two results: the activation goes to C below, its derivative to C2 here
            float d2[8];
            if (out_f32) {
#pragma unroll
              for (int e = 0; e < 8; ++e) gemm_act_pair<false>(v[e] + bias_v[e], g.act, v[e], d2[e]);
            } else {
#pragma unroll
              for (int e = 0; e < 8; ++e) gemm_act_pair<true>(v[e] + bias_v[e], g.act, v[e], d2[e]);
            }
            if (vec_store && !out_f32) {
              uint4 o;
              o.x = (uint32_t)nbk_f32_to_bf16(d2[0]) | ((uint32_t)nbk_f32_to_bf16(d2[1]) << 16);
              o.y = (uint32_t)nbk_f32_to_bf16(d2[2]) | ((uint32_t)nbk_f32_to_bf16(d2[3]) << 16);
              o.z = (uint32_t)nbk_f32_to_bf16(d2[4]) | ((uint32_t)nbk_f32_to_bf16(d2[5]) << 16);
              o.w = (uint32_t)nbk_f32_to_bf16(d2[6]) | ((uint32_t)nbk_f32_to_bf16(d2[7]) << 16);
              *(uint4*)((uint16_t*)g.C2 + idx) = o;
            } else {
#pragma unroll
              for (int e = 0; e < 8; ++e)
                if (col + e < g.N) {
                  if (out_f32) ((float*)g.C2)[idx + e] = d2[e];
                  else ((uint16_t*)g.C2)[idx + e] = nbk_f32_to_bf16(d2[e]);
                }
            }
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float x = gemm_act(v[e] + bias_v[e], g.act);
              v[e] = !g.residual ? x : (g.res_mul ? x * res[e] : x + res[e]);
            }
          }
        }
        if (vec_store && !out_f32) {
          uint4 o;
          o.x = (uint32_t)nbk_f32_to_bf16(v[0]) | ((uint32_t)nbk_f32_to_bf16(v[1]) << 16);
          o.y = (uint32_t)nbk_f32_to_bf16(v[2]) | ((uint32_t)nbk_f32_to_bf16(v[3]) << 16);
          o.z = (uint32_t)nbk_f32_to_bf16(v[4]) | ((uint32_t)nbk_f32_to_bf16(v[5]) << 16);
          o.w = (uint32_t)nbk_f32_to_bf16(v[6]) | ((uint32_t)nbk_f32_to_bf16(v[7]) << 16);
          if (g.c_stream) {
            const u32x4 ov = {o.x, o.y, o.z, o.w};
            __builtin_nontemporal_store(ov, (u32x4*)((uint16_t*)g.C + idx));
          } else {
            *(uint4*)((uint16_t*)g.C + idx) = o;
          }
        } else if (vec_store && out_f32) {
          float4* dst = (float4*)((float*)g.C + idx);
          dst[0] = make_float4(v[0], v[1], v[2], v[3]);
          dst[1] = make_float4(v[4], v[5], v[6], v[7]);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (col + e < g.N) {
              if (out_f32) ((float*)g.C)[idx + e] = v[e];
              else ((uint16_t*)g.C)[idx + e] = nbk_f32_to_bf16(v[e]);
            }
        }
      }
    };
    if constexpr (EPI == 2) {
#pragma unroll
      for (int pass = 0; pass < NP; ++pass) one_pass(pass, rpre[i][pass]);
    } else if constexpr (EPI == 4) {
#pragma unroll
      for (int pass = 0; pass < NP; ++pass) one_pass(pass, pre[i * NP + pass]);
    } else {
#pragma unroll 1
      for (int pass = 0; pass < NP; ++pass) one_pass(pass, make_uint4(0u, 0u, 0u, 0u));
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // slab reads done before the next tile row overwrites it
  });
}

// 32x32 MFMA blocks: D[i][j] lives in lane (j, (i / 4) % 2), register (i / 8) * 4 + i % 4.
template <int TM, int TN, int WN, bool FAST, int EPI>
__device__ __forceinline__ void gemm_epilogue(f32x16 (&acc)[TM][TN], const GemmArgs& g, int64_t m0,
                                              int64_t n0, int wm, int wn, int64_t c_off, const void* bias,
                                              int wave, int lane, const uint4* pre = nullptr) {
  const int li = lane & 31, kg = lane >> 5;
  gemm_epilogue_bands<TM, WN, FAST, EPI>(
      [&](auto ti, float* slab) {
        constexpr int i = decltype(ti)::value;
        static_for<TN>([&](auto tj) {
          constexpr int j = decltype(tj)::value;
          const f32x16 a = acc[i][j];
#pragma unroll
          for (int r = 0; r < 16; ++r)
            slab[((r >> 2) * 8 + kg * 4 + (r & 3)) * (WN + 4) + j * 32 + li] = a[r];
        });
      },
      g, m0, n0, wm, wn, c_off, bias, wave, lane, pre);
}

// 16x16 MFMA blocks: D[i][j] lives in lane (j, i / 4), register i % 4; a band is two block rows.
// (Storing straight from the registers, with the product transposed so that a lane holds four
// consecutive columns, was measured: the 32-byte row pieces it writes make the epilogue slower
// than the slab round trip with its whole 128-byte lines.)
template <int TM, int TN, int WN, bool FAST, int EPI>
__device__ __forceinline__ void gemm_epilogue(f32x4 (&acc)[TM][TN], const GemmArgs& g, int64_t m0,
                                              int64_t n0, int wm, int wn, int64_t c_off, const void* bias,
                                              int wave, int lane) {
  static_assert(TM % 2 == 0, "block rows per wave tile");
  const int p = lane & 15, q = lane >> 4;
  gemm_epilogue_bands<TM / 2, WN, FAST, EPI>(
      [&](auto ti, float* slab) {
        constexpr int i = decltype(ti)::value;
        static_for<2 * TN>([&](auto tb) {
          constexpr int ib = decltype(tb)::value / TN, j = decltype(tb)::value % TN;
          const f32x4 a = acc[2 * i + ib][j];
#pragma unroll
          for (int r = 0; r < 4; ++r) slab[(ib * 16 + 4 * q + r) * (WN + 4) + j * 16 + p] = a[r];
        });
      },
      g, m0, n0, wm, wn, c_off, bias, wave, lane);
}

// NW waves: 4 as 2 x 2, or 8 as 2 x 4 (two waves per SIMD, each with half the accumulators:
// they cover each other's waits at the price of 1.5 x the LDS fragment traffic).
template <int BM, int BN, bool A_KC, bool B_KC, bool EPI, int NW, bool B_Q = false>
__global__ __launch_bounds__(NW * 64) void gemm_bf16_kernel(const GemmArgs g) {
  constexpr int NT = NW * 64, WGN = NW / 2;
  // B_Q: B holds NF4 codes (one byte per weight, addressed like a dense B) and g.b_scales the
  // block scales; the tile loader dequantises on the way into LDS
  __shared__ float nf4_table[B_Q ? 16 : 1];
  if (B_Q) {
    if (threadIdx.x < 16) nf4_table[threadIdx.x] = nbk_nf4_levels[threadIdx.x];
    __syncthreads();
  }
  constexpr int WM = BM / 2, WN = BN / WGN;  // wave tile
  constexpr int TM = WM / 32, TN = WN / 32;
  constexpr int CA = TileGeom<BM, A_KC>::CHUNKS, CB = TileGeom<BN, B_KC>::CHUNKS;
  constexpr int TILE_CHUNKS = CA + CB;
  constexpr int PA = TileGeom<BM, A_KC>::PITCH * 16, PB = TileGeom<BN, B_KC>::PITCH * 16;  // bytes
  int tm_i, tn_i;
  gemm_tile_coords(blockIdx.x, g.tiles_m, g.tiles_n, tm_i, tn_i);
  const int64_t m0 = (int64_t)tm_i * BM, n0 = (int64_t)tn_i * BN;
  const int64_t bo = (int64_t)blockIdx.y / g.batch_inner, bi = (int64_t)blockIdx.y % g.batch_inner;
  const uint16_t* A = (const uint16_t*)g.A + bo * g.a_bs + bi * g.a_bs2;
  const GemmMember mem = gemm_member(g, bo, bi, 2);
  const uint16_t* B = (const uint16_t*)mem.B;
  const int64_t c_off = mem.c_off;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave / WGN) * WM, wn = (wave % WGN) * WN;
  const int li = lane & 31, kg = lane >> 5;

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = (f32x16)(0.f);

  TileLoader<BM, A_KC, NT> la;
  TileLoader<BN, B_KC, NT> lb;
  const int64_t K = gemm_slice_k(g, bo, bi, gridDim.y);
  const int64_t nk = (K + 63) / 64;
  // A is rows = m; for the loader a K-contiguous operand has (rs = row stride, k unit),
  // a row-contiguous one has (cs = k stride, row unit).
  la.load(A, g.a_rs, g.a_cs, m0, g.M, 0, K);
  if constexpr (B_Q) lb.load_nf4((const uint8_t*)g.B, g.b_scales, g.b_block, nf4_table, g.b_cs, g.b_rs, n0, g.N, 0, K);
  else lb.load(B, g.b_cs, g.b_rs, n0, g.N, 0, K);
  la.store(gemm_lds);
  lb.store(gemm_lds + CA);
  __syncthreads();

  // Fragment addresses.  swz(row, ks * 2 + kg) = (row * 8 | t) ^ (ks * 2) with
  // t = kg ^ (row % 8) ^ (row / 8 % 8): only a constant XOR moves with ks.
  // A k-major operand needs one byte offset per wave: lane p of group q = lane / 16 points at
  // k-row 8 * (q / 2) + p / 4, rows 16 * (q % 2) + 4 * (p % 4) of the wave's first tile; the
  // tile row, the k-step and the second half of the fragment are constant offsets.
  int a_addr[TM], b_addr[TN];
  const int tr_k = 8 * (lane >> 5) + ((lane & 15) >> 2), tr_r = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const int a_tr = tr_k * PA + (wm + tr_r) * 2, b_tr = CA * 16 + tr_k * PB + (wn + tr_r) * 2;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int row = wm + i * 32 + li;
    a_addr[i] = row * 8 + (kg ^ (row & 7) ^ ((row >> 3) & 7));
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int row = wn + j * 32 + li;
    b_addr[j] = CA + row * 8 + (kg ^ (row & 7) ^ ((row >> 3) & 7));
  }

  // Software pipeline.  A SIMD holds one or two waves of the tile, so little hides a
  // stall but the wave's own instruction stream; every load is therefore issued one
  // stage before its use and sits between matrix instructions:
  //   * fragments of k-step ks + 1 are read from LDS while the MFMAs of ks run
  //     (two fragment sets, frag[0] / frag[1]);
  //   * the tile of iteration kt + 1, fetched from global memory during iteration
  //     kt - 1, is written to the other LDS buffer during k-step 2;
  //   * the global loads of tile kt + 2 are issued behind those writes;
  //   * the workgroup barrier falls in the middle of k-step 3, whose remaining
  //     MFMAs cover the first fragment reads of the next tile.
  bf16x8 fa[2][TM], fb[2][TN];
  constexpr int NFRAG = TM + TN, NMFMA = TM * TN;
  // read fragment r (A tiles first, then B) of k-step ks from `tile` into set SET
  auto read_frag = [&](auto set, auto r, const u32x4* tile, int ks) {
    // order of use by the MFMAs (row-major over the wave's tiles): A0, every B, A1, A2 ...
    constexpr int SET = decltype(set)::value, R0 = decltype(r)::value;
    constexpr int R = R0 == 0 ? 0 : (R0 <= TN ? TM + R0 - 1 : R0 - TN);
    // The XOR is recomputed at every read: hoisted out of the K loop, the 4 x (TM + TN)
    // x 2 variants of these addresses would spill the accumulating kernel.
    int sel = ks * 2;
    asm volatile("" : "+s"(sel));
    if constexpr (R < TM) {
      if constexpr (A_KC) {
        const u32x4 u = tile[a_addr[R] ^ sel];
        fa[SET][R] = *(const bf16x8*)&u;
      } else {
        const char* p = (const char*)tile + a_tr + (R * 64 + ks * 16 * PA);
        const s16x4 lo = lds_read_tr(p), hi = lds_read_tr(p + 4 * PA);
        const s16x8 u = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        fa[SET][R] = *(const bf16x8*)&u;
      }
    } else {
      if constexpr (B_KC) {
        const u32x4 u = tile[b_addr[R - TM] ^ sel];
        fb[SET][R - TM] = *(const bf16x8*)&u;
      } else {
        const char* p = (const char*)tile + b_tr + ((R - TM) * 64 + ks * 16 * PB);
        const s16x4 lo = lds_read_tr(p), hi = lds_read_tr(p + 4 * PB);
        const s16x8 u = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        fb[SET][R - TM] = *(const bf16x8*)&u;
      }
    }
  };
  // LDS read instructions of fragment r in the order above: a k-major operand takes two
  auto frag_reads = [](int r0) constexpr {
    const int r = r0 == 0 ? 0 : (r0 <= TN ? TM + r0 - 1 : r0 - TN);
    return r < TM ? (A_KC ? 1 : 2) : (B_KC ? 1 : 2);
  };
  auto mfma = [&](auto set, auto q) {
    constexpr int SET = decltype(set)::value, Q = decltype(q)::value;
    constexpr int i = Q / TN, j = Q % TN;
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[SET][i], fb[SET][j], acc[i][j], 0, 0, 0);
  };
  // k-step on fragment set SET while set 1 - SET is filled for k-step `ks_next` of `tile`
  auto stage = [&](auto set, const u32x4* tile, int ks_next) {
    constexpr int SET = decltype(set)::value;
    static_for<NFRAG>([&](auto r) {
      read_frag(std::integral_constant<int, 1 - SET>{}, r, tile, ks_next);
    });
    static_for<NMFMA>([&](auto q) { mfma(set, q); });
    // interleave: one fragment read, then its share of the MFMAs
    static_for<NFRAG>([&](auto r) {
      constexpr int n = share(NMFMA, NFRAG, decltype(r)::value);
      __builtin_amdgcn_sched_group_barrier(0x100, frag_reads(decltype(r)::value), 0);  // DS read
      if constexpr (n > 0) __builtin_amdgcn_sched_group_barrier(0x008, n, 0);  // MFMAs
    });
    __builtin_amdgcn_sched_barrier(0);  // later stages' work (and its waits) stays behind
  };

  static_for<NFRAG>([&](auto r) { read_frag(std::integral_constant<int, 0>{}, r, gemm_lds, 0); });
  {
    const int64_t k1 = nk > 1 ? 64 : 0;  // a single-tile problem re-reads tile 0 (never stored)
    la.load(A, g.a_rs, g.a_cs, m0, g.M, k1, K);
    if constexpr (B_Q) lb.load_nf4((const uint8_t*)g.B, g.b_scales, g.b_block, nf4_table, g.b_cs, g.b_rs, n0, g.N, k1, K);
    else lb.load(B, g.b_cs, g.b_rs, n0, g.N, k1, K);
  }
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  for (int64_t kt = 0; kt + 1 < nk; ++kt) {
    const u32x4* cur = gemm_lds + (kt & 1) * TILE_CHUNKS;
    u32x4* nxt = gemm_lds + ((kt + 1) & 1) * TILE_CHUNKS;
    stage(S0{}, cur, 1);
    stage(S1{}, cur, 2);
    // k-step 2, with tile kt + 1 going from registers to LDS
    // (LDS reads and writes keep their program order, so they alternate in the source)
    {
      using LA = TileLoader<BM, A_KC, NT>;
      using LB = TileLoader<BN, B_KC, NT>;
      constexpr int NPA = LA::NPIECE, NP = LA::NPIECE + LB::NPIECE;
      constexpr int PER = (NP + NFRAG - 1) / NFRAG;
      static_for<NFRAG>([&](auto r) {
        read_frag(S1{}, r, cur, 3);
        static_for<PER>([&](auto e) {
          constexpr int P = decltype(r)::value * PER + decltype(e)::value;
          if constexpr (P < NPA) la.template store_piece<P>(nxt);
          else if constexpr (P < NP) lb.template store_piece<P - NPA>(nxt + CA);
        });
      });
      static_for<NMFMA>([&](auto q) { mfma(S0{}, q); });
      static_for<NFRAG>([&](auto r) {
        constexpr int n = share(NMFMA, NFRAG, decltype(r)::value);
        __builtin_amdgcn_sched_group_barrier(0x100, frag_reads(decltype(r)::value), 0);  // DS read
        if constexpr (n > 0) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
        __builtin_amdgcn_sched_group_barrier(0x200, PER, 0);  // DS writes
        if constexpr (n > 1) __builtin_amdgcn_sched_group_barrier(0x008, n - 1, 0);  // MFMA
      });
    }
    __builtin_amdgcn_sched_barrier(0);
    // k-step 3: fetch tile kt + 2 (the last iteration re-fetches tile nk - 1, unused),
    // half of the MFMAs, barrier, first fragments of the next tile, the other half
    {
      const int64_t k2 = (kt + 2 < nk ? kt + 2 : nk - 1) * 64;
      la.load(A, g.a_rs, g.a_cs, m0, g.M, k2, K);
      if constexpr (B_Q) lb.load_nf4((const uint8_t*)g.B, g.b_scales, g.b_block, nf4_table, g.b_cs, g.b_rs, n0, g.N, k2, K);
      else lb.load(B, g.b_cs, g.b_rs, n0, g.N, k2, K);
    }
    static_for<NMFMA / 2>([&](auto q) { mfma(S1{}, q); });
    {
      constexpr int NL = TileLoader<BM, A_KC, NT>::NREG + TileLoader<BN, B_KC, NT>::NREG;
      static_for<NMFMA / 2>([&](auto q) {
        constexpr int n = share(NL, NMFMA / 2, decltype(q)::value);
        if constexpr (n > 0) __builtin_amdgcn_sched_group_barrier(0x020, n, 0);  // VMEM reads
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      });
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    __builtin_amdgcn_sched_barrier(0);
    static_for<NFRAG>([&](auto r) { read_frag(S0{}, r, nxt, 0); });
    static_for<NMFMA / 2>([&](auto q) {
      mfma(S1{}, std::integral_constant<int, decltype(q)::value + NMFMA / 2>{});
    });
    static_for<NFRAG>([&](auto r) {
      constexpr int n = share(NMFMA / 2, NFRAG, decltype(r)::value);
      __builtin_amdgcn_sched_group_barrier(0x100, frag_reads(decltype(r)::value), 0);
      if constexpr (n > 0) __builtin_amdgcn_sched_group_barrier(0x008, n, 0);
    });
    __builtin_amdgcn_sched_barrier(0);
  }
  {
    // last tile: nothing left to stage
    const u32x4* cur = gemm_lds + ((nk - 1) & 1) * TILE_CHUNKS;
    stage(S0{}, cur, 1);
    stage(S1{}, cur, 2);
    stage(S0{}, cur, 3);
    static_for<NMFMA>([&](auto q) { mfma(S1{}, q); });
  }
  __syncthreads();  // the epilogue reuses the tile buffers as per-wave slabs

  gemm_epilogue<TM, TN, WN, false, EPI ? 2 : 0>(acc, g, m0, n0, wm, wn, c_off, mem.bias, wave, lane);
}

// ------------------------------------------------------------- bf16, direct-to-LDS loads
// The hot form (16-byte-aligned operands, K % 64 == 0): tiles go from global memory into LDS
// without passing through registers (global_load_lds_dwordx4: lane l of a wave deposits its
// 16 bytes at a wave-uniform LDS base + 16 l), so that the fragment reads are the only LDS
// instructions of the K loop and the lanes hold no staging registers.  Because the LDS side
// of such a load is linear in the lane, both layouts are unpadded and XOR-swizzled, and the
// swizzle is applied to the global address each lane fetches from:
//   K-contiguous operand   [row][8 chunks]: chunk c of row r sits at c ^ dl_kc_xor(r) (below);
//   row-contiguous operand [64 k][ROWS / 8 chunks]: chunk c of k-row k sits at
//     c ^ 2 * T[k % 4], T = {0, 3, 6, 5}, which sends the eight 32-byte segments that half a
//     wave touches in one transposing read to eight different bank groups.
// ds_read_b128 serves 16 lanes per cycle, and not neighbouring ones: lanes {0-3, 12-15, 20-23,
// 24-27} share a cycle, lanes {4-11, 16-19, 28-31} the next, and the same again 32 lanes up
// (measured with the bank-conflict counter, two lanes at a time).  The 16 chunks of such a group
// have to fall into 16 different 16-byte slots of the 256-byte bank window.
//   32 x 32 x 16 fragments (lane = row % 32, one chunk per half-wave): rows {0-3, 12-15, 20-23,
//     24-27} of a block at one chunk: c ^ (r % 8) ^ (r / 8 % 2) does it;
//   16 x 16 x 32 fragments (lane = row % 16 + 16 * chunk): rows {0-3, 12-15} at chunk c together
//     with rows {4-11} at chunk c ^ 1: the row pairs e = r / 2 % 8 of the first set go to
//     {0..3}, those of the second to {4..7}, so that c and c ^ 1 never meet.
template <bool MI16>
__device__ __forceinline__ int dl_kc_xor(int row) {
  if constexpr (MI16) {
    const int e = (row >> 1) & 7;
    return ((((e >> 1) ^ (e >> 2)) & 1) << 2) | (((e >> 2) & 1) << 1) | (e & 1);
  } else {
    return (row & 7) ^ ((row >> 3) & 1);
  }
}
__device__ __forceinline__ int dl_seg_xor(int k) { return (k & 3) ^ (((k & 3) << 1) & 7); }
// The 16x16x32 form reads k-rows k .. k + 3 and k + 8 .. k + 11 of one 32-byte segment in
// half a wave: bit 3 of k joins the swizzle.
// A k-row of 64 has four segments, two k-rows to a 256-byte window: bit 0 of k picks the half of the
// window, and bits 1 and 3 tell the segments of a half apart.
template <bool MI16, int ROWS>
__device__ __forceinline__ int dl_seg_xor_of(int k) {
  if constexpr (ROWS == 64) return ((k >> 1) & 1) | (((k >> 3) & 1) << 1);
  return MI16 ? dl_seg_xor(k) ^ ((k >> 3) & 1) : dl_seg_xor(k);
}

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) const void glb_void_t;

template <int ROWS, bool KC, int NW, bool MI16 = false>
struct DirectLoader {
  // ROWS * 8 chunks, 64 per wave instruction, dealt to the waves in consecutive runs
  static constexpr int N = ROWS / (8 * NW);
  static constexpr int NC = ROWS / 8;
  static_assert(N >= 1 && N % 2 == 0, "instructions per wave");
  static_assert(ROWS != 64 || MI16, "the swizzle of 64 rows is made for 16 x 16 x 32 fragments");
  int voff[N];         // byte offset of this lane's chunk from the tile's first element
  const char* base;    // operand + tile row offset (wave-uniform)
  int64_t kstep;       // bytes between consecutive K tiles (wave-uniform)
  int first;           // first instruction of this wave

  __device__ __forceinline__ void init(const uint16_t* op, int64_t rs, int64_t cs, int64_t row0,
                                       int64_t rows_total, int wave, int lane) {
    first = wave * N;
    if (KC) {
      base = (const char*)(op + row0 * rs);
      kstep = 128;
      const int64_t last = rows_total - 1 - row0;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const int row = (first + j) * 8 + (lane >> 3);
        const int c = (lane & 7) ^ dl_kc_xor<MI16>(row);
        const int64_t r = row < last ? row : last;
        voff[j] = (int)(r * rs * 2 + c * 16);
      }
    } else {
      base = (const char*)(op + row0);
      kstep = 128 * cs;
      const int64_t last = rows_total - 8 - row0;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const int l = (first + j) * 64 + lane;
        const int k = l / NC, c = (l % NC) ^ (dl_seg_xor_of<MI16, ROWS>(k) << 1);
        const int64_t r = c * 8 < last ? c * 8 : last;
        voff[j] = (int)(k * cs * 2 + r * 2);
      }
    }
  }
  // One K tile of a second, shallower operand (only k < kvalid of the tile's 64 k-rows exist),
  // laid out in `region` like any other tile: a lane whose chunk lies beyond kvalid writes zeros
  // to its LDS slot instead of fetching.  Keeps no state; (rs, cs) as for init.
  __device__ __forceinline__ static void issue_tail(u32x4* region, const uint16_t* op, int64_t rs,
                                                    int64_t cs, int64_t row0, int64_t rows_total,
                                                    int kvalid, int wave, int lane) {
    const int first_ = wave * N;
    static_for<N>([&](auto jj) {
      constexpr int j = decltype(jj)::value;
      const char* src;
      bool there;
      if (KC) {
        const int64_t last = rows_total - 1 - row0;
        const int row = (first_ + j) * 8 + (lane >> 3);
        const int c = (lane & 7) ^ dl_kc_xor<MI16>(row);
        const int64_t r = row < last ? row : last;
        src = (const char*)(op + row0 * rs) + (r * rs * 2 + c * 16);
        there = c * 8 < kvalid;
      } else {
        const int64_t last = rows_total - 8 - row0;
        const int l = (first_ + j) * 64 + lane;
        const int k = l / NC, c = (l % NC) ^ (dl_seg_xor_of<MI16, ROWS>(k) << 1);
        const int64_t r = c * 8 < last ? c * 8 : last;
        src = (const char*)(op + row0) + (k * cs * 2 + r * 2);
        there = k < kvalid;
      }
      if (there)
        __builtin_amdgcn_global_load_lds((glb_void_t*)src, (lds_void_t*)(region + (first_ + j) * 64),
                                         16, 0, 0);
      else
        region[(first_ + j) * 64 + lane] = (u32x4)(0u);
    });
  }
  // start the copy of K tile `kt` into `region` (this operand's part of a tile buffer)
  __device__ __forceinline__ const char* tile_src(int64_t kt) const { return base + kt * kstep; }
  template <int J>
  __device__ __forceinline__ void issue_one(u32x4* region, const char* src) const {
    __builtin_amdgcn_global_load_lds((glb_void_t*)(src + voff[J]),
                                     (lds_void_t*)(region + (first + J) * 64), 16, 0, 0);
  }
  __device__ __forceinline__ void issue(u32x4* region, int64_t kt) const {
    const char* src = tile_src(kt);
    static_for<N>([&](auto j) { issue_one<decltype(j)::value>(region, src); });
  }
};

// MI16: the matrix instruction is v_mfma_f32_16x16x32_bf16 (blocks of 16 x 16, 32 deep) instead
// of v_mfma_f32_32x32x16_bf16 (32 x 32, 16 deep).  Same LDS traffic and register budget; the
// 16 x 16 form does the same arithmetic for about a tenth less power, and these products run at
// the power limit (the clock under MFMA load settles where the limit puts it), so it is the
// faster one with two waves per SIMD to keep its shorter instructions back to back.
// KSS: k-steps (one MFMA deep) per fragment set.  A step of KSS k-steps is multiplied out of one
// set while the other is filled for the next step; small wave tiles take 2, so that a read has
// more than a handful of MFMAs to land.
// COLSUM: the launch also leaves sum_k B[k][n] (the bias gradient beside a weight gradient
// x^T dy, which reads dy anyway): the waves that hold the first block row of the first tile row
// multiply a fragment of ones into one more accumulator per block column, from the B fragments
// that are in registers for the product -- no byte is read twice.
// STAGES: tile buffers (a power of two).  With more than two a copy has STAGES - 1 tiles' time to land.
// (bx, by: tile and batch member, of ny)
template <int BM, int BN, bool A_KC, bool B_KC, int EPI, int NW, int KSS, bool MI16, bool COLSUM, int STAGES>
__device__ __forceinline__ void gemm_bf16_dl_body(const GemmArgs& g, int bx, int by, int ny) {
  static_assert((STAGES & (STAGES - 1)) == 0, "tile t is in buffer t % STAGES");
  constexpr int WGN = NW / 2;
  constexpr int WM = BM / 2, WN = BN / WGN;  // wave tile
  constexpr int FM = MI16 ? 16 : 32;          // rows / columns of an MFMA block
  constexpr int KQ = MI16 ? 32 : 16;          // depth of one MFMA
  constexpr int TM = WM / FM, TN = WN / FM;
  constexpr int CA = BM * 8, TILE_CHUNKS = (BM + BN) * 8;
  int tm_i, tn_i;
  gemm_tile_coords(bx, g.tiles_m, g.tiles_n, tm_i, tn_i);
  const int64_t m0 = (int64_t)tm_i * BM, n0 = (int64_t)tn_i * BN;
  const int64_t bo = (int64_t)by / g.batch_inner, bi = (int64_t)by % g.batch_inner;
  const uint16_t* A = (const uint16_t*)g.A + bo * g.a_bs + bi * g.a_bs2;
  const GemmMember mem = gemm_member(g, bo, bi, 2);
  const uint16_t* B = (const uint16_t*)mem.B;
  const int64_t c_off = mem.c_off;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = (wave / WGN) * WM, wn = (wave % WGN) * WN;
  const int li = lane & 31, kg = lane >> 5;

  using Acc = std::conditional_t<MI16, f32x4, f32x16>;
  Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = (Acc)(0.f);

  static_assert(!COLSUM || MI16, "column sums ride on the 16 x 16 x 32 instruction");
  f32x4 cs[COLSUM ? TN : 1];
  bool do_cs = false;
  if constexpr (COLSUM) {
#pragma unroll
    for (int j = 0; j < TN; ++j) cs[j] = (f32x4)(0.f);
    do_cs = tm_i == 0 && wm == 0 && g.colsum != nullptr;  // (uniform over the wave)
  }

  using LA = DirectLoader<BM, A_KC, NW, MI16>;
  using LB = DirectLoader<BN, B_KC, NW, MI16>;
  LA la;
  LB lb;
  // K tiles of the launch: the shallow pairs (one tile each; their offsets are dead before the
  // loop's are made), then A and B, then the deep pairs, which share the loop's lane offsets and
  // differ in the wave-uniform base only.  src_a(t) / src_b(t): where tile t starts in memory.
  // (tile numbers are 32-bit: the scalar unit compares those, 64-bit ones go through vector registers)
  // Two row-contiguous operands take any K: what is left over a multiple of 64 (of this slice, where
  // the product is split along K) is the first tile, like a shallow pair.
  const int64_t K = gemm_slice_k(g, bo, bi, ny);
  const int k_over = !A_KC && !B_KC ? (int)(K & 63) : 0;
  const int ns = k_over ? 1 : g.n_shallow;
  const int e0 = ns + (int)(K / 64);                                     // first tile past A and B
  const int e1 = e0 + (g.n_deep > 0 ? (int)(g.deep[0].K / 64) : 0);      // ... past the first deep pair
  const int nk = e1 + (g.n_deep > 1 ? (int)(g.deep[1].K / 64) : 0);
  if (k_over) {
    LA::issue_tail(gemm_lds, A + (K - k_over) * g.a_cs, g.a_rs, g.a_cs, m0, g.M, k_over, wave, lane);
    LB::issue_tail(gemm_lds + CA, B + (K - k_over) * g.b_rs, g.b_cs, g.b_rs, n0, g.N, k_over, wave, lane);
  } else if (ns > 0) {
    const auto& t0 = g.shallow[0];
    LA::issue_tail(gemm_lds, (const uint16_t*)t0.A, t0.a_rs, t0.a_cs, m0, g.M, (int)t0.K, wave, lane);
    LB::issue_tail(gemm_lds + CA, (const uint16_t*)t0.B, t0.b_cs, t0.b_rs, n0, g.N, (int)t0.K, wave, lane);
  }
  if (ns > 1) {
    const auto& t1 = g.shallow[1];
    LA::issue_tail(gemm_lds + TILE_CHUNKS, (const uint16_t*)t1.A, t1.a_rs, t1.a_cs, m0, g.M, (int)t1.K,
                   wave, lane);
    LB::issue_tail(gemm_lds + TILE_CHUNKS + CA, (const uint16_t*)t1.B, t1.b_cs, t1.b_rs, n0, g.N,
                   (int)t1.K, wave, lane);
  }
  la.init(A, g.a_rs, g.a_cs, m0, g.M, wave, lane);
  lb.init(B, g.b_cs, g.b_rs, n0, g.N, wave, lane);
  // base of every run of tiles, moved back by the tiles before it, so that tile t of the launch
  // is at base + t * kstep whichever run it belongs to (wave-uniform values, held in scalar
  // registers as 64-bit integers: the K loop has no vector register to spare)
  auto uniform = [](const char* p) {
    const uint64_t b = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    return ((uint64_t)hi << 32) | lo;
  };
  const uint64_t a_run0 = uniform(la.base - ns * la.kstep), b_run0 = uniform(lb.base - ns * lb.kstep);
  uint64_t a_run1 = a_run0, b_run1 = b_run0, a_run2 = a_run0, b_run2 = b_run0;
  if (g.n_deep > 0) {
    a_run1 = uniform(la.base + ((const char*)g.deep[0].A - (const char*)A) - (int64_t)e0 * la.kstep);
    b_run1 = uniform(lb.base + ((const char*)g.deep[0].B - (const char*)B) - (int64_t)e0 * lb.kstep);
  }
  if (g.n_deep > 1) {
    a_run2 = uniform(la.base + ((const char*)g.deep[1].A - (const char*)A) - (int64_t)e1 * la.kstep);
    b_run2 = uniform(lb.base + ((const char*)g.deep[1].B - (const char*)B) - (int64_t)e1 * lb.kstep);
  }
  const int64_t a_kstep = la.kstep, b_kstep = lb.kstep;
#define GEMM_SRC_A(t) ((const char*)(((t) < e0 ? a_run0 : ((t) < e1 ? a_run1 : a_run2)) + (uint64_t)((int64_t)(t) * a_kstep)))
#define GEMM_SRC_B(t) ((const char*)(((t) < e0 ? b_run0 : ((t) < e1 ? b_run1 : b_run2)) + (uint64_t)((int64_t)(t) * b_kstep)))
  if (ns == 0) {
    const char* sa = GEMM_SRC_A(0);
    const char* sb = GEMM_SRC_B(0);
    static_for<LA::N>([&](auto j) { la.template issue_one<decltype(j)::value>(gemm_lds, sa); });
    static_for<LB::N>([&](auto j) { lb.template issue_one<decltype(j)::value>(gemm_lds + CA, sb); });
  }

  // Fragment addresses, one per block row / column of the wave tile.  32 x 32 x 16:
  //   K-contiguous: byte address 16 ((row * 8 | t) ^ (2 ks)), t = kg ^ (row % 8) ^ (row / 8 % 2);
  //   row-contiguous: byte address of this lane's 8 bytes in the transposing read of k-step 0,
  //     first half; the k-step and the half are constant offsets.  Lane p of group q = lane / 16
  //     points at k-row 8 (q / 2) + p / 4, rows 16 (q % 2) + 4 (p % 4) .. + 4 of the block.
  // 16 x 16 x 32 (lane p of group q holds k = 8 q .. + 8 of row p):
  //   K-contiguous: 16 ((row * 8 | t) ^ (4 ks)), t = q ^ dl_kc_xor<true>(row);
  //   row-contiguous: k-row 8 q + p / 4, rows 4 (p % 4) .. + 4 of the block.
  int a_addr[TM], b_addr[TN];
  if constexpr (MI16) {
    const int p = lane & 15, q = lane >> 4;
    const int kl = 8 * q + (p >> 2), sxa = dl_seg_xor_of<true, BM>(kl), sxb = dl_seg_xor_of<true, BN>(kl);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row = wm + i * 16 + p;
      if (A_KC) a_addr[i] = (row * 8 + (q ^ dl_kc_xor<true>(row))) * 16;
      else a_addr[i] = kl * (BM * 2) + ((((wm >> 4) + i) ^ sxa) * 32) + 8 * (p & 3);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int row = wn + j * 16 + p;
      if (B_KC) b_addr[j] = (CA + row * 8 + (q ^ dl_kc_xor<true>(row))) * 16;
      else b_addr[j] = CA * 16 + kl * (BN * 2) + ((((wn >> 4) + j) ^ sxb) * 32) + 8 * (p & 3);
    }
  } else {
    const int p = lane & 15, q = lane >> 4;
    const int kl = 8 * (q >> 1) + (p >> 2), sx = dl_seg_xor(p >> 2);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row = wm + i * 32 + li;
      if (A_KC) a_addr[i] = (row * 8 + (kg ^ dl_kc_xor<false>(row))) * 16;
      else a_addr[i] = kl * (BM * 2) + ((((wm >> 4) + 2 * i + (q & 1)) ^ sx) * 32) + 8 * (p & 3);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int row = wn + j * 32 + li;
      if (B_KC) b_addr[j] = (CA + row * 8 + (kg ^ dl_kc_xor<false>(row))) * 16;
      else
        b_addr[j] = CA * 16 + kl * (BN * 2) + ((((wn >> 4) + 2 * j + (q & 1)) ^ sx) * 32) +
                    8 * (p & 3);
    }
  }

  bf16x8 fa[2][KSS * TM], fb[2][KSS * TN];
  constexpr int NSTEP = 64 / KQ / KSS;
  static_assert(NSTEP >= 2 && NSTEP % 2 == 0, "steps per tile");
  constexpr int NFRAG = KSS * (TM + TN), NMFMA = KSS * TM * TN;  // per step
  // read fragment r of step `step` from `tile` into set SET; order of use by the MFMAs
  // (k-step by k-step, row-major over the wave's blocks): A0, every B, A1, A2 ...
  auto read_frag = [&](auto set, auto r, const u32x4* tile, int step) {
    constexpr int SET = decltype(set)::value;
    constexpr int KL = decltype(r)::value / (TM + TN), R0 = decltype(r)::value % (TM + TN);
    constexpr int R = R0 == 0 ? 0 : (R0 <= TN ? TM + R0 - 1 : R0 - TN);
    const int ks = step * KSS + KL;
    if constexpr (R < TM) {
      if constexpr (A_KC) {
        int sel = ks * (KQ * 2);
        asm volatile("" : "+s"(sel));  // recomputed at every read: hoisted variants would spill
        fa[SET][KL * TM + R] = lds_read_b128(lds_addr(tile) + (a_addr[R] ^ sel));
      } else {
        const uint32_t p = lds_addr(tile) + a_addr[R];
        fa[SET][KL * TM + R] = lds_read_tr_pair(p, ks * KQ * (BM * 2), (ks * KQ + 4) * (BM * 2));
      }
    } else {
      if constexpr (B_KC) {
        int sel = ks * (KQ * 2);
        asm volatile("" : "+s"(sel));
        fb[SET][KL * TN + R - TM] = lds_read_b128(lds_addr(tile) + (b_addr[R - TM] ^ sel));
      } else {
        const uint32_t p = lds_addr(tile) + b_addr[R - TM];
        fb[SET][KL * TN + R - TM] = lds_read_tr_pair(p, ks * KQ * (BN * 2), (ks * KQ + 4) * (BN * 2));
      }
    }
  };
  // The compiler does not see the fragment reads (inline assembly): before the MFMAs of a
  // k-step may touch a fragment set, wait for LDS by hand, with the set's registers as
  // operands of the wait so that no MFMA can be moved in front of it.
  auto frags_ready = [&](auto set) {
    constexpr int SET = decltype(set)::value;
    __builtin_amdgcn_sched_barrier(0);
    lds_wait_for(fa[SET]);
    lds_wait_for(fb[SET]);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto mfma = [&](auto set, auto q) {
    constexpr int SET = decltype(set)::value, Q = decltype(q)::value;
    constexpr int kl = Q / (TM * TN), i = Q % (TM * TN) / TN, j = Q % TN;
    if constexpr (MI16)
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[SET][kl * TM + i], fb[SET][kl * TN + j],
                                                          acc[i][j], 0, 0, 0);
    else
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[SET][kl * TM + i], fb[SET][kl * TN + j],
                                                          acc[i][j], 0, 0, 0);
  };
  // column sums of the step whose B fragments are in set SET (still whole: reads fill the other)
  auto colsum_step = [&](auto set) {
    if constexpr (COLSUM) {
      constexpr int SET = decltype(set)::value;
      if (do_cs) {
        const uint32_t one2 = 0x3f803f80u;  // two bf16 ones
        const u32x4 ones4 = {one2, one2, one2, one2};
        const bf16x8 ones = __builtin_bit_cast(bf16x8, ones4);
#pragma unroll
        for (int kl = 0; kl < KSS; ++kl)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            cs[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, fb[SET][kl * TN + j], cs[j], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // step on fragment set SET while set 1 - SET is filled for step `step_next` of `tile`
  auto stage = [&](auto set, const u32x4* tile, int step_next) {
    constexpr int SET = decltype(set)::value;
    frags_ready(set);
    // the reads go out between the MFMAs of the first half (pinned: the scheduler would batch
    // them), so that they have the second half to land
    constexpr int SPREAD = NMFMA / 2;
    static_for<NMFMA>([&](auto q) {
      constexpr int Q = decltype(q)::value;
      static_for<NFRAG>([&](auto r) {
        if constexpr (decltype(r)::value * SPREAD / NFRAG == Q)
          read_frag(std::integral_constant<int, 1 - SET>{}, r, tile, step_next);
      });
      mfma(set, q);
      if constexpr (Q < SPREAD) __builtin_amdgcn_sched_barrier(0);
    });
    __builtin_amdgcn_sched_barrier(0);
    colsum_step(set);
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  // a workgroup barrier behind which every wave's copies have landed
  auto tile_barrier = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's copies are in LDS
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    __builtin_amdgcn_sched_barrier(0);
  };
  // ... but for its youngest IN_FLIGHT copies (no fence: the compiler waits for every copy in front of one)
  auto tile_barrier_behind = [&](auto in_flight) {
    constexpr int V = decltype(in_flight)::value;
    static_assert(V < 64, "vmcnt has six bits");
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(V) : "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // Tiles kt + 1 .. kt + STAGES - 1 are on their way while tile kt is multiplied; the barrier that
  // ends tile kt (in the middle of its last step, whose fragments are in registers by then)
  // frees its buffer for tile kt + STAGES, whose copies are started right behind that barrier.
  // A wave's copies land in the order of their requests and every tile past the first ones takes NL of
  // them, so that tile kt + 1 is there when no more than those of the STAGES - 2 behind it are missing.
  constexpr int NL = LA::N + LB::N;
#define GEMM_COPY_TILE(t, to)                                                                            \
  do {                                                                                                   \
    const char* sa = GEMM_SRC_A(t);                                                                      \
    const char* sb = GEMM_SRC_B(t);                                                                      \
    static_for<LA::N>([&](auto j) { la.template issue_one<decltype(j)::value>((to), sa); });             \
    static_for<LB::N>([&](auto j) { lb.template issue_one<decltype(j)::value>((to) + CA, sb); });        \
  } while (0)
  if constexpr (STAGES > 2) {
    if (nk > 1) {
      // (past the last tile: that one again, so that the count holds)
#pragma unroll
      for (int t = 1; t < STAGES; ++t) {
        const int src = t < nk ? t : nk - 1;
        if (t >= ns) GEMM_COPY_TILE(src, gemm_lds + t * TILE_CHUNKS);
      }
    }
    // (a shallow tile takes fewer copies)
    if (ns > 0 || nk == 1) tile_barrier();
    else tile_barrier_behind(std::integral_constant<int, (STAGES - 1) * NL>{});
    static_for<NFRAG>([&](auto r) { read_frag(S0{}, r, gemm_lds, 0); });
  } else {
    tile_barrier();
    static_for<NFRAG>([&](auto r) { read_frag(S0{}, r, gemm_lds, 0); });
    if (nk > 1 && ns < 2) GEMM_COPY_TILE(1, gemm_lds + TILE_CHUNKS);
  }
  for (int kt = 0; kt + 1 < nk; ++kt) {
    u32x4* cur = gemm_lds + (kt & (STAGES - 1)) * TILE_CHUNKS;
    const u32x4* nxt = gemm_lds + ((kt + 1) & (STAGES - 1)) * TILE_CHUNKS;
    static_for<NSTEP - 1>([&](auto st) {
      constexpr int ST = decltype(st)::value;
      stage(std::integral_constant<int, ST & 1>{}, cur, ST + 1);
    });
    frags_ready(S1{});  // the last step (NSTEP is even) is on set 1
    static_for<NMFMA / 2>([&](auto q) { mfma(S1{}, q); });
    if constexpr (STAGES > 2) tile_barrier_behind(std::integral_constant<int, (STAGES - 2) * NL>{});
    else tile_barrier();
    {
      // Behind the barrier: the first fragments of tile kt + 1, the copies of tile kt + STAGES and
      // the second half of the MFMAs, dealt out evenly and pinned in this order (the copies
      // and the reads both touch LDS, so the scheduler would otherwise leave the MFMAs last).
      // (past the last tile: it fetches tile nk - 1 again, into a buffer that
      // is not read any more, which keeps this block free of branches)
      constexpr int H = NMFMA / 2;
      const int k2 = kt + STAGES < nk ? kt + STAGES : nk - 1;
      const char* src_a2 = GEMM_SRC_A(k2);
      const char* src_b2 = GEMM_SRC_B(k2);
      static_for<H>([&](auto q) {
        constexpr int Q = decltype(q)::value;
        static_for<NFRAG>([&](auto r) {
          constexpr int R = decltype(r)::value;
          if constexpr (R >= NFRAG * Q / H && R < NFRAG * (Q + 1) / H) read_frag(S0{}, r, nxt, 0);
        });
        static_for<NL>([&](auto l) {
          constexpr int L = decltype(l)::value;
          if constexpr (L >= NL * Q / H && L < NL * (Q + 1) / H) {
            if constexpr (L < LA::N) la.template issue_one<L>(cur, src_a2);
            else lb.template issue_one<L - LA::N>(cur + CA, src_b2);
          }
        });
        mfma(S1{}, std::integral_constant<int, Q + H>{});
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    __builtin_amdgcn_sched_barrier(0);
    colsum_step(S1{});
  }
  {
    const u32x4* cur = gemm_lds + ((nk - 1) & (STAGES - 1)) * TILE_CHUNKS;
    static_for<NSTEP - 1>([&](auto st) {
      constexpr int ST = decltype(st)::value;
      stage(std::integral_constant<int, ST & 1>{}, cur, ST + 1);
    });
    frags_ready(S1{});
    static_for<NMFMA>([&](auto q) { mfma(S1{}, q); });
    colsum_step(S1{});
  }
  if constexpr (COLSUM) {
    // every row of a block holds the same sums: lanes 0..15 have row 0 of their column
    if (do_cs && lane < 16) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int64_t col = n0 + wn + j * 16 + lane;
        if (col < g.N) {
          const int64_t at = (int64_t)by * g.N + col;
          if (g.dtype_c == NBK_F32) ((float*)g.colsum)[at] = cs[j][0];
          else ((uint16_t*)g.colsum)[at] = nbk_f32_to_bf16(cs[j][0]);
        }
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): no copy may land in a slab
  __syncthreads();  // the epilogue reuses the tile buffers as per-wave slabs
  gemm_epilogue<TM, TN, WN, true, EPI>(acc, g, m0, n0, wm, wn, c_off, mem.bias, wave, lane);
#undef GEMM_COPY_TILE
#undef GEMM_SRC_A
#undef GEMM_SRC_B
}
template <int BM, int BN, bool A_KC, bool B_KC, int EPI, int NW, int KSS, bool MI16, bool COLSUM = false, int STAGES = 2>
__global__ __launch_bounds__(NW * 64) void gemm_bf16_dl_kernel(const GemmArgs g) {
  gemm_bf16_dl_body<BM, BN, A_KC, B_KC, EPI, NW, KSS, MI16, COLSUM, STAGES>(g, blockIdx.x, blockIdx.y, gridDim.y);
}

// ------------------------------------------------------------------- bf16, K <= 16
// C = alpha * A @ B (+ residual) with a contraction of at most 16 (the "up" product of a
// low-rank adapter): one MFMA deep, all memory traffic.  No K loop and no operand tiles in
// LDS: every lane reads its 8 k-values of an A row / a B column straight from global memory
// into the MFMA fragment, and the tile leaves through the shared epilogue.
template <bool B_KC, int EPI>
__global__ __launch_bounds__(256) void gemm_skinny_k_kernel(const GemmArgs g) {
  constexpr int TM = 2, TN = 2, WN = 64;
  int tm_i, tn_i;
  gemm_tile_coords(blockIdx.x, g.tiles_m, g.tiles_n, tm_i, tn_i);
  const int64_t m0 = (int64_t)tm_i * 128, n0 = (int64_t)tn_i * 128;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
  const int li = lane & 31, kg = lane >> 5;
  const uint16_t* A = (const uint16_t*)g.A;
  const uint16_t* B = (const uint16_t*)g.B;
  // 8 k-values from k0 = 8 kg on, zero past K; rows / columns past the edge are clamped
  // (their products are never stored)
  auto frag8 = [&](const uint16_t* p, int64_t stride, bool vec) {
    const int k0 = 8 * kg;
    u32x4 u = {0u, 0u, 0u, 0u};
    if (vec && k0 + 8 <= g.K) {
      u = *(const u32x4*)(p + k0);
    } else {
      uint32_t h[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) h[e] = k0 + e < g.K ? p[(k0 + e) * stride] : 0u;
      u.x = h[0] | (h[1] << 16); u.y = h[2] | (h[3] << 16);
      u.z = h[4] | (h[5] << 16); u.w = h[6] | (h[7] << 16);
    }
    return *(const bf16x8*)&u;
  };
  // The two 32-row bands of a wave's tile are worked off one after the other (not unrolled), so
  // that one band's accumulators, residual pieces and epilogue registers are all a lane holds:
  // four workgroups then fit a CU, and the 1024 tiles of an 8192 x 2048 result are resident at
  // once instead of leaving a quarter of them to a second, mostly empty round.
  // (EPI 4: the residual is on its way before the operands are, one memory latency for both)
  bf16x8 fb[TN];
  uint4 pre[WN / 16];
  u32x4 b_piece = {0u, 0u, 0u, 0u};
  if (!B_KC && g.b_vec) {
    const int k = threadIdx.x >> 4;
    const int64_t col = n0 + (threadIdx.x & 15) * 8;
    if (k < g.K && col + 8 <= g.N) b_piece = *(const u32x4*)(B + (int64_t)k * g.b_rs + col);
  }
  if constexpr (EPI == 4) gemm_residual_prefetch<1, WN>(g, m0, n0, wm, wn, lane, pre);
  if (!B_KC && g.b_vec) {
    // B given as [K][N] with whole 16-byte pieces of its rows readable: the workgroup's 16 x 128
    // piece goes to LDS k-major (one coalesced 16-byte load per lane, zeros past K and N; it was
    // requested above, ahead of the first band's residual) and
    // the fragments come out through the transposing read -- instead of eight strided 2-byte
    // loads per lane and column block.
    char* bst = (char*)gemm_lds + 4 * 32 * (64 + 4) * sizeof(float);
    *(u32x4*)(bst + (threadIdx.x >> 4) * 256 + (threadIdx.x & 15) * 16) = b_piece;
    __syncthreads();
    const int p = lane & 15, q = lane >> 4;
    const char* tr = bst + (8 * (q >> 1) + (p >> 2)) * 256 + (wn + 16 * (q & 1) + 4 * (p & 3)) * 2;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const s16x4 lo = lds_read_tr(tr + j * 64), hi = lds_read_tr(tr + j * 64 + 4 * 256);
      const s16x8 u = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      fb[j] = *(const bf16x8*)&u;
    }
  } else {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      int64_t col = n0 + wn + j * 32 + li;
      col = col < g.N ? col : g.N - 1;
      fb[j] = B_KC ? frag8(B + col * g.b_cs, 1, g.b_vec) : frag8(B + col, g.b_rs, false);
    }
  }
#pragma unroll 1
  for (int i = 0; i < TM; ++i) {
    if (EPI == 4 && i > 0) gemm_residual_prefetch<1, WN>(g, m0, n0, wm + i * 32, wn, lane, pre);
    int64_t row = m0 + wm + i * 32 + li;
    row = row < g.M ? row : g.M - 1;
    const bf16x8 fa = frag8(A + row * g.a_rs, 1, g.a_vec);
    f32x16 acc[1][TN];
#pragma unroll
    for (int j = 0; j < TN; ++j)
      acc[0][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, fb[j], (f32x16)(0.f), 0, 0, 0);
    gemm_epilogue<1, TN, WN, true, EPI>(acc, g, m0, n0, wm + i * 32, wn, 0, g.bias, wave, lane,
                                        EPI == 4 ? pre : nullptr);
  }
}

// ------------------------------------------------------------------- bf16, N <= 32
// C[M x N] = alpha * A[M x K] @ B[K x N] with at most 32 columns (the "down" product of a
// low-rank adapter and its transpose in the backward pass): A is read once and that is all the
// traffic there is.  One workgroup per 32 rows of A; its eight waves split K, each reads its
// part of the rows straight from global memory into MFMA fragments (one 32 x 32 accumulator
// tile; columns past N hold whatever the clamped or padded reads give and are never stored:
// a column of B only reaches the same column of C), and the eight partial tiles are added
// through LDS.
//   B_KC:  B given as [N][K] (K contiguous): fragments come straight from global memory too.
//   !B_KC: B given as [K][N] (N contiguous, N % 8 == 0): every wave stages its K range in LDS
//          k-major and reads fragments through the transposing read.
extern __shared__ __align__(16) u32x4 skinny_lds[];

constexpr int SKN_WAVES = 8;

template <bool B_KC>
__global__ __launch_bounds__(SKN_WAVES * 64) void gemm_skinny_n_kernel(const GemmArgs g,
                                                                        int pitch_chunks) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 31, kg = lane >> 5;
  const uint16_t* A = (const uint16_t*)g.A;
  const uint16_t* B = (const uint16_t*)g.B;
  const int64_t row0 = (int64_t)blockIdx.x * 32;
  // this wave's 64-wide K chunks
  const int chunks = (int)(g.K >> 6);
  const int per = (chunks + SKN_WAVES - 1) / SKN_WAVES;
  const int c_begin = wave * per;
  const int c_end = c_begin + per < chunks ? c_begin + per : chunks;
  float* red = (float*)skinny_lds;                                   // [waves][16 regs][64 lanes]
  char* stage = (char*)(skinny_lds + SKN_WAVES * 16 * 64 / 4);        // behind the reduction area
  const int pitch = pitch_chunks * 16;                                // bytes per staged k-row
  const char* tr_ptr = nullptr;
  const uint16_t* bp = nullptr;
  if (B_KC) {
    const int64_t col = li < g.N ? li : g.N - 1;
    bp = B + col * g.b_cs + 8 * kg;
  } else {
    // (rows [64 c_begin, 64 c_end) of B are staged below, behind the first requests for A)
    // lane p of group q = lane / 16: k-row 8 (q / 2) + p / 4, columns 16 (q % 2) + 4 (p % 4) .. + 4
    // (every lane of a group takes part in the exchange, also those that point at padding)
    const int p = lane & 15, q = lane >> 4;
    const int col0 = 16 * (q & 1) + 4 * (p & 3);
    tr_ptr = stage + (8 * (q >> 1) + (p >> 2)) * pitch + col0 * 2;
  }
  f32x16 acc = (f32x16)(0.f);
  // A streams through a 4 KB slab per wave (the bytes that later hold this wave's partial tile):
  // a 32-row x 64-k chunk arrives in four fully coalesced loads (eight lanes per 128-byte row
  // piece; fetching the 32-byte pieces of 32 rows that an MFMA fragment consists of straight
  // from memory runs at a quarter of that rate), is written to the slab swizzled and read back
  // as fragments.  The slab belongs to one wave, whose LDS accesses execute in order, so no
  // workgroup barrier is involved.  Three chunks are in flight in registers.
  u32x4* slab = (u32x4*)(red + wave * 16 * 64);
  const int lrow = lane >> 3, lch = lane & 7;
  const uint16_t* arow_p[4];
  int w_at[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int r = p * 8 + lrow;
    const int64_t gr = row0 + r < g.M ? row0 + r : g.M - 1;
    arow_p[p] = A + gr * g.a_rs + 8 * lch;
    w_at[p] = r * 8 + (lch ^ dl_kc_xor<false>(r));
  }
  const int r_at = li * 8, r_x = dl_kc_xor<false>(li);
  constexpr int AHEAD = 3;
  u32x4 an[AHEAD][4], bn[AHEAD][4];
  auto fetch = [&](auto slot, int c) {
    constexpr int J = decltype(slot)::value;
    const int64_t k0 = (int64_t)c * 64;
#pragma unroll
    for (int p = 0; p < 4; ++p) an[J][p] = *(const u32x4*)(arow_p[p] + k0);
    if (B_KC) {
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) bn[J][s4] = *(const u32x4*)(bp + k0 + 16 * s4);
    }
  };
  static_for<AHEAD>([&](auto j) {
    if (c_begin + decltype(j)::value < c_end) fetch(j, c_begin + decltype(j)::value);
  });
  if (!B_KC) {
    // stage rows [64 c_begin, 64 c_end) of B; a k-row holds N / 8 chunks (pitch_chunks >= that);
    // four pieces per lane are on their way at a time
    const int nch = (int)(g.N >> 3);
    const int total = (c_end - c_begin) * 64 * nch;
    for (int t0 = 0; t0 < total; t0 += 256) {
      u32x4 piece[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = t0 + u * 64 + lane;
        const int k = t / nch, c = t - k * nch;
        const int64_t gk = (int64_t)c_begin * 64 + k;
        if (t < total) piece[u] = *(const u32x4*)(B + gk * g.b_rs + c * 8);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = t0 + u * 64 + lane;
        const int k = t / nch, c = t - k * nch;
        const int64_t gk = (int64_t)c_begin * 64 + k;
        if (t < total) *(u32x4*)(stage + (size_t)gk * pitch + c * 16) = piece[u];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  for (int c = c_begin; c < c_end; c += AHEAD) {
    static_for<AHEAD>([&](auto j) {
      constexpr int J = decltype(j)::value;
      const int cc = c + J;
      if (cc < c_end) {  // (uniform over the wave)
        const int64_t k0 = (int64_t)cc * 64;
#pragma unroll
        for (int p = 0; p < 4; ++p) slab[w_at[p]] = an[J][p];
        bf16x8 fa[4], fb[4];
        if (B_KC) {
#pragma unroll
          for (int s4 = 0; s4 < 4; ++s4) fb[s4] = *(const bf16x8*)&bn[J][s4];
        } else {
#pragma unroll
          for (int s4 = 0; s4 < 4; ++s4) {
            const char* a0 = tr_ptr + (k0 + 16 * s4) * pitch;
            const s16x4 lo = lds_read_tr(a0), hi = lds_read_tr(a0 + 4 * pitch);
            const s16x8 u = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            fb[s4] = *(const bf16x8*)&u;
          }
        }
        if (cc + AHEAD < c_end) fetch(j, cc + AHEAD);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) {
          const u32x4 u = slab[r_at + ((2 * s4 + kg) ^ r_x)];
          fa[s4] = *(const bf16x8*)&u;
        }
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4)
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[s4], fb[s4], acc, 0, 0, 0);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
    });
  }
  // (the slab is this wave's part of the reduction area: its last fragments are in registers)
#pragma unroll
  for (int r = 0; r < 16; ++r) red[(wave * 16 + r) * 64 + lane] = acc[r];
  __syncthreads();
  const int64_t col = li;
  if (col >= g.N) return;
  // Every wave adds up its share of the tile: left to one wave, the 128 reads in a row are a quarter of the launch
  // (1000 x 8 x 1024 8.1 -> 4.4 us with the form for few rows, 8192 x 16 x 1024 7.7 -> 5.5, 8192 x 16 x 2048 10.7 ->
  // 8.6, 20000 x 16 x 1024 15.5 -> 11.2).  Sixteen waves that halve the K of each gain nothing (4.4, 5.0, 7.4, 13.8).
#pragma unroll
  for (int r0 = 0; r0 < 16 / SKN_WAVES; ++r0) {
    const int r = wave * (16 / SKN_WAVES) + r0;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < SKN_WAVES; ++w) v += red[(w * 16 + r) * 64 + lane];
    const int64_t row = row0 + 8 * (r >> 2) + 4 * kg + (r & 3);
    if (row < g.M) nbk_store_from_f32(g.C, row * g.ldc + col, g.dtype_c, v * g.alpha);
  }
}

// ------------------------------------------------------ fp32 against NF4-coded weights
// 128 x 128 x 16 tile, LDS k-major ([k][rows], rows padded by 4 floats).
template <bool B_KC>
__global__ __launch_bounds__(256) void gemm_f32_nf4_kernel(const GemmArgs g) {
  constexpr int BM = 128, BN = 128, BK = 16, LD = 128 + 4;
  __shared__ float As[2][BK][LD];
  __shared__ float Bs[2][BK][LD];
  __shared__ float nf4_table[16];  // (B holds NF4 codes, g.b_scales the block scales)
  if (threadIdx.x < 16) nf4_table[threadIdx.x] = nbk_nf4_levels[threadIdx.x];
  __syncthreads();
  int tm_i, tn_i;
  gemm_tile_coords(blockIdx.x, g.tiles_m, g.tiles_n, tm_i, tn_i);
  const int64_t m0 = (int64_t)tm_i * BM, n0 = (int64_t)tn_i * BN;
  const float* A = (const float*)g.A;
  const int64_t K = g.K;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
  const int li = lane & 31, kg = lane >> 5;

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (f32x16)(0.f);

  // each lane stages 8 floats of A and 8 of B per k-tile (128*16 / 256)
  float ra[8], rb[8];
  auto load_a = [&](int64_t k0, float* r) {
    // lane -> (row = tid/2, 8 consecutive k)
    const int64_t gr = m0 + (tid >> 1), gk = k0 + (tid & 1) * 8;
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = (gr < g.M && gk + e < K) ? A[gr * g.a_rs + gk + e] : 0.f;
  };
  // B from NF4 codes: the same eight elements per lane, dequantised
  auto load_b = [&](int64_t k0, float* r) {
    if (B_KC) {
      const int64_t gr = n0 + (tid >> 1), gk = k0 + (tid & 1) * 8;
      nf4_load8((const uint8_t*)g.B, g.b_scales, g.b_block, nf4_table, gr * g.b_cs + gk, gr < g.N ? K - gk : 0, r);
    } else {
      const int64_t gk = k0 + (tid >> 4), gr = n0 + (tid & 15) * 8;
      nf4_load8((const uint8_t*)g.B, g.b_scales, g.b_block, nf4_table, gk * g.b_rs + gr, gk < K ? g.N - gr : 0, r);
    }
  };
  auto store_tile = [&](float (*S)[LD], bool kc, const float* r) {
    if (kc) {
      const int row = tid >> 1, kk = (tid & 1) * 8;
#pragma unroll
      for (int e = 0; e < 8; ++e) S[kk + e][row] = r[e];
    } else {
      const int kk = tid >> 4, rr = (tid & 15) * 8;
#pragma unroll
      for (int e = 0; e < 8; ++e) S[kk][rr + e] = r[e];
    }
  };

  const int64_t nk = (K + BK - 1) / BK;
  load_a(0, ra);
  load_b(0, rb);
  store_tile(As[0], true, ra);
  store_tile(Bs[0], B_KC, rb);
  __syncthreads();
  for (int64_t kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    const bool more = kt + 1 < nk;
    if (more) {
      load_a((kt + 1) * BK, ra);
      load_b((kt + 1) * BK, rb);
    }
#pragma unroll
    for (int ks = 0; ks < BK / 2; ++ks) {
      const int k = ks * 2 + kg;
      float fa[2], fb[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) fa[i] = As[cur][k][wm + i * 32 + li];
#pragma unroll
      for (int j = 0; j < 2; ++j) fb[j] = Bs[cur][k][wn + j * 32 + li];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
    if (more) {
      store_tile(As[cur ^ 1], true, ra);
      store_tile(Bs[cur ^ 1], B_KC, rb);
    }
    __syncthreads();
  }
  float* C = (float*)g.C;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t col = n0 + wn + j * 32 + li;
      if (col >= g.N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t row = m0 + wm + i * 32 + (r >> 2) * 8 + kg * 4 + (r & 3);
        if (row < g.M) C[row * g.ldc + col] = acc[i][j][r] * g.alpha;
      }
    }
}

// --------------------------------------------------------------- fp32
// Rows of one operand of a workgroup's K tile on their way from memory through registers to LDS, as
// [row][k] with four floats of padding: a fragment is then one 16-byte LDS read of four k values of a
// row, without bank conflicts for every pitch used (20, 36, 68 floats: 16 rows start on 16 different
// groups of four banks).  The 16-byte chunks of a row are permuted by bits 4 and 5 of its number,
// which spreads the transposed writes of a row-contiguous operand over all banks too.  Global
// reads are 16-byte pieces at any 4-byte alignment.
template <int N>
using f32_piece = float __attribute__((ext_vector_type(N)));
template <int N>
using f32_piece_any = float __attribute__((ext_vector_type(N), aligned(4)));
__device__ __forceinline__ int f32_at(int row, int chunk, int ld) { return row * ld + (chunk ^ (row >> 4 & 3)) * 4; }
template <int ROWS, int BK, bool KC, int NT>
struct F32Rows {
  static constexpr int LD = BK + 4;
  static constexpr int RB = 2;  // row-contiguous operand: blocks of RB rows x 2 k
  static constexpr int V = KC ? 4 : RB, Q = KC ? 1 : 2;  // a piece: Q accesses of V floats
  static constexpr int PAD = KC ? 0 : V - 1;  // LDS rows in front of the tile (place)
  static constexpr int PIECES = ROWS * BK / NT / (V * Q);
  static_assert(PIECES >= 1, "at least one piece per lane");
  f32_piece<V> r[2][PIECES][Q];  // two K tiles in flight
  // Where the pieces of the next K tile begin: worked out once (a product of 64 bits per request and
  // tile was a tenth of the kernel: 128 x 256 x 784 11.3 us, then 10.7).
  const float* at[PIECES];
  int64_t stride;

  // Where a piece lies in the tile.  The pieces of a row-contiguous operand past its end lie where its
  // last one does, which ends with the last row (and may begin before the tile): the edge of a
  // result is loaded like the rest of it.  Element by element, the workgroups there took half as long
  // again as the others: 79 x 150 x 1188 as x^T dy 29.0 us, 16.5 now, 576 x 248 x 2608 54.0 -> 29.9.
  __device__ static __forceinline__ void place(int p, int64_t left, bool whole, int& row, int& kk) {
    const int idx = (int)threadIdx.x + NT * p;
    if constexpr (KC) {
      row = idx / (BK / 4);
      kk = idx % (BK / 4) * 4;
    } else {
      row = idx % (ROWS / RB) * RB;
      kk = idx / (ROWS / RB) * 2;
      if (whole) row = (int)min((int64_t)row, left - V);
    }
  }
  // Whether the operand has rows for a whole piece.
  __device__ static __forceinline__ bool pieces(int64_t rows) { return KC || rows >= V; }
  // `stride`: between rows (KC) or between k (row-contiguous).  Rows past the end repeat the last one or
  // are left as they are in LDS (their results are not stored).
  __device__ __forceinline__ void init(const float* P, int64_t stride_, int64_t row0, int64_t rows) {
    stride = stride_;
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      int row, kk;
      place(p, rows - row0, pieces(rows), row, kk);
      at[p] = KC ? P + min(row0 + row, rows - 1) * stride + kk : P + kk * stride + row0 + row;
    }
  }
  __device__ __forceinline__ void next() {
#pragma unroll
    for (int p = 0; p < PIECES; ++p) at[p] += KC ? (int64_t)BK : BK * stride;
  }
  // A K tile that lies inside K, in whole pieces.
  template <int SET>
  __device__ __forceinline__ void load() {
#pragma unroll
    for (int p = 0; p < PIECES; ++p)
#pragma unroll
      for (int q = 0; q < Q; ++q) r[SET][p][q] = *(const f32_piece_any<V>*)(KC || q == 0 ? at[p] : at[p] + stride);
    next();
  }
  // Any other K tile, element by element, `left` k before the end; k past it reads as zero.
  template <int SET>
  __device__ __forceinline__ void load_each(int64_t row0, int64_t rows, int64_t left) {
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      int row, kk;
      place(p, rows - row0, pieces(rows), row, kk);
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const int64_t over = KC ? 0 : min(row0 + row + e, rows - 1) - (row0 + row);  // (past the last row: the last)
          const float* src = KC ? at[p] + e : at[p] + q * stride + over;
          r[SET][p][q][e] = kk + (KC ? e : q) < left ? *src : 0.f;
        }
    }
    next();
  }
  template <int SET>
  __device__ __forceinline__ void store(float* S, int64_t row0, int64_t rows) {
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      int row, kk;
      place(p, rows - row0, pieces(rows), row, kk);
      // (the pieces stay as they were loaded until here: pairing two k of a row any earlier would
      // wait for the loads right behind their request)
#pragma unroll
      for (int q = 0; q < Q; ++q) asm volatile("" : "+v"(r[SET][p][q]));
      if constexpr (KC) {
        *(f32_piece<4>*)(S + f32_at(row, kk >> 2, LD)) = r[SET][p][0];
      } else {
#pragma unroll
        for (int e = 0; e < RB; ++e)
          *(float2*)(S + f32_at(row + e, kk >> 2, LD) + (kk & 2)) = make_float2(r[SET][p][0][e], r[SET][p][1][e]);
      }
    }
  }
};

// Small results: a workgroup of WK waves owns a tile of T x T (32 or 16) and splits every K tile of 16 WK; their sums
// meet in LDS at the end.  Bound by the length of a workgroup's K loop: two K tiles are requested ahead.
// Lane l of a v_mfma_f32_32x32x2f32 supplies A[row l % 32][k = l / 32] and B[k = l / 32][col l % 32] (of a
// 16x16x4f32: l % 16, l / 16); which k values share an instruction is free as long as A and B agree, so the lane
// with part h = l / T owns four consecutive k of a step and issues four instructions.  Where which form
// runs, and the times: nbk_gemm.  Two workgroups of up to eight waves have to fit a CU (the second launch
// bound); four waves with no row-contiguous operand are two to five per cent faster without.
template <bool A_KC, bool B_KC, int T, int WK>
__device__ __forceinline__ void gemm_f32_body(const GemmArgs& g, int bx, int by, int ny) {
  constexpr int BM = T, BN = T, KS = T / 16, BK = 16 * WK, LD = BK + 4;  // (a step: 8 or 16 k, in four instructions)
  constexpr int R = T * T / 64;                                           // results of a lane
  typedef float acc_t __attribute__((ext_vector_type(R)));
  typedef F32Rows<BM, BK, A_KC, 64 * WK> RowsA;
  typedef F32Rows<BN, BK, B_KC, 64 * WK> RowsB;
  constexpr int A0 = RowsA::PAD * LD, B0 = A0 + (BM + RowsB::PAD) * LD;
  constexpr int SET = B0 + BN * LD;  // (two of them)
  extern __shared__ __align__(16) u32x4 gemm_lds[];
  float* lds = (float*)gemm_lds;
  static_assert(WK * R * 64 <= 2 * SET, "the partial sums fit");
  int tm_i, tn_i;
  gemm_tile_coords(bx, g.tiles_m, g.tiles_n, tm_i, tn_i);
  const int64_t m0 = (int64_t)tm_i * BM, n0 = (int64_t)tn_i * BN;
  const int64_t bo = (int64_t)by / g.batch_inner, bi = (int64_t)by % g.batch_inner;
  const float* A = (const float*)g.A + bo * g.a_bs + bi * g.a_bs2;
  const GemmMember mem = gemm_member(g, bo, bi, 4);
  const float* B = (const float*)mem.B;
  const int64_t c_off = mem.c_off;
  const int64_t K = gemm_slice_k(g, bo, bi, ny);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane % T, h = lane / T;
  const int64_t a_stride = A_KC ? g.a_rs : g.a_cs, b_stride = B_KC ? g.b_cs : g.b_rs;

  acc_t acc = (acc_t)(0.f);

  RowsA la;
  RowsB lb;
  const int64_t nk = (K + BK - 1) / BK;
  const bool pieces = la.pieces(g.M) && lb.pieces(g.N);
  // (one branch for both operands: with a branch each, the second one's requests wait for the
  // data of the first, 576 x 256 x 2608 40 us instead of 31)
  la.init(A, a_stride, m0, g.M);
  lb.init(B, b_stride, n0, g.N);
  auto load = [&](auto set, int64_t kt) {  // (tile after tile)
    if (pieces && (kt + 1) * BK <= K) {
      la.template load<set.value>();
      lb.template load<set.value>();
    } else {
      la.template load_each<set.value>(m0, g.M, K - kt * BK);
      lb.template load_each<set.value>(n0, g.N, K - kt * BK);
    }
  };
  auto store = [&](auto set) {
    float* S = lds + set.value * SET;
    la.template store<set.value>(S + A0, m0, g.M);
    lb.template store<set.value>(S + B0, n0, g.N);
  };
  auto tile = [&](auto cur, auto next, int64_t kt) {
    if (kt + 2 < nk) load(cur, kt + 2);  // (its registers went to LDS an iteration ago)
    const float* As = lds + cur.value * SET + A0;
    const float* Bs = lds + cur.value * SET + B0;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const f32x4 fa = *(const f32x4*)(As + f32_at(li, (wave * KS + s) * (64 / T) + h, LD));
      const f32x4 fb = *(const f32x4*)(Bs + f32_at(li, (wave * KS + s) * (64 / T) + h, LD));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (T == 32) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[e], fb[e], acc, 0, 0, 0);
        else acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fb[e], acc, 0, 0, 0);
      }
    }
    if (kt + 1 < nk) store(next);
    __syncthreads();
  };
  const std::integral_constant<int, 0> s0{};
  const std::integral_constant<int, 1> s1{};
  load(s0, 0);
  if (nk > 1) load(s1, 1);
  store(s0);
  __syncthreads();
  for (int64_t kt = 0; kt < nk; kt += 2) {
    tile(s0, s1, kt);
    if (kt + 1 < nk) tile(s1, s0, kt + 1);
  }

  // D register r of lane (col li, part h) is row (r / 4) * 8 + h * 4 + r % 4
  float* C = (float*)g.C;
  auto put = [&](int r, float sum) {
    const int64_t row = m0 + (r >> 2) * 8 + h * 4 + (r & 3), col = n0 + li;
    if (row >= g.M || col >= g.N) return;
    const int64_t idx = c_off + row * g.ldc + col;
    const float x = sum * g.alpha + (mem.bias ? ((const float*)mem.bias)[col] : 0.f);
    float v;
    if (g.C2) {
      float dv;
      gemm_act_pair<false>(x, g.act, v, dv);
      ((float*)g.C2)[idx] = dv;
    } else {
      v = gemm_act(x, g.act);
    }
    if (g.residual) v = g.res_mul ? v * ((const float*)g.residual)[idx] : v + ((const float*)g.residual)[idx];
    C[idx] = v;
  };
  // (every read of the last K tile lies before its barrier) each wave sums its share of the registers
#pragma unroll
  for (int r = 0; r < R; ++r) lds[(wave * R + r) * 64 + lane] = acc[r];
  __syncthreads();
  const float* part = lds + lane;
#pragma unroll
  for (int q = 0; q < (R + WK - 1) / WK; ++q) {
    const int r = q * WK + wave;
    if (r >= R) break;
    float sum[WK];
#pragma unroll
    for (int w = 0; w < WK; ++w) sum[w] = part[(w * R + r) * 64];
#pragma unroll
    for (int n = WK / 2; n > 0; n /= 2)
#pragma unroll
      for (int w = 0; w < n; ++w) sum[w] = sum[2 * w] + sum[2 * w + 1];
    put(r, sum[0]);
  }
}
template <bool A_KC, bool B_KC, int T, int WK>
__global__ __launch_bounds__(64 * WK, WK > 8 || (WK == 4 && A_KC && B_KC) ? 1 : 2) void gemm_f32_kernel(const GemmArgs g) {
  gemm_f32_body<A_KC, B_KC, T, WK>(g, blockIdx.x, blockIdx.y, gridDim.y);
}
// LDS of a workgroup of gemm_f32_kernel: two K tiles, each with rows in front of a row-contiguous operand.
template <bool A_KC, bool B_KC, int T, int WK>
constexpr size_t gemm_f32_lds() {
  return 2 * (size_t)(2 * T + !A_KC + !B_KC) * (16 * WK + 4) * sizeof(float);
}

// --------------------------------------------------------------- fp32 out of bf16 parts
// One operand's rows of a workgroup's K tile on their way through registers: a lane takes pieces of 8
// consecutive k of a row, which it splits when they have landed (split_f32.h).
template <int ROWS, int NT, bool KC>
struct SplitRows {
  static constexpr int PIECES = ROWS * 4 / NT;
  static_assert(PIECES >= 1 && PIECES * NT == ROWS * 4, "whole pieces per lane");
  const float* at[PIECES];  // the piece's first element in the next K tile
  int64_t stride, left;     // between k of a row-contiguous operand; k from the next tile's first to the end
  float r[2][KC ? 1 : PIECES][8];  // two K tiles in flight, of either form
  sp_f4 r4[2][KC ? PIECES : 1][2];
  __device__ __forceinline__ static void place(int p, int& row, int& c) {
    const int idx = (int)threadIdx.x + NT * p;
    row = KC ? idx >> 2 : idx % ROWS;
    c = KC ? idx & 3 : idx / ROWS;
  }
  // (rows past the end repeat the last one: their results are not stored)
  __device__ __forceinline__ void init(const float* P, int64_t stride_, int64_t row0, int64_t rows, int64_t K) {
    stride = stride_;
    left = K;
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      int row, c;
      place(p, row, c);
      const int64_t m = min(row0 + row, rows - 1);
      at[p] = KC ? P + m * stride + c * 8 : P + (c * 8) * stride + m;
    }
  }
  // Whether the next K tile lies inside K (one branch for both operands: with a branch each, the second
  // one's requests wait for the data of the first).
  __device__ __forceinline__ bool whole() const { return left >= SPLIT_BK; }
  template <int SET>
  __device__ __forceinline__ void load() {
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      if constexpr (KC) {
#pragma unroll
        for (int h = 0; h < 2; ++h) r4[SET][p][h] = *(const sp_f4_any*)(at[p] + 4 * h);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) r[SET][p][e] = at[p][e * stride];
      }
    }
    next();
  }
  // The last tile of a contraction that is no multiple of 32.
  template <int SET>
  __device__ __forceinline__ void load_tail() {
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      int row, c;
      place(p, row, c);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = c * 8 + e < left ? at[p][KC ? e : e * stride] : 0.f;
        if constexpr (KC) r4[SET][p][e >> 2][e & 3] = x;
        else r[SET][p][e] = x;
      }
    }
    next();
  }
  __device__ __forceinline__ void next() {
    left -= SPLIT_BK;
#pragma unroll
    for (int p = 0; p < PIECES; ++p) at[p] += KC ? (int64_t)SPLIT_BK : SPLIT_BK * stride;
  }
  template <int SET>
  __device__ __forceinline__ void store(sp_u4* tile) {
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      int row, c;
      place(p, row, c);
      float x[8];
      // (the numbers stay as they were loaded until here: split any earlier, they would be waited for
      // right behind their request)
      if constexpr (KC) {
#pragma unroll
        for (int h = 0; h < 2; ++h) asm volatile("" : "+v"(r4[SET][p][h]));
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) asm volatile("" : "+v"(r[SET][p][e]));
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = KC ? r4[SET][p][e >> 2][e & 3] : r[SET][p][e];
      split_store<ROWS>(tile, row, c, x);
    }
  }
};

// C = A B of float32 numbers: tiles of BM x BN, NWM x NWN waves, two K tiles of 32 in LDS.
template <int BM, int BN, int NWM, int NWN, int NM, bool A_KC, bool B_KC, bool FULL>
__device__ __forceinline__ void gemm_f32_split_body(const GemmArgs& g, int bx, int by, int ny) {
  constexpr int NT = NWM * NWN * 64, WM = BM / NWM, WN = BN / NWN, TM = WM / 16, TN = WN / 16;
  constexpr int TILE = (BM + BN) * 12;  // 16-byte chunks: three parts of four chunks a row
  extern __shared__ __align__(16) u32x4 gemm_lds[];
  sp_u4* lds = (sp_u4*)gemm_lds;
  int tm_i, tn_i;
  gemm_tile_coords(bx, g.tiles_m, g.tiles_n, tm_i, tn_i);
  const int64_t m0 = (int64_t)tm_i * BM, n0 = (int64_t)tn_i * BN;
  const int64_t bo = (int64_t)by / g.batch_inner, bi = (int64_t)by % g.batch_inner;
  const float* A = (const float*)g.A + bo * g.a_bs + bi * g.a_bs2;
  const GemmMember mem = gemm_member(g, bo, bi, 4);
  const float* B = (const float*)mem.B;
  const int64_t c_off = mem.c_off;
  const int64_t K = gemm_slice_k(g, bo, bi, ny);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / NWN * WM, wn = wave % NWN * WN;
  SplitRows<BM, NT, A_KC> la;
  SplitRows<BN, NT, B_KC> lb;
  la.init(A, A_KC ? g.a_rs : g.a_cs, m0, g.M, K);
  lb.init(B, B_KC ? g.b_cs : g.b_rs, n0, g.N, K);
  SplitAcc<TM, TN, NM> acc;
  acc.zero();
  const int nk = (int)((K + SPLIT_BK - 1) / SPLIT_BK);
#define SPLIT_LOAD(SET)                                                  \
  do {                                                                   \
    if (la.whole()) { la.template load<SET>(); lb.template load<SET>(); } \
    else { la.template load_tail<SET>(); lb.template load_tail<SET>(); }  \
  } while (0)
#define SPLIT_STORE(SET) do { la.template store<SET>(lds + SET * TILE); lb.template store<SET>(lds + SET * TILE + BM * 12); } while (0)
  // tile kt, with tile kt + 2 requested and tile kt + 1 split into the other buffer meanwhile
#define SPLIT_TILE(SET, REQUEST, MORE)                                                                   \
  do {                                                                                                   \
    REQUEST;                                                                                             \
    acc.template multiply<BM, BN, SET>(lds + SET * TILE, lds + SET * TILE + BM * 12, wm, wn, lane);      \
    if (MORE) SPLIT_STORE((1 - SET));                                                                    \
    __syncthreads();                                                                                     \
  } while (0)
  SPLIT_LOAD(0);
  if (nk > 1) SPLIT_LOAD(1);
  SPLIT_STORE(0);
  __syncthreads();
  int kt = 0;
  // (while the requests are whole tiles they stand in no branch: behind one, the compiler waits for the
  // youngest request before it lets the splitting have the older ones)
  for (; kt + 3 < (int)(K / SPLIT_BK); kt += 2) {
    SPLIT_TILE(0, (la.template load<0>(), lb.template load<0>()), true);
    SPLIT_TILE(1, (la.template load<1>(), lb.template load<1>()), true);
  }
  for (; kt < nk; ++kt) {
    SPLIT_TILE(0, if (kt + 2 < nk) SPLIT_LOAD(0), kt + 1 < nk);
    if (++kt < nk) SPLIT_TILE(1, if (kt + 2 < nk) SPLIT_LOAD(1), kt + 1 < nk);
  }
#undef SPLIT_TILE
#undef SPLIT_STORE
#undef SPLIT_LOAD
  float* C = (float*)g.C;
  // sum(i, j, r) of the results that `put` is to store, and the others, a bit each
  auto store = [&](auto sum, auto put) {
    uint32_t left = 0;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int64_t col = n0 + wn + j * 16 + (lane & 15);
        if (col >= g.N) continue;
        const float bias = mem.bias ? ((const float*)mem.bias)[col] : 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int64_t row = m0 + wm + i * 16 + (lane >> 4) * 4 + r;
          if (row >= g.M) continue;
          const float s = sum(i, j, r);
          const uint32_t bit = 1u << ((i * TN + j) * 4 + r);
          if (!put(s, bit)) {
            left |= bit;
            continue;
          }
          const int64_t idx = c_off + row * g.ldc + col;
          const float x = s * g.alpha + bias;
          float v;
          if (FULL && g.C2) {
            float dv;
            gemm_act_pair<false>(x, g.act, v, dv);
            ((float*)g.C2)[idx] = dv;
          } else {
            v = FULL ? gemm_act(x, g.act) : g.act == NBK_ACT_RELU ? fmaxf(x, 0.f) : x;
          }
          if (FULL && g.residual) v = g.res_mul ? v * ((const float*)g.residual)[idx] : v + ((const float*)g.residual)[idx];
          C[idx] = v;
        }
      }
    return left;
  };
  static_assert(TM * TN * 4 <= 32, "a bit for each of a lane's results");
  // (a contraction of one number is a product, rounded once: six rounded together are up to 0.78 of the last place off)
  const bool one = K == 1;
  const uint32_t left = store([&](int i, int j, int r) { return acc.sum(i, j, r); },
                              [&](float s, uint32_t) { return fabsf(s) < INFINITY && !one; });
  // (us, numbers that have parts / one infinity / NaN throughout: 1024 x 1024 x 1024 25 / 52 / 55, 4096 x 4096 x 1024
  // 193 / 336 / 585, where the float32 instruction alone takes 37 and 313; a lane at a time 1660 and 13700 at last)
  if (one) {
    static_assert(WM <= 64, "a row for each lane");
    const float x = A[min(m0 + wm + min(lane, WM - 1), g.M - 1) * g.a_rs];
    float y[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) y[j] = B[min(n0 + wn + j * 16 + (lane & 15), g.N - 1) * g.b_cs];
    float mine[TM][4];  // (shuffled here: the lanes past an edge leave `store`)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) mine[i][r] = __shfl(x, i * 16 + (lane >> 4) * 4 + r);
    store([&](int i, int j, int r) { return mine[i][r] * y[j]; }, [](float, uint32_t) { return true; });
  } else if (__any(left != 0)) {
    const float* pa[TM];
    const float* pb[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) pa[i] = A + min(m0 + wm + i * 16 + (lane & 15), g.M - 1) * g.a_rs;
#pragma unroll
    for (int j = 0; j < TN; ++j) pb[j] = B + min(n0 + wn + j * 16 + (lane & 15), g.N - 1) * g.b_cs;
    auto at = [&](const float* p, int64_t k, int64_t stride, auto inside) {
      if constexpr (inside.value) return p[k * stride];
      const float x = p[min(k, K - 1) * stride];
      return k < K ? x : 0.f;
    };
    acc.again(0, K, lane, [&](int i, int64_t k, auto inside) { return at(pa[i], k, A_KC ? 1 : g.a_cs, inside); },
              [&](int j, int64_t k, auto inside) { return at(pb[j], k, B_KC ? 1 : g.b_rs, inside); });
    store([&](int i, int j, int r) { return acc.sum_again(i, j, r); }, [&](float, uint32_t bit) { return (left & bit) != 0; });
  }
}
template <int BM, int BN, int NWM, int NWN, int NM, bool A_KC, bool B_KC, bool FULL>
__global__ __launch_bounds__(NWM * NWN * 64) void gemm_f32_split_kernel(const GemmArgs g) {
  gemm_f32_split_body<BM, BN, NWM, NWN, NM, A_KC, B_KC, FULL>(g, blockIdx.x, blockIdx.y, gridDim.y);
}

template <int BM, int BN, int NW = 4>
static int launch_bf16(const GemmArgs& a, bool akc, bool bkc, int64_t batch, hipStream_t st) {
  GemmArgs g = a;
  g.tiles_m = (int)((a.M + BM - 1) / BM);
  g.tiles_n = (int)((a.N + BN - 1) / BN);
  dim3 grid((unsigned)(g.tiles_m * g.tiles_n), (unsigned)batch);
  const size_t pipe_of[2][2] = {
      {2 * (size_t)(TileGeom<BM, false>::CHUNKS + TileGeom<BN, false>::CHUNKS) * 16,
       2 * (size_t)(TileGeom<BM, false>::CHUNKS + TileGeom<BN, true>::CHUNKS) * 16},
      {2 * (size_t)(TileGeom<BM, true>::CHUNKS + TileGeom<BN, false>::CHUNKS) * 16,
       2 * (size_t)(TileGeom<BM, true>::CHUNKS + TileGeom<BN, true>::CHUNKS) * 16}};
  const size_t pipe = pipe_of[akc][bkc];
  const size_t slabs = NW * 32 * (size_t)(BN / (NW / 2) + 4) * sizeof(float);
  const size_t lds = pipe > slabs ? pipe : slabs;
  const bool epi = a.bias != nullptr || a.residual != nullptr || a.act != NBK_ACT_NONE;
#define NBK_LAUNCH_BF16(AK, BK_)                                                              \
  do {                                                                                        \
    if (epi) NBK_LAUNCH_BF16_E(AK, BK_, true);                                                \
    else NBK_LAUNCH_BF16_E(AK, BK_, false);                                                   \
  } while (0)
#define NBK_LAUNCH_BF16_E(AK, BK_, EP)                                                        \
  do {                                                                                        \
    auto kern = gemm_bf16_kernel<BM, BN, AK, BK_, EP, NW>;                              \
    static bool attr_set = false; /* idempotent, so a race only repeats the call */          \
    if (!attr_set) {                                                                          \
      NBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                  (int)lds));                                                 \
      attr_set = true;                                                                        \
    }                                                                                         \
    hipLaunchKernelGGL(kern, grid, dim3(NW * 64), lds, st, g);                                \
  } while (0)
  if (akc && bkc) NBK_LAUNCH_BF16(true, true);
  else if (akc && !bkc) NBK_LAUNCH_BF16(true, false);
  else if (!akc && bkc) NBK_LAUNCH_BF16(false, true);
  else NBK_LAUNCH_BF16(false, false);
#undef NBK_LAUNCH_BF16
#undef NBK_LAUNCH_BF16_E
  return nbk_check_launch("gemm_bf16_kernel");
}

// MI16: whether two K-contiguous operands are multiplied with the 16 x 16 x 32 instruction (the other
// layouts always are).
template <int BM, int BN, int NW, int KSS, bool MI16, int STAGES = 2>
static int launch_bf16_dl(const GemmArgs& a, bool akc, bool bkc, int64_t batch, hipStream_t st) {
  GemmArgs g = a;
  g.tiles_m = (int)((a.M + BM - 1) / BM);
  g.tiles_n = (int)((a.N + BN - 1) / BN);
  dim3 grid((unsigned)(g.tiles_m * g.tiles_n), (unsigned)batch);
  const size_t pipe = STAGES * (size_t)(BM + BN) * 8 * 16;
  const size_t slabs = NW * 32 * (size_t)(BN / (NW / 2) + 4) * sizeof(float);
  const size_t lds = pipe > slabs ? pipe : slabs;
  const int epi = (a.residual != nullptr || a.act != NBK_ACT_NONE) ? 2 : (a.bias != nullptr ? 1 : 0);
#define NBK_LAUNCH_DL(AK, BK_, EP)                                                            \
  do {                                                                                        \
    auto kern = gemm_bf16_dl_kernel<BM, BN, AK, BK_, EP, NW, KSS, MI16 || !(AK && BK_), false, STAGES>; \
    static bool attr_set = false; /* idempotent, so a race only repeats the call */          \
    if (!attr_set) {                                                                          \
      NBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                  (int)lds));                                                 \
      attr_set = true;                                                                        \
    }                                                                                         \
    hipLaunchKernelGGL(kern, grid, dim3(NW * 64), lds, st, g);                                \
  } while (0)
#define NBK_LAUNCH_DL2(AK, BK_)                                                               \
  do {                                                                                        \
    if (epi == 2) NBK_LAUNCH_DL(AK, BK_, 2);                                                  \
    else if (epi == 1) NBK_LAUNCH_DL(AK, BK_, 1);                                             \
    else NBK_LAUNCH_DL(AK, BK_, 0);                                                           \
  } while (0)
  if (akc && bkc) NBK_LAUNCH_DL2(true, true);
  else if (akc && !bkc) NBK_LAUNCH_DL2(true, false);
  else if (!akc && bkc) NBK_LAUNCH_DL2(false, true);
  else NBK_LAUNCH_DL2(false, false);
#undef NBK_LAUNCH_DL
#undef NBK_LAUNCH_DL2
  return nbk_check_launch("gemm_bf16_dl_kernel");
}

// The same launch with the column sums of B as a second result (both operands row-contiguous,
// no epilogue: the weight gradient x^T dy beside the bias gradient).
template <int BM, int BN, int NW, int STAGES = 2>
static int launch_bf16_dl_colsum(const GemmArgs& a, int64_t batch, hipStream_t st) {
  GemmArgs g = a;
  g.tiles_m = (int)((a.M + BM - 1) / BM);
  g.tiles_n = (int)((a.N + BN - 1) / BN);
  dim3 grid((unsigned)(g.tiles_m * g.tiles_n), (unsigned)batch);
  const size_t pipe = STAGES * (size_t)(BM + BN) * 8 * 16;
  const size_t slabs = NW * 32 * (size_t)(BN / (NW / 2) + 4) * sizeof(float);
  const size_t lds = pipe > slabs ? pipe : slabs;
  auto kern = gemm_bf16_dl_kernel<BM, BN, false, false, 0, NW, 1, true, true, STAGES>;
  static bool attr_set = false; /* idempotent, so a race only repeats the call */
  if (!attr_set) {
    NBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set = true;
  }
  hipLaunchKernelGGL(kern, grid, dim3(NW * 64), lds, st, g);
  return nbk_check_launch("gemm_bf16_dl_kernel (column sums)");
}

template <int T, int WK>
static int launch_f32(const GemmArgs& args, bool akc, bool bkc, int64_t batch, hipStream_t st) {
  GemmArgs a = args;
  const int64_t tiles_m = (a.M + T - 1) / T, tiles_n = (a.N + T - 1) / T;
  NBK_REQUIRE(tiles_m * tiles_n <= 0x7fffffffLL, "gemm: launch too large");
  a.tiles_m = (int)tiles_m;
  a.tiles_n = (int)tiles_n;
  const dim3 grid((unsigned)(tiles_m * tiles_n), (unsigned)batch);
#define NBK_LAUNCH_F32(AK, BK_)                                                                              \
  do {                                                                                                       \
    auto kern = gemm_f32_kernel<AK, BK_, T, WK>;                                                             \
    constexpr size_t lds = gemm_f32_lds<AK, BK_, T, WK>();                                                   \
    static bool attr_set = false; /* idempotent, so a race only repeats the call */                          \
    if (!attr_set) {                                                                                         \
      NBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)); \
      attr_set = true;                                                                                       \
    }                                                                                                        \
    hipLaunchKernelGGL(kern, grid, dim3(64 * WK), lds, st, a);                                               \
  } while (0)
  if (akc && bkc) NBK_LAUNCH_F32(true, true);
  else if (akc) NBK_LAUNCH_F32(true, false);
  else if (bkc) NBK_LAUNCH_F32(false, true);
  else NBK_LAUNCH_F32(false, false);
#undef NBK_LAUNCH_F32
  return nbk_check_launch("gemm_f32_kernel");
}

template <int BM, int BN, int NWM, int NWN, int NM>
static int launch_f32_split(const GemmArgs& args, bool akc, bool bkc, int64_t batch, hipStream_t st) {
  GemmArgs a = args;
  const int64_t tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
  NBK_REQUIRE(tiles_m * tiles_n <= 0x7fffffffLL, "gemm: launch too large");
  a.tiles_m = (int)tiles_m;
  a.tiles_n = (int)tiles_n;
  const dim3 grid((unsigned)(tiles_m * tiles_n), (unsigned)batch);
  const size_t lds = 2 * (size_t)(BM + BN) * 12 * 16;
  const bool full = a.C2 || a.residual || a.act == NBK_ACT_GELU;
#define NBK_LAUNCH_SPLIT(AK, BK_, F)                                                                     \
  do {                                                                                                   \
    auto kern = gemm_f32_split_kernel<BM, BN, NWM, NWN, NM, AK, BK_, F>;                                 \
    static bool attr_set = false; /* idempotent, so a race only repeats the call */                     \
    if (!attr_set) {                                                                                     \
      NBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)); \
      attr_set = true;                                                                                   \
    }                                                                                                    \
    hipLaunchKernelGGL(kern, grid, dim3(NWM * NWN * 64), lds, st, a);                                    \
  } while (0)
#define NBK_LAUNCH_SPLIT2(AK, BK_)                                 \
  do {                                                             \
    if (full) NBK_LAUNCH_SPLIT(AK, BK_, true);                     \
    else NBK_LAUNCH_SPLIT(AK, BK_, false);                         \
  } while (0)
  if (akc && bkc) NBK_LAUNCH_SPLIT2(true, true);
  else if (akc) NBK_LAUNCH_SPLIT2(true, false);
  else if (bkc) NBK_LAUNCH_SPLIT2(false, true);
  else NBK_LAUNCH_SPLIT2(false, false);
#undef NBK_LAUNCH_SPLIT2
#undef NBK_LAUNCH_SPLIT
  return nbk_check_launch("gemm_f32_split_kernel");
}

// What the products of one A have of their own (nbk_gemm_members).
struct GemmMembers { int n; const void* const* B; const void* const* bias; void* const* C; };

// Checks a description and fills the kernels' arguments.
static int gemm_prepare(const nbk_gemm_desc* d, const GemmMembers& own, GemmArgs& a) {
  NBK_REQUIRE(d != nullptr, "gemm: null descriptor");
  NBK_REQUIRE(d->A && d->B && d->C, "gemm: null operand pointer");
  NBK_REQUIRE(d->M > 0 && d->N > 0 && d->K > 0, "gemm: empty problem %lld x %lld x %lld",
              (long long)d->M, (long long)d->N, (long long)d->K);
  NBK_REQUIRE(d->batch >= 1 && d->batch <= 65535, "gemm: batch %lld out of range",
              (long long)d->batch);
  NBK_REQUIRE(d->dtype_ab == NBK_F32 || d->dtype_ab == NBK_BF16, "gemm: operand dtype %d",
              d->dtype_ab);
  NBK_REQUIRE(d->dtype_c == NBK_F32 || d->dtype_c == NBK_BF16, "gemm: result dtype %d",
              d->dtype_c);
  NBK_REQUIRE(d->dtype_ab == NBK_BF16 || d->dtype_c == NBK_F32,
              "gemm: fp32 operands need an fp32 result");
  NBK_REQUIRE(d->a_rs == 1 || d->a_cs == 1, "gemm: A needs a unit stride (rs=%lld, cs=%lld)",
              (long long)d->a_rs, (long long)d->a_cs);
  NBK_REQUIRE(d->b_rs == 1 || d->b_cs == 1, "gemm: B needs a unit stride (rs=%lld, cs=%lld)",
              (long long)d->b_rs, (long long)d->b_cs);
  NBK_REQUIRE(d->ldc >= d->N, "gemm: ldc %lld < N %lld", (long long)d->ldc, (long long)d->N);
  NBK_REQUIRE(d->batch_reduce == 0, "gemm: batch_reduce is folded into K by the caller");
  const int members = own.n;
  NBK_REQUIRE(members == 0 || (d->batch == 1 && d->residual == nullptr && d->C_aux == nullptr && d->colsum == nullptr &&
                               d->n_terms == 0 && d->k_last == 0),
              "gemm: several products of one A go without batches, residual, second result, column sums, "
              "further operand pairs and k_last");
  const int64_t batch = members > 0 ? members : d->batch;
  a = {};
  a.A = d->A; a.B = d->B; a.C = d->C; a.bias = d->bias; a.residual = d->residual;
  a.M = d->M; a.N = d->N; a.K = d->K;
  a.a_rs = d->a_rs; a.a_cs = d->a_cs; a.b_rs = d->b_rs; a.b_cs = d->b_cs; a.ldc = d->ldc;
  if (members == 0) {  // (the products of one A have one A and their own pointers to the rest)
    a.a_bs = d->a_bs; a.b_bs = d->b_bs; a.c_bs = d->c_bs;
  }
  a.batch_inner = d->batch_inner > 1 ? d->batch_inner : 1;
  NBK_REQUIRE(d->batch % a.batch_inner == 0, "gemm: batch %lld is not a multiple of batch_inner %lld",
              (long long)d->batch, (long long)a.batch_inner);
  a.a_bs2 = a.batch_inner > 1 ? d->a_bs2 : 0;
  a.b_bs2 = a.batch_inner > 1 ? d->b_bs2 : 0;
  a.c_bs2 = a.batch_inner > 1 ? d->c_bs2 : 0;
  a.dtype_c = d->dtype_c; a.act = d->act; a.alpha = d->alpha;
  // A result beyond the 256 MiB last-level cache does not survive until its consumer runs: it is
  // streamed (non-temporal stores), which leaves the cache to the operands.  Smaller results are
  // stored normally: measured inside the decoder step, streaming them takes as much from the
  // kernels that read them next as it gives the product.
  a.c_stream = d->M * d->N * batch * (d->dtype_c == NBK_F32 ? 4 : 2) > (256ll << 20) ? 1 : 0;
  NBK_REQUIRE(d->aux_op == NBK_AUX_NONE || d->aux_op == NBK_AUX_ACT_GRAD, "gemm: aux_op %d", d->aux_op);
  NBK_REQUIRE((d->aux_op == NBK_AUX_NONE) == (d->C_aux == nullptr),
              "gemm: C_aux and aux_op go together");
  NBK_REQUIRE(d->aux_op == NBK_AUX_NONE || (d->act != NBK_ACT_NONE && d->residual == nullptr),
              "gemm: the derivative of the activation needs an activation and no residual");
  a.C2 = d->C_aux;
  NBK_REQUIRE(d->residual_op == NBK_RES_ADD || d->residual_op == NBK_RES_MUL,
              "gemm: residual_op %d", d->residual_op);
  a.res_mul = d->residual_op == NBK_RES_MUL;
  a.colsum = d->colsum;
  // (a slice longer than K would read behind both operands)
  NBK_REQUIRE(d->k_last >= 0 && d->k_last <= d->K && (d->k_last == 0 || d->n_terms == 0),
              "gemm: k_last %d (at most K = %lld, and 0 with more operand pairs)", d->k_last, (long long)d->K);
  a.k_last = d->k_last;
  // K-contiguous when the stride along k is 1 (ties: a single row / column counts as K-contiguous)
  const bool akc = d->a_cs == 1;
  const bool bkc = d->b_rs == 1;
  NBK_REQUIRE(d->n_terms >= 0 && d->n_terms <= NBK_GEMM_MAX_TERMS, "gemm: n_terms %d", d->n_terms);
  const bool tail = d->n_terms > 0;
  if (tail) {
    NBK_REQUIRE(d->dtype_ab == NBK_BF16 && batch == 1 && d->colsum == nullptr,
                "gemm: more operand pairs go with one bf16 product without column sums");
    for (int i = 0; i < d->n_terms; ++i) {
      const nbk_gemm_term& t = d->term[i];
      NBK_REQUIRE(t.A && t.B && t.K > 0, "gemm: term %d is empty", i);
      NBK_REQUIRE(t.a_rs == 1 || t.a_cs == 1, "gemm: A of term %d needs a unit stride", i);
      NBK_REQUIRE(t.b_rs == 1 || t.b_cs == 1, "gemm: B of term %d needs a unit stride", i);
    }
  }
  const int esz = d->dtype_ab == NBK_F32 ? 4 : 2;
  auto vec_ok = [&](const void* p, int64_t other_stride, int64_t bs, int64_t bs2) {
    const int64_t q = 16 / esz;
    return ((uintptr_t)p % 16 == 0) && (other_stride % q == 0) && (bs % q == 0) && (bs2 % q == 0);
  };
  a.a_vec = vec_ok(d->A, akc ? d->a_rs : d->a_cs, a.a_bs, a.a_bs2);
  a.b_vec = vec_ok(d->B, bkc ? d->b_cs : d->b_rs, a.b_bs, a.b_bs2);
  const int esz_c = d->dtype_c == NBK_F32 ? 4 : 2;
  a.n_members = members;
  for (int i = 0; i < members; ++i) {
    NBK_REQUIRE(own.B[i] && own.C[i] && ((uintptr_t)own.C[i] - (uintptr_t)d->C) % 16 == 0, "gemm: product %d of one A", i);
    a.member[i] = {own.B[i], own.bias[i], (int64_t)((intptr_t)own.C[i] - (intptr_t)d->C) / esz_c};
    if (own.bias[i]) a.bias = own.bias[i];  // (whether there is one at all)
    a.b_vec = a.b_vec && (uintptr_t)own.B[i] % 16 == 0;
  }
  // (checked before any kernel is chosen: no path may take the product and drop the sums)
  NBK_REQUIRE(d->colsum == nullptr || (d->dtype_ab == NBK_BF16 && !akc && !bkc),
              "gemm: column sums need bf16 operands that are both row-contiguous (a_rs == b_cs == 1)");
  return NBK_OK;
}

// Whether the direct-to-LDS kernels take a product.
static bool gemm_direct(const nbk_gemm_desc* d, const GemmArgs& a) {
  // (they keep per-lane byte offsets within a tile in 32 bits: 256 rows or 64 k-rows times the stride)
  const bool akc = d->a_cs == 1, bkc = d->b_rs == 1;
  const int64_t a_stride = akc ? d->a_rs : d->a_cs, b_stride = bkc ? d->b_cs : d->b_rs;
  const bool k_whole = d->K % 64 == 0 && d->k_last % 64 == 0;
  return a.a_vec && a.b_vec && (k_whole || (!akc && !bkc && d->n_terms == 0)) && (akc || d->M % 8 == 0) &&
         (bkc || d->N % 8 == 0) && d->M >= 8 && d->N >= 8 &&
         a_stride >= 0 && b_stride >= 0 && a_stride < (1 << 22) && b_stride < (1 << 22);
}

// How a float32 product is added up: tiles of 16 or 32 by so many waves, each with a share of K, on the float32
// instruction, or out of bf16 parts.  A function of the product alone: products that share a launch (nbk_gemm_members,
// nbk_gemm_group) have the sums they have by themselves.
enum F32Form { F32_16_BY_16, F32_16_BY_8, F32_32_BY_8, F32_32_BY_4, F32_PARTS };
static F32Form gemm_f32_form(int64_t M, int64_t N, int64_t K, int64_t batch) {
  // Out of bf16 parts where a launch gives most CUs a tile of 64 x 64; below that the K loop of one workgroup
  // is what a launch waits for, and four waves that share a fragment of 32 x 32 on the float32
  // instruction have the shorter one.  us, 32 x 32 / 64 x 64 out of parts: 1024 x 512 x 512 (128 tiles of 64)
  // 12.9 / 15.9, 512 x 2048 x 1024 (256) 34 / 27 and as x^T dy 40 / 27, 1024 x 1024 x 200 (256) 15.1 / 10.3.
  // Tiles of 64 that are half padding are no more work than two of 32: 300 x (20 x 20 x 64) 4.8 / 7.4, 128 x (32 x 128 x
  // 64) 5.1 / 6.9, 32 x 16384 x 1024 20 / 26, 64 x (16 x 224 x 704) 16.5 / 20; past two of 32 to a CU the two are even (8 x
  // 32768 x 256 12.6 / 12.5, 64 x (40 x 224 x 704) 27 / 21).
  auto tiles = [&](int64_t edge) { return ((M + edge - 1) / edge) * ((N + edge - 1) / edge) * batch; };
  const int64_t cus = nbk_num_cus(), t16 = tiles(16), t32 = tiles(32);
  if (tiles(64) * 4 >= cus * 3 && t32 > 2 * cus) return F32_PARTS;
  // The float32 instruction does 256 operations a cycle and CU, so a tile's K loop on one CU is bound by it:
  // tiles of 16 x 16 while two to a CU hold the result spread it over four times as many.  us, tiles of 32
  // by four waves / 16 by eight: 128 x 256 x 784 (128 tiles of 16) 10.8 / 6.1, 300 x 300 x 300 (361) 7.0 / 5.6,
  // 2048 x 64 x 1024 (512) 12.2 / 8.2, 784 x 256 x 128 (784) 4.8 / 5.8; the longest contractions by sixteen waves:
  // 128 x 128 x 4096 36.7 / 15.6 / 13.3.  Tiles of 32 by eight waves, where a CU holds all its workgroups and
  // a K tile of 128 is filled: 512 x 512 x 1024 (256 tiles) 12.0 / 10.8, 1024 x 512 x 2048 (512) 32.1 / 31.1 (K-contiguous
  // 28.9 / 26.5); 64 x (96 x 64 x 96) (384) 6.2 / 6.9, 16 x (300 x 64 x 300) (320) 9.0 / 9.4.
  if (t16 <= 2 * cus) return t16 <= cus && K >= 2048 ? F32_16_BY_16 : F32_16_BY_8;
  return K >= 128 && (t32 <= cus || (t32 <= 2 * cus && K % 128 == 0)) ? F32_32_BY_8 : F32_32_BY_4;
}

// LDS of gemm_skinny_n_kernel: the partial sums of its waves, and a copy of a B that is not K-contiguous, in rows of so
// many 16-byte chunks.
constexpr size_t SKN_SUMS = SKN_WAVES * 16 * 64 * sizeof(float);
static int skn_pitch(int64_t N) { return N <= 8 ? 1 : N <= 16 ? 2 : 4; }
static size_t skn_stage(int64_t N, int64_t K) { return (size_t)K * skn_pitch(N) * 16 + 64; }
// Whether gemm_skinny_n_kernel takes a product.  Planner._few_columns (backend/planner.py) asks the same.
static bool gemm_few_columns(const nbk_gemm_desc* d, const GemmArgs& a, int64_t batch) {
  const bool akc = d->a_cs == 1, bkc = d->b_rs == 1;
  // (few rows too, where a workgroup's share of B is small, us on this kernel / on 64 x 64 tiles: 1000 x 8 x 1024
  // 4.4 / 8.1, 1000 x 8 x 4096 8.3 / 20.3, 1000 x 32 x 2048 6.9 / 11.8; and many rows until a workgroup's copy of a
  // B of eight columns fills the LDS: 8192 x 8 x 4096 18.9 / 20.3, 20000 x 8 x 4096 41.0 / 31.7)
  const bool tall = d->M >= 1024 ? d->M <= 8192 || bkc || d->N > 8 || d->K < 4096
                                 : d->M >= 16 && d->K * (d->N <= 16 ? 1 : 2) <= 4096;
  return d->n_terms == 0 && d->k_last == 0 && d->dtype_ab == NBK_BF16 && d->N <= 32 && tall && d->K >= 256 && d->K % 64 == 0 &&
         akc && a.a_vec && batch == 1 && d->bias == nullptr && d->residual == nullptr && d->act == NBK_ACT_NONE &&
         a.b_vec && (bkc || (d->N % 8 == 0 && SKN_SUMS + skn_stage(d->N, d->K) <= 160 * 1024 - 512)) &&
         (d->M + 31) / 32 <= 0x7fffffff;
}

static int gemm_launch(const nbk_gemm_desc* d, const GemmMembers& own, void* stream) {
  GemmArgs a;
  { const int rc = gemm_prepare(d, own, a); if (rc != NBK_OK) return rc; }
  hipStream_t st = (hipStream_t)stream;
  const int64_t batch = own.n > 0 ? own.n : d->batch;
  const bool akc = d->a_cs == 1, bkc = d->b_rs == 1, tail = d->n_terms > 0;
  if (gemm_few_columns(d, a, batch)) {
    // 32 rows per workgroup, K split over its eight waves
    const int pitch_chunks = skn_pitch(d->N);
    dim3 grid((unsigned)((d->M + 31) / 32));
    if (bkc) {
      hipLaunchKernelGGL((gemm_skinny_n_kernel<true>), grid, dim3(SKN_WAVES * 64), SKN_SUMS, st, a, pitch_chunks);
    } else {
      static bool attr_set = false; /* idempotent, so a race only repeats the call */
      if (!attr_set) {
        NBK_HIP(hipFuncSetAttribute((const void*)gemm_skinny_n_kernel<false>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        attr_set = true;
      }
      hipLaunchKernelGGL((gemm_skinny_n_kernel<false>), grid, dim3(SKN_WAVES * 64), SKN_SUMS + skn_stage(d->N, d->K), st,
                         a, pitch_chunks);
    }
    return nbk_check_launch("gemm_skinny_n_kernel");
  }
  if (!tail && d->k_last == 0 && d->dtype_ab == NBK_BF16 && d->K <= 16 && akc && batch == 1 && d->N % 8 == 0 &&
      d->ldc % 8 == 0 && ((uintptr_t)d->C & 15) == 0 && ((uintptr_t)d->residual & 15) == 0 &&
      (d->K == 16 ? a.a_vec : d->K == 8 && (d->a_rs % 8 == 0) && ((uintptr_t)d->A & 15) == 0)) {
    // (the vector path reads whole 16-byte pieces of A rows: K = 16 or 8)
    a.a_vec = 1;
    // (K-contiguous B: whole fragments from memory; row-contiguous B: whole row pieces into LDS)
    a.b_vec = bkc ? (d->K == 16 ? a.b_vec : (d->b_cs % 8 == 0) && ((uintptr_t)d->B & 15) == 0)
                  : (d->b_cs == 1 && d->b_rs % 8 == 0 && ((uintptr_t)d->B & 15) == 0);
    a.tiles_m = (int)((d->M + 127) / 128);
    a.tiles_n = (int)((d->N + 127) / 128);
    dim3 grid((unsigned)(a.tiles_m * a.tiles_n));
    const size_t lds = 4 * 32 * (size_t)(64 + 4) * sizeof(float) + 16 * 256;  // slabs + a B piece
    // 0 plain; 3 a bias and / or an added residual (the adapter's update on top of the base
    // product: all memory traffic, so the lean epilogue that keeps four waves per SIMD); 2 the rest
    const bool any = a.bias != nullptr || a.residual != nullptr || a.act != NBK_ACT_NONE;
    // (4: the same with the residual requested before the operands -- bf16 results only)
    const int epi = !any ? 0 : ((a.act == NBK_ACT_NONE && a.C2 == nullptr && !a.res_mul)
                                    ? (a.residual != nullptr && d->dtype_c == NBK_BF16 ? 4 : 3) : 2);
#define NBK_LAUNCH_SKK(BK_)                                                                        \
  do {                                                                                             \
    if (epi == 0) hipLaunchKernelGGL((gemm_skinny_k_kernel<BK_, 0>), grid, dim3(256), lds, st, a); \
    else if (epi == 4) hipLaunchKernelGGL((gemm_skinny_k_kernel<BK_, 4>), grid, dim3(256), lds, st, a); \
    else if (epi == 3) hipLaunchKernelGGL((gemm_skinny_k_kernel<BK_, 3>), grid, dim3(256), lds, st, a); \
    else hipLaunchKernelGGL((gemm_skinny_k_kernel<BK_, 2>), grid, dim3(256), lds, st, a);         \
  } while (0)
    if (bkc) NBK_LAUNCH_SKK(true);
    else NBK_LAUNCH_SKK(false);
#undef NBK_LAUNCH_SKK
    return nbk_check_launch("gemm_skinny_k_kernel");
  }
  if (d->dtype_ab == NBK_BF16) {
    const bool fast = gemm_direct(d, a);
    if (tail) {
      // In the accumulator of the direct-to-LDS kernels when every pair is laid out like A and B
      // and 16-byte aligned: shallow pairs (one K tile each, at most two) and deep pairs with
      // exactly the strides of A and B (at most two); otherwise one product after the other,
      // each adding itself to the result so far (plain products only: an epilogue would have to
      // wait for the last one).
      bool inside = fast && d->M >= 128 && d->N >= 128;
      a.n_shallow = 0;
      a.n_deep = 0;
      for (int i = 0; inside && i < d->n_terms; ++i) {
        const nbk_gemm_term& t = d->term[i];
        const bool tkc_a = t.a_cs == 1, tkc_b = t.b_rs == 1;
        const int64_t sa = tkc_a ? t.a_rs : t.a_cs, sb = tkc_b ? t.b_cs : t.b_rs;
        if (tkc_a != akc || tkc_b != bkc || ((uintptr_t)t.A & 15) || ((uintptr_t)t.B & 15) || sa % 8 ||
            sb % 8 || sa < 0 || sb < 0 || sa >= (1 << 22) || sb >= (1 << 22)) {
          inside = false;
        } else if (t.K <= 64 && t.K % 8 == 0 && a.n_shallow < 2) {
          GemmArgs::Shallow& sh = a.shallow[a.n_shallow++];
          sh.A = t.A; sh.B = t.B; sh.K = t.K;
          sh.a_rs = t.a_rs; sh.a_cs = t.a_cs; sh.b_rs = t.b_rs; sh.b_cs = t.b_cs;
        } else if (t.K % 64 == 0 && a.n_deep < 2 && t.a_rs == d->a_rs && t.a_cs == d->a_cs &&
                   t.b_rs == d->b_rs && t.b_cs == d->b_cs) {
          GemmArgs::Deep& dp = a.deep[a.n_deep++];
          dp.A = t.A; dp.B = t.B; dp.K = t.K;
        } else {
          inside = false;
        }
      }
      if (!inside) {
        NBK_REQUIRE(d->bias == nullptr && d->residual == nullptr && d->act == NBK_ACT_NONE &&
                        d->C_aux == nullptr && d->alpha == 1.f,
                    "gemm: operand pairs outside the direct kernels' conditions go with a plain "
                    "product only");
        nbk_gemm_desc one = *d;
        one.n_terms = 0;
        int rc = nbk_gemm(&one, stream);
        for (int i = 0; rc == NBK_OK && i < d->n_terms; ++i) {
          const nbk_gemm_term& t = d->term[i];
          one.A = t.A; one.B = t.B; one.K = t.K;
          one.a_rs = t.a_rs; one.a_cs = t.a_cs; one.b_rs = t.b_rs; one.b_cs = t.b_cs;
          one.residual = d->C;  // (every kernel reads a residual element in the lane that writes it)
          one.residual_op = NBK_RES_ADD;
          rc = nbk_gemm(&one, stream);
        }
        return rc;
      }
    }
    // 64 x 64 tiles while two of them per CU hold the whole result: such a launch is bound by the
    // latency of its K loop, not by the LDS reads a small tile repeats (a wave reads four fragments
    // for four MFMAs, the 128 x 128 tile eight for sixteen).  Measured on operands in the nearest cache,
    // 64 / 128: 1998 x 512 x 512 6.3 / 9.5 us, 512 x 512 x 1998 (x^T dy) 12.4 / 20.5, 1800 x 1024 x 1024 (464
    // small tiles) 11.2 / 14.4; past two per CU it turns: 1000 x 4096 x 1024 (1024 small tiles) 17.1 / 14.9.
    // A batch of products of one large tile each is the exception from one small tile per CU on: the four
    // small ones lie on different XCDs, and each fetches its part of the operands again.  It shows where
    // a row-contiguous operand ends inside a tile, whose rows lie across cache lines (90 x (104 x 104 x
    // 512) as x^T dy 14.0 / 10.4, x 128 7.1 / 6.3), and on long contractions (128 x (128 x 128 x 512)
    // 13.5 / 12.1, x 128 7.2 / 7.5).
    const bool ragged = (!akc && d->M % 64 != 0) || (!bkc && d->N % 64 != 0);
    const int64_t tiles_64 = ((d->M + 63) / 64) * ((d->N + 63) / 64) * batch;
    const bool one_each = batch > 1 && d->M <= 128 && d->N <= 128 && tiles_64 > 256 &&
                          (d->M > 64 || d->N > 64) &&
                          ((ragged && d->K >= 128) || (d->K >= 512 && d->M % 64 == 0 && d->N % 64 == 0));
    const bool small = tiles_64 <= 512 && !one_each;
    // Four tile buffers where a launch leaves the LDS for them: a copy requested one tile ahead takes
    // longer than the tile's few instructions, and a K loop of one workgroup per CU waited for every
    // one.  Two against four buffers, us: 64 x 64 tiles 1024 x 1024 x 1024 12.0 / 9.0 (nn), 11.8 / 8.2 (xT
    // dy), 520 x 520 x 768 9.8 / 7.7, 1000 x 1024 x 4096 34.5 / 21.6; on short contractions the requests in
    // front of the loop cost more (1024 x 1024 x 512 5.7 / 5.8, x 256 4.7 / 4.9).  Two small tiles per CU are
    // one of 64 x 128 with its four buffers: 1800 x 1024 x 1024 13.0 / 11.4, x 512 8.9 / 8.6, x 384 7.65 / 7.73.
    // 128 x 128 tiles, where all run at once: 1800 x 2048 x 1024 17.7 / 15.3, x 384 10.9 / 10.5, x 256 9.3 / 9.3.
    const int64_t cus = nbk_num_cus();
    const bool deep = d->K > 512;
    const bool wide = tiles_64 > cus && d->K >= 512 && d->N > 64;
    const bool one_round = ((d->M + 127) / 128) * ((d->N + 127) / 128) * batch <= cus && d->K > 256;
    if (d->colsum != nullptr) {
      NBK_REQUIRE(fast && !akc && !bkc && d->bias == nullptr &&
                      d->residual == nullptr && d->act == NBK_ACT_NONE && d->alpha == 1.f,
                  "gemm: column sums go with a plain bf16 product of two row-contiguous, 16-byte "
                  "aligned operands (M %% 8 == 0, N %% 8 == 0)");
      if (small && wide) return launch_bf16_dl_colsum<64, 128, 4, 4>(a, batch, st);
      if (small) return deep ? launch_bf16_dl_colsum<64, 64, 4, 4>(a, batch, st)
                             : launch_bf16_dl_colsum<64, 64, 4>(a, batch, st);
      return one_round ? launch_bf16_dl_colsum<128, 128, 4, 4>(a, batch, st)
                       : launch_bf16_dl_colsum<128, 128, 4>(a, batch, st);
    }
    if (!fast) return launch_bf16<128, 128>(a, akc, bkc, batch, st);
    // 256 x 256 tiles run at about twice the rate of 128 x 128 ones per CU, one workgroup
    // per CU at a time: take them when the rounds of workgroups they need are at least
    // 60 % full (256 tiles on 256 CUs is the ideal case, 128 or 300 tiles are not).
    const int64_t big_tiles = ((d->M + 255) / 256) * ((d->N + 255) / 256) * batch;
    const int64_t rounds = (big_tiles + cus - 1) / cus;
    // (a K loop of one or two iterations is all prologue and epilogue: there two co-resident
    // 128 x 128 workgroups per CU overlap better than one 256 x 256)
    // (eight waves on the big tile: 8-16 % faster than four on every shape measured)
    if (big_tiles * 10 >= rounds * cus * 6 && d->M >= 256 && d->N >= 256 && d->K > 128)
      return launch_bf16_dl<256, 256, 8, 1, true>(a, akc, bkc, batch, st);
    if (small && wide) return launch_bf16_dl<64, 128, 4, 1, true, 4>(a, akc, bkc, batch, st);
    if (small) return deep ? launch_bf16_dl<64, 64, 4, 1, true, 4>(a, akc, bkc, batch, st)
                           : launch_bf16_dl<64, 64, 4, 1, true>(a, akc, bkc, batch, st);
    // (a 256 x 128 tile was measured and is no faster than 128 x 128 on mid-sized problems:
    // with one workgroup per CU a short K loop is bound by load latency, and two co-resident
    // 128 x 128 workgroups hide it better)
    // (the 16 x 16 x 32 instruction is 3-8 % faster on every shape and layout of the big tile; on
    // this one it gains 4-9 % with a row-contiguous operand and loses 5-10 % with two K-contiguous)
    return one_round ? launch_bf16_dl<128, 128, 4, 1, false, 4>(a, akc, bkc, batch, st)
                     : launch_bf16_dl<128, 128, 4, 1, false>(a, akc, bkc, batch, st);
  }
  const int64_t cus = nbk_num_cus();
  switch (gemm_f32_form(d->M, d->N, d->K, d->batch)) {
    case F32_16_BY_16: return launch_f32<16, 16>(a, akc, bkc, batch, st);
    case F32_16_BY_8: return launch_f32<16, 8>(a, akc, bkc, batch, st);
    case F32_32_BY_8: return launch_f32<32, 8>(a, akc, bkc, batch, st);
    case F32_32_BY_4: return launch_f32<32, 4>(a, akc, bkc, batch, st);
    default: break;
  }
  // 128 x 128 tiles run one to a CU, two of 64 x 64 do; a round of the former does the work of two of the
  // latter in 1.7 of one's time: 4096 x 4096 x 1024 (4 rounds / 8) 197 / 251, 4096 x 1024 x 64 (1 / 2) 12.4 /
  // 14.2, 64 x (333 x 333 x 64) (3 / 5) 33 / 29, 2048 x 1024 x 1024 (1 / 1) 44 / 39.  (A sum is the same in either.)
  auto tiles = [&](int64_t edge) { return ((d->M + edge - 1) / edge) * ((d->N + edge - 1) / edge) * batch; };
  const int64_t rounds_64 = (tiles(64) + 2 * cus - 1) / (2 * cus), rounds_128 = (tiles(128) + cus - 1) / cus;
  if (rounds_128 * 17 <= rounds_64 * 10) return launch_f32_split<128, 128, 2, 4, 2>(a, akc, bkc, batch, st);
  return launch_f32_split<64, 64, 2, 2, 2>(a, akc, bkc, batch, st);
}

extern "C" int nbk_gemm(const nbk_gemm_desc* d, void* stream) { return gemm_launch(d, {}, stream); }
extern "C" int nbk_gemm_few_columns(const nbk_gemm_desc* d) {
  GemmArgs a;
  return gemm_prepare(d, {}, a) == NBK_OK && gemm_few_columns(d, a, d->batch) ? 1 : 0;
}

// ------------------------------------------------------------------ products that share a launch
// Weight gradients of small layers: each has a fraction of the workgroups the GPU holds, and nothing reads
// them before the end of a step.  A workgroup finds its product from the running counts and runs the
// body of the kernel that the product would have had to itself.  us, one after the other / together: 4096 x 8,
// 8 x 1024, 1024 x 8 and 8 x 4096 over 1000 rows in bf16 32 / 10.5; six of 512 x 512 to 512 x 2048 over 1998 rows 52 / 27, over
// 1024 rows in float32 102 / 75; the adapters of a decoder layer over 8192 rows 44 / 34.
constexpr int GEMM_GROUP_MAX = 7;
struct GemmGroup {
  int32_t n;
  int32_t first[GEMM_GROUP_MAX + 1];  // workgroups before each product
  int32_t batch[GEMM_GROUP_MAX];
  int32_t bm[GEMM_GROUP_MAX], bn[GEMM_GROUP_MAX];  // tile of each product
  GemmArgs a[GEMM_GROUP_MAX];
};
static_assert(sizeof(GemmGroup) <= 4096, "kernel arguments");
template <typename Body>
__device__ __forceinline__ void gemm_group_run(const GemmGroup& G, Body&& body) {
  int i = 0;
  while (i + 1 < G.n && (int)blockIdx.x >= G.first[i + 1]) ++i;
  const GemmArgs& g = G.a[i];
  const int local = (int)blockIdx.x - G.first[i], tiles = g.tiles_m * g.tiles_n;
  const int by = local / tiles;
  body(g, local - by * tiles, by, G.batch[i], G.bm[i]);
}
template <int BM, int BN, int STAGES>
__global__ __launch_bounds__(256) void gemm_bf16_group_kernel(const GemmGroup G) {
  gemm_group_run(G, [](const GemmArgs& g, int bx, int by, int ny, int) {
    gemm_bf16_dl_body<BM, BN, false, false, 0, 4, 1, true, true, STAGES>(g, bx, by, ny);
  });
}
// (tiles of 16 and of 32 by eight waves: one kernel for both)
template <int WK>
__global__ __launch_bounds__(64 * WK, WK > 8 ? 1 : 2) void gemm_f32_group_kernel(const GemmGroup G) {
  gemm_group_run(G, [](const GemmArgs& g, int bx, int by, int ny, int tile) {
    if constexpr (WK == 16) gemm_f32_body<false, false, 16, WK>(g, bx, by, ny);
    else if constexpr (WK == 4) gemm_f32_body<false, false, 32, WK>(g, bx, by, ny);
    else if (tile == 16) gemm_f32_body<false, false, 16, WK>(g, bx, by, ny);
    else gemm_f32_body<false, false, 32, WK>(g, bx, by, ny);
  });
}
__global__ __launch_bounds__(256) void gemm_f32_split_group_kernel(const GemmGroup G) {
  gemm_group_run(G, [](const GemmArgs& g, int bx, int by, int ny, int) {
    gemm_f32_split_body<64, 64, 2, 2, 2, false, false, false>(g, bx, by, ny);
  });
}
template <auto KERN>
static int launch_group(GemmGroup& G, int threads, size_t lds, hipStream_t st) {
  int64_t blocks = 0;
  for (int i = 0; i < G.n; ++i) {
    GemmArgs& a = G.a[i];
    a.tiles_m = (int)((a.M + G.bm[i] - 1) / G.bm[i]);
    a.tiles_n = (int)((a.N + G.bn[i] - 1) / G.bn[i]);
    G.first[i] = (int32_t)blocks;
    blocks += (int64_t)a.tiles_m * a.tiles_n * G.batch[i];
    NBK_REQUIRE(blocks <= 0x7fffffffLL, "gemm_group: launch too large");
  }
  G.first[G.n] = (int32_t)blocks;
  static bool attr_set = false; /* idempotent, so a race only repeats the call */
  if (!attr_set) {
    NBK_HIP(hipFuncSetAttribute((const void*)KERN, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set = true;
  }
  hipLaunchKernelGGL(KERN, dim3((unsigned)blocks), dim3((unsigned)threads), lds, st, G);
  return nbk_check_launch("gemm group kernel");
}
template <int BM, int BN, int STAGES>
static int launch_bf16_group(GemmGroup& G, hipStream_t st) {
  const size_t pipe = STAGES * (size_t)(BM + BN) * 8 * 16, slabs = 4 * 32 * (size_t)(BN / 2 + 4) * sizeof(float);
  for (int i = 0; i < G.n; ++i) { G.bm[i] = BM; G.bn[i] = BN; }
  return launch_group<gemm_bf16_group_kernel<BM, BN, STAGES>>(G, 256, pipe > slabs ? pipe : slabs, st);
}
template <int WK>
static int launch_f32_group(GemmGroup& G, hipStream_t st) {
  constexpr int T = WK > 8 ? 16 : 32;  // (the larger where there are two)
  return launch_group<gemm_f32_group_kernel<WK>>(G, 64 * WK, gemm_f32_lds<false, false, T, WK>(), st);
}

extern "C" int nbk_gemm_group(const nbk_gemm_desc* const* d, int32_t n, void* stream) {
  NBK_REQUIRE(d != nullptr && n > 0, "gemm_group: no products");
  for (int32_t base = 0; base < n; base += GEMM_GROUP_MAX) {
    GemmGroup G;
    G.n = n - base < GEMM_GROUP_MAX ? n - base : GEMM_GROUP_MAX;
    bool together = G.n > 1, narrow = false, deep = false, long_k = true;
    int64_t t64 = 0, t128 = 0;
    F32Form form[GEMM_GROUP_MAX];
    const int ab = d[base] != nullptr ? d[base]->dtype_ab : -1;
    for (int i = 0; i < G.n; ++i) {
      const nbk_gemm_desc* p = d[base + i];
      const int rc = gemm_prepare(p, {}, G.a[i]);
      if (rc != NBK_OK) return rc;
      // (x^T dy: both operands row-contiguous, nothing behind the product)
      together = together && p->dtype_ab == ab && p->a_cs != 1 && p->b_rs != 1 && p->n_terms == 0 && p->bias == nullptr &&
                 p->residual == nullptr && p->act == NBK_ACT_NONE && p->K > 1 &&
                 (ab == NBK_F32 || (gemm_direct(p, G.a[i]) && (p->colsum == nullptr || p->alpha == 1.f)));
      G.batch[i] = (int32_t)p->batch;
      auto tiles = [&](int64_t edge) { return ((p->M + edge - 1) / edge) * ((p->N + edge - 1) / edge) * p->batch; };
      t64 += tiles(64); t128 += tiles(128);
      form[i] = gemm_f32_form(p->M, p->N, p->K, p->batch);
      narrow = narrow || p->M <= 64 || p->N <= 64;
      deep = deep || p->K > 512;
      long_k = long_k && p->K >= 512;
    }
    int rc = NBK_OK;
    hipStream_t st = (hipStream_t)stream;
    const int64_t cus = nbk_num_cus();
    if (!together) {
      for (int i = 0; rc == NBK_OK && i < G.n; ++i) rc = nbk_gemm(d[base + i], stream);
    } else if (ab == NBK_BF16) {  // (the lines of nbk_gemm, for all products together)
      if (narrow || (t64 <= 2 * cus && !(t64 > cus && long_k)))
        rc = deep ? launch_bf16_group<64, 64, 4>(G, st) : launch_bf16_group<64, 64, 2>(G, st);
      else if (t64 <= 2 * cus) rc = launch_bf16_group<64, 128, 4>(G, st);
      else if (t128 <= cus) rc = launch_bf16_group<128, 128, 4>(G, st);
      else rc = launch_bf16_group<128, 128, 2>(G, st);
    } else {  // (those of as many waves share a launch)
      for (F32Form of : {F32_16_BY_16, F32_16_BY_8, F32_32_BY_4, F32_PARTS}) {
        GemmGroup F;
        F.n = 0;
        int last = 0;
        for (int i = 0; i < G.n; ++i) {
          if (form[i] != of && !(of == F32_16_BY_8 && form[i] == F32_32_BY_8)) continue;
          F.a[F.n] = G.a[i];
          F.bm[F.n] = F.bn[F.n] = form[i] <= F32_16_BY_8 ? 16 : form[i] == F32_PARTS ? 64 : 32;
          F.batch[F.n++] = G.batch[i];
          last = i;
        }
        if (F.n == 0) continue;
        if (F.n == 1) rc = nbk_gemm(d[base + last], stream);
        else if (of == F32_16_BY_16) rc = launch_f32_group<16>(F, st);
        else if (of == F32_16_BY_8) rc = launch_f32_group<8>(F, st);
        else if (of == F32_32_BY_4) rc = launch_f32_group<4>(F, st);
        else rc = launch_group<gemm_f32_split_group_kernel>(F, 256, 2 * (64 + 64) * 12 * 16, st);
        if (rc != NBK_OK) return rc;
      }
    }
    if (rc != NBK_OK) return rc;
  }
  return NBK_OK;
}

extern "C" int nbk_gemm_members(const nbk_gemm_desc* d, int32_t n, const void* const* B, const void* const* bias,
                                void* const* C, void* stream) {
  NBK_REQUIRE(d != nullptr && B != nullptr && bias != nullptr && C != nullptr, "gemm_members: null argument");
  NBK_REQUIRE(n >= 2 && n <= GEMM_MAX_MEMBERS, "gemm_members: %d products", n);
  nbk_gemm_desc first = *d;
  first.B = B[0];
  first.bias = bias[0];
  first.C = C[0];
  return gemm_launch(&first, {n, B, bias, C}, stream);
}

// ------------------------------------------------------------------ NF4-coded weights
// A whole weight from its codes, eight per lane.  One byte is read and two or four are written per
// weight, yet weights of a usual size take what a launch and one trip to memory and back take: 4 M
// bf16 weights 7.1 us, 1.8 TB/s where a large copy reaches 7.0.
template <typename T>
__global__ __launch_bounds__(256) void nf4_decode_kernel(const uint8_t* codes, const float* scales, T* w,
                                                         uint32_t groups, uint32_t groups_per_block) {
  __shared__ float table[16];
  if (threadIdx.x < 16) table[threadIdx.x] = nbk_nf4_levels[threadIdx.x];
  __syncthreads();
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= groups) return;
  const uint64_t raw = ((const uint64_t*)codes)[i];
  const float s = scales[i / groups_per_block];
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = table[(raw >> (8 * e)) & 15] * s;
  if constexpr (sizeof(T) == 2) {
    u32x4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      r[e] = (uint32_t)nbk_f32_to_bf16(v[2 * e]) | ((uint32_t)nbk_f32_to_bf16(v[2 * e + 1]) << 16);
    ((u32x4*)w)[i] = r;
  } else {
    ((f32x4*)w)[2 * (int64_t)i] = f32x4{v[0], v[1], v[2], v[3]};
    ((f32x4*)w)[2 * (int64_t)i + 1] = f32x4{v[4], v[5], v[6], v[7]};
  }
}

// Further operand pairs of a product that has been launched: each adds itself to the result.
static int nf4_add_terms(const nbk_gemm_nf4_desc* d, int dtype_c, int64_t N, const nbk_gemm_term* term, int n_terms,
                         void* stream) {
  for (int i = 0; i < n_terms; ++i) {
    nbk_gemm_desc p = {};
    p.A = term[i].A; p.B = term[i].B; p.C = d->C; p.residual = d->C;
    p.M = d->M; p.N = N; p.K = term[i].K;
    p.a_rs = term[i].a_rs; p.a_cs = term[i].a_cs; p.b_rs = term[i].b_rs; p.b_cs = term[i].b_cs;
    p.ldc = d->ldc; p.batch = 1; p.batch_inner = 1;
    p.dtype_ab = d->dtype; p.dtype_c = dtype_c; p.alpha = 1.f;
    const int rc = nbk_gemm(&p, stream);
    if (rc != NBK_OK) return rc;
  }
  return NBK_OK;
}

// (The update of an adapter as one more K tile of the product out of the workspace: 1000 x 1024 x 4096 with rank 8
// 17.4 + 9.2 us in two launches and 7 of the sum in a row kernel, then 18.)
static int gemm_nf4(const nbk_gemm_nf4_desc* d, bool c_f32, const nbk_gemm_term* term, int n_terms, void* stream) {
  NBK_REQUIRE(d != nullptr, "gemm_nf4: null descriptor");
  NBK_REQUIRE(n_terms >= 0 && n_terms <= NBK_GEMM_MAX_TERMS && (n_terms == 0 || (term != nullptr && d->alpha == 1.f)),
              "gemm_nf4: %d further pairs, with alpha 1 only", n_terms);
  NBK_REQUIRE(d->A && d->codes && d->scales && d->C, "gemm_nf4: null pointer");
  NBK_REQUIRE(d->M > 0 && d->w_rows > 0 && d->w_cols > 0, "gemm_nf4: empty problem");
  NBK_REQUIRE(d->dtype == NBK_BF16 || d->dtype == NBK_F32, "gemm_nf4: dtype %d", d->dtype);
  NBK_REQUIRE(d->block > 0 && d->block % 8 == 0 && d->w_cols % 8 == 0,
              "gemm_nf4: the block length (%d) and the weight's width (%lld) must be multiples of 8",
              d->block, (long long)d->w_cols);
  NBK_REQUIRE(((uintptr_t)d->codes & 7) == 0, "gemm_nf4: codes must be 8-byte aligned");
  const int dtype_c = c_f32 ? NBK_F32 : d->dtype;
  // C = A @ W (K = rows of W, N = its columns) or A @ W^T (K = columns of W, N = its rows)
  const int64_t K = d->transpose_w ? d->w_cols : d->w_rows;
  const int64_t N = d->transpose_w ? d->w_rows : d->w_cols;
  NBK_REQUIRE(d->lda >= K && d->ldc >= N, "gemm_nf4: leading dimension too small");
  // The kernels that decode while they multiply look a level up for every weight and every 128 rows of
  // A, on 128 x 128 tiles whose K loop waits for it; decoding once leaves the tile that fits the
  // product.  Measured, us, bf16 (fp32): 1000 x 1024 x 4096 274 -> 42 (688 -> 138), 16 x 1024 x 4096
  // 225 -> 40 (547 -> 55), 8192 x 4096 x 2048 627 -> 127, 200 x 128 x 128 16 -> 7.5 (25 -> 8); shorter
  // contractions are two K tiles at most and keep their single launch.
  const int64_t weights = d->w_rows * d->w_cols;
  if (d->workspace != nullptr && K >= 128 && weights / 8 < (1ll << 32) - 256) {
    NBK_REQUIRE(((uintptr_t)d->workspace & 15) == 0 && d->workspace_bytes >= weights * (d->dtype == NBK_F32 ? 4 : 2),
                "gemm_nf4: the workspace takes %lld weights on 16-byte alignment", (long long)weights);
    const uint32_t groups = (uint32_t)(weights / 8), per = (uint32_t)(d->block / 8);
    const dim3 blocks((groups + 255) / 256);
    if (d->dtype == NBK_F32)
      hipLaunchKernelGGL((nf4_decode_kernel<float>), blocks, dim3(256), 0, (hipStream_t)stream,
                         (const uint8_t*)d->codes, (const float*)d->scales, (float*)d->workspace, groups, per);
    else
      hipLaunchKernelGGL((nf4_decode_kernel<uint16_t>), blocks, dim3(256), 0, (hipStream_t)stream,
                         (const uint8_t*)d->codes, (const float*)d->scales, (uint16_t*)d->workspace, groups, per);
    const int rc = nbk_check_launch("nf4_decode_kernel");
    if (rc != NBK_OK) return rc;
    nbk_gemm_desc p = {};
    p.A = d->A; p.B = d->workspace; p.C = d->C;
    p.M = d->M; p.N = N; p.K = K;
    p.a_rs = d->lda; p.a_cs = 1;
    p.b_rs = d->transpose_w ? 1 : d->w_cols;
    p.b_cs = d->transpose_w ? d->w_cols : 1;
    p.ldc = d->ldc; p.batch = 1; p.batch_inner = 1;
    p.dtype_ab = d->dtype; p.dtype_c = dtype_c; p.alpha = d->alpha;
    if (d->dtype == NBK_BF16) {
      p.n_terms = n_terms;
      for (int i = 0; i < n_terms; ++i) p.term[i] = term[i];
      return nbk_gemm(&p, stream);
    }
    const int prc = nbk_gemm(&p, stream);
    return prc != NBK_OK ? prc : nf4_add_terms(d, dtype_c, N, term, n_terms, stream);
  }
  GemmArgs a = {};
  a.A = d->A; a.B = d->codes; a.C = d->C;
  a.M = d->M; a.N = N; a.K = K;
  a.a_rs = d->lda; a.a_cs = 1;
  // the element (k, n) of the B operand is code k * b_rs + n * b_cs of the flattened weight
  a.b_rs = d->transpose_w ? 1 : d->w_cols;
  a.b_cs = d->transpose_w ? d->w_cols : 1;
  a.ldc = d->ldc; a.batch_inner = 1;
  a.dtype_c = dtype_c; a.act = NBK_ACT_NONE; a.alpha = d->alpha;
  a.b_scales = (const float*)d->scales; a.b_block = d->block;
  a.a_vec = ((uintptr_t)d->A % 16 == 0) && (d->lda % (d->dtype == NBK_F32 ? 4 : 8) == 0);
  a.b_vec = 0;
  a.tiles_m = (int)((a.M + 127) / 128);
  a.tiles_n = (int)((a.N + 127) / 128);
  NBK_REQUIRE((int64_t)a.tiles_m * a.tiles_n <= 0x7fffffffLL, "gemm_nf4: launch too large");
  dim3 grid((unsigned)(a.tiles_m * a.tiles_n), 1);
  hipStream_t st = (hipStream_t)stream;
  const bool bkc = d->transpose_w != 0;
  if (d->dtype == NBK_F32) {
    if (bkc) hipLaunchKernelGGL((gemm_f32_nf4_kernel<true>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((gemm_f32_nf4_kernel<false>), grid, dim3(256), 0, st, a);
    const int krc = nbk_check_launch("gemm_f32_nf4_kernel");
    return krc != NBK_OK ? krc : nf4_add_terms(d, dtype_c, N, term, n_terms, stream);
  }
  const size_t pipe = 2 * (size_t)(TileGeom<128, true>::CHUNKS +
                                   (bkc ? TileGeom<128, true>::CHUNKS : TileGeom<128, false>::CHUNKS)) * 16;
  const size_t slabs = 4 * 32 * (size_t)(64 + 4) * sizeof(float);
  const size_t lds = pipe > slabs ? pipe : slabs;
#define NBK_LAUNCH_NF4(BK_)                                                                   \
  do {                                                                                        \
    auto kern = gemm_bf16_kernel<128, 128, true, BK_, false, 4, true>;                        \
    static bool attr_set = false; /* idempotent, so a race only repeats the call */          \
    if (!attr_set) {                                                                          \
      NBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                  (int)lds));                                                 \
      attr_set = true;                                                                        \
    }                                                                                         \
    hipLaunchKernelGGL(kern, grid, dim3(256), lds, st, a);                                    \
  } while (0)
  if (bkc) NBK_LAUNCH_NF4(true);
  else NBK_LAUNCH_NF4(false);
#undef NBK_LAUNCH_NF4
  const int krc = nbk_check_launch("gemm_bf16_kernel (nf4)");
  return krc != NBK_OK ? krc : nf4_add_terms(d, dtype_c, N, term, n_terms, stream);
}

extern "C" int nbk_gemm_nf4(const nbk_gemm_nf4_desc* d, void* stream) { return gemm_nf4(d, false, nullptr, 0, stream); }
extern "C" int nbk_gemm_nf4_terms(const nbk_gemm_nf4_desc* d, const nbk_gemm_term* term, int32_t n_terms, void* stream) {
  return gemm_nf4(d, false, term, n_terms, stream);
}
extern "C" int nbk_gemm_nf4_terms_f32(const nbk_gemm_nf4_desc* d, const nbk_gemm_term* term, int32_t n_terms, void* stream) {
  return gemm_nf4(d, true, term, n_terms, stream);
}
