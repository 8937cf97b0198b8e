// Data-movement kernels: strided copy (materialise a view), fill, and the
// reduction over a middle axis.
#include "nbk_common.h"

struct CopyDesc {
  int rank;
  int64_t shape[NBK_MAX_RANK];
  int64_t sstride[NBK_MAX_RANK];
  int64_t dstride[NBK_MAX_RANK];
};

// Generic path: one lane per element, index decomposed innermost-first.
template <typename T_SRC, typename T_DST, bool CONVERT>
__global__ __launch_bounds__(256) void copy_strided_kernel(const void* __restrict__ src,
                                                           void* __restrict__ dst, CopyDesc d,
                                                           int64_t total, int dts, int dtd) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * 256) {
    int64_t rem = i, so = 0, dof = 0;
    for (int k = d.rank - 1; k >= 0; --k) {
      int64_t q = rem / d.shape[k];
      int64_t r = rem - q * d.shape[k];
      so += r * d.sstride[k];
      dof += r * d.dstride[k];
      rem = q;
    }
    if (CONVERT) {
      nbk_store_from_f32(dst, dof, dtd, nbk_load_as_f32(src, so, dts));
    } else {
      ((T_DST*)dst)[dof] = ((const T_SRC*)src)[so];
    }
  }
}

// 2-D transpose-style tile through LDS for the case where the source is
// unit-stride along some axis other than the last: both sides stay coalesced.
template <typename T>
__global__ __launch_bounds__(256) void copy_tile_kernel(const T* __restrict__ src,
                                                        T* __restrict__ dst, CopyDesc d,
                                                        int ax_s /* src-contiguous axis */) {
  // tile over (ax_s, last); the remaining axes are enumerated by blockIdx.z
  __shared__ T tile[64][65];
  const int last = d.rank - 1;
  const int64_t n_s = d.shape[ax_s], n_l = d.shape[last];
  int64_t rem = blockIdx.z, so = 0, dof = 0;
  for (int k = d.rank - 1; k >= 0; --k) {
    if (k == ax_s || k == last) continue;
    int64_t q = rem / d.shape[k];
    int64_t r = rem - q * d.shape[k];
    so += r * d.sstride[k];
    dof += r * d.dstride[k];
    rem = q;
  }
  const int64_t s0 = (int64_t)blockIdx.y * 64, l0 = (int64_t)blockIdx.x * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;  // 64 x 4
  // read: lanes run along ax_s (unit stride in src)
  for (int j = ty; j < 64; j += 4) {
    int64_t s = s0 + tx, l = l0 + j;
    if (s < n_s && l < n_l) tile[j][tx] = src[so + s * d.sstride[ax_s] + l * d.sstride[last]];
  }
  __syncthreads();
  // write: lanes run along the last axis (unit stride in dst)
  for (int j = ty; j < 64; j += 4) {
    int64_t s = s0 + j, l = l0 + tx;
    if (s < n_s && l < n_l) dst[dof + s * d.dstride[ax_s] + l * d.dstride[last]] = tile[tx][j];
  }
}

extern "C" int nbk_copy_strided(const void* src, void* dst, int32_t dts, int32_t dtd, int32_t rank,
                                const int64_t* shape, const int64_t* sstride,
                                const int64_t* dstride, void* stream) {
  NBK_REQUIRE(src && dst, "copy_strided: null pointer");
  NBK_REQUIRE(rank >= 0 && rank <= NBK_MAX_RANK, "copy_strided: rank %d exceeds %d", rank,
              NBK_MAX_RANK);
  NBK_REQUIRE(nbk_dtype_size(dts) > 0 && nbk_dtype_size(dtd) > 0, "copy_strided: bad dtype");
  CopyDesc d;
  d.rank = rank;
  int64_t total = 1;
  for (int k = 0; k < rank; ++k) {
    NBK_REQUIRE(shape[k] >= 0, "copy_strided: negative extent");
    d.shape[k] = shape[k];
    d.sstride[k] = sstride[k];
    d.dstride[k] = dstride[k];
    total *= shape[k];
  }
  if (total == 0) return NBK_OK;
  hipStream_t st = (hipStream_t)stream;
  const int es = nbk_dtype_size(dts);
  if (dts == dtd && rank >= 2 && d.dstride[rank - 1] == 1 && d.sstride[rank - 1] != 1 &&
      (es == 4 || es == 2)) {
    int ax = -1;
    for (int k = rank - 2; k >= 0; --k)
      if (d.sstride[k] == 1 && d.shape[k] >= 16) { ax = k; break; }
    if (ax >= 0 && d.shape[rank - 1] >= 16) {
      int64_t nz = total / (d.shape[ax] * d.shape[rank - 1]);
      int64_t gx = (d.shape[rank - 1] + 63) / 64, gy = (d.shape[ax] + 63) / 64;
      if (nz <= 65535 && gy <= 65535) {
        dim3 grid((unsigned)gx, (unsigned)gy, (unsigned)nz);
        if (es == 4)
          hipLaunchKernelGGL(copy_tile_kernel<uint32_t>, grid, dim3(256), 0, st,
                             (const uint32_t*)src, (uint32_t*)dst, d, ax);
        else
          hipLaunchKernelGGL(copy_tile_kernel<uint16_t>, grid, dim3(256), 0, st,
                             (const uint16_t*)src, (uint16_t*)dst, d, ax);
        return nbk_check_launch("copy_tile_kernel");
      }
    }
  }
  int64_t blocks = (total + 255) / 256;
  if (blocks > 1 << 20) blocks = 1 << 20;
  dim3 grid((unsigned)blocks);
  if (dts != dtd) {
    hipLaunchKernelGGL((copy_strided_kernel<float, float, true>), grid, dim3(256), 0, st, src, dst,
                       d, total, dts, dtd);
  } else if (es == 4) {
    hipLaunchKernelGGL((copy_strided_kernel<uint32_t, uint32_t, false>), grid, dim3(256), 0, st,
                       src, dst, d, total, dts, dtd);
  } else if (es == 2) {
    hipLaunchKernelGGL((copy_strided_kernel<uint16_t, uint16_t, false>), grid, dim3(256), 0, st,
                       src, dst, d, total, dts, dtd);
  } else if (es == 8) {
    hipLaunchKernelGGL((copy_strided_kernel<uint64_t, uint64_t, false>), grid, dim3(256), 0, st,
                       src, dst, d, total, dts, dtd);
  } else {
    hipLaunchKernelGGL((copy_strided_kernel<uint8_t, uint8_t, false>), grid, dim3(256), 0, st, src,
                       dst, d, total, dts, dtd);
  }
  return nbk_check_launch("copy_strided_kernel");
}

// ---- fill -------------------------------------------------------------------
__global__ __launch_bounds__(256) void fill_kernel(void* dst, int dt, int64_t n, float v,
                                                   int64_t iv) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    if (dt == NBK_I64) ((int64_t*)dst)[i] = iv;
    else if (dt == NBK_I32) ((int32_t*)dst)[i] = (int32_t)iv;
    else nbk_store_from_f32(dst, i, dt, v);
  }
}
extern "C" int nbk_fill(void* dst, int32_t dtype, int64_t n, double value, void* stream) {
  NBK_REQUIRE(dst || n == 0, "fill: null pointer");
  NBK_REQUIRE(nbk_dtype_size(dtype) > 0, "fill: bad dtype %d", dtype);
  if (n <= 0) return NBK_OK;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(fill_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, dst,
                     dtype, n, (float)value, (int64_t)value);
  return nbk_check_launch("fill_kernel");
}

// ---- reduction over a middle axis ---------------------------------------------
// in [outer, red, inner] -> out [outer, inner].  A workgroup of 256 lanes owns a strip of
// `lx` (1 .. 256, a power of two) neighbouring pieces of the row and walks the reduced axis
// 256 / lx rows abreast; the partial sums of a column meet across lanes, then in LDS.
// What bounds it is how many workgroups there are: one CU takes rows from the other XCDs' results
// at 15 to 35 GB/s whatever it keeps in flight (4 or 8 rows per lane measured the same), and
// a wavefront that waits for one row after the other is pure latency.  So the strip is as narrow
// as it takes to give every CU work (reduce_strip).  The earlier form had strips of 64 to 256
// pieces and rows four abreast, and where the row was shorter most of its lanes idled; times in
// us, before and after, behind a kernel that has just written the operand: 128x256 fp32 10.7 / 4.5,
// 200x32 15.1 / 3.5, 27 x (74x512) bf16 15.1 / 5.4, 32 x (256x1024) bf16 65.7 / 14.1, 64x4096
// fp32 17.7 / 3.3, 50 x (196x72) 16.2 / 5.7, the four halves of a split product 4x786432 11.0 / 9.3.
// (These, and the lines in reduce_layout, from before the combining function was a template's; by themselves in
// a row 32 x (256x1024) bf16 8.0 / 3.8 since then.)
// (A long axis over few columns is cut into slices by the caller: two launches, fp32 partials
// in between.)
__device__ __forceinline__ float red_comb(float a, float b, int kind) {
  return kind == NBK_RED_SUM ? a + b : (kind == NBK_RED_MAX ? fmaxf(a, b) : fminf(a, b));
}
// A piece of a row: 16 bytes where the rows allow it, else one element.
struct RedF32x4 {
  typedef uint4 raw;
  static constexpr int N = 4;
  static __device__ __forceinline__ void unpack(const uint4 u, int, float* v) {
    v[0] = __uint_as_float(u.x); v[1] = __uint_as_float(u.y);
    v[2] = __uint_as_float(u.z); v[3] = __uint_as_float(u.w);
  }
  static __device__ __forceinline__ uint4 load(const void* p, int64_t i, int) { return ((const uint4*)p)[i]; }
};
struct RedBf16x8 {
  typedef uint4 raw;
  static constexpr int N = 8;
  static __device__ __forceinline__ void unpack(const uint4 u, int, float* v) {
    v[0] = __uint_as_float(u.x << 16); v[1] = __uint_as_float(u.x & 0xffff0000u);
    v[2] = __uint_as_float(u.y << 16); v[3] = __uint_as_float(u.y & 0xffff0000u);
    v[4] = __uint_as_float(u.z << 16); v[5] = __uint_as_float(u.z & 0xffff0000u);
    v[6] = __uint_as_float(u.w << 16); v[7] = __uint_as_float(u.w & 0xffff0000u);
  }
  static __device__ __forceinline__ uint4 load(const void* p, int64_t i, int) { return ((const uint4*)p)[i]; }
};
struct RedF32 {
  typedef float raw;
  static constexpr int N = 1;
  static __device__ __forceinline__ void unpack(const float u, int, float* v) { v[0] = u; }
  static __device__ __forceinline__ float load(const void* p, int64_t i, int) { return ((const float*)p)[i]; }
};
struct RedBf16 {
  typedef uint16_t raw;
  static constexpr int N = 1;
  static __device__ __forceinline__ void unpack(const uint16_t u, int, float* v) { v[0] = nbk_bf16_to_f32(u); }
  static __device__ __forceinline__ uint16_t load(const void* p, int64_t i, int) { return ((const uint16_t*)p)[i]; }
};
struct RedAny {
  typedef float raw;
  static constexpr int N = 1;
  static __device__ __forceinline__ void unpack(const float u, int, float* v) { v[0] = u; }
  static __device__ __forceinline__ float load(const void* p, int64_t i, int dt) { return nbk_load_as_f32(p, i, dt); }
};
constexpr int RED_FLIGHT = 8;  // rows in flight per lane

// LINE: rows of one element, read 16 bytes at a time as if N of them were a row; the N sums meet at the end.
template <typename P, int kind, bool LINE>
__device__ __forceinline__ void reduce_strip_kind(const void* __restrict__ in, void* __restrict__ out,
                                                  int dti, int dto, int64_t red, int64_t inner,
                                                  int64_t bx, int64_t o, int lxs, float* part) {
  constexpr int N = P::N;
  if constexpr (LINE) red /= N;
  const int LX = LINE ? 1 : 1 << lxs, RY = LINE ? 256 : 256 >> lxs;
  const int64_t pieces = LINE ? 1 : inner / N;
  const int64_t at = bx * LX + (threadIdx.x & (LX - 1));
  const int64_t base = o * red * pieces + (at < pieces ? at : pieces - 1);
  const float ident = kind == NBK_RED_SUM ? 0.f : (kind == NBK_RED_MAX ? -INFINITY : INFINITY);
  // CHAINS sums of a lane's rows side by side, T rows at a time: where no rows stand abreast, one sum
  // would be rounded once a row.  Error against float64 of uniform numbers, one sum / these: 64 x (1024x4099)
  // fp32 4.2e-7 / 5.0e-8, 1024 x (12x1000) 5.4e-8 / 4.0e-8.  (Up to eight rows are added in their order.)
  constexpr int CHAINS = N == 1 ? 8 : 2, T = RED_FLIGHT / CHAINS;
  static_assert(T == 1 || T == 4, "a sum of one row or of four");
  float acc[CHAINS][N];
#pragma unroll
  for (int c = 0; c < CHAINS; ++c)
#pragma unroll
    for (int e = 0; e < N; ++e) acc[c][e] = ident;
  auto add = [&](int c, const typename P::raw u) {
    float v[N];
    P::unpack(u, dti, v);
#pragma unroll
    for (int e = 0; e < N; ++e) acc[c][e] = red_comb(acc[c][e], v[e], kind);
  };
  const int64_t step = (int64_t)RY * pieces;
  int64_t r = threadIdx.x >> lxs, i = base + r * pieces;
#pragma unroll 1
  for (; r + (RED_FLIGHT - 1) * RY < red; r += RED_FLIGHT * RY, i += RED_FLIGHT * step) {
    typename P::raw u[RED_FLIGHT];
#pragma unroll
    for (int q = 0; q < RED_FLIGHT; ++q) u[q] = P::load(in, i + q * step, dti);
    if (N > 1 && red == RED_FLIGHT) {
#pragma unroll
      for (int q = 0; q < RED_FLIGHT; ++q) add(0, u[q]);
    } else {
#pragma unroll
      for (int c = 0; c < CHAINS; ++c) {
        float v[T][N];
#pragma unroll
        for (int q = 0; q < T; ++q) P::unpack(u[c * T + q], dti, v[q]);
#pragma unroll
        for (int e = 0; e < N; ++e) {
          float x = v[0][e];
          if constexpr (T == 4) x = red_comb(red_comb(x, v[1][e], kind), red_comb(v[2][e], v[3][e], kind), kind);
          acc[c][e] = red_comb(acc[c][e], x, kind);
        }
      }
    }
  }
  if (r < red) {  // the rows left, requested together too
    typename P::raw u[RED_FLIGHT - 1];
#pragma unroll
    for (int q = 0; q < RED_FLIGHT - 1; ++q) u[q] = P::load(in, r + q * RY < red ? i + q * step : i, dti);
    if (N > 1 && red < RED_FLIGHT) {
#pragma unroll
      for (int q = 0; q < RED_FLIGHT - 1; ++q)
        if (r + q * RY < red) add(0, u[q]);
    } else {
#pragma unroll
      for (int q = 0; q < RED_FLIGHT - 1; ++q)
        if (r + q * RY < red) add(q % CHAINS, u[q]);
    }
  }
#pragma unroll
  for (int w = CHAINS / 2; w > 0; w /= 2)
#pragma unroll
    for (int c = 0; c < w; ++c)
#pragma unroll
      for (int e = 0; e < N; ++e) acc[c][e] = red_comb(acc[c][e], acc[c + w][e], kind);
  float(&sum)[N] = acc[0];
  if constexpr (LINE) {
#pragma unroll
    for (int w = N / 2; w > 0; w /= 2)
#pragma unroll
      for (int e = 0; e < w; ++e) sum[e] = red_comb(sum[e], sum[e + w], kind);
    for (int s = 1; s < 64; s <<= 1) sum[0] = red_comb(sum[0], __shfl_xor(sum[0], s), kind);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sum[0];
    __syncthreads();
    if (threadIdx.x == 0)
      nbk_store_from_f32(out, o, dto, red_comb(red_comb(part[0], part[1], kind), red_comb(part[2], part[3], kind), kind));
    return;
  }
  if (RY == 1) {  // a column is one lane's: no partial sums to meet
    if (at >= pieces) return;
    const int64_t to = o * pieces + at;
    const bool whole = N == 4 && ((uintptr_t)out & 15) == 0;
    if (whole && dto == NBK_F32) {
      ((float4*)out)[to] = make_float4(sum[0], sum[1 % N], sum[2 % N], sum[3 % N]);
    } else if (whole && dto == NBK_BF16) {
      ((uint2*)out)[to] = make_uint2((uint32_t)nbk_f32_to_bf16(sum[0]) | ((uint32_t)nbk_f32_to_bf16(sum[1 % N]) << 16),
                                     (uint32_t)nbk_f32_to_bf16(sum[2 % N]) | ((uint32_t)nbk_f32_to_bf16(sum[3 % N]) << 16));
    } else {
#pragma unroll
      for (int e = 0; e < N; ++e) nbk_store_from_f32(out, to * N + e, dto, sum[e]);
    }
    return;
  }
  for (int s = LX; s < 64; s <<= 1)  // rows that share a wavefront
#pragma unroll
    for (int e = 0; e < N; ++e) sum[e] = red_comb(sum[e], __shfl_xor(sum[e], s), kind);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lanes = LX < 64 ? LX : 64, across = LX >> 6 ? LX >> 6 : 1;
  if (lane < lanes)
#pragma unroll
    for (int e = 0; e < N; ++e) part[wave * (64 * N) + lane * N + e] = sum[e];
  __syncthreads();
  const int cols = lanes * N;  // of one wavefront
  for (int c = threadIdx.x; c < across * cols; c += 256) {
    const int64_t col = bx * LX * N + c;
    if (col >= inner) break;
    const float* p = part + (c / cols) * (64 * N) + c % cols;
    float v = p[0];
    for (int k = across; k < 4; k += across) v = red_comb(v, p[k * (64 * N)], kind);
    nbk_store_from_f32(out, o * inner + col, dto, v);
  }
}
// (a function chosen anew for every number was two thirds of the instructions: us, 2 x (3287x2624) bf16 27.4 / 12.7,
// 33 x (7479x56) 53 / 13.3, 42 x (105x4664) 16.6 / 11.0)
template <typename P, bool LINE = false>
__device__ __forceinline__ void reduce_strip_body(const void* __restrict__ in, void* __restrict__ out,
                                                  int dti, int dto, int64_t red, int64_t inner, int kind,
                                                  int64_t bx, int64_t o, int lxs, float* part) {
#define REDUCE_KIND(K) reduce_strip_kind<P, K, LINE>(in, out, dti, dto, red, inner, bx, o, lxs, part)
  if (kind == NBK_RED_SUM) REDUCE_KIND(NBK_RED_SUM);
  else if (kind == NBK_RED_MAX) REDUCE_KIND(NBK_RED_MAX);
  else REDUCE_KIND(NBK_RED_MIN);
#undef REDUCE_KIND
}
// How a reduction is laid out, a function of its own shape alone: the order of summation, and so
// the result, does not depend on how reductions are grouped into launches.
struct RedLayout {
  int mode;  // 1: bf16 by 16 bytes, 2: fp32 by 16 bytes; by element 3: bf16, 4: fp32, 0: other types; rows of one
             // element by 16 bytes 5: bf16, 6: fp32
  int lxs;   // log2 of the strip's width in pieces
  int64_t blocks_x;
};
// The strip: 256 pieces, halved while the launch has fewer than 1024 workgroups and there are rows
// left to put abreast.  Down to 256 bytes of a row the narrower strip is never slower; below that
// two workgroups share cache lines, which pays for launches that leave half of the chip idle (128
// bytes from 512 workgroups down: 32 x (256x1024) bf16 16.3 -> 14.1 us; 64 bytes only with more
// than eight rows per lane left: 64 x (1024x64) fp32 16.4 -> 12.2, but 27 x (74x512) bf16 5.4 -> 6.3).
static RedLayout reduce_layout(const void* in, int dti, int64_t outer, int64_t red, int64_t inner) {
  RedLayout L;
  const bool aligned = ((uintptr_t)in & 15) == 0;
  L.mode = dti == NBK_BF16 ? (aligned && inner % 8 == 0 ? 1 : 3) : dti == NBK_F32 ? (aligned && inner % 4 == 0 ? 2 : 4) : 0;
  // (a column of numbers behind each other, the sum of a loss, by 16 bytes a lane: 16384 bf16 are one trip to memory, and
  // up to 65536 one workgroup is faster than slices and the launch that adds them, which is where the planner's line is;
  // us, 8192 bf16 9.2 in slices / 4.7)
  if (inner == 1 && aligned && red >= 512 && (dti == NBK_BF16 ? red % 8 == 0 : dti == NBK_F32 && red % 4 == 0)) {
    L.mode = dti == NBK_BF16 ? 5 : 6;
    L.lxs = 0;
    L.blocks_x = 1;
    return L;
  }
  const int64_t pieces = inner / (L.mode == 1 ? 8 : L.mode == 2 ? 4 : 1);
  // (by element, two rows abreast at least: sixteen chains with the eight of a lane)
  const int widest = (L.mode == 1 || L.mode == 2 || red <= RED_FLIGHT) ? 8 : 7;
  int s = 0;
  while (s < widest && (1ll << s) < pieces) ++s;
  const int whole = L.mode == 1 || L.mode == 2 ? 4 : 5;  // 256 bytes of a row (fp32 by element: 128)
  // (a few long rows, the partial products of a GEMM split along K, are added in their order: a
  // strip of 256 is as fast there, 4 x 65536 2.1 us)
  const bool in_order = L.mode == 2 && red <= 8 && inner >= 65536;
  for (; !in_order && s > 0 && (256 >> s) < red; --s) {
    const int64_t blocks = outer * ((pieces + (1ll << s) - 1) >> s);
    const bool narrower = s > whole ? blocks < 1024 : s == whole ? blocks < 512
                        : s == whole - 1 && blocks < 256 && red * (1ll << s) > 8 * 256;
    if (!narrower) break;
  }
  L.lxs = s;
  L.blocks_x = (pieces + (1ll << s) - 1) >> s;
  return L;
}
template <typename P, bool LINE = false>
__global__ __launch_bounds__(256) void reduce_strip_kernel(const void* __restrict__ in, void* __restrict__ out,
                                                           int dti, int dto, int64_t red, int64_t inner, int kind,
                                                           int lxs) {
  __shared__ float part[4 * 64 * P::N];
  reduce_strip_body<P, LINE>(in, out, dti, dto, red, inner, kind, blockIdx.x, blockIdx.y, lxs, part);
}

// Integer tensors: exact, with a 64-bit accumulator.  The same [outer, red, inner] layout and
// 64 columns per workgroup; the four waves split `red` and meet in LDS.
__device__ __forceinline__ int64_t red_comb_i(int64_t a, int64_t b, int kind) {
  return kind == NBK_RED_SUM ? a + b : (kind == NBK_RED_MAX ? (a > b ? a : b) : (a < b ? a : b));
}
__device__ __forceinline__ int64_t load_as_i64(const void* p, int64_t i, int dt) {
  return dt == NBK_I64 ? ((const int64_t*)p)[i] : (int64_t)((const int32_t*)p)[i];
}
__global__ __launch_bounds__(256) void reduce_mid_int_kernel(const void* __restrict__ in,
                                                             void* __restrict__ out, int dti, int dto,
                                                             int64_t red, int64_t inner, int kind) {
  __shared__ int64_t part[4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t col = (int64_t)blockIdx.x * 64 + lane, o = blockIdx.y;
  int64_t acc = kind == NBK_RED_SUM ? 0 : (kind == NBK_RED_MAX ? INT64_MIN : INT64_MAX);
  if (col < inner) {
    const int64_t base = o * red * inner + col;
    for (int64_t r = w; r < red; r += 4) acc = red_comb_i(acc, load_as_i64(in, base + r * inner, dti), kind);
  }
  part[w][lane] = acc;
  __syncthreads();
  if (w == 0 && col < inner) {
    const int64_t v = red_comb_i(red_comb_i(part[0][lane], part[1][lane], kind),
                                 red_comb_i(part[2][lane], part[3][lane], kind), kind);
    const int64_t at = o * inner + col;
    if (dto == NBK_I64) ((int64_t*)out)[at] = v;
    else if (dto == NBK_I32) ((int32_t*)out)[at] = (int32_t)v;
    else nbk_store_from_f32(out, at, dto, (float)v);
  }
}

// Several independent reductions in one launch (the column sums behind the bias and norm
// gradients of a step are many, small and ready at the same time: one launch instead of one
// each).  A workgroup finds its task from the running block counts and runs the same body.
struct ReduceBatchArgs {
  int32_t n;
  int32_t first_block[NBK_REDUCE_BATCH_MAX + 1];
  int32_t blocks_x[NBK_REDUCE_BATCH_MAX];
  int16_t mode[NBK_REDUCE_BATCH_MAX];
  int16_t lxs[NBK_REDUCE_BATCH_MAX];
  nbk_reduce_task t[NBK_REDUCE_BATCH_MAX];
};

__global__ __launch_bounds__(256) void reduce_batch_kernel(const ReduceBatchArgs B) {
  __shared__ float part[4 * 64 * RedBf16x8::N];
  int i = 0;
  while (i + 1 < B.n && (int)blockIdx.x >= B.first_block[i + 1]) ++i;
  const nbk_reduce_task& t = B.t[i];
  const int lb = (int)blockIdx.x - B.first_block[i];
  const int64_t bx = lb % B.blocks_x[i], o = lb / B.blocks_x[i];
#define REDUCE_STRIP(...)                                                                                         \
  reduce_strip_body<__VA_ARGS__>(t.in, t.out, t.dtype_in, t.dtype_out, t.red, t.inner, t.kind, bx, o, B.lxs[i], part)
  switch (B.mode[i]) {
    case 1: REDUCE_STRIP(RedBf16x8); break;
    case 2: REDUCE_STRIP(RedF32x4); break;
    case 3: REDUCE_STRIP(RedBf16); break;
    case 4: REDUCE_STRIP(RedF32); break;
    case 5: REDUCE_STRIP(RedBf16x8, true); break;
    case 6: REDUCE_STRIP(RedF32x4, true); break;
    default: REDUCE_STRIP(RedAny);
  }
#undef REDUCE_STRIP
}

static int reduce_mid_slab(const RedLayout& L, const void* in, void* out, int32_t dti, int32_t dto,
                           int64_t outer, int64_t red, int64_t inner, int32_t kind, void* stream);

extern "C" int nbk_reduce_mid(const void* in, void* out, int32_t dti, int32_t dto, int64_t outer,
                              int64_t red, int64_t inner, int32_t kind, void* stream) {
  NBK_REQUIRE(in && out, "reduce_mid: null pointer");
  NBK_REQUIRE(outer > 0 && red > 0 && inner > 0, "reduce_mid: empty extent");
  NBK_REQUIRE(kind >= NBK_RED_SUM && kind <= NBK_RED_MIN, "reduce_mid: kind %d", kind);
  NBK_REQUIRE(nbk_dtype_size(dti) > 0 && nbk_dtype_size(dto) > 0, "reduce_mid: bad dtype");
  // `outer` rides on the grid's second dimension (65535 at most): longer ones go in slabs, all of
  // them laid out as the whole is
  const int64_t kSlab = 65535;
  const RedLayout L = reduce_layout(in, dti, outer, red, inner);
  for (int64_t o0 = 0; o0 < outer; o0 += kSlab) {
    const int64_t n = outer - o0 < kSlab ? outer - o0 : kSlab;
    const int rc = reduce_mid_slab(L, (const char*)in + o0 * red * inner * nbk_dtype_size(dti),
                                   (char*)out + o0 * inner * nbk_dtype_size(dto), dti, dto, n, red,
                                   inner, kind, stream);
    if (rc != NBK_OK) return rc;
  }
  return NBK_OK;
}

static int reduce_mid_slab(const RedLayout& L, const void* in, void* out, int32_t dti, int32_t dto,
                           int64_t outer, int64_t red, int64_t inner, int32_t kind, void* stream) {
  if (dti == NBK_I32 || dti == NBK_I64) {
    dim3 grid((unsigned)((inner + 63) / 64), (unsigned)outer);
    hipLaunchKernelGGL(reduce_mid_int_kernel, grid, dim3(256), 0, (hipStream_t)stream, in, out, dti,
                       dto, red, inner, kind);
    return nbk_check_launch("reduce_mid_int_kernel");
  }
  dim3 grid((unsigned)L.blocks_x, (unsigned)outer);
#define REDUCE_STRIP(...)                                                                                         \
  hipLaunchKernelGGL((reduce_strip_kernel<__VA_ARGS__>), grid, dim3(256), 0, (hipStream_t)stream, in, out, dti, dto, red, \
                     inner, kind, L.lxs)
  switch (L.mode) {
    case 1: REDUCE_STRIP(RedBf16x8); break;
    case 2: REDUCE_STRIP(RedF32x4); break;
    case 3: REDUCE_STRIP(RedBf16); break;
    case 4: REDUCE_STRIP(RedF32); break;
    case 5: REDUCE_STRIP(RedBf16x8, true); break;
    case 6: REDUCE_STRIP(RedF32x4, true); break;
    default: REDUCE_STRIP(RedAny);
  }
#undef REDUCE_STRIP
  return nbk_check_launch("reduce_strip_kernel");
}

extern "C" int nbk_reduce_mid_batch(const nbk_reduce_task* tasks, int32_t n, void* stream) {
  NBK_REQUIRE(tasks != nullptr && n > 0, "reduce_mid_batch: no tasks");
  for (int32_t i = 0; i < n; ++i)
    if (tasks[i].dtype_in == NBK_I32 || tasks[i].dtype_in == NBK_I64) {
      // integer tensors take the exact kernel, one launch each; the float ones share launches
      int32_t n_float = 0;
      nbk_reduce_task rest[NBK_REDUCE_BATCH_MAX];
      for (int32_t j = 0; j < n; ++j) {
        const nbk_reduce_task& t = tasks[j];
        if (t.dtype_in == NBK_I32 || t.dtype_in == NBK_I64) {
          const int rc = nbk_reduce_mid(t.in, t.out, t.dtype_in, t.dtype_out, t.outer, t.red, t.inner,
                                        t.kind, stream);
          if (rc != NBK_OK) return rc;
        } else {
          rest[n_float++] = t;
          if (n_float == NBK_REDUCE_BATCH_MAX) {
            const int rc = nbk_reduce_mid_batch(rest, n_float, stream);
            if (rc != NBK_OK) return rc;
            n_float = 0;
          }
        }
      }
      return n_float > 0 ? nbk_reduce_mid_batch(rest, n_float, stream) : NBK_OK;
    }
  for (int32_t base = 0; base < n; base += NBK_REDUCE_BATCH_MAX) {
    ReduceBatchArgs B;
    B.n = n - base < NBK_REDUCE_BATCH_MAX ? n - base : NBK_REDUCE_BATCH_MAX;
    int64_t blocks = 0;
    for (int i = 0; i < B.n; ++i) {
      const nbk_reduce_task& t = tasks[base + i];
      NBK_REQUIRE(t.in && t.out, "reduce_mid_batch: task %d: null pointer", base + i);
      NBK_REQUIRE(t.outer > 0 && t.red > 0 && t.inner > 0, "reduce_mid_batch: task %d: empty extent", base + i);
      NBK_REQUIRE(t.kind >= NBK_RED_SUM && t.kind <= NBK_RED_MIN, "reduce_mid_batch: task %d: kind %d", base + i, t.kind);
      NBK_REQUIRE(nbk_dtype_size(t.dtype_in) > 0 && nbk_dtype_size(t.dtype_out) > 0,
                  "reduce_mid_batch: task %d: bad dtype", base + i);
      const RedLayout L = reduce_layout(t.in, t.dtype_in, t.outer, t.red, t.inner);
      B.mode[i] = (int16_t)L.mode;
      B.lxs[i] = (int16_t)L.lxs;
      B.blocks_x[i] = (int32_t)L.blocks_x;
      B.first_block[i] = (int32_t)blocks;
      blocks += L.blocks_x * t.outer;
      NBK_REQUIRE(blocks <= 0x7fffffffLL, "reduce_mid_batch: launch too large");
      B.t[i] = t;
    }
    B.first_block[B.n] = (int32_t)blocks;
    hipLaunchKernelGGL(reduce_batch_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, B);
  }
  return nbk_check_launch("reduce_batch_kernel");
}
