// conv2d (NHWC x RSCK) forward, input gradient and filter gradient as implicit
// GEMMs.  No im2col buffer is materialised: the tile loaders gather straight from the image.
//
//   forward : M = N*Ho*Wo   Ng = Cout   K = R*S*Cin   (k = (r, s, c), c fastest)
//             A[m,k] = x[n, ho*sh-pt+r, wo*sw-pl+s, c]      B[k,j] = w[r,s,c,j]
//   dgrad   : M = N*H*W     Ng = Cin    K = R*S*Cout  (k = (r, s, co))
//             A[m,k] = dy[n, (h+pt-r)/sh, (w+pl-s)/sw, co]  B[k,j] = w[r,s,j,co]
//   wgrad   : M = R*S*Cin   Ng = Cout   K = N*Ho*Wo   (k = output pixel)
//             A[m,k] = x[n, ho*sh-pt+r, wo*sw-pl+s, c]      B[k,j] = dy[n,ho,wo,j]
// Out-of-image taps read zero, which is the zero padding of the reference op.
//
// Forward and dgrad multiply out of bf16 parts (split_f32.h), the filter gradient and filters of
// a few numbers on the float32 instruction.  Address arithmetic is kept out of the K loop: a lane decomposes its pixels or filter
// rows once and steps through the taps.
// wgrad contracts over every output pixel of the batch while its result is tiny,
// so it is split along K over blockIdx.z into a workspace and summed by a second
// kernel in a fixed order (no atomics: results do not depend on scheduling).
//
// us, before (float32 instruction, channel counts that are no multiple of 16 gathered one by one) / now:
// 64 x 32 x 32, 64 -> 128 channels forward 98 / 79, dgrad 107 / 83; 64 x 16 x 16, 128 -> 256 107 / 67, 138 / 80;
// 50 x 28 x 28, 24 -> 40 44 / 25, 96 / 23; 50 x 14 x 14, 40 -> 72 48 / 22, 123 / 22; 5 x 13 x 13, 24 -> 40 31 / 12, 71 / 15.
#include "nbk_common.h"
#include "split_f32.h"

typedef float f32x16 __attribute__((ext_vector_type(16)));

enum { CONV_FWD = 0, CONV_DGRAD = 1, CONV_WGRAD = 2 };

// Division of a number below 2^31 by a divisor fixed for the launch as a multiplication: the
// host finds mul = ceil(2^(31 + shift) / d) with shift = ceil(log2 d), which fits 32 bits, and
// n / d = (n * mul) >> (31 + shift) exactly for 0 <= n < 2^31 (five instructions where the
// division takes twenty-odd).
struct ConvDiv {
  uint32_t mul, shift, d, pad;
  __host__ void set(int64_t div) {
    d = (uint32_t)div;
    shift = 0;
    while ((1ull << shift) < (uint64_t)div) ++shift;
    mul = (uint32_t)(((1ull << (31 + shift)) + (uint64_t)div - 1) / (uint64_t)div);
  }
  __device__ __forceinline__ int quot(int n) const {
    return (int)(((uint64_t)(uint32_t)n * mul) >> (31 + shift));
  }
  // quotient and remainder of n >= 0
  __device__ __forceinline__ int divmod(int n, int& rem) const {
    const int q = quot(n);
    rem = n - q * (int)d;
    return q;
  }
};

struct ConvArgs {
  nbk_conv_desc d;
  const float* a;     // x (fwd, wgrad) or dy (dgrad)
  const float* b;     // w (fwd, dgrad) or dy (wgrad)
  const float* bias;  // fwd only
  float* out;         // result, or the [splits, M, Ng] workspace when splits > 1
  int64_t M, Ng, K;
  int64_t k_per_split;  // multiple of 16
  int32_t tiles_m, tiles_n, splits;
  ConvDiv by_cin, by_cout, by_s, by_w, by_h, by_wo, by_ho, by_sh, by_sw;
  __host__ void set_divisors() {
    by_cin.set(d.Cin); by_cout.set(d.Cout); by_s.set(d.S);
    by_w.set(d.W); by_h.set(d.H); by_wo.set(d.Wo); by_ho.set(d.Ho);
    by_sh.set(d.stride_h); by_sw.set(d.stride_w);
  }
};

// ---- element-wise gather (any channel count) ----------------------------------------------
// (every extent that is divided here fits 32 bits, checked on the host: 64-bit divisions would
// cost ten times the instructions, eight times per element)
template <int MODE>
__device__ __forceinline__ float conv_load_a(const ConvArgs& g, int64_t m64, int64_t k64, int64_t k_end) {
  const nbk_conv_desc& d = g.d;
  if (m64 >= g.M || k64 >= k_end) return 0.f;
  const int m = (int)m64, k = (int)k64;
  const int Cin = (int)d.Cin, Cout = (int)d.Cout, S = (int)d.S, H = (int)d.H, W = (int)d.W,
            Ho = (int)d.Ho, Wo = (int)d.Wo;
  if (MODE == CONV_FWD) {
    int c, s, wo, ho;
    const int rs = g.by_cin.divmod(k, c);
    const int r = g.by_s.divmod(rs, s);
    const int t = g.by_wo.divmod(m, wo);
    const int n = g.by_ho.divmod(t, ho);
    const int h = ho * d.stride_h - d.pad_t + r, w = wo * d.stride_w - d.pad_l + s;
    if (h < 0 || h >= H || w < 0 || w >= W) return 0.f;
    return g.a[(int64_t)((n * H + h) * W + w) * Cin + c];
  } else if (MODE == CONV_DGRAD) {
    int co, s, w, h;
    const int rs = g.by_cout.divmod(k, co);
    const int r = g.by_s.divmod(rs, s);
    const int t = g.by_w.divmod(m, w);
    const int n = g.by_h.divmod(t, h);
    const int hn = h + d.pad_t - r, wn = w + d.pad_l - s;
    if (hn < 0 || wn < 0) return 0.f;
    int between_h, between_w;
    const int ho = g.by_sh.divmod(hn, between_h), wo = g.by_sw.divmod(wn, between_w);
    if (between_h != 0 || between_w != 0 || ho >= Ho || wo >= Wo) return 0.f;
    return g.a[(int64_t)((n * Ho + ho) * Wo + wo) * Cout + co];
  } else {
    int c, s, wo, ho;
    const int rs = g.by_cin.divmod(m, c);
    const int r = g.by_s.divmod(rs, s);
    const int t = g.by_wo.divmod(k, wo);
    const int n = g.by_ho.divmod(t, ho);
    const int h = ho * d.stride_h - d.pad_t + r, w = wo * d.stride_w - d.pad_l + s;
    if (h < 0 || h >= H || w < 0 || w >= W) return 0.f;
    return g.a[(int64_t)((n * H + h) * W + w) * Cin + c];
  }
}

template <int MODE>
__device__ __forceinline__ float conv_load_b(const ConvArgs& g, int64_t k, int64_t j, int64_t k_end) {
  const nbk_conv_desc& d = g.d;
  if (k >= k_end || j >= g.Ng) return 0.f;
  if (MODE == CONV_FWD) return g.b[k * d.Cout + j];  // w viewed as [R*S*Cin, Cout]
  if (MODE == CONV_DGRAD) {
    int co;
    const int rs = g.by_cout.divmod((int)k, co);
    return g.b[((int64_t)rs * d.Cin + j) * d.Cout + co];
  }
  return g.b[k * d.Cout + j];  // dy viewed as [N*Ho*Wo, Cout]
}

__device__ __forceinline__ void conv_ld8(const float* p, bool ok, float* r) {
  float4 v0 = make_float4(0.f, 0.f, 0.f, 0.f), v1 = v0;
  if (ok) {
    v0 = *(const float4*)p;
    v1 = *(const float4*)(p + 4);
  }
  r[0] = v0.x; r[1] = v0.y; r[2] = v0.z; r[3] = v0.w;
  r[4] = v1.x; r[5] = v1.y; r[6] = v1.z; r[7] = v1.w;
}

// Filter gradient on the float32 instruction, channel counts that are multiples of 8.
// NJ: 32-column MFMA tiles per wave along the output's channel axis: 2 for a 128 x 128
// workgroup tile, 1 for 128 x 64 (channel counts up to 64 would waste half of the wider tile).
template <int NJ>
__global__ __launch_bounds__(256) void conv_wgrad_kernel(const ConvArgs g) {
  // Tiles sit in LDS k-major, [k][128 rows], with the rows of k-row k rotated by 32 places when
  // (k ^ k / 8) is odd.  The two halves of a wave read k-rows 2 ks and 2 ks + 1 of one MFMA
  // step, and either way the halves land 32 banks apart.
  constexpr int BK = 16, LD = 128, BN = 64 * NJ;
  __shared__ float As[2][BK][LD];
  __shared__ float Bs[2][BK][LD];
  auto rot = [](int k, int col) { return (col + 32 * ((k ^ (k >> 3)) & 1)) & 127; };
  const nbk_conv_desc& d = g.d;
  const int tm_i = blockIdx.x % g.tiles_m, tn_i = blockIdx.x / g.tiles_m;
  const int64_t m0 = (int64_t)tm_i * 128, n0 = (int64_t)tn_i * BN;
  const int64_t k_begin = (int64_t)blockIdx.z * g.k_per_split;
  const int64_t k_end = min(g.K, k_begin + g.k_per_split);
  float* out = g.out + (g.splits > 1 ? (int64_t)blockIdx.z * g.M * g.Ng : 0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 32 * NJ;
  const int li = lane & 31, kg = lane >> 5;

  f32x16 acc[2][NJ];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = (f32x16)(0.f);

  // the lane's first filter row and, as running state, the pixel of its K column
  const int w_kk = tid >> 4, w_rr = (tid & 15) * 8;  // pixel column, 8 filter rows
  const int64_t m = m0 + w_rr;
  const bool f_ok = m < g.M;
  const int mm = f_ok ? (int)m : 0;
  const int f_c = mm % (int)d.Cin, rs = mm / (int)d.Cin;
  const int f_s = rs % (int)d.S, f_r = rs / (int)d.S;
  const int64_t px = k_begin + w_kk;  // < 2^31 (checked on the host)
  int p_x = (int)(px % d.Wo);
  const int t = (int)(px / d.Wo);
  int p_y = t % (int)d.Ho, p_n = t / (int)d.Ho;

  float ra[8], rb[8];
  auto load = [&](int64_t k0) {
    // pixel (p_n, p_y, p_x) is column k0 + w_kk; taps of rows m0 + w_rr .. + 7
    const int64_t k = k0 + w_kk, j = n0 + w_rr;
    const int h = p_y * d.stride_h - d.pad_t + f_r, w = p_x * d.stride_w - d.pad_l + f_s;
    const bool ok = f_ok && k < k_end && h >= 0 && h < d.H && w >= 0 && w < d.W;
    conv_ld8(g.a + (((int64_t)p_n * d.H + h) * d.W + w) * d.Cin + f_c, ok, ra);
    // advance the pixel by one K step
    p_x += BK;
    while (p_x >= d.Wo) {
      p_x -= (int)d.Wo;
      if (++p_y >= d.Ho) { p_y = 0; ++p_n; }
    }
    conv_ld8(g.b + k * d.Cout + j, k < k_end && j < g.Ng, rb);  // dy, [K, Cout] row-major
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int e = 0; e < 8; ++e) As[buf][w_kk][rot(w_kk, w_rr) + e] = ra[e];
#pragma unroll
    for (int e = 0; e < 8; ++e) Bs[buf][w_kk][rot(w_kk, w_rr) + e] = rb[e];
  };

  const int64_t nk = (k_end - k_begin + BK - 1) / BK;
  load(k_begin);
  store(0);
  __syncthreads();
  for (int64_t kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    const bool more = kt + 1 < nk;
    if (more) load(k_begin + (kt + 1) * BK);
#pragma unroll
    for (int ks = 0; ks < BK / 2; ++ks) {
      const int k = ks * 2 + kg;
      float fa[2], fb[NJ];
#pragma unroll
      for (int i = 0; i < 2; ++i) fa[i] = As[cur][k][rot(k, wm + i * 32 + li)];
#pragma unroll
      for (int j = 0; j < NJ; ++j) fb[j] = Bs[cur][k][rot(k, wn + j * 32 + li)];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
    if (more) store(cur ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int64_t col = n0 + wn + j * 32 + li;
      if (col >= g.Ng) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t row = m0 + wm + i * 32 + (r >> 2) * 8 + kg * 4 + (r & 3);
        if (row < g.M) out[row * g.Ng + col] = acc[i][j][r];
      }
    }
}

// Filter gradient of up to 32 filter rows (a first layer: 3 x 3 taps of one or three channels), any channel counts and
// alignment.  All of it is reading dy once, so nothing is staged: a lane is one filter row, its tap fixed for the
// launch, and what an MFMA step wants of x and of dy it loads itself, STEPS of them in flight.  The eight half waves of a
// workgroup take an eighth of its slice of pixels each (which pixels share an instruction is free as long as both
// operands agree), and the waves' sums meet in LDS.
// us with the sum of the slices (2 to 5), the kernels for any number of rows / this one: 64 x 32 x 32, 3 -> 64 channels
// 22.9 / 13.1 (dy once: 2.4), 96 x 40 x 40 38 / 24, 50 x 28 x 28, 1 -> 24 17.5 / 11.3, 2 x 14 x 14, 3 -> 16 12.9 / 7.7; one
// tap, 64 x 32 x 32, 32 -> 64 20.3 / 13.5, 8 -> 512 80 / 44, 50 x 14 x 14, 16 -> 40 12.1 / 10.7.  Error against float64 0.41 to
// 0.6 of what one chain a slice has (3 -> 64 2.5e-7 -> 1.2e-7).
template <int NB>
__global__ __launch_bounds__(256) void conv_wgrad_few_kernel(const ConvArgs g) {
  constexpr int STEPS = 16;
  __shared__ float part[4][NB * 16][64];
  const nbk_conv_desc& d = g.d;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 31, h = lane >> 5;
  const int64_t n0 = (int64_t)blockIdx.x * (32 * NB);
  const int64_t k_begin = (int64_t)blockIdx.z * g.k_per_split, k_end = min(g.K, k_begin + g.k_per_split);
  const int run = (int)((k_end - k_begin + 7) / 8);
  const int64_t first = k_begin + (int64_t)(wave * 2 + h) * run;
  int left = (int)max((int64_t)0, min((int64_t)run, k_end - first));
  const int px = left > 0 ? (int)first : 0;  // < 2^31 (checked on the host)
  // (filter rows and columns past the end repeat the last one: their results are not stored)
  int f_c, f_s, x, y;
  const int f_rs = g.by_cin.divmod(min(li, (int)g.M - 1), f_c);
  const int q_h = g.by_s.divmod(f_rs, f_s) - d.pad_t, q_w = f_s - d.pad_l;
  const int t = g.by_wo.divmod(px, x);
  int n = g.by_ho.divmod(t, y);
  const float* b[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) b[j] = g.b + (int64_t)px * d.Cout + min(n0 + j * 32 + li, g.Ng - 1);
  f32x16 acc[2][NB];  // (two chains a wave: half the roundings in a row)
#pragma unroll
  for (int j = 0; j < NB; ++j) acc[0][j] = acc[1][j] = (f32x16)(0.f);
  for (int t0 = 0; t0 < run; t0 += STEPS) {
    float fa[STEPS], fb[NB][STEPS];
#pragma unroll
    for (int e = 0; e < STEPS; ++e) {
      const bool live = left > 0;
      const int ih = y * d.stride_h + q_h, iw = x * d.stride_w + q_w;
      const bool in = live && ih >= 0 && ih < d.H && iw >= 0 && iw < d.W;
      const float v = g.a[in ? (int64_t)((n * (int)d.H + ih) * (int)d.W + iw) * d.Cin + f_c : 0];
      fa[e] = in ? v : 0.f;
      --left;
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const float w = *b[j];
        fb[j][e] = live ? w : 0.f;
        b[j] += left > 0 ? d.Cout : 0;  // (the last pixel again)
      }
      if (++x == d.Wo) {
        x = 0;
        if (++y == d.Ho) { y = 0; ++n; }
      }
    }
#pragma unroll
    for (int e = 0; e < STEPS; ++e)
#pragma unroll
      for (int j = 0; j < NB; ++j)
        acc[e & 1][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[e], fb[j][e], acc[e & 1][j], 0, 0, 0);
  }
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave][j * 16 + r][lane] = acc[0][j][r] + acc[1][j][r];
  __syncthreads();
  // D register r of lane (column li, half h) is row (r / 4) * 8 + h * 4 + r % 4; a wave sums its share of the registers
  float* out = g.out + (g.splits > 1 ? (int64_t)blockIdx.z * g.M * g.Ng : 0);
#pragma unroll
  for (int q = 0; q < NB * 4; ++q) {
    const int at = wave * (NB * 4) + q, r = at & 15;
    const int64_t row = (r >> 2) * 8 + h * 4 + (r & 3), col = n0 + (at >> 4) * 32 + li;
    const float sum = (part[0][at][lane] + part[1][at][lane]) + (part[2][at][lane] + part[3][at][lane]);
    if (row < g.M && col < g.Ng) out[row * g.Ng + col] = sum;
  }
}

// Forward of filters with up to 2 STEPS numbers a channel of the result (a first layer), any channel counts and
// alignment: as above, nothing is staged.  A lane is a pixel and knows the taps of the numbers that it supplies (k = 2 e + h
// of step e); the filter stays in registers while a wave goes from block to block of 32 pixels.
// us, the former tiles on the float32 instruction / tiles out of bf16 parts / this kernel: 64 x 32 x 32, 3 -> 64 channels
// 14.2 / 15.6 / 10.4, 96 x 40 x 40 24 / 32 / 19, 1 -> 64 19 / 32 / 14, 50 x 28 x 28, 1 -> 24 9.7 / 9.5 / 5.3, 5 x 5 taps
// 64 x 30 x 30, 1 -> 32 12.4 / 10.6 / 7.4; one tap 64 x 32 x 32, 32 -> 64 11.8 / 13.4 / 10.7, 8 -> 512 52 / 69 / 33.  Bound by the
// result's writes where it is large (3 -> 64: 2.4 us of them).  Error against float64 0.78 to 0.93 of one chain's.
template <int NB, int STEPS>
__global__ __launch_bounds__(256, 2) void conv_fwd_few_kernel(const ConvArgs g) {
  const nbk_conv_desc& d = g.d;
  const int lane = threadIdx.x & 63, li = lane & 31, h = lane >> 5;
  const int64_t n0 = (int64_t)blockIdx.y * (32 * NB);
  float fb[NB][STEPS];
  int off[STEPS], tap[STEPS];
#pragma unroll
  for (int e = 0; e < STEPS; ++e) {
    const int k = 2 * e + h;
    const bool ok = k < g.K;
    int c, s;
    const int r = g.by_s.divmod(g.by_cin.divmod(ok ? k : 0, c), s);
    off[e] = ok ? (r * (int)d.W + s) * (int)d.Cin + c : -1;
    tap[e] = r << 8 | s;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const float v = g.b[(ok ? k : 0) * d.Cout + min(n0 + j * 32 + li, g.Ng - 1)];
      fb[j][e] = ok ? v : 0.f;
    }
  }
  float bias[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) bias[j] = g.bias ? g.bias[min(n0 + j * 32 + li, g.Ng - 1)] : 0.f;
  const bool relu = d.act == NBK_ACT_RELU;
  const int64_t step = (int64_t)gridDim.x * 128;
  for (int64_t m0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 32; m0 < g.M; m0 += step) {
    // (pixels past the end repeat the last one: their results are not stored)
    int x, y;
    const int t = g.by_wo.divmod((int)min(m0 + li, g.M - 1), x);
    const int n = g.by_ho.divmod(t, y);
    const int h0 = y * d.stride_h - d.pad_t, w0 = x * d.stride_w - d.pad_l;
    const int64_t base = (((int64_t)n * d.H + h0) * d.W + w0) * d.Cin;
    float fa[STEPS];
#pragma unroll
    for (int e = 0; e < STEPS; ++e) {
      const int ih = h0 + (tap[e] >> 8), iw = w0 + (tap[e] & 255);
      const bool in = off[e] >= 0 && ih >= 0 && ih < d.H && iw >= 0 && iw < d.W;
      const float v = g.a[in ? base + off[e] : 0];
      fa[e] = in ? v : 0.f;
    }
    f32x16 acc[2][NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[0][j] = acc[1][j] = (f32x16)(0.f);
#pragma unroll
    for (int e = 0; e < STEPS; ++e)
#pragma unroll
      for (int j = 0; j < NB; ++j)
        acc[e & 1][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[e], fb[j][e], acc[e & 1][j], 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int64_t row = m0 + (r >> 2) * 8 + h * 4 + (r & 3), col = n0 + j * 32 + li;
        const float v = acc[0][j][r] + acc[1][j][r] + bias[j];
        if (row < g.M && col < g.Ng) g.out[row * g.Ng + col] = relu ? fmaxf(v, 0.f) : v;
      }
  }
}

// ---- out of bf16 parts (split_f32.h) --------------------------------------------------------
// Tiles of BM x BN on NWM x NWN waves, K tiles of 32 in two LDS buffers.  A lane takes pieces of 8
// consecutive k of a row: forward and dgrad, 8 channels of a pixel at one tap (channel counts that are
// multiples of 8: FAST), each piece with its own tap; wgrad, one filter row at 8 pixels.  The pieces of the
// next tile but one are requested before a tile is multiplied and split behind it.
// The launch's K loop is the sum of its matrix instructions and of what it costs to gather and to split
// (5.5 instructions a number), which the two waves of a SIMD cover for each other only in part.
template <int MODE, bool FAST, int ROWS, int NT, bool IS_A>
struct ConvRows {
  static constexpr int PIECES = ROWS * 4 > NT ? ROWS * 4 / NT : 1;
  static_assert(PIECES == 1 || PIECES * NT == ROWS * 4, "whole pieces per lane");
  // (a tile of fewer pieces than lanes: the lanes behind them request the first number of the tensor)
  static __device__ __forceinline__ bool mine() { return ROWS * 4 >= NT || (int)threadIdx.x < ROWS * 4; }
  // whether a piece's 8 numbers stand side by side in memory
  static constexpr bool WHOLE = FAST && MODE != CONV_WGRAD && (IS_A || MODE == CONV_DGRAD);
  int row[PIECES], c[PIECES];
  // forward / dgrad: pixel at tap (0, 0) of an A piece; wgrad: the tap's offset from a pixel
  int q_h[PIECES], q_w[PIECES], q_pix[PIECES], ch[PIECES];
  bool ok[PIECES];
  int t_r[PIECES], t_s[PIECES], t_c[PIECES];  // the next K tile's tap and first channel; wgrad: pixel (n, y, x)
  float r[2][PIECES][8];

  __device__ __forceinline__ void init(const ConvArgs& g, int64_t row0, int64_t k_begin) {
    const nbk_conv_desc& d = g.d;
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      const int idx = (int)threadIdx.x + NT * p;
      row[p] = WHOLE ? idx >> 2 : idx % ROWS;
      c[p] = WHOLE ? idx & 3 : idx / ROWS;
      const int64_t m = row0 + row[p];
      const int k = (int)k_begin + c[p] * 8;
      ok[p] = mine() && m < (IS_A ? g.M : g.Ng);
      const int mm = ok[p] ? (int)m : 0;
      if (MODE == CONV_WGRAD) {
        if (IS_A) {
          int s;
          const int rs = g.by_cin.divmod(mm, ch[p]);
          const int rr = g.by_s.divmod(rs, s);
          q_h[p] = rr - d.pad_t;
          q_w[p] = s - d.pad_l;
          const int t = g.by_wo.divmod(k, t_c[p]);
          t_r[p] = g.by_ho.divmod(t, t_s[p]);
        }
      } else {
        const ConvDiv& by = MODE == CONV_FWD ? g.by_cin : g.by_cout;
        const int tap = by.divmod(k, t_c[p]);
        t_r[p] = g.by_s.divmod(tap, t_s[p]);
        if (IS_A) {
          int x, y;
          const int t = (MODE == CONV_FWD ? g.by_wo : g.by_w).divmod(mm, x);
          const int n = (MODE == CONV_FWD ? g.by_ho : g.by_h).divmod(t, y);
          if (MODE == CONV_FWD) {
            q_h[p] = y * d.stride_h - d.pad_t;
            q_w[p] = x * d.stride_w - d.pad_l;
            q_pix[p] = (n * (int)d.H + q_h[p]) * (int)d.W + q_w[p];
          } else {
            q_h[p] = y + d.pad_t;
            q_w[p] = x + d.pad_l;
            q_pix[p] = n;
          }
        }
      }
    }
  }
  // Forward / dgrad: where channel `chan` of piece p's pixel lies at tap (r, s), and whether it is inside.
  __device__ __forceinline__ bool where(const ConvArgs& g, int p, int r, int s, int chan, int64_t& at) const {
    const nbk_conv_desc& d = g.d;
    if (MODE == CONV_FWD) {
      const int h = q_h[p] + r, w = q_w[p] + s;
      at = (int64_t)(q_pix[p] + r * (int)d.W + s) * d.Cin + chan;
      return h >= 0 && h < d.H && w >= 0 && w < d.W;
    }
    const int hn = q_h[p] - r, wn = q_w[p] - s;
    int ho = hn, wo = wn;
    bool in = hn >= 0 && wn >= 0;
    if (d.stride_h != 1 || d.stride_w != 1) {
      int between_h, between_w;
      ho = g.by_sh.divmod(max(hn, 0), between_h);
      wo = g.by_sw.divmod(max(wn, 0), between_w);
      in = in && between_h == 0 && between_w == 0;
    }
    at = (int64_t)((q_pix[p] * (int)d.Ho + ho) * (int)d.Wo + wo) * d.Cout + chan;
    return in && ho < d.Ho && wo < d.Wo;
  }
  // K tile at k0 into set SET; the pieces move on to the next.
  template <int SET>
  __device__ __forceinline__ void load(const ConvArgs& g, int64_t row0, int64_t k0, int64_t k_end) {
    const nbk_conv_desc& d = g.d;
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      const int64_t k = k0 + c[p] * 8, m = row0 + row[p];
      float* x = r[SET][p];
      if constexpr (!FAST && !IS_A) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = ok[p] ? conv_load_b<MODE>(g, k + e, m, k_end) : 0.f;
      } else if constexpr (!FAST) {  // every number has a tap of its own
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          int chan, s;
          const int tap = (MODE == CONV_FWD ? g.by_cin : g.by_cout).divmod((int)k + e, chan);
          const int rr = g.by_s.divmod(tap, s);
          int64_t at;
          const bool in = ok[p] && k + e < k_end && where(g, p, rr, s, chan, at);
          const float v = g.a[in ? at : 0];
          x[e] = in ? v : 0.f;
        }
      } else if constexpr (MODE == CONV_WGRAD && IS_A) {
        // 8 pixels in a row of the output, or across its end
        int n = t_r[p], y = t_s[p], w = t_c[p];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int ih = y * d.stride_h + q_h[p], iw = w * d.stride_w + q_w[p];
          const bool in = ok[p] && k + e < k_end && ih >= 0 && ih < d.H && iw >= 0 && iw < d.W;
          const int64_t at = in ? (int64_t)((n * (int)d.H + ih) * (int)d.W + iw) * d.Cin + ch[p] : 0;
          const float v = g.a[at];
          x[e] = in ? v : 0.f;
          if (++w == d.Wo) {
            w = 0;
            if (++y == d.Ho) { y = 0; ++n; }
          }
        }
      } else if constexpr (WHOLE) {
        bool in = ok[p] && k < k_end;
        int64_t at;
        if (!IS_A) {  // dgrad: w[r, s, j, co]
          at = ((int64_t)(t_r[p] * (int)d.S + t_s[p]) * d.Cin + m) * d.Cout + t_c[p];
        } else {
          in = in && where(g, p, t_r[p], t_s[p], t_c[p], at);
        }
        // (what lies outside reads the first numbers of the tensor: no branch around the request)
        const float* src = (IS_A ? g.a : g.b) + (in ? at : 0);
        const sp_f4 v0 = *(const sp_f4_any*)src, v1 = *(const sp_f4_any*)(src + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[e] = in ? v0[e] : 0.f;
          x[4 + e] = in ? v1[e] : 0.f;
        }
      } else {  // [K, Cout] row-major: w for the forward product, dy for wgrad
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const bool in = ok[p] && k + e < k_end;
          const float v = g.b[in ? (k + e) * d.Cout + m : 0];
          x[e] = in ? v : 0.f;
        }
      }
      if constexpr (FAST && MODE == CONV_WGRAD && IS_A) {
        t_c[p] += SPLIT_BK;
        while (t_c[p] >= d.Wo) {
          t_c[p] -= (int)d.Wo;
          if (++t_s[p] >= d.Ho) { t_s[p] = 0; ++t_r[p]; }
        }
      } else if constexpr (WHOLE) {
        const int ck = MODE == CONV_FWD ? (int)d.Cin : (int)d.Cout;
        t_c[p] += SPLIT_BK;
        while (t_c[p] >= ck) {
          t_c[p] -= ck;
          if (++t_s[p] == (int)d.S) { t_s[p] = 0; ++t_r[p]; }
        }
      }
    }
  }
  template <int SET>
  __device__ __forceinline__ void store(sp_u4* tile) {
    if (mine())
#pragma unroll
      for (int p = 0; p < PIECES; ++p) split_store<ROWS>(tile, row[p], c[p], r[SET][p]);
  }
};

// SHORT: contractions of up to SPLIT_SHORT tiles, without requests past the end.  us, in the loop / so: forward 83 x 32 x 32, 3 ->
// 172 channels, 5 x 5 taps 85 / 59, 64 x 32 x 32, 3 -> 64 26 / 21.5, 32 x 64 x 64, 12 -> 130 (four tiles) 155 / 112, input gradients
// 90 x 53 x 53, 78 -> 3 111 / 68; with channels in pieces of eight 64 x 32 x 32, 128 -> 16, one tap 12.2 / 10.7.
constexpr int SPLIT_SHORT = 4;
// (Three workgroups of 64 x 64 share a CU where the gather leaves the registers for it: input gradients 64 x 56 x 56, 36 ->
// 100 459 us, with two 534.)
template <int MODE, bool FAST, int BM, int BN, int NWM, int NWN, bool SHORT>
__global__ __launch_bounds__(NWM * NWN * 64, BM == 64 && (MODE != CONV_FWD || FAST) ? 3 : 1) void conv_split_kernel(const ConvArgs g) {
  constexpr int NT = NWM * NWN * 64, WM = BM / NWM, WN = BN / NWN, TM = WM / 16, TN = WN / 16;
  constexpr int TILE = (BM + BN) * 12;
  extern __shared__ __align__(16) sp_u4 conv_lds[];
  const int tm_i = blockIdx.x % g.tiles_m, tn_i = blockIdx.x / g.tiles_m;
  const int64_t m0 = (int64_t)tm_i * BM, n0 = (int64_t)tn_i * BN;
  const int64_t k_begin = (int64_t)blockIdx.z * g.k_per_split;
  const int64_t k_end = min(g.K, k_begin + g.k_per_split);
  float* out = g.out + (g.splits > 1 ? (int64_t)blockIdx.z * g.M * g.Ng : 0);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / NWN * WM, wn = wave % NWN * WN;
  ConvRows<MODE, FAST, BM, NT, true> la;
  ConvRows<MODE, FAST, BN, NT, false> lb;
  la.init(g, m0, k_begin);
  lb.init(g, n0, k_begin);
  SplitAcc<TM, TN, 2> acc;
  acc.zero();
  const int nk = (int)((k_end - k_begin + SPLIT_BK - 1) / SPLIT_BK);
#define CONV_LOAD(SET, T)                                                  \
  do {                                                                     \
    const int64_t k0 = k_begin + (int64_t)(T) * SPLIT_BK;                  \
    la.template load<SET>(g, m0, k0, k_end);                               \
    lb.template load<SET>(g, n0, k0, k_end);                               \
  } while (0)
#define CONV_STORE(SET)                                                    \
  do {                                                                     \
    la.template store<SET>(conv_lds + SET * TILE);                         \
    lb.template store<SET>(conv_lds + SET * TILE + BM * 12);               \
  } while (0)
#define CONV_MULTIPLY(SET) acc.template multiply<BM, BN, SET>(conv_lds + SET * TILE, conv_lds + SET * TILE + BM * 12, wm, wn, lane)
  // (past the end: zeros.  Where every number has a tap of its own, such a request costs more than a tile's
  // multiplication; but with conditions in front of them the loop became slower by up to half.)
  CONV_LOAD(0, 0);
  if constexpr (SHORT) {
    if (nk > 1) CONV_LOAD(1, 1);
    CONV_STORE(0);
    __syncthreads();
    if (nk > 2) CONV_LOAD(0, 2);
    CONV_MULTIPLY(0);
    if (nk > 1) {
      CONV_STORE(1);
      __syncthreads();
      if (nk > 3) CONV_LOAD(1, 3);
      CONV_MULTIPLY(1);
    }
    if (nk > 2) {
      CONV_STORE(0);
      __syncthreads();
      CONV_MULTIPLY(0);
    }
    if (nk > 3) {
      CONV_STORE(1);
      __syncthreads();
      CONV_MULTIPLY(1);
    }
  } else {
    CONV_LOAD(1, 1);
    CONV_STORE(0);
    __syncthreads();
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
      CONV_LOAD(0, kt + 2);
      CONV_MULTIPLY(0);
      CONV_STORE(1);
      __syncthreads();
      CONV_LOAD(1, kt + 3);
      CONV_MULTIPLY(1);
      CONV_STORE(0);
      __syncthreads();
    }
    if (kt < nk) CONV_MULTIPLY(0);
  }
#undef CONV_MULTIPLY
#undef CONV_STORE
#undef CONV_LOAD
  const bool relu = MODE == CONV_FWD && g.d.act == NBK_ACT_RELU;
  // sum(i, j, r) of the results that `put` is to store, and the others, a bit each
  auto store = [&](auto sum, auto put) {
    uint32_t left = 0;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int64_t col = n0 + wn + j * 16 + (lane & 15);
        if (col >= g.Ng) continue;
        const float bias = g.bias ? g.bias[col] : 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int64_t row = m0 + wm + i * 16 + (lane >> 4) * 4 + r;
          if (row >= g.M) continue;
          const float s = sum(i, j, r);
          const uint32_t bit = 1u << ((i * TN + j) * 4 + r);
          if (put(s, bit)) out[row * g.Ng + col] = relu ? fmaxf(s + bias, 0.f) : s + bias;
          else left |= bit;
        }
      }
    return left;
  };
  static_assert(TM * TN * 4 <= 32, "a bit for each of a lane's results");
  const uint32_t left = store([&](int i, int j, int r) { return acc.sum(i, j, r); },
                              [](float s, uint32_t) { return fabsf(s) < INFINITY; });
  // (us, numbers that have parts / one infinity / NaN throughout: 64 x 32 x 32, 64 -> 128 channels 73 / 136 / 345, its
  // input gradient 84 / 251 / 643: it gathers number by number; a lane at a time 7870 and 15480 at last)
  if (__any(left != 0)) {
    const int64_t row = m0 + wm + (lane & 15), col = n0 + wn + (lane & 15);
    acc.again(k_begin, k_end, lane, [&](int i, int64_t k, auto) { return conv_load_a<MODE>(g, row + i * 16, k, k_end); },
              [&](int j, int64_t k, auto) { return conv_load_b<MODE>(g, k, col + j * 16, k_end); });
    store([&](int i, int j, int r) { return acc.sum_again(i, j, r); }, [&](float, uint32_t bit) { return (left & bit) != 0; });
  }
}

// Results of one product each (the input gradient of one output channel and one tap, the filter gradient of one pixel):
// rounded once, where the six products of the parts would be rounded together.  A wave has 16 rows, a lane a column.  us,
// 64 x 32 x 32, 128 -> 1 channels: 8.2, out of parts 27 (its writes: 4.8).
template <int MODE>
__global__ __launch_bounds__(256) void conv_outer_kernel(const ConvArgs g) {
  constexpr int ROWS = 16;
  const int lane = threadIdx.x & 63;
  const int64_t m0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * ROWS;
  const float x = conv_load_a<MODE>(g, m0 + (lane & (ROWS - 1)), 0, 1);
  for (int64_t n = lane; n - lane < g.Ng; n += 64) {
    const float w = conv_load_b<MODE>(g, 0, n, 1);
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const float xr = __shfl(x, r);
      if (m0 + r < g.M && n < g.Ng) g.out[(m0 + r) * g.Ng + n] = xr * w;
    }
  }
}
template <int MODE>
static int conv_launch_outer(ConvArgs& a, hipStream_t st) {
  a.set_divisors();
  const int64_t blocks = (a.M + 63) / 64;
  NBK_REQUIRE(blocks <= 0x7fffffffLL, "conv2d: launch too large");
  hipLaunchKernelGGL(conv_outer_kernel<MODE>, dim3((unsigned)blocks), dim3(256), 0, st, a);
  return nbk_check_launch("conv_outer_kernel");
}

// out[i] = sum over z of partial[z][i].  Eight loads in flight are a trip to memory, and a lane that adds every
// slice of a small filter by itself makes one trip behind the other on a few CUs; so ZG lanes share a sum,
// each with every ZG-th slice, and meet in LDS.  The order of the additions is fixed: the result
// does not depend on scheduling.
template <int ZG>
__global__ __launch_bounds__(256) void conv_sum_partials(const float* partial, float* out, int64_t n, int splits) {
  constexpr int COLS = 256 / ZG;
  __shared__ float part[ZG][COLS];
  const int col = (int)threadIdx.x % COLS, zg = (int)threadIdx.x / COLS;
  const int64_t i = (int64_t)blockIdx.x * COLS + col;
  float s = 0.f;
  if (i < n) {
    int z = zg;
    for (; z + 7 * ZG < splits; z += 8 * ZG) {
      float v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = partial[(int64_t)(z + q * ZG) * n + i];
      s += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
    for (; z < splits; z += ZG) s += partial[(int64_t)z * n + i];
  }
  if constexpr (ZG > 1) {
    part[zg][col] = s;
    __syncthreads();
    if (zg > 0) return;
    float v[ZG];
#pragma unroll
    for (int q = 0; q < ZG; ++q) v[q] = part[q][col];
#pragma unroll
    for (int w = ZG / 2; w > 0; w /= 2)
#pragma unroll
      for (int q = 0; q < w; ++q) v[q] += v[q + w];
    s = v[0];
  }
  if (i < n) out[i] = s;
}

static int conv_check(const nbk_conv_desc* d) {
  NBK_REQUIRE(d != nullptr, "conv2d: null descriptor");
  NBK_REQUIRE(d->dtype == NBK_F32, "conv2d: only fp32 is implemented (dtype %d)", d->dtype);
  NBK_REQUIRE(d->N > 0 && d->H > 0 && d->W > 0 && d->Cin > 0 && d->R > 0 && d->S > 0 &&
                  d->Cout > 0 && d->Ho > 0 && d->Wo > 0,
              "conv2d: empty extent");
  NBK_REQUIRE(d->act == NBK_ACT_NONE || d->act == NBK_ACT_RELU, "conv2d: act %d", d->act);
  NBK_REQUIRE(d->stride_h > 0 && d->stride_w > 0, "stride values must be > 0");
  NBK_REQUIRE(d->pad_t >= 0 && d->pad_b >= 0 && d->pad_l >= 0 && d->pad_r >= 0,
              "padding values must be >= 0");
  const int64_t ho = (d->H + d->pad_t + d->pad_b - d->R) / d->stride_h + 1;
  const int64_t wo = (d->W + d->pad_l + d->pad_r - d->S) / d->stride_w + 1;
  NBK_REQUIRE(ho == d->Ho && wo == d->Wo, "conv2d: output size %lld x %lld does not match %lld x %lld",
              (long long)d->Ho, (long long)d->Wo, (long long)ho, (long long)wo);
  NBK_REQUIRE(d->N * d->H * d->W < 0x7fffffffLL && d->N * d->Ho * d->Wo < 0x7fffffffLL &&
                  d->R * d->S * d->Cin < 0x7fffffffLL && d->R * d->S * d->Cout < 0x7fffffffLL,
              "conv2d: extent beyond 2^31 elements");
  return NBK_OK;
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

template <int MODE, bool FAST, int BM, int BN, int NWM, int NWN, bool SHORT = false>
static int conv_launch_tile(ConvArgs& a, hipStream_t st) {
  a.tiles_m = (int)((a.M + BM - 1) / BM);
  a.tiles_n = (int)((a.Ng + BN - 1) / BN);
  const int64_t blocks = (int64_t)a.tiles_m * a.tiles_n;
  NBK_REQUIRE(blocks <= 0x7fffffffLL, "conv2d: launch too large");
  const size_t lds = 2 * (size_t)(BM + BN) * 12 * 16;
  auto kern = conv_split_kernel<MODE, FAST, BM, BN, NWM, NWN, SHORT>;
  static bool attr_set = false; /* idempotent, so a race only repeats the call */
  if (!attr_set) {
    NBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set = true;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks, 1, (unsigned)a.splits), dim3(NWM * NWN * 64), lds, st, a);
  return nbk_check_launch("conv_split_kernel");
}
// Forward and dgrad.  128 x 128 tiles run one to a CU and two of 64 x 64 do; a round of the former does the work of
// two of the latter in 1.7 of one's time.  us, 128 x 128 / 64 x 64: 64 x 32 x 32, 64 -> 128 channels, 79 / 108; 64 x 16
// x 16, 128 -> 256, 67 / 100, its input gradient (128 columns: 128 tiles) 108 / 80; 90 x 20 x 20, 56 -> 120 72 / 71.
// Up to 32 channels of results, tiles of 128 x 32 from one per CU on: 50 x 28 x 28, 1 -> 24 9.1 against 11.0,
// input gradient of 24 -> 40 23 against 29; below that 1 x 32 x 32, 16 -> 32 12.0 against 10.3.
// (128 x 64 tiles: 5 % less than 64 x 64 at best.)  Number by number, the gather is most of a forward tile, and two of 64
// x 64 have no third beside them: 1.5 there (32 x 64 x 64, 12 -> 130 129 / 155 in the loop).
template <int MODE, bool FAST, bool SHORT>
static int conv_launch_length(ConvArgs& a, hipStream_t st) {
  const int64_t cus = nbk_num_cus(), m128 = (a.M + 127) / 128;
  const int64_t t64 = ((a.M + 63) / 64) * ((a.Ng + 63) / 64);
  if (a.Ng <= 32 && m128 >= cus) return conv_launch_tile<MODE, FAST, 128, 32, 4, 1, SHORT>(a, st);
  const int64_t rounds_128 = (m128 * ((a.Ng + 127) / 128) + cus - 1) / cus, rounds_64 = (t64 + 2 * cus - 1) / (2 * cus);
  if (rounds_128 * (MODE == CONV_FWD && !FAST ? 15 : 17) <= rounds_64 * 10)
    return conv_launch_tile<MODE, FAST, 128, 128, 2, 4, SHORT>(a, st);
  return conv_launch_tile<MODE, FAST, 64, 64, 2, 2, SHORT>(a, st);
}
template <int MODE, bool FAST>
static int conv_launch(ConvArgs& a, hipStream_t st) {
  a.set_divisors();
  return a.K <= SPLIT_SHORT * SPLIT_BK ? conv_launch_length<MODE, FAST, true>(a, st) : conv_launch_length<MODE, FAST, false>(a, st);
}

// The filter gradient of channel counts that are multiples of 8 stays on the float32 instruction: its pieces
// of 8 k are 8 pixels, whose gather costs more than the instruction saves (64 x 32 x 32, 64 -> 128 channels 139
// us against 112).  Others gather number by number there, too (before the sum of slices took many lanes 3 -> 64 44 against 51).
static int conv_launch_wgrad(ConvArgs& a, bool fast, hipStream_t st) {
  if (a.K == 1) return conv_launch_outer<CONV_WGRAD>(a, st);
  a.set_divisors();
  if (a.M <= 32) {  // one block of 32 filter rows: faster at every size above
    const int64_t nb = a.Ng <= 32 ? 1 : 2, columns = (a.Ng + 32 * nb - 1) / (32 * nb);
    NBK_REQUIRE(columns <= 0x7fffffffLL, "conv2d: launch too large");
    const dim3 grid((unsigned)columns, 1, (unsigned)a.splits);
    if (nb == 1) hipLaunchKernelGGL((conv_wgrad_few_kernel<1>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((conv_wgrad_few_kernel<2>), grid, dim3(256), 0, st, a);
    return nbk_check_launch("conv_wgrad_few_kernel");
  }
  if (!fast)
    return a.k_per_split <= SPLIT_SHORT * SPLIT_BK ? conv_launch_tile<CONV_WGRAD, true, 64, 64, 2, 2, true>(a, st)
                                                   : conv_launch_tile<CONV_WGRAD, true, 64, 64, 2, 2>(a, st);
  // the narrow workgroup tile when the last 128-wide column tile would be at most half full,
  // or when the wide tiling gives fewer workgroups than the GPU has CUs
  const int64_t wide = ((a.M + 127) / 128) * ((a.Ng + 127) / 128) * a.splits;
  const bool narrow = (a.Ng - 1) % 128 < 64 || wide < nbk_num_cus();
  const int bn = narrow ? 64 : 128;
  a.tiles_m = (int)((a.M + 127) / 128);
  a.tiles_n = (int)((a.Ng + bn - 1) / bn);
  const int64_t blocks = (int64_t)a.tiles_m * a.tiles_n;
  NBK_REQUIRE(blocks <= 0x7fffffffLL, "conv2d: launch too large");
  const dim3 grid((unsigned)blocks, 1, (unsigned)a.splits);
  if (narrow) hipLaunchKernelGGL((conv_wgrad_kernel<1>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((conv_wgrad_kernel<2>), grid, dim3(256), 0, st, a);
  return nbk_check_launch("conv_wgrad_kernel");
}

template <int NB, int STEPS>
static int conv_launch_fwd_few(const ConvArgs& a, hipStream_t st) {
  const int64_t blocks = (a.M + 127) / 128, most = 4 * (int64_t)nbk_num_cus();
  const dim3 grid((unsigned)(blocks < most ? blocks : most), (unsigned)((a.Ng + 32 * NB - 1) / (32 * NB)));
  hipLaunchKernelGGL((conv_fwd_few_kernel<NB, STEPS>), grid, dim3(256), 0, st, a);
  return nbk_check_launch("conv_fwd_few_kernel");
}

extern "C" int nbk_conv2d_fwd(const nbk_conv_desc* d, const void* x, const void* w,
                              const void* bias, void* y, void* stream) {
  int rc = conv_check(d);
  if (rc) return rc;
  NBK_REQUIRE(x && w && y, "conv2d: null pointer");
  ConvArgs a;
  a.d = *d;
  a.a = (const float*)x; a.b = (const float*)w; a.bias = (const float*)bias; a.out = (float*)y;
  a.M = d->N * d->Ho * d->Wo; a.Ng = d->Cout; a.K = d->R * d->S * d->Cin;
  a.splits = 1; a.k_per_split = (a.K + 15) / 16 * 16;
  // (offsets inside a filter stand in 32 bits, the launch's second axis ends at 65535)
  // sixteen steps are what the registers hold; faster at every size above
  if (a.K <= 32 && d->R * d->W * d->Cin < 0x7fffffffLL && d->Cout <= 65535 * 32) {
    a.set_divisors();
    hipStream_t st = (hipStream_t)stream;
    if (a.Ng <= 32) return a.K <= 16 ? conv_launch_fwd_few<1, 8>(a, st) : conv_launch_fwd_few<1, 16>(a, st);
    return a.K <= 16 ? conv_launch_fwd_few<2, 8>(a, st) : conv_launch_fwd_few<2, 16>(a, st);
  }
  return d->Cin % 8 == 0 ? conv_launch<CONV_FWD, true>(a, (hipStream_t)stream)
                         : conv_launch<CONV_FWD, false>(a, (hipStream_t)stream);
}

extern "C" int nbk_conv2d_dgrad(const nbk_conv_desc* d, const void* dy, const void* w, void* dx,
                                void* stream) {
  int rc = conv_check(d);
  if (rc) return rc;
  NBK_REQUIRE(dy && w && dx, "conv2d: null pointer");
  NBK_REQUIRE(d->act == NBK_ACT_NONE, "conv2d: an activation goes with the forward product only");
  ConvArgs a;
  a.d = *d;
  a.a = (const float*)dy; a.b = (const float*)w; a.bias = nullptr; a.out = (float*)dx;
  a.M = d->N * d->H * d->W; a.Ng = d->Cin; a.K = d->R * d->S * d->Cout;
  a.splits = 1; a.k_per_split = (a.K + 15) / 16 * 16;
  if (a.K == 1) return conv_launch_outer<CONV_DGRAD>(a, (hipStream_t)stream);
  return d->Cout % 8 == 0 ? conv_launch<CONV_DGRAD, true>(a, (hipStream_t)stream)
                          : conv_launch<CONV_DGRAD, false>(a, (hipStream_t)stream);
}

// K split of the filter-gradient product: as many workgroups as the GPU holds at once (two per
// CU) and no more -- a handful beyond that would run as a second round behind the first and
// nearly double the launch (515 workgroups for 512 places: 129 us, 500: 90) --, at least four
// K steps each.
static void wgrad_split(const nbk_conv_desc* d, int* splits, int64_t* k_per_split) {
  const int64_t M = d->R * d->S * d->Cin, K = d->N * d->Ho * d->Wo;
  // (conv_launch_wgrad's tiles: 64 x 64 out of bf16 parts.  Slices for tiles of 128 gave those up to four rounds of
  // workgroups on short slices: us, 81 x 14 x 14, 140 -> 114 channels at stride 2 51 / 37, 16 x 28 x 28, 50 -> 50 38 / 29, 64 x
  // 28 x 28, 30 -> 60 63 / 48.  A CU holds three: for two 41 / 30 / 54, for four 41 / 38 / 57)
  const int64_t edge = M > 32 && (d->Cin % 8 != 0 || d->Cout % 8 != 0) ? 64 : 128;
  const int64_t tiles = ((M + edge - 1) / edge) * ((d->Cout + edge - 1) / edge);
  int64_t want = (edge == 64 ? 3 : 2) * (int64_t)nbk_num_cus() / tiles;
  const int64_t most = K / 64 > 0 ? K / 64 : 1;
  if (want > most) want = most;
  if (want < 1) want = 1;
  int64_t kps = (K + want - 1) / want;
  kps = (kps + 15) / 16 * 16;
  *k_per_split = kps;
  *splits = (int)((K + kps - 1) / kps);
}

extern "C" int64_t nbk_conv2d_wgrad_workspace(const nbk_conv_desc* d) {
  if (conv_check(d) != NBK_OK) return -1;
  int splits;
  int64_t kps;
  wgrad_split(d, &splits, &kps);
  if (splits <= 1) return 0;
  return (int64_t)splits * d->R * d->S * d->Cin * d->Cout * (int64_t)sizeof(float);
}

extern "C" int nbk_conv2d_wgrad(const nbk_conv_desc* d, const void* x, const void* dy, void* dw,
                                void* workspace, int64_t workspace_bytes, void* stream) {
  int rc = conv_check(d);
  if (rc) return rc;
  NBK_REQUIRE(x && dy && dw, "conv2d: null pointer");
  NBK_REQUIRE(d->act == NBK_ACT_NONE, "conv2d: an activation goes with the forward product only");
  ConvArgs a;
  a.d = *d;
  a.a = (const float*)x; a.b = (const float*)dy; a.bias = nullptr; a.out = (float*)dw;
  a.M = d->R * d->S * d->Cin; a.Ng = d->Cout; a.K = d->N * d->Ho * d->Wo;
  int splits;
  int64_t kps;
  wgrad_split(d, &splits, &kps);
  const int64_t need = (int64_t)splits * a.M * a.Ng * (int64_t)sizeof(float);
  if (splits > 1 && (workspace == nullptr || workspace_bytes < need || !aligned16(workspace))) {
    splits = 1;  // no room for partial sums: one pass over all of K
    kps = (a.K + 15) / 16 * 16;
  }
  a.splits = splits;
  a.k_per_split = kps;
  if (splits > 1) a.out = (float*)workspace;
  const bool fast = d->Cin % 8 == 0 && d->Cout % 8 == 0 && aligned16(x) && aligned16(dy);
  rc = conv_launch_wgrad(a, fast, (hipStream_t)stream);
  if (rc || splits == 1) return rc;
  const int64_t n = a.M * a.Ng;
  auto sum = [&](auto kern, int cols) {
    hipLaunchKernelGGL(kern, dim3((unsigned)((n + cols - 1) / cols)), dim3(256), 0, (hipStream_t)stream,
                       (const float*)workspace, (float*)dw, n, splits);
  };
  // (the fewer results, the fewer lanes to add them.  us with the product, one lane a sum / these: 64 x 32 x 32, 3 -> 64
  // channels (1728 results, 512 slices) 43 / 23, 50 x 28 x 28, 1 -> 24 35 / 17.6, 50 x 14 x 14, 24 -> 40 17.7 / 14.9; by four
  // 50 x 14 x 14, 40 -> 72 29.4 / 26.8, 64 x 32 x 32, 64 -> 128 109 / 107; 128 -> 256 is the same either way)
  if (n <= 64 * (int64_t)nbk_num_cus()) sum(conv_sum_partials<16>, 16);
  else if (n <= 512 * (int64_t)nbk_num_cus()) sum(conv_sum_partials<4>, 64);
  else sum(conv_sum_partials<1>, 256);
  return nbk_check_launch("conv_sum_partials");
}
