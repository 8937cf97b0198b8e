// Row-program interpreter: fused elementwise chains and last-axis reductions for which the
// library carries no compiled kernel.
//
// The host decodes a program once (rp_vm_decode; the result is kept by the program's contents):
// values that several phases of a program compute are computed once, constants leave the row
// loop, inputs become slots that are requested together, registers are assigned anew.  One kernel
// template runs it:
//   * ROW: a row is held in registers by a workgroup, one 4-column chunk per lane, or two where the
//     program needs few registers; SUB: by 1 to 32 lanes of a wavefront, so that short rows share a wavefront;
//   * LOOP: longer rows, one workgroup per row, segment by segment over the chunks;
//   * FLAT: programs without reductions, one chunk per lane.
// What bounds them is decoding, not memory: an instruction costs a wavefront some 30 scalar instructions
// and branches, a request of the scalar cache, and for every chunk 12 register moves with a wave-uniform
// index beside the 4 operations that compute.  So what helps is to run fewer instructions per element (two
// chunks a lane share all of the scalar part), to find the commonest ones by few comparisons, and never to
// wait inside one: the next instruction is requested behind the wait for the present one, and the inputs
// of a row together at its start, without a branch between them, into the first registers (an interpreted
// load writes a register chosen at run time and has to wait for its own data).  Measured over 6001 rows of
// 1003 floats, of 11.7 wavefronts a SIMD: a product 1.94 us with one chunk a lane, 0.75 with two; a
// reduction 7.4, then 3.5; a step of two programs (layer norm, gate, softmax, squared error and their
// gradients) 249 us, then 159; 4096 rows of 12000 in a loop (one chunk) 3090, then 2300.
#include "rowprog_vm.h"
#include "rowprog_device.h"
#include <stddef.h>
#include <algorithm>
#include <memory>
#include <mutex>
#include <string>
#include <type_traits>
#include <unordered_map>
#include <vector>

enum { K_FLAT = 0, K_SUB = 1, K_ROW = 2, K_LOOP = 3 };
// A launch's `flags`: every input that is requested ahead has four bytes an element; C is no multiple of 4.
enum { RPVM_WORDS = 1, RPVM_RAGGED = 2 };
// What a launch writes into rp_vm_ins::two so that the commonest instructions are found by one or two
// comparisons: products, sums and differences of two vectors, or of a vector and a scalar; stores of contiguous
// elements of four bytes, or in bfloat16.
enum { RPVM_TWO_WORDS = 1, RPVM_TWO_BF16 = 2, RPVM_TWO_MUL = 4, RPVM_TWO_MUL_S = 8 };
#define RPVM_WIDE_REGS 8  /* vector registers of the form with two chunks a lane */

typedef float vf16 __attribute__((ext_vector_type(16)));
typedef float vf32 __attribute__((ext_vector_type(32)));
typedef uint32_t rp_u4b __attribute__((ext_vector_type(4), aligned(1)));
static_assert(NBK_RP_NSCL == 16, "the scalar file is a 16-wide vector");

// The program is read where the launch put it, in the kernel arguments, through the scalar cache
// (a dependent read takes about 60 ns there, and the next instruction is read ahead).
typedef const __attribute__((address_space(4))) rp_vm* rp_prog;
typedef const __attribute__((address_space(4))) uint64_t* rp_pc;
__device__ __forceinline__ rp_vm_ins rp_fetch(rp_pc pc) { return __builtin_bit_cast(rp_vm_ins, *pc); }
static_assert(sizeof(rp_vm_ins) == 8 && offsetof(rp_vm, ins) % 8 == 0, "instructions are read with 8-byte accesses");
static_assert(sizeof(rp_vm) + 24 <= 4096, "kernel arguments");

// (the compiler has no builtin of that name)
__device__ int rp_writelane(int v, int lane, int old) __asm("llvm.amdgcn.writelane.i32");

// Vector registers: N chunks each of 16 / N registers.  Two chunks: a chunk's components side by side, as a load
// leaves them.
template <int N> struct RpFile;
template <> struct RpFile<1> {
  vf16 x, y, z, w;
  __device__ __forceinline__ float4 get(int i, int) const { return make_float4(x[i], y[i], z[i], w[i]); }
  __device__ __forceinline__ void set(int i, int, float4 v) { x[i] = v.x; y[i] = v.y; z[i] = v.z; w[i] = v.w; }
};
template <> struct RpFile<2> {
  vf32 c[2];
  __device__ __forceinline__ float4 get(int i, int j) const {
    return make_float4(c[j][i * 4], c[j][i * 4 + 1], c[j][i * 4 + 2], c[j][i * 4 + 3]);
  }
  __device__ __forceinline__ void set(int i, int j, float4 v) {
    c[j][i * 4] = v.x; c[j][i * 4 + 1] = v.y; c[j][i * 4 + 2] = v.z; c[j][i * 4 + 3] = v.w;
  }
};

// Per-row scalars.  Where a wavefront works on one row they are uniform and sixteen of them
// share one vector register, a lane each; else every lane holds its own row's.
template <bool UNIFORM> struct RpScalars;
template <> struct RpScalars<true> {
  int v;
  __device__ __forceinline__ float get(int i) const { return __int_as_float(__builtin_amdgcn_readlane(v, i)); }
  __device__ __forceinline__ void set(int i, float x) {
    // (a vector register's number, or none: a lane that no scalar has)
    v = rp_writelane(__builtin_amdgcn_readfirstlane(__float_as_int(x)), i & 63, v);
  }
};
template <> struct RpScalars<false> {
  vf16 v;
  __device__ __forceinline__ float get(int i) const { return v[i]; }
  __device__ __forceinline__ void set(int i, float x) {
    const bool hit = i >= 0 && i < NBK_RP_NSCL;
    const float keep = v[0];
    v[hit ? i : 0] = hit ? x : keep;
  }
};

__device__ __forceinline__ int64_t rp_off(rp_prog P, int k, const uint32_t* li) {
  const auto& o = P->operand[k];
  const int n_lead = P->n_lead;
  int64_t off = 0;
  if (n_lead > 0) off = (int64_t)li[0] * o.lead_stride[0];
  if (n_lead > 1) off += (int64_t)li[1] * o.lead_stride[1];
  if (n_lead > 2) off += (int64_t)li[2] * o.lead_stride[2] + (int64_t)li[3] * o.lead_stride[3];
  return off;
}

// The instruction loop has wave-uniform branches only: one divergent branch in it, and the
// compiler turns the whole dispatch into predicated flow (three scalar instructions more at every
// node).  So lanes outside a row store nothing by an execution mask set for one instruction, load
// from an address inside it and reduce the identity.
#define RPVM_STORE(INSN, PTR, DATA, MASK)                                                       \
  {                                                                                             \
    uint64_t saved_;                                                                            \
    asm volatile("s_and_saveexec_b64 %0, %1\n\t" INSN " %2, %3, off\n\ts_mov_b64 exec, %0\n\ts_nop 1" \
                 : "=&s"(saved_) : "s"(MASK), "v"(PTR), "v"(DATA) : "memory", "scc");           \
  }
typedef uint32_t rp_v4 __attribute__((ext_vector_type(4)));
typedef uint32_t rp_v2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint64_t rp_ballot(bool b) { return __builtin_amdgcn_ballot_w64(b); }
__device__ __forceinline__ uint32_t rp_pack_bf16(float a, float b) {
  return (uint32_t)nbk_f32_to_bf16(a) | ((uint32_t)nbk_f32_to_bf16(b) << 16);
}
// One element to `p`, in the lanes of `mask`.
__device__ __forceinline__ void rp_store1_masked(void* p, int dt, float v, uint64_t mask) {
  if (dt == NBK_F32 || dt == NBK_I32) {
    RPVM_STORE("global_store_dword", p, v, mask)
  } else if (dt == NBK_BF16 || dt == NBK_F16) {
    uint32_t u = dt == NBK_BF16 ? nbk_f32_to_bf16(v) : (uint32_t)__builtin_bit_cast(uint16_t, __float2half(v));
    RPVM_STORE("global_store_short", p, u, mask)
  } else if (dt == NBK_I64) {
    const int i = rp_int(v);
    const rp_v2 u = {(uint32_t)i, (uint32_t)(i >> 31)};
    RPVM_STORE("global_store_dwordx2", p, u, mask)
  } else {
    const uint32_t u = v != 0.f;
    RPVM_STORE("global_store_byte", p, u, mask)
  }
}
// A chunk of `valid` contiguous columns of four bytes each to `p`.
__device__ __forceinline__ void rp_store4_words(char* p, int valid, float4 v) {
  const uint64_t whole = rp_ballot(valid == 4), part = rp_ballot(valid > 0) & ~whole;
  const rp_v4 u = {__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z), __float_as_uint(v.w)};
  RPVM_STORE("global_store_dwordx4", p, u, whole)
  if (part) {
    RPVM_STORE("global_store_dword", p, v.x, part)
    RPVM_STORE("global_store_dword", p + 4, v.y, rp_ballot(valid > 1) & part)
    RPVM_STORE("global_store_dword", p + 8, v.z, rp_ballot(valid > 2) & part)
  }
}
// The same in bfloat16.
__device__ __forceinline__ void rp_store4_bf16(char* p, int valid, float4 v) {
  const uint64_t whole = rp_ballot(valid == 4), part = rp_ballot(valid > 0) & ~whole;
  const rp_v2 u = {rp_pack_bf16(v.x, v.y), rp_pack_bf16(v.z, v.w)};
  RPVM_STORE("global_store_dwordx2", p, u, whole)
  if (part) {
    const uint32_t second = u.x >> 16;
    RPVM_STORE("global_store_short", p, u.x, part)
    RPVM_STORE("global_store_short", p + 2, second, rp_ballot(valid > 1) & part)
    RPVM_STORE("global_store_short", p + 4, u.y, rp_ballot(valid > 2) & part)
  }
}
// A chunk of `valid` columns of stride `cs` elements to `p`.
__device__ __forceinline__ void rp_store4_masked(char* p, int dt, int64_t cs, int valid, float4 v) {
  const int64_t es = dt == NBK_U8 ? 1 : (dt == NBK_BF16 || dt == NBK_F16) ? 2 : dt == NBK_I64 ? 8 : 4;
  uint64_t whole = 0;
  if (cs == 1) {
    whole = rp_ballot(valid == 4);
    if (dt == NBK_F32 || dt == NBK_I32) {
      const rp_v4 u = {__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z), __float_as_uint(v.w)};
      RPVM_STORE("global_store_dwordx4", p, u, whole)
    } else if (dt == NBK_BF16) {
      const rp_v2 u = {rp_pack_bf16(v.x, v.y), rp_pack_bf16(v.z, v.w)};
      RPVM_STORE("global_store_dwordx2", p, u, whole)
    } else if (dt == NBK_F16) {
      const rp_v2 u = {__builtin_bit_cast(uint32_t, __floats2half2_rn(v.x, v.y)),
                       __builtin_bit_cast(uint32_t, __floats2half2_rn(v.z, v.w))};
      RPVM_STORE("global_store_dwordx2", p, u, whole)
    } else if (dt == NBK_U8) {
      const uint32_t u = (uint32_t)(v.x != 0.f) | ((uint32_t)(v.y != 0.f) << 8) | ((uint32_t)(v.z != 0.f) << 16) |
                         ((uint32_t)(v.w != 0.f) << 24);
      RPVM_STORE("global_store_dword", p, u, whole)
    } else {
      whole = 0;
    }
  }
  if (rp_ballot(valid > 0) & ~whole) {
    rp_store1_masked(p, dt, v.x, rp_ballot(valid > 0) & ~whole);
    rp_store1_masked(p + cs * es, dt, v.y, rp_ballot(valid > 1) & ~whole);
    rp_store1_masked(p + 2 * cs * es, dt, v.z, rp_ballot(valid > 2) & ~whole);
    rp_store1_masked(p + 3 * cs * es, dt, v.w, rp_ballot(valid > 3) & ~whole);
  }
}
// A chunk at element `e`, column by column; columns past the row's end repeat its last.
__device__ __forceinline__ float4 rp_load4_inside(const void* p, int dt, int64_t e, int64_t cs, int valid) {
  const int last = valid > 1 ? valid - 1 : 0;
  return make_float4(rp_load1(p, e, dt), rp_load1(p, e + cs * (last < 1 ? last : 1), dt),
                     rp_load1(p, e + cs * (last < 2 ? last : 2), dt), rp_load1(p, e + cs * last, dt));
}
__device__ __forceinline__ float rp_acc4_inside(float acc, float4 a, int kind, int valid) {
  const float id = rp_identity(kind);
  acc = rp_combine(acc, valid > 0 ? a.x : id, kind);
  acc = rp_combine(acc, valid > 1 ? a.y : id, kind);
  acc = rp_combine(acc, valid > 2 ? a.z : id, kind);
  return rp_combine(acc, valid > 3 ? a.w : id, kind);
}
// This lane's part of a reduction over the row.
__device__ __forceinline__ float rp_part(float4 a, int kind, int valid) {
  return rp_acc4_inside(rp_identity(kind), a, kind, valid);
}

// Lane totals over groups of `lanes` (1 .. 32) neighbouring lanes.
__device__ __forceinline__ float rp_group_reduce(float v, int kind, int lanes) {
  if (lanes > 1) v = rp_dpp_step<0xB1, 0xf>(v, kind);
  if (lanes > 2) v = rp_dpp_step<0x4E, 0xf>(v, kind);
  if (lanes > 4) v = rp_dpp_step<0x141, 0xf>(v, kind);
  if (lanes > 8) v = rp_dpp_step<0x140, 0xf>(v, kind);
  if (lanes > 16) v = rp_combine(v, __shfl_xor(v, 16), kind);
  return v;
}
// Total over the first sixteen lanes (one partial per wavefront of the workgroup), uniform.
__device__ __forceinline__ float rp_reduce16(float v, int kind) {
  v = rp_dpp_step<0xB1, 0xf>(v, kind);
  v = rp_dpp_step<0x4E, 0xf>(v, kind);
  v = rp_dpp_step<0x141, 0xf>(v, kind);
  v = rp_dpp_step<0x140, 0xf>(v, kind);
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

#define RPVM_U(OP) case OP: RPVM_ALL(r.v[j] = rp_un4<OP>(r.v[j])) break;
#define RPVM_B(OP) case OP: RPVM_ALL(r.v[j] = rp_bin4<OP>(r.v[j], b.v[j])) break;
#define RPVM_S1(OP) case OP: x = rp_unary(OP, a); break;
#define RPVM_S2(OP) case OP: x = rp_binary(OP, a, b); break;
// Components one at a time, for functions whose code would fill the instruction cache four times.
#define RPVM_EACH(EXPR)                                                                     \
  _Pragma("unroll 1") for (int k = 0; k < 4 * N; ++k) {                                     \
    float t, u;                                                                             \
    RPVM_ALL(if (k == 4 * j) { t = r.v[j].x; u = b.v[j].x; }                                \
             if (k == 4 * j + 1) { t = r.v[j].y; u = b.v[j].y; }                            \
             if (k == 4 * j + 2) { t = r.v[j].z; u = b.v[j].z; }                            \
             if (k == 4 * j + 3) { t = r.v[j].w; u = b.v[j].w; })                           \
    (void)u;                                                                                \
    const float v = EXPR;                                                                   \
    RPVM_ALL(if (k == 4 * j) r.v[j].x = v;                                                  \
             if (k == 4 * j + 1) r.v[j].y = v;                                              \
             if (k == 4 * j + 2) r.v[j].z = v;                                              \
             if (k == 4 * j + 3) r.v[j].w = v;)                                             \
  }

__device__ __forceinline__ float rp_rare_unary(int op, float t) {
  switch (op) {
    case NBK_OP_LOG: return rp_unary(NBK_OP_LOG, t);
    case NBK_OP_ERF: return rp_unary(NBK_OP_ERF, t);
    case NBK_OP_GELU: return rp_unary(NBK_OP_GELU, t);
    case NBK_OP_DGELU: return rp_unary(NBK_OP_DGELU, t);
    case NBK_OP_TANH: return rp_unary(NBK_OP_TANH, t);
    case NBK_OP_SIN: return rp_unary(NBK_OP_SIN, t);
    case NBK_OP_COS: return rp_unary(NBK_OP_COS, t);
    default: return t;
  }
}

// `N` chunks a lane share every decoded instruction.  With two a lane holds 64 registers of values and as many
// of other things, so three wavefronts fit a SIMD (four with one chunk; forced to four it spills 38).
template <int K, bool RARE, int N>
__global__ __launch_bounds__(K == K_ROW ? 1024 / N : K == K_LOOP ? 512 : 256, RARE || N > 1 ? 3 : 4)
void rp_vm_kernel(const rp_vm, uint32_t rows, uint32_t cpr, uint64_t total, uint32_t flags) {
  constexpr bool UNIFORM = K == K_ROW || K == K_LOOP;
  static_assert(N == 1 || K == K_ROW, "a lane's chunks are of one row");
  static_assert(RPVM_SLOTS <= 16 / N && 16 / N == (N == 1 ? NBK_RP_NVEC : RPVM_WIDE_REGS), "inputs come into the first registers");
  typedef typename std::conditional<K == K_ROW || K == K_SUB, int, int64_t>::type column;  // (such rows have up to 4096)
  __shared__ float red_buf[128];
  const rp_prog P = (rp_prog)__builtin_amdgcn_kernarg_segment_ptr();  // (the first argument)
  RpScalars<UNIFORM> S = {};
  float acc[NBK_RP_NACC] = {0.f, 0.f, 0.f, 0.f};
  int phase = 0;
  const int lanes = K == K_SUB ? P->lanes : 1;
  const int nw = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t C = P->C;
  int first = 0;  // (what no row changes runs with the first)

  // A row, a group of rows or 256 chunks at a time.
  const uint64_t n_at = K == K_FLAT ? (total + 255) / 256
                        : K == K_SUB ? ((uint64_t)rows * (uint32_t)lanes + 255) / 256 : rows;
  for (uint64_t at = blockIdx.x; at < n_at; at += gridDim.x) {
    // where this lane is: its row, the row's leading indices, its columns
    uint32_t row, cc = threadIdx.x;
    bool inside = true;
    if (K == K_FLAT) {
      uint64_t g = at * 256 + threadIdx.x;
      inside = g < total;
      if (!inside) g = total - 1;
      row = 0;
      cc = (uint32_t)g;
      if (P->n_lead > 0 && cpr < total) {
        row = total <= 0xffffffffull ? (uint32_t)g / cpr : (uint32_t)(g / cpr);
        cc = (uint32_t)(g - (uint64_t)row * cpr);
      }
    } else if (K == K_SUB) {
      row = (uint32_t)at * (256u / (uint32_t)lanes) + threadIdx.x / (uint32_t)lanes;
      inside = row < rows;
      if (!inside) row = rows - 1;
      cc = threadIdx.x & (uint32_t)(lanes - 1);
    } else {
      row = (uint32_t)at;
    }
    const bool writer = cc == 0 && inside;
    uint32_t li[NBK_RP_MAX_LEAD];
    rp_decompose_row(row, P->n_lead, (uint32_t)P->lead_dim[1], (uint32_t)P->lead_dim[2], (uint32_t)P->lead_dim[3], li);

    // scalars of the row
    {
      float rs[RPVM_ROW_SLOTS];
#pragma unroll
      for (int k = 0; k < RPVM_ROW_SLOTS; ++k) {
        rs[k] = 0.f;
        if (k < P->n_row_slots) {
          const int i = P->row_slots[k];
          rs[k] = ((const float*)P->operand[i].ptr)[rp_off(P, i, li)];
        }
      }
      if (P->n_row_slots > 0) {
#pragma unroll
        for (int k = 0; k < RPVM_ROW_SLOTS; ++k) S.set((int)P->row_dst[k] - RPVM_SCALAR, rs[k]);
      }
    }

    int q1 = K == K_LOOP ? first : P->n_ins;
    do {
      int q0 = first, s0 = 0, n_in = P->n_slots;
      int64_t c0 = 0, c_end = 1;
      if (K == K_LOOP) {  // the next segment of the row
        const rp_vm_ins seg = rp_fetch((rp_pc)P->ins + q1);
        q0 = q1 + 1;
        q1 = q0 + seg.aux;
        s0 = seg.c;
        n_in = seg.a;
        if (seg.b) c_end = C;
      }
      do {
        column col[N];
        int valid[N];
#pragma unroll
        for (int j = 0; j < N; ++j) {
          col[j] = (column)c0 + (((column)cc + (column)(j * (int)blockDim.x)) << 2);
          const column left = (column)C - col[j];
          valid[j] = !inside || left <= 0 ? 0 : left >= 4 ? 4 : (int)left;
        }
        RpFile<N> F;
        // The inputs: 16 bytes from where the lane is, or the last 16 of the row where its end is nearer,
        // into the first registers.  One form of load for every type and every lane keeps the requests of
        // a row in one straight line; where every input has four bytes an element (nearly all programs)
        // nothing is asked about types.
        {
          const bool words = (flags & RPVM_WORDS) != 0, ragged = (flags & RPVM_RAGGED) != 0;
          auto operand_of = [&](int k) { return K == K_LOOP ? (int)P->slots[s0 + k] : k; };
          auto shift_of = [&](int k) {
            if (words) return 2;
            const int dt = P->operand[operand_of(k)].dtype;
            return dt == NBK_U8 ? 0 : (dt == NBK_BF16 || dt == NBK_F16) ? 1 : 2;
          };
          rp_u4b bits[RPVM_SLOTS][N];
#pragma unroll
          for (int k = 0; k < RPVM_SLOTS; ++k)
            if (k < n_in) {
              const int i = operand_of(k), es = shift_of(k);
              const char* at_row = (const char*)P->operand[i].ptr + (rp_off(P, i, li) << es);
              const column b1 = ((column)C << es) - 16;
#pragma unroll
              for (int j = 0; j < N; ++j) {
                const column b0 = col[j] << es;
                bits[k][j] = *(const rp_u4b*)(at_row + (b0 > b1 ? b1 : b0));
              }
            }
#pragma unroll
          for (int k = 0; k < RPVM_SLOTS; ++k)
            if (k < n_in) {
              const int es = shift_of(k);
              const column b1 = ((column)C << es) - 16;
#pragma unroll
              for (int j = 0; j < N; ++j) {
                uint32_t u0 = bits[k][j].x, u1 = bits[k][j].y, u2 = bits[k][j].z, u3 = bits[k][j].w;
                if (ragged || !words) {  // (else the lanes past the row hold what nobody reads)
                  const column past = (col[j] << es) - b1;
                  if (rp_ballot(past > 0)) {  // (lanes at the end of a row)
                    const int back = past > 15 ? 15 : past > 0 ? (int)past : 0;
                    if (back & 8) { u0 = u2; u1 = u3; }
                    if (back & 4) { u0 = u1; u1 = u2; u2 = u3; }
                    const uint32_t sh = (uint32_t)back & 3;
                    u0 = __builtin_amdgcn_alignbyte(u1, u0, sh);
                    u1 = __builtin_amdgcn_alignbyte(u2, u1, sh);
                  }
                  if (!words) {
                    const int dt = P->operand[operand_of(k)].dtype;
                    if (dt == NBK_BF16) {
                      u3 = u1 & 0xffff0000u; u2 = u1 << 16; u1 = u0 & 0xffff0000u; u0 <<= 16;
                    } else if (dt == NBK_F16) {
                      const float2 f0 = __half22float2(__builtin_bit_cast(__half2, u0)),
                                   f1 = __half22float2(__builtin_bit_cast(__half2, u1));
                      u0 = __float_as_uint(f0.x); u1 = __float_as_uint(f0.y);
                      u2 = __float_as_uint(f1.x); u3 = __float_as_uint(f1.y);
                    } else if (dt == NBK_U8) {
                      u3 = __float_as_uint((float)(u0 >> 24)); u2 = __float_as_uint((float)((u0 >> 16) & 0xff));
                      u1 = __float_as_uint((float)((u0 >> 8) & 0xff)); u0 = __float_as_uint((float)(u0 & 0xff));
                    }
                  }
                }
                F.set(k, j, make_float4(__uint_as_float(u0), __uint_as_float(u1), __uint_as_float(u2), __uint_as_float(u3)));
              }
            }
        }
        struct Chunks { float4 v[N]; };
        auto get_vec = [&](int i) {
          Chunks g;
#pragma unroll
          for (int j = 0; j < N; ++j) g.v[j] = F.get(i, j);
          return g;
        };
        auto splat = [&](int i) {
          Chunks g;
          const float s = S.get(i - RPVM_SCALAR);
#pragma unroll
          for (int j = 0; j < N; ++j) g.v[j] = make_float4(s, s, s, s);
          return g;
        };
        auto get = [&](int i) { return i < RPVM_SCALAR ? get_vec(i) : splat(i); };
#define RPVM_ALL(EXPR) { _Pragma("unroll") for (int j = 0; j < N; ++j) { EXPR; } }
        rp_pc pc = (rp_pc)P->ins + q0;  // (of the instruction that is read ahead)
        rp_vm_ins nxt = rp_fetch(pc);
#pragma unroll 1
        for (int q = q0; q < q1; ++q) {
          const rp_vm_ins in = nxt;
          // (waits for this instruction before the next is requested: the two would be waited for together)
          __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
          ++pc;
          asm volatile("" : "+s"(pc));
          nxt = rp_fetch(pc);
          const int op = in.op;
          Chunks r;
          int d = in.dst;
          float sv = 0.f;
          auto set_scalar = [&](const rp_vm_ins& by, float x) {
            if (UNIFORM) S.set((int)by.dst - RPVM_SCALAR, x);
            else sv = x;
          };
          if (in.two >= RPVM_TWO_MUL) {  // the commonest: of two vectors, or of a vector and a scalar
            r = get_vec(in.a);
            const Chunks b = in.two < RPVM_TWO_MUL_S ? get_vec(in.b) : splat(in.b);
            const int what = in.two & 3;
            if (what == 0) RPVM_ALL(r.v[j] = rp_bin4<NBK_OP_MUL>(r.v[j], b.v[j]))
            else if (what == 1) RPVM_ALL(r.v[j] = rp_bin4<NBK_OP_ADD>(r.v[j], b.v[j]))
            else RPVM_ALL(r.v[j] = rp_bin4<NBK_OP_SUB>(r.v[j], b.v[j]))
          } else {
          RPVM_ALL(r.v[j] = make_float4(0.f, 0.f, 0.f, 0.f))
          if (op >= NBK_OP_MOV && in.dst >= RPVM_SCALAR) {  // of scalars
            const float a = S.get(in.a - RPVM_SCALAR), b = S.get(in.b - RPVM_SCALAR), c = S.get(in.c - RPVM_SCALAR);
            float x = a;
            switch (op) {
              case NBK_OP_WHERE: x = rp_where(a, b, c); break;
              case NBK_OP_FMA: x = fmaf(a, b, c); break;
              RPVM_S1(NBK_OP_NEG) RPVM_S1(NBK_OP_RELU) RPVM_S1(NBK_OP_EXP) RPVM_S1(NBK_OP_SQRT) RPVM_S1(NBK_OP_RSQRT)
              RPVM_S1(NBK_OP_SIGMOID) RPVM_S1(NBK_OP_ABS) RPVM_S1(NBK_OP_RBF16) RPVM_S1(NBK_OP_NOT) RPVM_S1(NBK_OP_TRUNC)
              RPVM_S1(NBK_OP_NEZ) RPVM_S1(NBK_OP_INEG) RPVM_S1(NBK_OP_IABS) RPVM_S1(NBK_OP_IRELU) RPVM_S1(NBK_OP_I2F)
              RPVM_S1(NBK_OP_F2I) RPVM_S1(NBK_OP_INEZ)
              RPVM_S2(NBK_OP_ADD) RPVM_S2(NBK_OP_SUB) RPVM_S2(NBK_OP_MUL) RPVM_S2(NBK_OP_DIV) RPVM_S2(NBK_OP_MAX)
              RPVM_S2(NBK_OP_MIN) RPVM_S2(NBK_OP_GT) RPVM_S2(NBK_OP_GE) RPVM_S2(NBK_OP_EQ) RPVM_S2(NBK_OP_NE)
              RPVM_S2(NBK_OP_LT) RPVM_S2(NBK_OP_LE) RPVM_S2(NBK_OP_AND) RPVM_S2(NBK_OP_OR) RPVM_S2(NBK_OP_IADD)
              RPVM_S2(NBK_OP_ISUB) RPVM_S2(NBK_OP_IMUL) RPVM_S2(NBK_OP_IMAX) RPVM_S2(NBK_OP_IMIN) RPVM_S2(NBK_OP_IGT)
              RPVM_S2(NBK_OP_IGE) RPVM_S2(NBK_OP_IEQ) RPVM_S2(NBK_OP_INE) RPVM_S2(NBK_OP_ILT) RPVM_S2(NBK_OP_ILE)
              default:
                if (RARE) x = op == NBK_OP_POW ? powf(a, b) : rp_rare_unary(op, a);
            }
            set_scalar(in, x);
          } else if (op >= NBK_OP_MOV) {
            r = get(in.a);
            if (in.two) {
              const Chunks b = get(in.b);
              switch (op) {
                RPVM_B(NBK_OP_ADD) RPVM_B(NBK_OP_SUB) RPVM_B(NBK_OP_MUL) RPVM_B(NBK_OP_DIV) RPVM_B(NBK_OP_MAX)
                RPVM_B(NBK_OP_MIN) RPVM_B(NBK_OP_GT) RPVM_B(NBK_OP_GE) RPVM_B(NBK_OP_EQ) RPVM_B(NBK_OP_NE)
                RPVM_B(NBK_OP_LT) RPVM_B(NBK_OP_LE) RPVM_B(NBK_OP_AND) RPVM_B(NBK_OP_OR) RPVM_B(NBK_OP_IADD)
                RPVM_B(NBK_OP_ISUB) RPVM_B(NBK_OP_IMUL) RPVM_B(NBK_OP_IMAX) RPVM_B(NBK_OP_IMIN) RPVM_B(NBK_OP_IGT)
                RPVM_B(NBK_OP_IGE) RPVM_B(NBK_OP_IEQ) RPVM_B(NBK_OP_INE) RPVM_B(NBK_OP_ILT) RPVM_B(NBK_OP_ILE)
                case NBK_OP_WHERE: {
                  const Chunks c = get(in.c);
                  RPVM_ALL(r.v[j] = rp_where4(r.v[j], b.v[j], c.v[j]))
                  break;
                }
                case NBK_OP_FMA: {
                  const Chunks c = get(in.c);
                  RPVM_ALL(r.v[j] = rp_fma4(r.v[j], b.v[j], c.v[j]))
                  break;
                }
                default:
                  if (RARE) RPVM_EACH(powf(t, u))
              }
            } else {
              const Chunks& b = r;
              switch (op) {
                RPVM_U(NBK_OP_NEG) RPVM_U(NBK_OP_RELU) RPVM_U(NBK_OP_EXP) RPVM_U(NBK_OP_SQRT)
                RPVM_U(NBK_OP_RSQRT) RPVM_U(NBK_OP_SIGMOID) RPVM_U(NBK_OP_ABS) RPVM_U(NBK_OP_RBF16) RPVM_U(NBK_OP_NOT)
                RPVM_U(NBK_OP_TRUNC) RPVM_U(NBK_OP_NEZ) RPVM_U(NBK_OP_INEG) RPVM_U(NBK_OP_IABS) RPVM_U(NBK_OP_IRELU)
                RPVM_U(NBK_OP_I2F) RPVM_U(NBK_OP_F2I) RPVM_U(NBK_OP_INEZ)
                default: if (RARE && op != NBK_OP_MOV) RPVM_EACH(rp_rare_unary(op, t))
              }
            }
          } else if (op == RPVM_STG) {
            const auto& o = P->operand[in.c];
            r = get(in.a);
            if (in.two == RPVM_TWO_WORDS) {  // (four bytes an element, contiguous)
              char* at_row = (char*)o.ptr + (rp_off(P, in.c, li) << 2);
#pragma unroll
              for (int j = 0; j < N; ++j) rp_store4_words(at_row + ((int64_t)col[j] << 2), valid[j], r.v[j]);
            } else if (in.two == RPVM_TWO_BF16) {
              char* at_row = (char*)o.ptr + (rp_off(P, in.c, li) << 1);
#pragma unroll
              for (int j = 0; j < N; ++j) rp_store4_bf16(at_row + ((int64_t)col[j] << 1), valid[j], r.v[j]);
            } else {
              const int dt = o.dtype;
              const int64_t cs = o.col_stride, e = rp_off(P, in.c, li);
              const int64_t es = dt == NBK_U8 ? 1 : (dt == NBK_BF16 || dt == NBK_F16) ? 2 : dt == NBK_I64 ? 8 : 4;
#pragma unroll
              for (int j = 0; j < N; ++j)
                rp_store4_masked((char*)o.ptr + (e + col[j] * cs) * es, dt, cs, valid[j], r.v[j]);
            }
          } else if (K != K_FLAT && op == RPVM_RED) {
            // neighbouring reductions (at most 4); between the wavefronts of a workgroup they
            // share one barrier: each leaves its part in bank[k * 16 + wave], and two banks alternate
            const int n = UNIFORM ? in.aux : 1;
            float* bank = red_buf + ((phase++ & 1) << 6);
#pragma unroll 1
            for (int k = n - 1; k >= 0; --k) {
              const rp_vm_ins rk = k ? rp_fetch(pc + (k - 1)) : in;
              float v;
              if (K == K_LOOP) {
                v = rk.c == 0 ? acc[0] : rk.c == 1 ? acc[1] : rk.c == 2 ? acc[2] : acc[3];
              } else {
                r = get(rk.a);
                auto part = [&](int kind) {
                  v = rp_part(r.v[0], kind, valid[0]);
#pragma unroll
                  for (int j = 1; j < N; ++j) v = rp_combine(v, rp_part(r.v[j], kind, valid[j]), kind);
                };
                if (rk.b == NBK_RED_SUM) part(NBK_RED_SUM); else part(rk.b);
              }
              if (rk.b == NBK_RED_SUM) v = UNIFORM ? rp_wave_reduce(v, NBK_RED_SUM) : rp_group_reduce(v, NBK_RED_SUM, lanes);
              else v = UNIFORM ? rp_wave_reduce(v, rk.b) : rp_group_reduce(v, rk.b, lanes);
              if (UNIFORM && nw > 1) bank[k * 16 + wave] = v;  // (every lane the same)
              else set_scalar(rk, v);
            }
            if (UNIFORM && nw > 1) {
              rp_lds_barrier();
              const int ln = threadIdx.x & 15;
#pragma unroll 1
              for (int k = n - 1; k >= 0; --k) {
                const rp_vm_ins rk = k ? rp_fetch(pc + (k - 1)) : in;
                float part = bank[k * 16 + ln];
                asm volatile("" : "+v"(part));  // (read by every lane, not in a branch)
                part = ln < nw ? part : rp_identity(rk.b);
                set_scalar(rk, rk.b == NBK_RED_SUM ? rp_reduce16(part, NBK_RED_SUM) : rp_reduce16(part, rk.b));
              }
            }
            if (n > 1) {
              q += n - 1;
              pc += n - 1;
              nxt = rp_fetch(pc);
            }
          } else if (op == RPVM_LDG) {
            const auto& o = P->operand[in.c];
#pragma unroll
            for (int j = 0; j < N; ++j) {
              float4& t = r.v[j];
              t = rp_load4_inside(o.ptr, o.dtype, rp_off(P, in.c, li) + (valid[j] > 0 ? col[j] : 0) * o.col_stride,
                                  o.col_stride, valid[j]);
              // (waits here, so that the common tail has no load to wait for: it would wait for stores too)
              asm volatile("" : "+v"(t.x), "+v"(t.y), "+v"(t.z), "+v"(t.w));
            }
          } else if (op == RPVM_LDR) {
            const auto& o = P->operand[in.c];
            float x = rp_load1(o.ptr, rp_off(P, in.c, li), o.dtype);
            asm volatile("" : "+v"(x));
            set_scalar(in, x);
          } else if (op == RPVM_STR) {
            const auto& o = P->operand[in.c];
            const float v = S.get(in.a - RPVM_SCALAR);
            const int dt = o.dtype;
            const int64_t es = dt == NBK_U8 ? 1 : (dt == NBK_BF16 || dt == NBK_F16) ? 2 : dt == NBK_I64 ? 8 : 4;
            rp_store1_masked((char*)o.ptr + rp_off(P, in.c, li) * es, dt, v, rp_ballot(writer));
          } else if (op == RPVM_IMM) {
            set_scalar(in, P->imm[in.c]);
          } else if (op == RPVM_COLIDX) {
            RPVM_ALL(r.v[j] = rp_colidx4(col[j], in.c != 0))
          } else if (op == RPVM_LEADIDX) {
            const int k = in.c;
            const int v = (int)(k == 0 ? li[0] : k == 1 ? li[1] : k == 2 ? li[2] : li[3]);
            set_scalar(in, in.b != 0 ? rp_ibits(v) : (float)v);
          } else if (K == K_LOOP && op == RPVM_ACC) {
            r = get(in.a);
#pragma unroll
            for (int k = 0; k < NBK_RP_NACC; ++k)
              if (in.c == k) RPVM_ALL(acc[k] = rp_acc4_inside(acc[k], r.v[j], in.b, valid[j]))
          } else if (K == K_LOOP && op == RPVM_ACCINIT) {
#pragma unroll
            for (int k = 0; k < NBK_RP_NACC; ++k)
              if (in.c == k) acc[k] = rp_identity(in.b);
          }
            // Every instruction writes a register, one without such a result what is there already: a
            // write under a branch makes the compiler copy the whole file (16 moves) around it.
            if (in.dst >= NBK_RP_NVEC) {
              r = get_vec(0);
              d = 0;
            }
          }
          RPVM_ALL(F.set(d, j, r.v[j]))
          if (!UNIFORM) S.set((int)in.dst - RPVM_SCALAR, sv);
        }
        c0 += (int64_t)blockDim.x * (4 * N);
      } while (K == K_LOOP && c0 < c_end);
    } while (K == K_LOOP && q1 < P->n_ins);
    first = P->n_once;
  }
}

// ------------------------------------------------------------------ decoding (host)
namespace {

bool is_unary(int op) {
  return (op >= NBK_OP_MOV && op < NBK_OP_ADD) || op == NBK_OP_DGELU || op == NBK_OP_SIN || op == NBK_OP_COS ||
         (op >= NBK_OP_INEG && op <= NBK_OP_INEZ);
}

// Functions of many instructions and constants, compiled into kernels of their own: beside them
// the others would lose a third of their wavefronts to registers.
bool is_rare(int op) {
  return op == NBK_OP_LOG || op == NBK_OP_ERF || op == NBK_OP_GELU || op == NBK_OP_DGELU || op == NBK_OP_TANH ||
         op == NBK_OP_SIN || op == NBK_OP_COS || op == NBK_OP_POW;
}

// Whether an input can be requested ahead: contiguous columns, at least 16 bytes of them.
bool rp_vm_ahead(const nbk_rowprog* p, int operand) {
  const nbk_operand& o = p->operand[operand];
  return o.col_stride == 1 && o.dtype != NBK_I64 && p->C * nbk_dtype_size(o.dtype) >= 16;
}

// One computed value.  `op` is an rp_vm_op or an elementwise nbk_rp_op; a, b, c are values, x an
// operand, immediate, slot, axis or accumulator, y a dtype or reduction kind.
struct Val {
  int op = 0, a = -1, b = -1, c = -1, x = 0, y = 0;
  bool scalar = false, once = false, used = false;
  int reg = -1, last = -1;  // register, position of the last use
  int own = -1;             // the register the program gave it (level 2)
};
enum ItemKind { DEF, STG, STR, ACCINIT, ACC, BODY_BEGIN, BODY_END };
struct Item {
  ItemKind kind;
  int val;   // DEF: the value; STG / STR / ACC: what is stored or accumulated
  int x, y;  // operand or accumulator; reduction kind.  BODY_BEGIN: first slot of its inputs and their number
};

class Decoder {
 public:
  // `level` 0: values shared between phases; 1: vector values shared inside a phase only; 2: the
  // program as it stands, every value in the register it was given and every load in its place.  Level 2
  // takes any program that is looped over its rows or has none to reduce.
  // At most `slots` inputs are requested ahead.
  Decoder(const nbk_rowprog* p, int mode, int level, int slots)
      : p_(p), mode_(mode), level_(level), max_slots_(slots) {}

  // False if the mode or this level does not take the program.
  bool run(rp_vm* out) {
    out_ = out;
    if (!build()) return false;
    mark_used();
    return assign() && emit();
  }

 private:
  const nbk_rowprog* p_;
  const int mode_, level_, max_slots_;
  rp_vm* out_ = nullptr;
  std::vector<Val> vals_;
  std::vector<Item> items_;
  std::vector<int> known_vec_, known_scl_;
  int n_slots_ = 0, n_row_slots_ = 0, body_slots_ = 0;

  bool written(int operand) const {
    for (int i = 0; i < p_->n_ins; ++i)
      if ((p_->ins[i].op == NBK_OP_STG || p_->ins[i].op == NBK_OP_STR) && p_->ins[i].dst == operand) return true;
    return false;
  }
  int find(const Val& v) const {
    for (int id : v.scalar ? known_scl_ : known_vec_) {
      const Val& w = vals_[id];
      if (w.op == v.op && w.a == v.a && w.b == v.b && w.c == v.c && w.x == v.x && w.y == v.y) return id;
    }
    return -1;
  }
  int define(const Val& v, bool shared) {
    shared &= level_ < 2;
    if (shared) {
      const int got = find(v);
      if (got >= 0) return got;
    }
    const int id = (int)vals_.size();
    vals_.push_back(v);
    items_.push_back({DEF, id, 0, 0});
    if (shared) (v.scalar ? known_scl_ : known_vec_).push_back(id);
    return id;
  }
  // The slot that requests `operand` for this body (LOOP) or row; -1 if there is none left.
  int slot_of(int operand) {
    const int first = mode_ == RPVM_LOOP ? n_slots_ - body_slots_ : 0;
    for (int k = first; k < n_slots_; ++k)
      if (out_->slots[k] == operand) return k - first;
    if (n_slots_ - first >= max_slots_ || n_slots_ >= (int)sizeof out_->slots) return -1;
    out_->slots[n_slots_++] = (uint8_t)operand;
    ++body_slots_;
    return n_slots_ - 1 - first;
  }
  int row_slot_of(int operand) {
    if (nbk_dtype_size(p_->operand[operand].dtype) != 4) return -1;
    for (int k = 0; k < n_row_slots_; ++k)
      if (out_->row_slots[k] == operand) return k;
    if (n_row_slots_ >= RPVM_ROW_SLOTS) return -1;
    out_->row_slots[n_row_slots_] = (uint8_t)operand;
    return n_row_slots_++;
  }

  bool build() {
    int vec[NBK_RP_NVEC], scl[NBK_RP_NSCL];
    struct { int init = -1, kind = -1, val = -1, n = 0; } acc[NBK_RP_NACC];
    for (int& v : vec) v = -1;
    for (int& v : scl) v = -1;
    bool op_written[NBK_RP_MAX_OPERANDS];
    for (int i = 0; i < p_->n_operands; ++i) op_written[i] = written(i);
    auto reg = [&](int r) {
      int& v = r < NBK_RP_NVEC ? vec[r] : scl[r - NBK_RP_NVEC];
      if (v < 0) {  // read before it is written: zero
        Val z;
        z.scalar = true; z.op = RPVM_IMM; z.x = NBK_RP_MAX_IMM;  // (the decoded program's own)
        if (level_ == 2) z.own = r & (NBK_RP_NVEC - 1);
        if (level_ == 2 && r < NBK_RP_NVEC) {  // (in the register itself: is it greater than itself?)
          z.scalar = false; z.op = NBK_OP_GT; z.a = z.b = (int)vals_.size();
        }
        v = define(z, true);
      }
      return v;
    };
    auto operands = [&](Val& v, const nbk_ins& in) {
      v.op = in.op;
      v.a = reg(in.a);
      if (!is_unary(in.op)) v.b = reg(in.b);
      if (in.op == NBK_OP_WHERE || in.op == NBK_OP_FMA) v.c = reg(in.c);
    };
    int pc = 0;
    while (pc < p_->n_ins && p_->ins[pc].op != NBK_OP_HALT) {
      const nbk_ins in = p_->ins[pc];
      if (in.op == NBK_OP_BODY) {
        // (an input that a row starts with is one value in one register for the whole program: a
        // second value on its slot would lose the register when the first is used up)
        if (mode_ == RPVM_LOOP) known_vec_.clear();
        else if (level_ > 0)
          known_vec_.erase(std::remove_if(known_vec_.begin(), known_vec_.end(),
                                          [&](int id) { return vals_[id].op != RPVM_LD; }),
                           known_vec_.end());
        if (mode_ == RPVM_LOOP)
          for (int& v : vec) v = -1;  // (a chunk's values do not outlive it)
        const size_t begin = items_.size();
        const int first_slot = n_slots_;
        body_slots_ = 0;
        items_.push_back({BODY_BEGIN, 0, 0, 0});
        for (int q = pc + 1; q <= pc + in.aux; ++q) {
          const nbk_ins b = p_->ins[q];
          if (b.op == NBK_OP_STG) {
            items_.push_back({STG, reg(b.a), b.dst, 0});
          } else if (b.op == NBK_OP_ACC) {
            if (mode_ == RPVM_LOOP) {
              items_.push_back({ACC, reg(b.a), b.dst, b.b});
            } else {
              auto& s = acc[b.dst];
              if (s.n++) return false;
              s.val = reg(b.a);
              s.kind = b.b;
            }
          } else {
            Val v;
            bool shared = true;
            if (b.op == NBK_OP_LDG) {
              const int slot = op_written[b.a] || !rp_vm_ahead(p_, b.a) ? -1 : slot_of(b.a);
              v.op = slot >= 0 ? RPVM_LD : RPVM_LDG;
              v.x = slot >= 0 ? slot : b.a;
              v.y = slot >= 0 ? p_->operand[b.a].dtype : 0;
              shared = !op_written[b.a];
            } else if (b.op == NBK_OP_COLIDX) {
              v.op = RPVM_COLIDX;
              v.x = b.a != 0;
            } else {
              operands(v, b);
            }
            if (level_ == 2) v.own = b.dst;
            vec[b.dst] = define(v, shared);
          }
        }
        items_[begin].x = first_slot;
        items_[begin].y = n_slots_ - first_slot;
        items_.push_back({BODY_END, 0, 0, 0});
        pc += 1 + in.aux;
        continue;
      }
      ++pc;
      if (in.op == NBK_OP_STR) {
        items_.push_back({STR, reg(in.a), in.dst, 0});
        continue;
      }
      if (in.op == NBK_OP_ACCINIT) {
        if (mode_ == RPVM_LOOP) items_.push_back({ACCINIT, 0, in.dst, in.a});
        acc[in.dst] = {in.a, -1, -1, 0};
        continue;
      }
      Val v;
      v.scalar = true;
      bool shared = true;
      if (level_ == 2) v.own = in.dst - NBK_RP_NVEC;
      if (in.op == NBK_OP_IMM) {
        v.op = RPVM_IMM;
        v.x = in.a;
        v.once = true;
      } else if (in.op == NBK_OP_LDR) {
        bool moves = op_written[in.a];
        for (int k = 0; k < p_->n_lead; ++k) moves |= p_->operand[in.a].lead_stride[k] != 0;
        const int slot = moves && !op_written[in.a] && level_ < 2 ? row_slot_of(in.a) : -1;
        v.op = slot >= 0 ? RPVM_LDS : RPVM_LDR;
        v.x = slot >= 0 ? slot : in.a;
        v.once = !moves;
        shared &= !op_written[in.a];
      } else if (in.op == NBK_OP_LEADIDX) {
        v.op = RPVM_LEADIDX;
        v.x = in.a;
        v.y = in.b != 0;
      } else if (in.op == NBK_OP_RED) {
        v.op = RPVM_RED;
        v.y = in.b;
        if (mode_ == RPVM_LOOP) {
          v.x = in.a;
          shared = false;
        } else {
          const auto& s = acc[in.a];
          if (s.n != 1 || s.init != in.b || s.kind != in.b) return false;
          v.a = s.val;
        }
      } else {
        operands(v, in);
        v.once = vals_[v.a].once && (v.b < 0 || vals_[v.b].once) && (v.c < 0 || vals_[v.c].once);
      }
      if (level_ >= 2) v.once = false;
      scl[in.dst - NBK_RP_NVEC] = define(v, shared);
    }
    return true;
  }

  template <typename Fn>
  void sources(const Val& v, Fn fn) const {
    if (v.a >= 0) fn(v.a);
    if (v.b >= 0) fn(v.b);
    if (v.c >= 0) fn(v.c);
  }

  void mark_used() {
    for (int i = (int)items_.size() - 1; i >= 0; --i) {
      const Item& it = items_[i];
      if (it.kind == STG || it.kind == STR || it.kind == ACC) vals_[it.val].used = true;
      if (it.kind == DEF && vals_[it.val].used)
        sources(vals_[it.val], [&](int s) { vals_[s].used = true; });
    }
  }

  bool assign() {
    const int n = (int)items_.size();
    std::vector<int> body_end(n, -1);
    for (int i = 0, begin = -1; i < n; ++i) {
      if (items_[i].kind == BODY_BEGIN) begin = i;
      if (items_[i].kind == BODY_END)
        for (int q = begin; q <= i; ++q) body_end[q] = i;
    }
    auto use = [&](int v, int at) {
      // (a body that is looped over needs its scalars until it ends)
      if (mode_ == RPVM_LOOP && vals_[v].scalar && body_end[at] >= 0) at = body_end[at];
      vals_[v].last = std::max(vals_[v].last, at);
    };
    for (int i = 0; i < n; ++i) {
      const Item& it = items_[i];
      if (it.kind == STG || it.kind == STR || it.kind == ACC) use(it.val, i);
      if (it.kind == DEF && vals_[it.val].used && !vals_[it.val].once)
        sources(vals_[it.val], [&](int s) { use(s, i); });
    }
    bool vec_busy[NBK_RP_NVEC] = {}, scl_busy[NBK_RP_NSCL] = {};
    auto take = [&](Val& v) {
      bool* busy = v.scalar ? scl_busy : vec_busy;
      const int r0 = v.own >= 0 ? v.own : 0;
      const int r1 = v.own >= 0 ? v.own + 1 : v.scalar ? NBK_RP_NSCL : NBK_RP_NVEC;
      for (int r = r0; r < r1; ++r)
        if (!busy[r]) {
          busy[r] = true;
          v.reg = r;
          return true;
        }
      return false;
    };
    // what is there before the program starts
    std::vector<int> live;
    for (const Item& it : items_) {
      if (it.kind != DEF || !vals_[it.val].used) continue;
      Val& v = vals_[it.val];
      if (v.once && !take(v)) return false;
    }
    auto start = [&](size_t i0, size_t i1, int op) {
      for (size_t i = i0; i < i1; ++i) {
        if (items_[i].kind != DEF || vals_[items_[i].val].op != op) continue;
        Val& v = vals_[items_[i].val];
        bool* busy = v.scalar ? scl_busy : vec_busy;
        if (op == RPVM_LD) {  // (an unused one is loaded all the same: its register is free after that)
          v.reg = v.x;
          if (!v.used) continue;
          busy[v.reg] = true;
        } else {
          if (!v.used) continue;
          if (!take(v)) return false;
          out_->row_dst[v.x] = (uint8_t)(RPVM_SCALAR + v.reg);
        }
        live.push_back(items_[i].val);
      }
      return true;
    };
    for (uint8_t& d : out_->row_dst) d = RPVM_NONE;
    if (!start(0, items_.size(), RPVM_LDS)) return false;
    if (mode_ != RPVM_LOOP) start(0, items_.size(), RPVM_LD);
    for (int i = 0; i < n; ++i) {
      // what is read here for the last time makes room for what is written
      for (size_t k = 0; k < live.size();) {
        Val& v = vals_[live[k]];
        if (v.last <= i) {
          (v.scalar ? scl_busy : vec_busy)[v.reg] = false;
          live[k] = live.back();
          live.pop_back();
        } else {
          ++k;
        }
      }
      const Item& it = items_[i];
      if (it.kind == BODY_BEGIN && mode_ == RPVM_LOOP) start((size_t)i, (size_t)body_end[i], RPVM_LD);
      if (it.kind != DEF) continue;
      Val& v = vals_[it.val];
      if (!v.used || v.once || v.op == RPVM_LD || v.op == RPVM_LDS) continue;
      if (!take(v)) return false;
      live.push_back(it.val);
    }
    return true;
  }

  int code(int v) const { return vals_[v].scalar ? RPVM_SCALAR + vals_[v].reg : vals_[v].reg; }

  rp_vm_ins encode(int id) const {
    const Val& v = vals_[id];
    rp_vm_ins in = {};
    in.op = (uint8_t)v.op;
    in.dst = (uint8_t)code(id);
    if (v.a >= 0) in.a = (uint8_t)code(v.a);
    if (v.op >= NBK_OP_MOV) {
      // (an instruction of scalars reads all three: an operand that it does not have is the first)
      const uint8_t none = v.scalar ? in.a : 0;
      in.b = v.b >= 0 ? (uint8_t)code(v.b) : none;
      in.c = v.c >= 0 ? (uint8_t)code(v.c) : none;
      in.two = v.b >= 0;
    } else {
      in.b = (uint8_t)v.y;
      in.c = (uint8_t)v.x;
    }
    return in;
  }

  bool emit() {
    std::vector<rp_vm_ins> list;
    const bool loop = mode_ == RPVM_LOOP;
    int open = -1;
    auto begin = [&](bool per_chunk, int slot, int n_slots) {
      open = (int)list.size();
      rp_vm_ins in = {};
      in.op = RPVM_SEG;
      in.dst = RPVM_NONE;
      in.a = (uint8_t)n_slots;
      in.b = per_chunk;
      in.c = (uint8_t)slot;
      list.push_back(in);
    };
    auto end = [&]() {
      list[open].aux = (uint16_t)(list.size() - (size_t)open - 1);
      if (list[open].aux == 0) list.resize((size_t)open);  // (nothing of it is used)
    };
    if (loop) begin(false, 0, 0);
    for (const Item& it : items_)
      if (it.kind == DEF && vals_[it.val].used && vals_[it.val].once) list.push_back(encode(it.val));
    if (loop) end();
    out_->n_once = (int)list.size();
    if (loop) begin(false, 0, 0);
    for (const Item& it : items_) {
      rp_vm_ins in = {};
      in.dst = RPVM_NONE;
      switch (it.kind) {
        case DEF:
          if (!vals_[it.val].used || vals_[it.val].once || vals_[it.val].op == RPVM_LD ||
              vals_[it.val].op == RPVM_LDS)
            continue;
          in = encode(it.val);
          break;
        case STG: in.op = RPVM_STG; break;
        case STR: in.op = RPVM_STR; break;
        case ACC: in.op = RPVM_ACC; break;
        case ACCINIT: in.op = RPVM_ACCINIT; break;
        case BODY_BEGIN:
          if (loop) { end(); begin(true, it.x, it.y); }
          continue;
        case BODY_END:
          if (loop) { end(); begin(false, 0, 0); }
          continue;
      }
      if (it.kind != DEF) {
        in.c = (uint8_t)it.x;
        in.b = (uint8_t)it.y;
        if (it.kind != ACCINIT) in.a = (uint8_t)code(it.val);
      }
      list.push_back(in);
    }
    if (loop) end();
    if ((int)list.size() >= RPVM_MAX_INS) return false;
    // reductions that stand together share one exchange between the wavefronts (one over a scalar
    // has its own: the scalar may be the result of its neighbour)
    auto joins = [&](size_t k) { return list[k].op == RPVM_RED && list[k].a < RPVM_SCALAR; };
    for (size_t i = 0; i < list.size();) {
      size_t k = i + 1;
      if (list[i].op == RPVM_RED) {
        while (k < list.size() && k - i < 4 && joins(i) && joins(k)) ++k;
        list[i].aux = (uint16_t)(k - i);
      }
      i = k;
    }
    out_->n_ins = (int)list.size();
    for (const rp_vm_ins& in : list) out_->rare |= is_rare(in.op);
    out_->n_slots = n_slots_;
    out_->n_row_slots = n_row_slots_;
    std::copy(list.begin(), list.end(), out_->ins);
    return true;
  }
};

// Decoded programs, by contents.  A step launches the same few again and again; a process that
// makes new ones without end starts over at the limit.
constexpr size_t kMaxDecoded = 512;
std::mutex g_decoded_mu;
std::unordered_map<std::string, std::shared_ptr<const rp_vm>>* g_decoded = nullptr;

// Everything the decoded form depends on: instructions, immediates, and of the operands their
// types and whether they move with the row.
std::string program_key(const nbk_rowprog* p, int mode) {
  std::string k;
  k.reserve((size_t)p->n_ins * 8 + 160);
  const int32_t head[5] = {mode, p->n_ins, p->n_operands, p->n_imm, p->n_lead};
  k.append((const char*)head, sizeof head);
  k.append((const char*)p->ins, (size_t)p->n_ins * sizeof(nbk_ins));
  k.append((const char*)p->imm, (size_t)p->n_imm * sizeof(float));
  for (int i = 0; i < p->n_operands; ++i) {
    bool moves = false;
    for (int a = 0; a < p->n_lead; ++a) moves |= p->operand[i].lead_stride[a] != 0;
    k.push_back((char)(p->operand[i].dtype * 4 + moves * 2 + rp_vm_ahead(p, i)));
  }
  return k;
}

// nullptr where the mode does not take the program.
std::shared_ptr<const rp_vm> decoded(const nbk_rowprog* p, int mode) {
  const std::string key = program_key(p, mode);
  std::lock_guard<std::mutex> lk(g_decoded_mu);
  if (!g_decoded) g_decoded = new std::unordered_map<std::string, std::shared_ptr<const rp_vm>>();
  auto it = g_decoded->find(key);
  if (it != g_decoded->end()) return it->second;
  if (g_decoded->size() >= kMaxDecoded) g_decoded->clear();
  auto vm = std::make_shared<rp_vm>();
  if (!rp_vm_decode(p, mode, vm.get())) vm.reset();
  (*g_decoded)[key] = vm;
  return vm;
}

int occupancy(const void* fn, int block, int* out) {
  static std::mutex mu;
  static std::unordered_map<uint64_t, int>* cache = nullptr;
  const uint64_t key = (uint64_t)(uintptr_t)fn ^ ((uint64_t)block << 48);
  std::lock_guard<std::mutex> lk(mu);
  if (!cache) cache = new std::unordered_map<uint64_t, int>();
  auto it = cache->find(key);
  if (it == cache->end()) {
    int n = 0;
    NBK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, block, 0));
    it = cache->emplace(key, n < 1 ? 1 : n).first;
  }
  *out = it->second;
  return NBK_OK;
}

}  // namespace

bool rp_vm_decode(const nbk_rowprog* p, int mode, rp_vm* out) {
  // From the fewest instructions to the fewest registers.
  static const struct { int level, slots; } kTry[] = {{0, RPVM_SLOTS}, {1, RPVM_SLOTS}, {1, 4}, {1, 0}, {2, 0}};
  for (const auto& t : kTry) {
    *out = {};
    if (Decoder(p, mode, t.level, t.slots).run(out)) return true;
  }
  return false;
}

// The instructions as the kernel runs them: operands renamed by `at`, the commonest operations marked.  Returns
// the largest vector register.
static int rp_vm_finish(const nbk_rowprog* p, const uint8_t* at, rp_vm* vm) {
  int top = 0;
  for (int q = 0; q < vm->n_ins; ++q) {
    rp_vm_ins& in = vm->ins[q];
    if (in.dst < NBK_RP_NVEC) {
      top = std::max<int>(top, in.dst);
      if (in.op == NBK_OP_MUL || in.op == NBK_OP_ADD || in.op == NBK_OP_SUB) {
        if (in.a >= RPVM_SCALAR && in.op != NBK_OP_SUB) std::swap(in.a, in.b);
        const int what = in.op == NBK_OP_MUL ? 0 : in.op == NBK_OP_ADD ? 1 : 2;
        if (in.a < RPVM_SCALAR) in.two = (uint8_t)((in.b < RPVM_SCALAR ? RPVM_TWO_MUL : RPVM_TWO_MUL_S) + what);
      }
    }
    if (in.op == RPVM_STG || in.op == RPVM_STR || in.op == RPVM_LDG || in.op == RPVM_LDR) {
      const nbk_operand& o = p->operand[in.c];
      if (in.op == RPVM_STG && o.col_stride == 1 && (o.dtype == NBK_F32 || o.dtype == NBK_I32)) in.two = RPVM_TWO_WORDS;
      if (in.op == RPVM_STG && o.col_stride == 1 && o.dtype == NBK_BF16) in.two = RPVM_TWO_BF16;
      in.c = at[in.c];
    }
  }
  return top;
}

int rp_vm_launch(const nbk_rowprog* p, int64_t rows, hipStream_t stream) {
  const int64_t chunks = (p->C + 3) >> 2;
  int mode = p->has_reduce ? RPVM_ROW : RPVM_FLAT;
  std::shared_ptr<const rp_vm> d;
  if (mode == RPVM_FLAT || chunks <= 1024) d = decoded(p, mode);
  if (mode == RPVM_ROW && !d) {
    mode = RPVM_LOOP;
    d = decoded(p, mode);
  }
  NBK_REQUIRE(d, "rowprog: the program cannot be decoded");
  rp_vm vm = *d;
  for (int k = 0; k < NBK_RP_MAX_LEAD; ++k) vm.lead_dim[k] = p->lead_dim[k];
  vm.C = p->C;
  vm.n_lead = p->n_lead;
  for (int i = 0; i < p->n_imm; ++i) vm.imm[i] = p->imm[i];
  // Where a row's inputs are requested once they are the first operands: their descriptions are read
  // without a look at the list of slots.
  uint8_t at[NBK_RP_MAX_OPERANDS];
  for (int i = 0; i < NBK_RP_MAX_OPERANDS; ++i) at[i] = (uint8_t)i;
  if (mode != RPVM_LOOP) {
    bool slot[NBK_RP_MAX_OPERANDS] = {};
    for (int k = 0; k < vm.n_slots; ++k) slot[vm.slots[k]] = true;
    int next = vm.n_slots;
    for (int i = 0; i < p->n_operands; ++i) at[i] = slot[i] ? 0 : (uint8_t)next++;
    for (int k = 0; k < vm.n_slots; ++k) at[vm.slots[k]] = (uint8_t)k;
  }
  for (int i = 0; i < p->n_operands; ++i) vm.operand[at[i]] = p->operand[i];
  for (int k = 0; k < vm.n_row_slots; ++k) vm.row_slots[k] = at[vm.row_slots[k]];
  const int top_reg = rp_vm_finish(p, at, &vm);
  uint32_t flags = p->C % 4 ? RPVM_WORDS | RPVM_RAGGED : RPVM_WORDS;
  const int n_listed = mode == RPVM_LOOP ? (int)sizeof vm.slots : vm.n_slots;
  for (int k = 0; k < n_listed && k < d->n_slots; ++k) {
    const int dt = p->operand[d->slots[k]].dtype;
    if (dt != NBK_F32 && dt != NBK_I32) flags &= ~(uint32_t)RPVM_WORDS;
  }
  // Two chunks a lane where a row has more than one wavefront's and the program up to eight vector registers: half
  // the decoding per element (20000 rows of 270 floats 383 -> 212 us, 3000 of 4001 510 -> 413).  On few rows too, where
  // half the wavefronts of a row are a longer chain each and share the scalar unit with fewer others (two programs, us:
  // 32 x 300 floats 17.2 + 12.8 -> 15.9 + 10.7, 250 x 2051 24.6 + 17.2 -> 21.7 + 14.5, 250 x 300 bf16 16.6 + 12.5 -> 16.8 + 11.4).
  // (Looped programs keep one: their accumulators and offsets leave no room, 4096 rows of 12000 bfloat16 3477 -> 3684 us.)
  const bool wide = mode == RPVM_ROW && chunks > 64 && top_reg < RPVM_WIDE_REGS;
#define RPVM_PICK(K, N) (d->rare ? (const void*)rp_vm_kernel<K, true, N> : (const void*)rp_vm_kernel<K, false, N>)
  const void* fn;
  int block = 256;
  uint64_t groups = (uint64_t)rows;  // workgroups' worth of work
  if (mode == RPVM_FLAT) {
    fn = RPVM_PICK(K_FLAT, 1);
    groups = ((uint64_t)rows * (uint64_t)chunks + 255) / 256;
  } else if (mode == RPVM_LOOP) {
    fn = RPVM_PICK(K_LOOP, 1);
    block = p->block;  // (the lanes of the generated kernels: sums associate as theirs do)
  } else if (chunks <= 32) {
    fn = RPVM_PICK(K_SUB, 1);
    vm.lanes = 1;
    while (vm.lanes < chunks) vm.lanes *= 2;
    groups = ((uint64_t)rows * (uint64_t)vm.lanes + 255) / 256;
  } else {
    fn = wide ? RPVM_PICK(K_ROW, 2) : RPVM_PICK(K_ROW, 1);
    const int64_t per_lane = wide ? 2 : 1;
    block = vm.lanes = (int)((chunks + 64 * per_lane - 1) / (64 * per_lane) * 64);
  }
  int per_cu = 0;
  { const int rc = occupancy(fn, block, &per_cu); if (rc != NBK_OK) return rc; }
  const uint64_t cap = (uint64_t)nbk_num_cus() * (uint64_t)per_cu;
  if (groups > cap) groups = cap;
  uint32_t rows_arg = (uint32_t)rows, cpr = (uint32_t)chunks;
  uint64_t total = (uint64_t)rows * (uint64_t)chunks;
  void* args[5] = {&vm, &rows_arg, &cpr, &total, &flags};
  NBK_HIP(hipLaunchKernel(fn, dim3((unsigned)groups), dim3((unsigned)block), args, 0, stream));
  return NBK_OK;
}
