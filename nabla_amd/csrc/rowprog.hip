// Row programs: fused elementwise chains and last-axis reductions.
//
// Checks a program, finds the compiled kernel the library carries for it (generated ahead of time
// or written by hand) and launches that, or hands the program to the interpreter (rowprog_vm.hip).
#include "nbk_common.h"
#include "rowprog_spec.h"
#include "rowprog_vm.h"
#include <stddef.h>
#include <mutex>
#include <unordered_map>

static bool rp_is_unary(int op) {
  return (op >= NBK_OP_MOV && op < NBK_OP_ADD) || op == NBK_OP_DGELU || op == NBK_OP_SIN ||
         op == NBK_OP_COS || (op >= NBK_OP_INEG && op <= NBK_OP_INEZ);
}
static bool rp_is_binary(int op) {
  return (op >= NBK_OP_ADD && op < NBK_OP_WHERE) || (op >= NBK_OP_IADD && op <= NBK_OP_ILE);
}
static bool rp_is_ew(int op) {
  return rp_is_unary(op) || rp_is_binary(op) || op == NBK_OP_WHERE || op == NBK_OP_FMA;
}

// ------------------------------------------------------------------ host side
static int rp_validate(const nbk_rowprog* p) {
  NBK_REQUIRE(p != nullptr, "rowprog: null program");
  NBK_REQUIRE(p->n_lead >= 0 && p->n_lead <= NBK_RP_MAX_LEAD, "rowprog: n_lead %d out of range",
              p->n_lead);
  NBK_REQUIRE(p->n_operands >= 0 && p->n_operands <= NBK_RP_MAX_OPERANDS,
              "rowprog: %d operands exceed the limit %d", p->n_operands, NBK_RP_MAX_OPERANDS);
  NBK_REQUIRE(p->n_ins > 0 && p->n_ins <= NBK_RP_MAX_INS, "rowprog: %d instructions (limit %d)",
              p->n_ins, NBK_RP_MAX_INS);
  NBK_REQUIRE(p->n_imm >= 0 && p->n_imm <= NBK_RP_MAX_IMM, "rowprog: %d immediates (limit %d)",
              p->n_imm, NBK_RP_MAX_IMM);
  NBK_REQUIRE(p->C > 0, "rowprog: row length %lld", (long long)p->C);
  for (int k = 0; k < p->n_lead; ++k)
    NBK_REQUIRE(p->lead_dim[k] > 0, "rowprog: leading dim %d is %lld", k,
                (long long)p->lead_dim[k]);
  for (int i = 0; i < p->n_operands; ++i) {
    const nbk_operand& o = p->operand[i];
    NBK_REQUIRE(o.ptr != nullptr, "rowprog: operand %d has a null pointer", i);
    NBK_REQUIRE(nbk_dtype_size(o.dtype) > 0, "rowprog: operand %d has dtype %d", i, o.dtype);
    NBK_REQUIRE(o.stage_slot < NBK_RP_MAX_STAGE, "rowprog: operand %d stage slot %d", i,
                o.stage_slot);
    if (o.vec_ok) {
      NBK_REQUIRE(o.col_stride == 1, "rowprog: operand %d vec_ok needs unit column stride", i);
      const int64_t a = 4 * nbk_dtype_size(o.dtype);
      NBK_REQUIRE(((uintptr_t)o.ptr % (uintptr_t)a) == 0,
                  "rowprog: operand %d pointer not aligned for 4-wide access", i);
      for (int k = 0; k < p->n_lead; ++k)
        NBK_REQUIRE(o.lead_stride[k] % 4 == 0,
                    "rowprog: operand %d lead stride %d not a multiple of 4", i, k);
    }
  }
  // instruction stream: register / operand indices in range, bodies closed
  int pc = 0;
  bool halted = false;
  while (pc < p->n_ins) {
    const nbk_ins in = p->ins[pc];
    if (in.op == NBK_OP_HALT) { halted = true; break; }
    if (in.op == NBK_OP_BODY) {
      NBK_REQUIRE(pc + 1 + in.aux <= p->n_ins, "rowprog: body at %d runs past the end", pc);
      for (int q = pc + 1; q < pc + 1 + in.aux; ++q) {
        const nbk_ins b = p->ins[q];
        const int op = b.op;
        if (op == NBK_OP_LDG) {
          NBK_REQUIRE(b.a < p->n_operands && b.dst < NBK_RP_NVEC, "rowprog: bad LDG at %d", q);
        } else if (op == NBK_OP_STG) {
          NBK_REQUIRE(b.dst < p->n_operands && b.a < 32, "rowprog: bad STG at %d", q);
        } else if (op == NBK_OP_ACC) {
          NBK_REQUIRE(p->has_reduce && b.dst < NBK_RP_NACC && b.a < 32 && b.b <= NBK_RED_MIN,
                      "rowprog: bad ACC at %d", q);
        } else if (op == NBK_OP_COLIDX) {
          NBK_REQUIRE(b.dst < NBK_RP_NVEC, "rowprog: bad COLIDX at %d", q);
        } else if (rp_is_ew(op)) {
          NBK_REQUIRE(b.dst < NBK_RP_NVEC && b.a < 32 && b.b < 32 && b.c < 32,
                      "rowprog: bad register at %d", q);
        } else {
          NBK_REQUIRE(false, "rowprog: opcode %d not allowed in a body (at %d)", op, q);
        }
      }
      pc += 1 + in.aux;
      continue;
    }
    const int op = in.op;
    const bool sreg_dst = in.dst >= NBK_RP_NVEC && in.dst < 32;
    if (op == NBK_OP_IMM) {
      NBK_REQUIRE(sreg_dst && in.a < p->n_imm, "rowprog: bad IMM at %d", pc);
    } else if (op == NBK_OP_LDR) {
      NBK_REQUIRE(sreg_dst && in.a < p->n_operands, "rowprog: bad LDR at %d", pc);
    } else if (op == NBK_OP_STR) {
      NBK_REQUIRE(in.dst < p->n_operands && in.a >= NBK_RP_NVEC && in.a < 32,
                  "rowprog: bad STR at %d", pc);
    } else if (op == NBK_OP_LEADIDX) {
      NBK_REQUIRE(sreg_dst && in.a < p->n_lead, "rowprog: bad LEADIDX at %d", pc);
    } else if (op == NBK_OP_ACCINIT) {
      NBK_REQUIRE(in.dst < NBK_RP_NACC && in.a <= NBK_RED_MIN, "rowprog: bad ACCINIT at %d", pc);
    } else if (op == NBK_OP_RED) {
      NBK_REQUIRE(p->has_reduce && sreg_dst && in.a < NBK_RP_NACC && in.b <= NBK_RED_MIN,
                  "rowprog: bad RED at %d", pc);
    } else if (rp_is_ew(op)) {
      NBK_REQUIRE(sreg_dst && in.a >= NBK_RP_NVEC && in.a < 32, "rowprog: bad scalar op at %d",
                  pc);
      if (!rp_is_unary(op))
        NBK_REQUIRE(in.b >= NBK_RP_NVEC && in.b < 32, "rowprog: bad scalar op at %d", pc);
      if (op == NBK_OP_WHERE || op == NBK_OP_FMA)
        NBK_REQUIRE(in.c >= NBK_RP_NVEC && in.c < 32, "rowprog: bad scalar op at %d", pc);
    } else {
      NBK_REQUIRE(false, "rowprog: opcode %d not allowed in a prologue (at %d)", op, pc);
    }
    ++pc;
  }
  NBK_REQUIRE(halted, "rowprog: program has no HALT");
  return NBK_OK;
}

// ---- specialised kernels -------------------------------------------------------
// A program's name: FNV-1a over its canonical bytes (same bytes as program_bytes() in
// nabla_amd/backend/specialize.py): header, per-operand (dtype, stride class,
// vec_ok, stage slot), instructions, immediates.  Extents and addresses are not
// part of it.
static uint64_t rp_program_hash(const nbk_rowprog* p) {
  uint64_t h = 0xCBF29CE484222325ULL;
  auto eat = [&](const void* data, size_t n) {
    const uint8_t* b = (const uint8_t*)data;
    for (size_t i = 0; i < n; ++i) h = (h ^ b[i]) * 0x100000001B3ULL;
  };
  const uint8_t head[6] = {(uint8_t)(p->has_reduce ? 1 : 0), (uint8_t)p->n_operands,
                           (uint8_t)(p->n_ins & 0xff), (uint8_t)(p->n_ins >> 8),
                           (uint8_t)p->n_imm, (uint8_t)p->n_stage};
  eat(head, 6);
  for (int i = 0; i < p->n_operands; ++i) {
    const nbk_operand& o = p->operand[i];
    const uint8_t ob[4] = {(uint8_t)o.dtype,
                           (uint8_t)(o.col_stride == 0 ? 0 : (o.col_stride == 1 ? 1 : 2)),
                           (uint8_t)(o.vec_ok ? 1 : 0), (uint8_t)(int8_t)o.stage_slot};
    eat(ob, 4);
  }
  for (int i = 0; i < p->n_ins; ++i) {
    const nbk_ins& in = p->ins[i];
    const uint8_t ib[8] = {in.op, in.dst, in.a, in.b, in.c, 0, (uint8_t)(in.aux & 0xff),
                           (uint8_t)(in.aux >> 8)};
    eat(ib, 8);
  }
  eat(p->imm, sizeof(float) * (size_t)p->n_imm);
  return h;
}

// What a compiled kernel is found by: the same without what it does not depend on.  A kernel reads
// immediates from the program it is launched with (a row length that a mean divides by is one), takes
// operands at any alignment, and only its generic form depends on what is staged (rp_stage_sig).  (Kernels with
// approximate functions are found by the whole hash above: they serve the programs they were chosen for.)
// Same bytes as key_bytes() in nabla_amd/backend/specialize.py.
static uint64_t rp_program_key(const nbk_rowprog* p) {
  uint64_t h = 0xCBF29CE484222325ULL;
  auto eat = [&](uint8_t b) { h = (h ^ b) * 0x100000001B3ULL; };
  eat(p->has_reduce ? 1 : 0);
  eat((uint8_t)p->n_operands);
  for (int i = 0; i < p->n_operands; ++i) {
    const nbk_operand& o = p->operand[i];
    eat((uint8_t)o.dtype);
    eat((uint8_t)(o.col_stride == 0 ? 0 : (o.col_stride == 1 ? 1 : 2)));
  }
  for (int i = 0; i < p->n_ins; ++i) {
    const nbk_ins& in = p->ins[i];
    for (uint8_t b : {in.op, in.dst, in.a, in.b, in.c, (uint8_t)(in.aux & 0xff), (uint8_t)(in.aux >> 8)}) eat(b);
  }
  return h;
}
// Which operand is staged where, three bits each.
static uint64_t rp_stage_sig(const nbk_rowprog* p) {
  uint64_t sig = 0;
  for (int i = 0; i < p->n_operands; ++i) sig |= (uint64_t)((p->operand[i].stage_slot + 1) & 7) << (3 * i);
  return sig;
}
static_assert(NBK_RP_MAX_OPERANDS * 3 <= 64 && NBK_RP_MAX_STAGE + 1 <= 7, "the signature of what is staged");

struct RpSpec {
  const void* kernel[5];
  const void* kernel_full[5];
  const void* kernel_stream[5];
  const void* kernel_flat;
  const void* kernel_stage16;
  const rp_hand_entry* hand;
  uint64_t stage_sig;
  int block_mode;
  bool has_approx;  // g_approx holds kernels for a program of this key
  bool approximate;
  bool lds_attr_set;
  bool lds16_attr_set;
};
static std::mutex g_spec_mu;
static std::unordered_map<uint64_t, RpSpec>* g_specs = nullptr;   // by key
static std::unordered_map<uint64_t, RpSpec>* g_approx = nullptr;  // by hash: the chosen programs alone

static RpSpec* rp_find_spec(const nbk_rowprog* p) {
  const uint64_t key = rp_program_key(p);
  std::lock_guard<std::mutex> lk(g_spec_mu);
  if (!g_specs) {
    g_approx = new std::unordered_map<uint64_t, RpSpec>();
    g_specs = new std::unordered_map<uint64_t, RpSpec>();
#define RP_TABLE(I) rp_spec_table_##I,
#define RP_COUNT(I) rp_spec_count_##I,
    const rp_spec_entry* tabs[NBK_RP_SPEC_FILES] = {NBK_RP_SPEC_EACH(RP_TABLE)};
    const int counts[NBK_RP_SPEC_FILES] = {NBK_RP_SPEC_EACH(RP_COUNT)};
#undef RP_TABLE
#undef RP_COUNT
    for (int t = 0; t < NBK_RP_SPEC_FILES; ++t)
      for (int i = 0; i < counts[t]; ++i)
      {
        RpSpec e;
        for (int k = 0; k < 5; ++k) {
          e.kernel[k] = tabs[t][i].kernel[k];
          e.kernel_full[k] = tabs[t][i].kernel_full[k];
          e.kernel_stream[k] = tabs[t][i].kernel_stream[k];
        }
        e.kernel_flat = tabs[t][i].kernel_flat;
        e.kernel_stage16 = tabs[t][i].kernel_stage16;
        e.block_mode = tabs[t][i].block_mode;
        e.stage_sig = tabs[t][i].stage_sig;
        e.lds_attr_set = false;
        e.lds16_attr_set = false;
        e.hand = nullptr;
        e.has_approx = false;
        e.approximate = tabs[t][i].approx_hash != 0;
        if (tabs[t][i].approx_hash) (*g_approx)[tabs[t][i].approx_hash] = e;
        else (*g_specs)[tabs[t][i].key] = e;
      }
    for (int t = 0; t < NBK_RP_SPEC_FILES; ++t)
      for (int i = 0; i < counts[t]; ++i)
        if (tabs[t][i].approx_hash) g_specs->at(tabs[t][i].key).has_approx = true;
    // (a hand-scheduled kernel stands beside generated ones, which take the launches it declines)
    for (int i = 0; i < rp_hand_count; ++i) {
      auto it = g_specs->find(rp_hand_table[i].key);
      if (it != g_specs->end()) it->second.hand = &rp_hand_table[i];
    }
  }
  auto it = g_specs->find(key);
  if (it == g_specs->end()) return nullptr;
  if (it->second.has_approx) {
    auto a = g_approx->find(rp_program_hash(p));
    if (a != g_approx->end()) return &a->second;
  }
  return &it->second;
}

// Resident workgroups per CU of a kernel at a block size (no dynamic LDS); cached.
static int rp_occupancy(const void* fn, int block, int* out) {
  static std::mutex mu;
  static std::unordered_map<uint64_t, int>* cache = nullptr;
  const uint64_t key = (uint64_t)(uintptr_t)fn ^ ((uint64_t)block << 48);
  std::lock_guard<std::mutex> lk(mu);
  if (!cache) cache = new std::unordered_map<uint64_t, int>();
  auto it = cache->find(key);
  if (it == cache->end()) {
    int n = 0;
    NBK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, block, 0));
    if (n < 1) n = 1;
    it = cache->emplace(key, n).first;
  }
  *out = it->second;
  return NBK_OK;
}

// 1: interpreter only (debug / comparison); read once.
static bool rp_specs_disabled() {
  static int v = -1;
  if (v < 0) {
    const char* e = getenv("NBK_ROWPROG_INTERPRET");
    v = (e && e[0] == '1') ? 1 : 0;
  }
  return v == 1;
}

// 1: generated kernels only (comparison of a hand-scheduled kernel with them); read once.
static bool rp_hand_disabled() {
  static int v = -1;
  if (v < 0) {
    const char* e = getenv("NBK_ROWPROG_HAND");
    v = (e && e[0] == '0') ? 1 : 0;
  }
  return v == 1;
}

extern "C" int nbk_rowprog_is_specialized(const nbk_rowprog* prog) {
  if (rp_validate(prog) != NBK_OK || rp_specs_disabled()) return 0;
  RpSpec* spec = rp_find_spec(prog);
  if (!spec) return 0;
  return (spec->hand && !rp_hand_disabled() && spec->hand->fits(prog)) ? 2 : spec->approximate ? 3 : 1;
}

extern "C" uint64_t nbk_rowprog_hash(const nbk_rowprog* prog) {
  if (rp_validate(prog) != NBK_OK) return 0;
  return rp_program_hash(prog);
}

extern "C" int nbk_rowprog_launch(const nbk_rowprog* prog, void* stream) {
  int rc = rp_validate(prog);
  if (rc != NBK_OK) return rc;
  // normalised copy: unused leading dims get extent 1 and stride 0 so the kernels
  // can index all four unconditionally
  nbk_rowprog norm = *prog;
  for (int k = norm.n_lead; k < NBK_RP_MAX_LEAD; ++k) {
    norm.lead_dim[k] = 1;
    for (int i = 0; i < norm.n_operands; ++i) norm.operand[i].lead_stride[k] = 0;
  }
  const nbk_rowprog* p = &norm;
  RpSpec* spec = (rp_specs_disabled() || prog->reserved == 1) ? nullptr
                                                               : rp_find_spec(prog);
  if (spec && spec->block_mode != (p->has_reduce ? 1 : 0)) spec = nullptr;
  hipStream_t st = (hipStream_t)stream;
  int64_t rows = 1;
  for (int k = 0; k < p->n_lead; ++k) rows *= p->lead_dim[k];
  if (p->has_reduce) {
    const int block = p->block;
    NBK_REQUIRE(block >= 64 && block <= 512 && (block & (block - 1)) == 0,
                "rowprog: workgroup size %d must be a power of two in [64, 512]", block);
    NBK_REQUIRE(rows <= 0x7fffffffLL, "rowprog: %lld rows exceed the grid limit", (long long)rows);
    const int64_t c_pad = (p->C + 3) & ~(int64_t)3;
    size_t lds = (size_t)p->n_stage * (size_t)c_pad * sizeof(float);
    NBK_REQUIRE(p->n_stage >= 0 && p->n_stage <= NBK_RP_MAX_STAGE, "rowprog: n_stage %d",
                p->n_stage);
    NBK_REQUIRE(lds <= 64 * 1024, "rowprog: staging %zu bytes of LDS exceeds 64 KiB", lds);
    // persistent workgroups: enough to fill every CU at this block size / LDS use
    const int per_cu = lds > 48 * 1024 ? 2 : (block >= 512 ? 2 : (block >= 256 ? 4 : 8));
    int64_t grid = (int64_t)nbk_num_cus() * per_cu;
    if (grid > rows) grid = rows;
    if (spec) {
      int64_t rows_arg = rows;
      void* args[2] = {(void*)p, (void*)&rows_arg};
      if (spec->hand && !rp_hand_disabled() && spec->hand->fits(p)) {
        int64_t bytes = 0;
        for (int i = 0; i < p->n_operands; ++i)
          if (p->operand[i].col_stride != 0)
            bytes += rows * p->C * (int64_t)nbk_dtype_size(p->operand[i].dtype);
        const void* fn = bytes > (256ll << 20) ? spec->hand->kernel_stream : spec->hand->kernel;
        int per_cu = 0;
        { const int orc = rp_occupancy(fn, spec->hand->block, &per_cu); if (orc != NBK_OK) return orc; }
        int64_t g2 = (int64_t)nbk_num_cus() * per_cu;
        if (g2 > rows) g2 = rows;
        NBK_HIP(hipLaunchKernel(fn, dim3((unsigned)g2), dim3(spec->hand->block), args, 0, st));
        return NBK_OK;
      }
      // register-resident form: lanes own ceil(chunks / block) chunks each
      const int64_t n_chunks = c_pad >> 2;
      const int64_t need = (n_chunks + block - 1) / block;
      int slot = need <= 1 ? 1 : need <= 2 ? 2 : need <= 4 ? 3 : need <= 8 ? 4 : 0;
      if (slot && spec->kernel[slot]) {
        static const int cpt_of[5] = {0, 1, 2, 4, 8};
        const bool full = p->C == (int64_t)4 * cpt_of[slot] * block && spec->kernel_full[slot];
        const void* fn = spec->kernel[slot];
        if (full) {
          // bytes of the row-shaped operands; beyond the 256 MiB last-level cache nothing
          // written here survives until a consumer runs, so stream it
          int64_t bytes = 0;
          for (int i = 0; i < p->n_operands; ++i)
            if (p->operand[i].col_stride != 0)
              bytes += rows * p->C * (int64_t)nbk_dtype_size(p->operand[i].dtype);
          fn = (bytes > (256ll << 20) && spec->kernel_stream[slot]) ? spec->kernel_stream[slot]
                                                                    : spec->kernel_full[slot];
        }
        // persistent workgroups, exactly as many as are resident at once: the program
        // descriptor is read from kernel-argument memory once per workgroup, not once per
        // row, and no second partial wave of workgroups trails behind the first
        int per_cu = 0;
        { const int orc = rp_occupancy(fn, block, &per_cu); if (orc != NBK_OK) return orc; }
        int64_t g2 = (int64_t)nbk_num_cus() * per_cu;
        if (g2 > rows) g2 = rows;
        NBK_HIP(hipLaunchKernel(fn, dim3((unsigned)g2), dim3(block), args, 0, st));
        return NBK_OK;
      }
      if (spec->kernel_stage16 && p->n_stage == 0 && (p->C & 3) == 0 && c_pad * 2 <= 64000) {
        // a long 16-bit row that several phases read: one copy in LDS as stored, two
        // workgroups per CU so that one row's traffic overlaps the other's arithmetic
        if (!spec->lds16_attr_set) {
          NBK_HIP(hipFuncSetAttribute(spec->kernel_stage16, hipFuncAttributeMaxDynamicSharedMemorySize,
                                      64 * 1024));
          spec->lds16_attr_set = true;
        }
        int64_t g2 = (int64_t)nbk_num_cus() * 2;
        if (g2 > rows) g2 = rows;
        NBK_HIP(hipLaunchKernel(spec->kernel_stage16, dim3((unsigned)g2), dim3(block), args,
                                (size_t)c_pad * 2, st));
        return NBK_OK;
      }
      if (spec->stage_sig == rp_stage_sig(p)) {
        if (lds > 32 * 1024 && !spec->lds_attr_set) {
          NBK_HIP(hipFuncSetAttribute(spec->kernel[0], hipFuncAttributeMaxDynamicSharedMemorySize,
                                      64 * 1024));
          spec->lds_attr_set = true;
        }
        NBK_HIP(hipLaunchKernel(spec->kernel[0], dim3((unsigned)grid), dim3(block), args, lds, st));
        return NBK_OK;
      }
    }
    return rp_vm_launch(p, rows, st);
  }
  NBK_REQUIRE(rows <= 0xffffffffLL, "rowprog: %lld rows exceed 2^32", (long long)rows);
  for (int k = 0; k < p->n_lead; ++k)
    NBK_REQUIRE(p->lead_dim[k] <= 0xffffffffLL, "rowprog: leading dim too large");
  const uint64_t cpr = (uint64_t)((p->C + 3) >> 2);
  NBK_REQUIRE(cpr <= 0xffffffffULL, "rowprog: row too long for a flat launch");
  const uint64_t total = (uint64_t)rows * cpr;
  uint64_t blocks = (total + 255) / 256;
  const uint64_t cap = (uint64_t)nbk_num_cus() * 8;
  if (blocks > cap) blocks = cap;
  if (spec) {
    uint32_t cpr_arg = (uint32_t)cpr;
    uint64_t total_arg = total;
    void* args[3] = {(void*)p, (void*)&cpr_arg, (void*)&total_arg};
    const void* fn = (rows == 1 && spec->kernel_flat) ? spec->kernel_flat : spec->kernel[0];
    NBK_HIP(hipLaunchKernel(fn, dim3((unsigned)blocks), dim3(256), args, 0, st));
    return NBK_OK;
  }
  return rp_vm_launch(p, rows, st);
}
