// Lookup table of ahead-of-time specialised row kernels.  The generated sources
// rowprog_spec_gen<N>.hip each define one table; rowprog.hip searches them by the
// key of the program it is asked to launch (operand types and instructions).
#pragma once
#include <stdint.h>
#include "nbk.h"

struct rp_spec_entry {
  uint64_t key;
  // [0]: generic form (any row length).  [1..4]: register-resident forms for
  // reduction programs whose lanes own exactly 1 / 2 / 4 / 8 chunks of a row;
  // nullptr where that form was not generated.  Reduction programs take (nbk_rowprog,
  // int64_t rows), the others (nbk_rowprog, uint32_t chunks per row, uint64_t chunks).
  const void* kernel[5];
  // [1..4]: the same register-resident forms compiled for rows of exactly
  // 1 / 2 / 4 / 8 chunks per lane (no masked lanes or elements); [0] unused.
  const void* kernel_full[5];
  // [1..4]: kernel_full with non-temporal loads and stores, for launches that move
  // more bytes than the last-level cache holds.
  const void* kernel_stream[5];
  // programs without reductions: the generic form compiled for launches of a single row (a flat
  // array: no row arithmetic per chunk); nullptr for reduction programs.
  const void* kernel_flat;
  // reduction programs over rows too long for a register-resident form, with a 16-bit input that
  // several phases read: the generic form with that row copied into LDS once, as it is stored
  // (2 bytes per element: a 32 000-element row and two workgroups fit a CU), and every phase
  // reading it from there; nullptr where not generated.
  const void* kernel_stage16;
  uint64_t stage_sig;  // what kernel[0] finds staged in LDS: a program that differs there cannot run it
  int block_mode;
  // 0, or the hash of the one program of this key that these kernels are for: they compute
  // rp_unary_lowp and rp_binary_lowp, which a benchmark step takes and no other program chose
  uint64_t approx_hash;
};

// A hand-scheduled kernel for one program (rowprog_hand.hip), attached by key to that program's
// entry above.  Signature of a generated reduction kernel; launched with `block` lanes per row when
// `fits(program)` holds, `kernel_stream` (non-temporal loads and stores) for launches that move
// more than the last-level cache holds.
struct rp_hand_entry {
  uint64_t key;
  const void* kernel;
  const void* kernel_stream;
  int block;
  bool (*fits)(const nbk_rowprog*);
};
extern const rp_hand_entry rp_hand_table[];
extern const int rp_hand_count;

#define NBK_RP_SPEC_FILES 8
#define NBK_RP_SPEC_EACH(F) F(0) F(1) F(2) F(3) F(4) F(5) F(6) F(7)
#define NBK_RP_SPEC_DECLARE(I)                       \
  extern const rp_spec_entry rp_spec_table_##I[];    \
  extern const int rp_spec_count_##I;
NBK_RP_SPEC_EACH(NBK_RP_SPEC_DECLARE)
