// The form in which the row-program interpreter runs a program (rowprog_vm.hip).
#pragma once
#include "nbk_common.h"

// What a decoded instruction does; elementwise instructions keep their nbk_rp_op number.
enum rp_vm_op {
  RPVM_STG = 1,     // operand c <- a
  RPVM_STR,         // operand c <- scalar a (one lane per row)
  RPVM_LD,          // (an input that a row or segment starts with: never executed)
  RPVM_LDG,         // dst <- operand c, requested in place
  RPVM_LDS,         // (a scalar that a row starts with: never executed)
  RPVM_LDR,         // scalar dst <- operand c at the row, requested in place
  RPVM_COLIDX,      // dst <- column index (c: as int32)
  RPVM_RED,         // scalar dst <- vector a (ROW) or accumulator c (LOOP) reduced over the row, kind b; aux: how
                    // many follow in one exchange
  RPVM_ACCINIT,     // accumulator c <- identity of kind b
  RPVM_ACC,         // accumulator c <- combined with vector a, kind b
  RPVM_IMM,         // scalar dst <- imm[c]
  RPVM_LEADIDX,     // scalar dst <- index of leading dim c (b: as int32)
  RPVM_SEG          // the aux instructions behind it run once per chunk (b) or row; slots[c ..) are its inputs, a of them
};

#define RPVM_SCALAR 32     /* register numbers from here on are scalars     */
#define RPVM_NONE 255      /* no result                                     */
#define RPVM_SLOTS 8       /* inputs of a row or chunk requested at once: registers 0, 1, ... */
#define RPVM_ROW_SLOTS 4   /* and scalars of a row                          */
/* Decoded instructions and one read ahead: a program's NBK_RP_MAX_INS and, where it is looped over, a
   segment for the scalars behind every body (a third of them at most) and for those before the first. */
#define RPVM_MAX_INS (NBK_RP_MAX_INS + NBK_RP_MAX_INS / 3 + 6)

struct rp_vm_ins {
  uint8_t op, dst, a, b, c;
  uint8_t two;  // elementwise: whether there is a second operand
  uint16_t aux;
};

// Kernel argument of the interpreter.
struct rp_vm {
  int64_t lead_dim[NBK_RP_MAX_LEAD];
  int64_t C;
  int32_t n_lead;
  // ins[0 .. n_once): scalar instructions that no row or chunk changes; ins[n_once .. n_ins): the program
  int32_t n_once, n_ins;
  int32_t n_slots, n_row_slots;
  int32_t lanes;     // lanes per row (power of two up to 32, or a multiple of 64)
  int32_t rare;      // whether it calls one of the long functions (logarithm, erf, powers, ...)
  uint8_t slots[44]; // operand of every input slot (per segment in a looped program)
  uint8_t row_slots[RPVM_ROW_SLOTS], row_dst[RPVM_ROW_SLOTS];  // operands and registers of a row's scalars
  float imm[NBK_RP_MAX_IMM + 1];  // (and a zero)
  nbk_operand operand[NBK_RP_MAX_OPERANDS];
  rp_vm_ins ins[RPVM_MAX_INS];
};

// How a program is launched: one chunk per lane without reductions; a row held by some lanes of a
// wavefront or by a workgroup; a row walked in chunks.
enum rp_vm_mode { RPVM_FLAT = 0, RPVM_ROW = 1, RPVM_LOOP = 2 };

// Decodes `p` (validated) into `out`; false where `mode` cannot run it (the accumulators of a row
// held in registers must be started, fed once and reduced with one kind).
bool rp_vm_decode(const nbk_rowprog* p, int mode, rp_vm* out);
// Launches a program on the interpreter.
int rp_vm_launch(const nbk_rowprog* p, int64_t rows, hipStream_t stream);
