// Device form of the parameter/coefficient bytecode (see lb_program.cpp).
#pragma once

#include <string>
#include <vector>

#include "lb_device.h"

struct LbProgram {
  std::vector<DevInstr> instr;
  std::vector<int32_t> expr_start;     // n_compounds + K + 1
  std::vector<int32_t> compound_slot;  // n_compounds (hidden ones included)
  std::vector<uint8_t> compound_dyn;
  std::vector<uint8_t> coef_dyn;
  int n_compounds = 0;
  int n_slots = 0;  // original slots + hidden cache slots
  int max_depth = 0;
};

// Three-address form of time-dependent expressions (DevVOp, lb_device.h).
struct LbVector {
  int n_slots = 0;                     // slots of a copy: the program's, constants, time, temporaries
  int time_slot = -1;
  std::vector<int32_t> const_slot;     // slot of each constant
  std::vector<double> const_value;     // re, im
  std::vector<DevVOp> ops;             // steps x LB_VOP_LANES
  int steps = 0;
};

// The expressions `list` of `prog` (in evaluation order; each reads slots
// written by earlier ones), expression e into slot dst[i] or (dst[i] < 0)
// coefficient row entry -dst[i] - 1, as steps of independent operations of
// one opcode.  Slots are numbered from first_slot on.  A program that would take
// more than max_bytes with `copies` copies of its slots gets no steps.
LbVector lb_vector_program(const LbProgram& prog, const std::vector<int32_t>& list, const std::vector<int32_t>& dst,
                           int first_slot, int copies, int64_t max_bytes);

// Returns 0 on success, -1 (with `why`) on a malformed expression.
int lb_build_program(const lb_plan_desc* d, const std::vector<uint8_t>& dyn_slot,
                     const std::vector<uint8_t>& compound_dyn, const std::vector<uint8_t>& coef_dyn,
                     LbProgram* out, std::string& why);
