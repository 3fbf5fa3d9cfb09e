// Host-side checks shared by the elementwise and contraction entry points (contract.hip).
#pragma once

#include "common.h"

namespace pdh {

// A program in full: opcodes, registers, operand slots and dims in range (ndim < 0: any).
int check_program(const pdh_ew_program* p, int ndim, bool allow_acc, const char* fn);
// A view of the program's lattice: non-negative strides, its largest offset under 2^31.
int check_view(const pdh_ew_program* p, const int64_t* stride, const char* fn, const char* what);

// How fp32 contractions run at this moment (pdh_contract_set_f32_mode): 0 VALU
// fma; 1, 3 or 6 bf16 MFMA products per term. Another thread may change it:
// read once per call, and handed on.
int f32_contract_mode();

}  // namespace pdh
