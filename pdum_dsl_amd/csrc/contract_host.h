// Host-side checks shared by the elementwise and contraction entry points (contract.hip).
#pragma once

#include "common.h"

namespace pdh {

// A program in full: opcodes, registers, operand slots and dims in range (ndim < 0: any).
int check_program(const pdh_ew_program* p, int ndim, bool allow_acc, const char* fn);
// A view of the program's lattice: non-negative strides, its largest offset under 2^31.
int check_view(const pdh_ew_program* p, const int64_t* stride, const char* fn, const char* what);

}  // namespace pdh
