// Runtime specialization of elementwise programs (jit.hip).
#pragma once

#include "common.h"

namespace pdh {

enum class JitKind { MapChain, Contract };

constexpr int kJitFns = 3;  // kernels of one specialized module, at most

bool jit_enabled();
// The kernels specialized for program p and element type dt; false when the
// interpreter kernels must run it (disabled, or the compile failed). Map chain:
// fns[0] four elements per lane, fns[1] one. Contraction: fns[0] 128 x 128
// tiles, fns[1] 64 x 64 tiles; at 16 bits also fns[2], the finish of a k split.
// lay: the operands' layouts (LAY of the contraction bodies);
// red: the fp32 row-partial reduction (ContractArgs::rowred, -1 for none);
// f32_mode: how an fp32 contraction runs (0 VALU fma; 1, 3 or 6 bf16 MFMA
// products per term), the mode its caller launches by: pdh_contract_set_f32_mode
// may change the process's at any time, so none of these functions reads it.
bool jit_get(JitKind kind, const pdh_ew_program& p, int dt, hipFunction_t fns[kJitFns], int lay = 0, int red = -1,
             int f32_mode = 6);
// The row-reduce kernels specialized for (summand, epilogue): fns[0] one wave
// per output, fns[1] the column variant; or false.
bool jit_get_reduce(const pdh_ew_program& ps, const pdh_ew_program& pe, int dt, hipFunction_t fns[kJitFns]);
// The fp32 contraction with operand prologues (pa / pb null: read as a view),
// specialized: fns[0] the 128 x 128-tile (or fp32-mode-0 VALU) kernel, fns[1]
// the 64 x 64-tile one; or false.
bool jit_get_pro(const pdh_ew_program& pe, const pdh_ew_program* pa, const pdh_ew_program* pb, hipFunction_t fns[kJitFns],
                 int lay, int dt, int f32_mode);
void jit_count_launch();

}  // namespace pdh
