// The fp32 attention kernels on the fp32 matrix cores (attn_f32.hip): the
// forward and backward of heads with e == od in {64, 128}, which
// pdh_flash_fwd and pdh_flash_bwd (flash_fwd.hip, flash_bwd.hip) send here.
#pragma once

#include "common.h"

namespace pdh {

struct AttnF32Args {
  const float* q;
  const float* k;
  const float* v;
  // forward: o written, the row statistics optional; backward: o and dout read
  float* o;
  float* m_out;
  float* den_out;
  float* lse_out;
  const float* dout;
  const float* lse;
  const float* m_in;
  const float* den_in;
  float* dq;
  float* dk;
  float* dv;
  float* ws;  // backward: [3][rows] -delta, lse log2(e), masked-entry probability
  int64_t rows;  // batch * heads * t
  int heads, heads_kv, group;
  int t, s;
  int64_t q_sb, q_sh, q_st, k_sb, k_sh, k_st, v_sb, v_sh, v_st, o_sb, o_sh, o_st;
  float scale, fill;
  int masked;
  int band_lo, band_hi;  // the band clamped to +-(2^29 + 64): t, s <= 2^29 compare against it as against 64 bits
  int prune;             // dead tiles may be skipped (every row has a live key)
  int ninst_kv, nqb, nkb;
};

// Whether the matrix-core kernels take this geometry: e == od in {64, 128},
// t and s within 32-bit row arithmetic, and the rows of a staged tile (64 at
// D = 64, 32 at D = 128) within 2 GiB of each other for every operand.
bool attn_f32_takes(const pdh_attn_geom& g);

// Geometry, mask and scale of `a` (tensor pointers are the caller's to set).
AttnF32Args attn_f32_args(const pdh_attn_geom& g, float scale, float fill, int masked, int64_t band_lo,
                          int64_t band_hi, int prune);

int attn_f32_forward(AttnF32Args a, const pdh_attn_geom& g, hipStream_t st);
int attn_f32_backward(AttnF32Args a, const pdh_attn_geom& g, hipStream_t st);

}  // namespace pdh
