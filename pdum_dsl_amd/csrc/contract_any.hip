// pdh_contract_any: the 16-bit contraction over operands stored either way
// round (k contiguous, or rows contiguous as a weight [k][n] is), with its k
// split over workgroups where the output's tiles cannot fill the chip. The
// kernels are the bodies of contract_core.h; the epilogue's come specialized
// from jit.hip.
#include <type_traits>

#include "common.h"
#include "contract_core.h"
#include "contract_host.h"
#include "jit.h"

namespace pdh {
namespace {

template <int DT, int LAY>
__global__ __launch_bounds__(256, 2) void contract_part(ContractArgs a, float* ws) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[contract_lds<32>()];
  contract_part_body<DT, LAY>(a, ws, smem);
}

int compute_units() {
  static const int cus = pdh_device_cus() > 0 ? pdh_device_cus() : 256;
  return cus;
}

// k slices: 1 where 64 x 64 tiles give every compute unit a workgroup or k is
// short; otherwise the cheapest under what a slice costs: a 64-wide k tile
// takes kTile us, the finish kFin us plus its planes' traffic. 458 x 320 x
// 6144 (40 tiles): 28.2 -> 12.7 us; 64 x 512 x 4096 (8): 19.7 -> 11.1; 24 x 6144
// x 4096 (96): 19.9 -> 15.5. Over half a tile per compute unit two slices pass one
// workgroup a unit and are not taken; two a unit have not been measured.
int pick_split(int64_t batch, int64_t m, int64_t n, int64_t k) {
  constexpr double kTile = 0.27, kFin = 3.5, kBytesPerUs = 4e6;
  const int64_t tiles = batch * ((m + 63) / 64) * ((n + 63) / 64), kt = (k + kBK - 1) / kBK;
  int best = 1;
  double cost = kTile * static_cast<double>(kt);
  for (int s = 2; s <= 16 && s * 2 <= kt && tiles * s <= compute_units(); ++s) {
    const int64_t per = (kt + s - 1) / s;
    if ((s - 1) * per >= kt) continue;  // an empty slice
    const double c = kTile * static_cast<double>(per) + kFin +
                     2.0 * s * static_cast<double>(batch * m * n) * 4.0 / kBytesPerUs;
    if (c < cost) {
      cost = c;
      best = s;
    }
  }
  return best;
}

}  // namespace
}  // namespace pdh

using namespace pdh;

extern "C" size_t pdh_contract_any_workspace(int64_t batch, int64_t m, int64_t n, int64_t k) {
  if (batch < 1 || m < 1 || n < 1 || k < 1) return 0;
  const int s = pick_split(batch, m, n, k);
  return s > 1 ? static_cast<size_t>(s) * static_cast<size_t>(batch * m * n) * sizeof(float) : 0;
}

extern "C" int pdh_contract_any(const void* a, int64_t sa_b, int64_t sa_r, int64_t sa_k, const void* bt, int64_t sb_b,
                                int64_t sb_r, int64_t sb_k, int64_t batch, int64_t m, int64_t n, int64_t k,
                                const pdh_ew_program* epi, const void* const* operands, void* out, int dtype,
                                void* ws, size_t ws_bytes, void* stream) {
  const char* fn = "pdh_contract_any";
  PDH_REQUIRE(dtype == PDH_BF16 || dtype == PDH_F16, PDH_EUNSUPPORTED, "%s: 16-bit operands only (fp32: pdh_contract_views)",
              fn);
  PDH_REQUIRE(a && bt && out, PDH_EINVAL, "%s: null pointer", fn);
  PDH_REQUIRE(batch >= 1 && m >= 1 && n >= 1 && k >= 1 && k % 8 == 0, PDH_EINVAL,
              "%s: need batch, m, n >= 1 and k a positive multiple of 8", fn);
  PDH_REQUIRE(batch * m * n <= INT32_MAX && m <= INT32_MAX / 2 && n <= INT32_MAX / 2 && k <= INT32_MAX / 2, PDH_EINVAL,
              "%s: output too large for one call", fn);
  // every 1 KB load is made of 16-byte chunks of a row: rows (of k values, or
  // k rows of values) and slices start on 16 bytes and do not overlap
  auto layout_ok = [&](const void* p, int64_t sb, int64_t sr, int64_t sk, int64_t rows) {
    return aligned16(p) && sb >= 0 && sb % 8 == 0 &&
           ((sk == 1 && sr >= k && sr % 8 == 0) || (sr == 1 && sk >= rows && sk % 8 == 0 && rows % 8 == 0));
  };
  PDH_REQUIRE(layout_ok(a, sa_b, sa_r, sa_k, m) && layout_ok(bt, sb_b, sb_r, sb_k, n), PDH_EINVAL,
              "%s: an operand needs k contiguous, or its rows contiguous with their number a multiple of 8, and 16-byte rows",
              fn);
  PDH_REQUIRE((m + 128) * sa_r * 2 + (k + 64) * sa_k * 2 < (int64_t{1} << 31) &&
                  (n + 128) * sb_r * 2 + (k + 64) * sb_k * 2 < (int64_t{1} << 31),
              PDH_EINVAL, "%s: a batch entry of a / bt must span under 2 GiB", fn);
  int rc = check_program(epi, 3, true, fn);
  if (rc) return rc;
  PDH_REQUIRE(epi->shape[0] == batch && epi->shape[1] == m && epi->shape[2] == n, PDH_EINVAL,
              "%s: epilogue shape must be {batch, m, n}", fn);
  PDH_REQUIRE(epi->n_operands == 0 || operands != nullptr, PDH_EINVAL, "%s: null operand table", fn);
  if ((rc = check_view(epi, epi->out_stride, fn, "output"))) return rc;
  EwOperands ops{};
  for (int i = 0; i < epi->n_operands; ++i) {
    PDH_REQUIRE(operands[i] != nullptr, PDH_EINVAL, "%s: operand %d is null", fn, i);
    if ((rc = check_view(epi, epi->in_stride[i], fn, "operand"))) return rc;
    ops.p[i] = operands[i];
  }
  const int split = pick_split(batch, m, n, k);
  const size_t need = pdh_contract_any_workspace(batch, m, n, k);
  PDH_REQUIRE(need == 0 || (ws != nullptr && ws_bytes >= need && aligned16(ws)), PDH_EINVAL,
              "%s: ws must be 16-byte aligned and hold %zu bytes (got %zu)", fn, need, ws_bytes);
  const int lay = (sa_k != 1 ? 1 : 0) | (sb_k != 1 ? 2 : 0);
  hipFunction_t fns[kJitFns];
  PDH_REQUIRE(jit_get(JitKind::Contract, *epi, dtype, fns, lay, -1), PDH_EUNSUPPORTED,
              "%s: needs the runtime-specialized kernels (disabled, or their compile failed)", fn);
  const int64_t kt = (k + kBK - 1) / kBK, kp = (kt + split - 1) / split * kBK;
  ContractArgs ca{a, bt, out, static_cast<int>(batch * split), static_cast<int>(m), static_cast<int>(n),
                  static_cast<int>(k), static_cast<int>(kp), 0, 0, dtype, sa_b, sa_r, sb_b, sb_r, split, sa_k, sb_k, -1};
  const int cus = compute_units();
  // the big tiles where they fill the chip and their k is long enough to hide
  // its loads (contract_launch's rule); else 64 x 64 tiles
  const bool small = batch * ((m + 127) / 128) * ((n + 127) / 128) < cus || m <= 64 || n <= 64 || k <= 2 * kBK;
  const int bm = small ? 64 : 128;
  ca.tiles_m = static_cast<int>((m + bm - 1) / bm);
  ca.tiles_n = static_cast<int>((n + bm - 1) / bm);
  const int64_t nblk = batch * split * ca.tiles_m * ca.tiles_n;
  PDH_REQUIRE(nblk <= INT32_MAX, PDH_EINVAL, "%s: grid too large", fn);
  hipStream_t st = as_stream(stream);
  pdh_ew_program pe = *epi;
  auto launch = [&](hipFunction_t f, int64_t blocks, void** args) {
    PDH_REQUIRE(hipModuleLaunchKernel(f, static_cast<unsigned>(blocks), 1, 1, 256, 1, 1, 0, st, args, nullptr) ==
                    hipSuccess,
                PDH_ELAUNCH, "%s: specialized launch failed", fn);
    jit_count_launch();
    return PDH_OK;
  };
  if (split == 1) {
    void* args[] = {&ca, &pe, &ops};
    return launch(fns[small ? 1 : 0], nblk, args);
  }
  float* wsf = static_cast<float*>(ws);
  auto part = [&](auto dt, auto lay_c) {
    contract_part<decltype(dt)::value, decltype(lay_c)::value><<<dim3(static_cast<unsigned>(nblk)), 256, 0, st>>>(ca, wsf);
  };
  auto part_lay = [&](auto dt) {
    if (lay == 0)
      part(dt, std::integral_constant<int, 0>{});
    else if (lay == 1)
      part(dt, std::integral_constant<int, 1>{});
    else if (lay == 2)
      part(dt, std::integral_constant<int, 2>{});
    else
      part(dt, std::integral_constant<int, 3>{});
  };
  if (dtype == PDH_BF16)
    part_lay(std::integral_constant<int, PDH_BF16>{});
  else
    part_lay(std::integral_constant<int, PDH_F16>{});
  if ((rc = check_launch(fn))) return rc;
  const int64_t lanes = batch * m * ((n + 3) / 4);
  void* args[] = {&ca, &pe, &ops, &wsf};
  return launch(fns[2], (lanes + 255) / 256, args);
}
