// fp32 attention, forward and backward, on the fp32 matrix cores
// (v_mfma_f32_16x16x4_f32: exact fp32 products and sums, 256 FLOP per cycle
// and compute unit, twice the unpacked VALU rate), e == od == D in {64, 128}.
//
// Layout. A wave owns 16 rows of its side (queries in the forward and in dQ,
// keys in dK / dV) as the columns of every product and sweeps the other
// side's rows in tiles of 16 or 32 staged in LDS, so a score tile comes out
// with its swept rows 4 G + i and owned row c on lane 16 G + c. The k index of
// a product may be taken in any order that both operands share, which removes
// every shuffle and transpose:
//   * scores: lane (G, c) reads 16 bytes of a row, features 16 s + 4 G ..+3,
//     and its j-th float is the k = G element of the j-th 16x16x4 product;
//   * the second contraction sums over swept rows: product j takes rows
//     4 G + j, so a lane's score accumulators are its B operand as they
//     stand, and the A operand is a 4-byte LDS read of feature c.
// LDS rows are unpadded; the 16-byte slot that holds chunk x of row r is
// x ^ (r & 15). Row reads (ds_read_b128: lane 16 G + c, row c, chunk 4 s + G)
// and feature reads (ds_read_b32: row 4 G + j, floats 16 f + c) both hit
// distinct banks under the bank rule tests/test_lds_layout.py states.
//
// What bounds it: the matrix pipe. A 16-column wave spends 4096 cycles of
// products per 32 swept rows and 16 columns in dK / dV (D = 64) against about
// 1000 of VALU and a quarter of the CU's LDS cycles, so 16 columns a wave is
// enough reuse, and it leaves the small blocks that balance a causal sweep
// over 256 CUs. Against the VALU kernels this replaced (one wave per row; one
// row per lane in the forward): 24 causal heads x 1000, D = 64, backward 7070
// -> 157 us and forward 182 -> 56 us (matrix pipe 48% and 36% busy: the causal
// tail); 32 heads x 2048, D = 64, all keys live: forward 115 TFLOP/s, backward 117
// (seven products, the dQ role recomputes two) of the 157 the fp32 matrix cores
// peak at, 72% and 75% busy; one head x 256: 29 -> 7.2 us.
// The distance to 64 bits is smaller than the VALU kernels' (o 1.8e-7, dK 3.9e-7 of
// the norm at 24 x 1000, against 2.6e-7 and 8.1e-7).
#include "attn_f32.h"

#include "attn_common.h"

#include <type_traits>

namespace pdh {
namespace {

constexpr float kInf = __builtin_inff();
constexpr int64_t kMaxRows32 = int64_t{1} << 29;

// The most rows any kernel here stages as one tile, and the row strides (in
// elements) under which such a tile's byte offsets stay under 2^31.
constexpr int tile_rows(int64_t D) { return D == 64 ? 64 : 32; }
constexpr int64_t max_stride(int64_t D) { return (int64_t{1} << 31) / (4 * tile_rows(D)); }

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// max / sum over the four lanes 16 G + c of one column
__device__ __forceinline__ float col_max(float m) {
  m = fmaxf(m, __shfl_xor(m, 32, 64));
  return fmaxf(m, __shfl_xor(m, 16, 64));
}
__device__ __forceinline__ float col_sum(float v) {
  v += __shfl_xor(v, 32, 64);
  return v + __shfl_xor(v, 16, 64);
}

__device__ __forceinline__ float exp_nat(float x) { return fast_exp2(x * kLog2e); }

// A tile of ROWS rows staged by W waves. AL: rows start on 16-byte boundaries
// (16 bytes per lane and load); otherwise 4 bytes per lane, the same layout.
template <int D, int ROWS, int W, bool AL>
struct Tile {
  static constexpr int ROWB = D * 4, BYTES = ROWS * ROWB;
  static constexpr int LD = AL ? 1024 : 256;         // bytes one load instruction of a wave brings
  static constexpr int N = BYTES / LD / W;           // loads per wave
  static_assert(BYTES % (LD * W) == 0, "a tile splits evenly over the waves");
  static_assert(ROWS <= tile_rows(D), "attn_f32_takes bounds the row strides for this tile");

  // rows [row0, row0 + ROWS) of a tensor (rows past `ext` read zeros, or the
  // last row's bytes where rows overlap: callers mask them)
  __device__ __forceinline__ static void stage(const float* base, int64_t st, int row0, int ext, unsigned char* lds,
                                               int lane, int w) {
    const int left = ext - row0 < ROWS ? ext - row0 : ROWS;
    const uint32_t gr = static_cast<uint32_t>(st) * 4u;
    const rsrc_t r = make_rsrc(base + static_cast<int64_t>(row0) * st, static_cast<uint32_t>(left - 1) * gr + ROWB);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int blk = i * W + w;
      if constexpr (AL) {
        constexpr int SL = D / 4, RPK = 64 / SL;  // slots per row, rows per load
        const int row = blk * RPK + lane / SL, slot = lane % SL;
        dma16(r, lds + blk * LD, (lane / SL) * gr + ((slot ^ (row & 15)) << 4), blk * RPK * gr);
      } else {
        constexpr int LPR = ROWB / LD;  // loads per row
        const int row = blk / LPR, slot = blk % LPR * 16 + lane / 4;
        dma4(r, lds + blk * LD, ((slot ^ (row & 15)) << 4) + (lane & 3) * 4, static_cast<uint32_t>(row) * gr);
      }
    }
  }
};

// Per-lane LDS offsets into a tile, the same for every tensor.
template <int D>
struct LaneOff {
  static constexpr int ROWB = D * 4, NS = D / 16;
  int rowr[4];     // row reads: row c, chunk 4 s + G for s < 4 (s >= 4: + 256 bytes)
  int feat[4][4];  // feature reads: row 4 G + j, floats 16 f + c for f < 4 (f >= 4: + 256 bytes)
  __device__ __forceinline__ void init(int lane) {
    const int G = lane >> 4, c = lane & 15;
#pragma unroll
    for (int s = 0; s < 4; ++s) rowr[s] = c * ROWB + (((4 * s + G) ^ c) << 4);
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        feat[f][j] = (4 * G + j) * ROWB + (((4 * f + (c >> 2)) ^ (4 * G + j)) << 4) + ((c & 3) << 2);
  }
  __device__ __forceinline__ f32x4 row(const unsigned char* t, int half, int s) const {
    return *reinterpret_cast<const f32x4*>(t + half * 16 * ROWB + rowr[s & 3] + (s >> 2) * 256);
  }
  __device__ __forceinline__ float feature(const unsigned char* t, int half, int f, int j) const {
    return *reinterpret_cast<const float*>(t + half * 16 * ROWB + feat[f & 3][j] + (f >> 2) * 256);
  }
};

// A wave's 16 owned rows as a product's B operand: lane (G, c) holds features
// 16 s + 4 G ..+3 of row row0 + c (zero past `ext`).
template <int D>
__device__ __forceinline__ void load_cols(f32x4 (&x)[D / 16], const float* base, int64_t st, int row0, int ext,
                                          int lane) {
  const int G = lane >> 4, r = row0 + (lane & 15);
  const bool ok = r < ext;
  const float* p = base + static_cast<int64_t>(ok ? r : ext - 1) * st + 4 * G;
#pragma unroll
  for (int s = 0; s < D / 16; ++s) {
    const f32x4 y = *reinterpret_cast<const f32x4u*>(p + 16 * s);
    x[s] = ok ? y : f32x4{0.f, 0.f, 0.f, 0.f};
  }
}

// Workgroup -> logical position: dispatch goes round-robin over the 8 XCDs,
// so XCD x takes a contiguous run and its L2 holds the instances it sweeps.
__device__ __forceinline__ int64_t xcd_position() {
  const int64_t n = gridDim.x, bid = blockIdx.x, x = bid & 7, per = n >> 3, rem = n & 7;
  return x * per + (x < rem ? x : rem) + (bid >> 3);
}

// Position -> (instance, rank): groups of four instances are taken rank by
// rank, heaviest first, so a group's long blocks start together.
__device__ __forceinline__ void instance_rank(int64_t pos, int ninst, int nb, int& inst, int& rank) {
  const int64_t g = pos / (4 * nb);
  const int r = static_cast<int>(pos - g * 4 * nb);
  const int left = ninst - static_cast<int>(4 * g);
  const int n = left < 4 ? left : 4;
  inst = __builtin_amdgcn_readfirstlane(static_cast<int>(4 * g) + r % n);  // uniform: keep them scalar
  rank = __builtin_amdgcn_readfirstlane(r / n);
}

// ---------------------------------------------------------------- forward
//
// WQ x WK waves: wave (wq, wk) owns query rows 16 wq .. of the block's 16 WQ
// and, of each staged step of 16 KH WK keys, the run of 16 KH keys at index
// wk; the WK partial states (m, l, o) merge through LDS at the end with the
// associative combine (zoo/attention.py:40-46). Key steps sit on the absolute
// key grid and a masked score inside a swept step is the fill, whose
// exponential vanishes against a live row's maximum: pruned and unpruned
// sweeps agree bit for bit.
template <int D, int WQ, int WK, int KH, bool AL>
__global__ __launch_bounds__(64 * WQ * WK, 2) void attn_f32_fwd(AttnF32Args a) {
  constexpr int W = WQ * WK, NS = D / 16, STEP = 16 * KH * WK, BM = 16 * WQ;
  using T = Tile<D, STEP, W, AL>;
  constexpr int MERGE = (WK - 1) * WQ * (NS * 4 + 2) * 64 * 4;
  constexpr int LDS = 4 * T::BYTES > MERGE ? 4 * T::BYTES : MERGE;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[LDS];
  const int lane = threadIdx.x & 63, w = wave_id(), c = lane & 15, G = lane >> 4;
  const int wq = w % WQ, wk = w / WQ;

  int inst, rank;
  instance_rank(xcd_position(), a.ninst_kv * a.group, a.nqb, inst, rank);
  const int qb = a.nqb - 1 - rank;  // late query blocks see the most keys of a causal band
  const int64_t b = inst / a.heads, hq = inst % a.heads, hk = hq / a.group;
  const float* kp = a.k + b * a.k_sb + hk * a.k_sh;
  const float* vp = a.v + b * a.v_sb + hk * a.v_sh;
  const int q0 = qb * BM, qw = q0 + 16 * wq, qrow = qw + c;

  f32x4 q[NS], o[NS];
  load_cols<D>(q, a.q + b * a.q_sb + hq * a.q_sh, a.q_st, qw, a.t, lane);
#pragma unroll
  for (int f = 0; f < NS; ++f) o[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -kInf, l = 0.f;

  int lo = 0, hi = (a.s + STEP - 1) / STEP;
  if (a.masked && a.prune) {
    const int qlast = q0 + BM - 1 < a.t ? q0 + BM - 1 : a.t - 1;
    const int smin = q0 + a.band_lo, smax = qlast + a.band_hi;
    if (smin > 0) lo = smin / STEP;
    hi = smax < 0 ? 0 : (smax / STEP + 1 < hi ? smax / STEP + 1 : hi);
  }
  LaneOff<D> off;
  off.init(lane);
  auto stage = [&](int buf, int kt) __attribute__((always_inline)) {
    unsigned char* t = smem + buf * 2 * T::BYTES;
    T::stage(kp, a.k_st, kt * STEP, a.s, t, lane, w);
    T::stage(vp, a.v_st, kt * STEP, a.s, t + T::BYTES, lane, w);
  };
  auto compute = [&](int kt, auto bufc) __attribute__((always_inline)) {
    constexpr int buf = decltype(bufc)::value;
    const int k0 = kt * STEP + 16 * KH * wk;  // this wave's keys: [k0, k0 + 16 KH)
    if (k0 >= a.s) return;
    bool cut = k0 + 16 * KH > a.s;
    if (a.masked) {
      const int dmin = k0 - (qw + 15), dmax = k0 + 16 * KH - 1 - qw;
      if (a.prune && (dmin > a.band_hi || dmax < a.band_lo)) return;
      cut = cut || dmin < a.band_lo || dmax > a.band_hi;
    }
    const unsigned char* kt_ = smem + buf * 2 * T::BYTES + 16 * KH * wk * T::ROWB;
    const unsigned char* vt_ = kt_ + T::BYTES;
    // Short chains of sums, as a wave's lanes had before the matrix cores: the
    // even and the odd chunks of D apart, and each step's P V added to o as a
    // whole. One chain over D and one over the keys was 1-4% faster but left o
    // 2.81e-7 from 64 bits at 24 heads x 1000 causal and 5.1e-7 at 64 heads x
    // 270 x 1232, D = 64 (the VALU kernel: 2.56e-7, 4.2e-7); these: 1.76e-7, 2.3e-7.
    f32x4 s[KH], s1[KH];
#pragma unroll
    for (int h = 0; h < KH; ++h) s[h] = s1[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < NS; ++x) {
      f32x4 kf[KH];
#pragma unroll
      for (int h = 0; h < KH; ++h) kf[h] = off.row(kt_, h, x);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int h = 0; h < KH; ++h) {
          f32x4& t = x & 1 ? s1[h] : s[h];
          t = mfma4(kf[h][j], q[x][j], t);
        }
    }
    float mx = m;
#pragma unroll
    for (int h = 0; h < KH; ++h) s[h] = (s[h] + s1[h]) * a.scale;
    if (cut) {
#pragma unroll
      for (int h = 0; h < KH; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = k0 + 16 * h + 4 * G + i, d = key - qrow;
          if (a.masked && (d < a.band_lo || d > a.band_hi)) s[h][i] = a.fill;
          if (key >= a.s) s[h][i] = -kInf;
        }
    }
#pragma unroll
    for (int h = 0; h < KH; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[h][i]);
    mx = col_max(mx);
    const float ref = mx == -kInf ? 0.f : mx;
    const float alpha = exp_nat(m - ref);
    float ps = 0.f;
#pragma unroll
    for (int h = 0; h < KH; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[h][i] = exp_nat(s[h][i] - ref);
        ps += s[h][i];
      }
    l = l * alpha + ps;
    m = mx;
#pragma unroll
    for (int f0 = 0; f0 < NS; f0 += 4) {
      f32x4 pv[4];
#pragma unroll
      for (int f = 0; f < 4; ++f) pv[f] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int h = 0; h < KH; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int f = 0; f < 4; ++f) pv[f] = mfma4(off.feature(vt_, h, f0 + f, j), s[h][j], pv[f]);
#pragma unroll
      for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[f0 + f][i] = __builtin_fmaf(o[f0 + f][i], alpha, pv[f][i]);
    }
  };
  auto step = [&](int kt, auto bufc) __attribute__((always_inline)) {
    wait_vmcnt0();
    __syncthreads();
    if (kt + 1 < hi) stage(1 - decltype(bufc)::value, kt + 1);
    compute(kt, bufc);
  };
  if (lo < hi) stage(0, lo);
  for (int kt = lo; kt < hi; kt += 2) {
    step(kt, std::integral_constant<int, 0>{});
    if (kt + 1 < hi) step(kt + 1, std::integral_constant<int, 1>{});
  }

  if constexpr (WK > 1) {  // merge the key groups' states: the tiles are done with
    __syncthreads();
    float* sm = reinterpret_cast<float*>(smem);
    constexpr int ST = (NS * 4 + 2) * 64;  // floats of one wave's state
    if (wk > 0) {
      float* p = sm + ((wk - 1) * WQ + wq) * ST;
#pragma unroll
      for (int f = 0; f < NS; ++f) *reinterpret_cast<f32x4*>(p + (f * 64 + lane) * 4) = o[f];
      p[NS * 256 + lane] = m;
      p[NS * 256 + 64 + lane] = l;
    }
    __syncthreads();
    if (wk != 0) return;
    float M = m;
#pragma unroll
    for (int i = 0; i < WK - 1; ++i) M = fmaxf(M, sm[(i * WQ + wq) * ST + NS * 256 + lane]);
    const float w0 = m == -kInf ? 0.f : exp_nat(m - M);
    l *= w0;
#pragma unroll
    for (int f = 0; f < NS; ++f) o[f] *= w0;
#pragma unroll
    for (int i = 0; i < WK - 1; ++i) {
      const float* p = sm + (i * WQ + wq) * ST;
      const float mi = p[NS * 256 + lane];
      const float wi = mi == -kInf ? 0.f : exp_nat(mi - M);
      l += p[NS * 256 + 64 + lane] * wi;
#pragma unroll
      for (int f = 0; f < NS; ++f) o[f] += *reinterpret_cast<const f32x4*>(p + (f * 64 + lane) * 4) * wi;
    }
    m = M;
  }
  l = col_sum(l);
  if (qrow >= a.t) return;
  const float inv = 1.0f / l;
  float* orow = a.o + b * a.o_sb + hq * a.o_sh + static_cast<int64_t>(qrow) * a.o_st + 4 * G;
#pragma unroll
  for (int f = 0; f < NS; ++f) *reinterpret_cast<f32x4u*>(orow + 16 * f) = o[f] * inv;
  if (G == 0) {
    const int64_t row = static_cast<int64_t>(inst) * a.t + qrow;
    if (a.m_out) a.m_out[row] = m;
    if (a.den_out) a.den_out[row] = l;
    if (a.lse_out) a.lse_out[row] = m + __logf(l);
  }
}

// A wave's own direct loads have landed: nothing after this reads the tile earlier.
__device__ __forceinline__ void wait_own_tile() {
  wait_vmcnt0();
  asm volatile("" ::: "memory");
}

// The forward on grids that cannot fill the chip: 16 query rows a workgroup,
// its W waves taking every W-th 16-key tile (on the absolute key grid), each
// through an LDS ring of its own: no wave shares a tile with another, so the
// sweep has no barrier. The states merge through LDS at the end, the waves
// sharing the features.
template <int D, int W, bool AL>
__global__ __launch_bounds__(64 * W, W / 4) void attn_f32_fwd_small(AttnF32Args a) {
  constexpr int NS = D / 16;
  using T = Tile<D, 16, 1, AL>;
  constexpr int RING = 4 * T::BYTES;  // a wave: two buffers of a K and a V tile
  static_assert(W * NS * 1024 + W * 512 <= W * RING, "the states fit the rings");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[W * RING];
  const int lane = threadIdx.x & 63, w = wave_id(), c = lane & 15, G = lane >> 4;
  int inst, rank;
  instance_rank(xcd_position(), a.ninst_kv * a.group, a.nqb, inst, rank);
  const int qb = a.nqb - 1 - rank;
  const int64_t b = inst / a.heads, hq = inst % a.heads, hk = hq / a.group;
  const float* kp = a.k + b * a.k_sb + hk * a.k_sh;
  const float* vp = a.v + b * a.v_sb + hk * a.v_sh;
  const int q0 = qb * 16, qrow = q0 + c;
  unsigned char* ring = smem + w * RING;

  int lo = 0, hi = (a.s + 15) / 16;
  if (a.masked && a.prune) {
    const int qlast = q0 + 15 < a.t ? q0 + 15 : a.t - 1;
    const int smin = q0 + a.band_lo, smax = qlast + a.band_hi;
    if (smin > 0) lo = smin / 16;
    hi = smax < 0 ? 0 : (smax / 16 + 1 < hi ? smax / 16 + 1 : hi);
  }
  const int first = lo + ((w - lo) & (W - 1));  // the first tile of [lo, hi) with index w mod W
  auto stage = [&](int buf, int kt) __attribute__((always_inline)) {
    T::stage(kp, a.k_st, kt * 16, a.s, ring + buf * 2 * T::BYTES, lane, 0);
    T::stage(vp, a.v_st, kt * 16, a.s, ring + buf * 2 * T::BYTES + T::BYTES, lane, 0);
  };
  if (first < hi) stage(0, first);
  f32x4 q[NS], o[NS];
  load_cols<D>(q, a.q + b * a.q_sb + hq * a.q_sh, a.q_st, q0, a.t, lane);
#pragma unroll
  for (int f = 0; f < NS; ++f) o[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -kInf, l = 0.f;
  LaneOff<D> off;
  off.init(lane);
  auto step = [&](int kt, auto bufc) __attribute__((always_inline)) {
    constexpr int buf = decltype(bufc)::value;
    const int k0 = kt * 16;
    wait_own_tile();
    if (kt + W < hi) stage(1 - buf, kt + W);
    const unsigned char* kt_ = ring + buf * 2 * T::BYTES;
    const unsigned char* vt_ = kt_ + T::BYTES;
    f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f}, s1 = s;  // two chains: even and odd feature runs
#pragma unroll
    for (int x = 0; x < NS; x += 2) {
      const f32x4 ka = off.row(kt_, 0, x), kb = off.row(kt_, 0, x + 1);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s = mfma4(ka[j], q[x][j], s);
        s1 = mfma4(kb[j], q[x + 1][j], s1);
      }
    }
    s = (s + s1) * a.scale;
    bool cut = k0 + 16 > a.s;
    if (a.masked) cut = cut || k0 - (q0 + 15) < a.band_lo || k0 + 15 - q0 > a.band_hi;
    if (cut) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = k0 + 4 * G + i, d = key - qrow;
        if (a.masked && (d < a.band_lo || d > a.band_hi)) s[i] = a.fill;
        if (key >= a.s) s[i] = -kInf;
      }
    }
    float mx = m;
#pragma unroll
    for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[i]);
    mx = col_max(mx);
    const float ref = mx == -kInf ? 0.f : mx;
    const float alpha = exp_nat(m - ref);
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[i] = exp_nat(s[i] - ref);
      ps += s[i];
    }
    l = l * alpha + ps;
    m = mx;
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int f = 0; f < NS; ++f) o[f] *= alpha;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int f = 0; f < NS; ++f) o[f] = mfma4(off.feature(vt_, 0, f, j), s[j], o[f]);
  };
  for (int kt = first; kt < hi; kt += 2 * W) {
    step(kt, std::integral_constant<int, 0>{});
    if (kt + W < hi) step(kt + W, std::integral_constant<int, 1>{});
  }
  __syncthreads();  // the rings become the states
  f32x4(*so)[NS][64] = reinterpret_cast<f32x4(*)[NS][64]>(smem);
  float(*sml)[2][64] = reinterpret_cast<float(*)[2][64]>(smem + W * NS * 1024);
#pragma unroll
  for (int f = 0; f < NS; ++f) so[w][f][lane] = o[f];
  sml[w][0][lane] = m;
  sml[w][1][lane] = l;
  __syncthreads();
  float M = -kInf, L = 0.f, wt[W];
#pragma unroll
  for (int i = 0; i < W; ++i) M = fmaxf(M, sml[i][0][lane]);
#pragma unroll
  for (int i = 0; i < W; ++i) {
    const float mi = sml[i][0][lane];
    wt[i] = mi == -kInf ? 0.f : exp_nat(mi - M);
    L += sml[i][1][lane] * wt[i];
  }
  L = col_sum(L);
  if (qrow >= a.t) return;
  const float inv = 1.0f / L;
  float* orow = a.o + b * a.o_sb + hq * a.o_sh + static_cast<int64_t>(qrow) * a.o_st + 4 * G;
  for (int f = w; f < NS; f += W) {
    f32x4 x = so[0][f][lane] * wt[0];
#pragma unroll
    for (int i = 1; i < W; ++i) x += so[i][f][lane] * wt[i];
    *reinterpret_cast<f32x4u*>(orow + 16 * f) = x * inv;
  }
  if (w == 0 && G == 0) {
    const int64_t row = static_cast<int64_t>(inst) * a.t + qrow;
    if (a.m_out) a.m_out[row] = M;
    if (a.den_out) a.den_out[row] = L;
    if (a.lse_out) a.lse_out[row] = M + __logf(L);
  }
}

// ---------------------------------------------------------------- backward
//
// attn_f32_bwd_stats: per query row -delta (delta = sum_d dO O), lse log2(e)
// and pm, the probability of a masked score (0 unless every key of the row is
// masked), as the 16-bit path defines them. D / 4 lanes per row.
template <int D>
__global__ __launch_bounds__(256) void attn_f32_bwd_stats(AttnF32Args a) {
  constexpr int LPR = D / 4, RPW = 64 / LPR;
  const int lane = threadIdx.x & 63, sub = lane % LPR;
  const int64_t row = (static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6)) * RPW + lane / LPR;
  float acc = 0.f;
  if (row < a.rows) {
    const int64_t inst = row / a.t, tq = row % a.t;
    const int64_t off = inst / a.heads * a.o_sb + inst % a.heads * a.o_sh + tq * a.o_st + sub * 4;
    const f32x4 x = *reinterpret_cast<const f32x4u*>(a.o + off), y = *reinterpret_cast<const f32x4u*>(a.dout + off);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = __builtin_fmaf(x[j], y[j], acc);
  }
#pragma unroll
  for (int off = LPR / 2; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (row < a.rows && sub == 0) {
    const float fill2 = a.fill * kLog2e;
    float lse2, pm = 0.f;
    if (a.m_in != nullptr) {
      const float m2 = a.m_in[row] * kLog2e, den = a.den_in[row];
      lse2 = m2 + __log2f(den);
      if (a.masked) pm = fast_exp2(fill2 - m2) / den;  // exact 1/den for a fully-masked row
    } else {
      lse2 = a.lse[row] * kLog2e;
      if (a.masked) pm = (lse2 - fill2 < 64.f) ? 1.0f / static_cast<float>(a.s) : fast_exp2(fill2 - lse2);
    }
    a.ws[row] = -acc;
    a.ws[a.rows + row] = lse2;
    a.ws[2 * a.rows + row] = pm;
  }
}

constexpr int kBW = 4, kBO = 16 * kBW;  // backward: waves and owned rows per workgroup

template <int D>
struct BwdLds {
  static constexpr int TB = 32 * D * 4;             // one staged tile
  static constexpr int STAT = 4 * TB;               // after two buffers of two tiles: [2][3][64] floats
  static constexpr int BYTES = STAT + 2 * 3 * 64 * 4;
};

// Tiles [lo, hi) of BT swept rows that hold a live pair for owned rows [o0, o0 + BO).
template <int BO, int BT>
__device__ __forceinline__ void sweep_range(const AttnF32Args& a, int o0, int ext, bool owner_is_query, int& lo,
                                            int& hi) {
  lo = 0;
  hi = (ext + BT - 1) / BT;
  if (!(a.masked && a.prune)) return;
  const int xmin = owner_is_query ? o0 + a.band_lo : o0 - a.band_hi;
  const int xmax = owner_is_query ? o0 + BO - 1 + a.band_hi : o0 + BO - 1 - a.band_lo;
  const int n = hi;
  lo = xmin <= 0 ? 0 : (xmin / BT < n ? xmin / BT : n);
  hi = xmax < 0 ? 0 : (xmax / BT + 1 < n ? xmax / BT + 1 : n);
}

// dK, dV of 64 keys: a wave keeps its 16 keys' K and V as B operands and
// sweeps query tiles (Q, dO and their statistics in LDS):
//   S = Q K^T, dP = dO V^T - delta, P = exp2(S scale log2(e) - lse2), dS = P dP
//   dV^T += dO^T P, dK^T += Q^T dS
// Short chains of sums, as in the forward: the even and the odd chunks of D
// apart, and each tile's products added to the gradient as a whole. With one
// chain over D and one over the swept rows the gradients were 1-6% further from
// 64 bits than the VALU kernels' (24 causal heads x 1000, D = 64: dQ 5.1e-7, dK
// 8.2e-7, dV 8.1e-7 of the norm; the VALU's 5.0, 8.1, 8.0; so 3.7, 3.9, 3.4) and
// the kernel 0-5% faster at D = 64 (that shape 154 us both ways, 24 heads x 2000,
// all keys live, 757 -> 791), 2% faster to 25% slower at D = 128 (64 heads x 700
// in a window 185 -> 189; 32 heads over 8 x 1024 causal 960 -> 740).
template <int D, bool AL>
__device__ __forceinline__ void bwd_dkdv(const AttnF32Args& a, int inst_kv, int kb, unsigned char* smem) {
  constexpr int NS = D / 16, FG = D == 64 ? 4 : 2;  // FG: feature blocks whose tile sums are in flight
  using T = Tile<D, 32, kBW, AL>;
  using L = BwdLds<D>;
  const int lane = threadIdx.x & 63, w = wave_id(), c = lane & 15, G = lane >> 4;
  const int64_t b = inst_kv / a.heads_kv, hk = inst_kv % a.heads_kv;
  const int k0 = kb * kBO, kw = k0 + 16 * w, key = kw + c;
  const float c2 = a.scale * kLog2e;
  f32x4 kf[NS], vf[NS], dk[NS], dv[NS];
  load_cols<D>(kf, a.k + b * a.k_sb + hk * a.k_sh, a.k_st, kw, a.s, lane);
  load_cols<D>(vf, a.v + b * a.v_sb + hk * a.v_sh, a.v_st, kw, a.s, lane);
#pragma unroll
  for (int f = 0; f < NS; ++f) dk[f] = dv[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  LaneOff<D> off;
  off.init(lane);
  int lo, hi;
  sweep_range<kBO, 32>(a, k0, a.t, false, lo, hi);
  const rsrc_t wsr = make_rsrc(a.ws, static_cast<uint32_t>(3 * a.rows * 4));

  auto stage = [&](int buf, int gq, int qt) __attribute__((always_inline)) {
    const int64_t hq = hk * a.group + gq;
    unsigned char* t = smem + buf * 2 * L::TB;
    T::stage(a.q + b * a.q_sb + hq * a.q_sh, a.q_st, qt * 32, a.t, t, lane, w);
    T::stage(a.dout + b * a.o_sb + hq * a.o_sh, a.o_st, qt * 32, a.t, t + L::TB, lane, w);
    if (w < 3) {  // wave x brings statistic x of the tile's rows (lanes 32.. repeat lanes 0..; the last row past t)
      const int r = qt * 32 + (lane & 31);
      const int64_t row = (b * a.heads + hq) * a.t + (r < a.t ? r : a.t - 1);
      dma4(wsr, smem + L::STAT + (buf * 3 + w) * 256, static_cast<uint32_t>((w * a.rows + row) * 4), 0);
    }
  };
  auto compute = [&](int qt, auto bufc) __attribute__((always_inline)) {
    constexpr int buf = decltype(bufc)::value;
    const int q0 = qt * 32;
    bool cut = q0 + 32 > a.t;
    if (a.masked) {
      const int dmin = kw - (q0 + 31), dmax = kw + 15 - q0;  // key - query
      if (a.prune && (dmin > a.band_hi || dmax < a.band_lo)) return;
      cut = cut || dmin < a.band_lo || dmax > a.band_hi;
    }
    const unsigned char* qt_ = smem + buf * 2 * L::TB;
    const unsigned char* ot_ = qt_ + L::TB;
    const float* stat = reinterpret_cast<const float*>(smem + L::STAT + buf * 3 * 256);
    f32x4 s[2], p[2], s1[2], p1[2];  // even and odd chunks of D apart, as in the forward
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s[h] = s1[h] = p1[h] = f32x4{0.f, 0.f, 0.f, 0.f};
      p[h] = *reinterpret_cast<const f32x4*>(stat + 16 * h + 4 * G);  // -delta
    }
#pragma unroll
    for (int x = 0; x < NS; ++x) {
      f32x4 qf[2], of[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        qf[h] = off.row(qt_, h, x);
        of[h] = off.row(ot_, h, x);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          f32x4 &t = x & 1 ? s1[h] : s[h], &u = x & 1 ? p1[h] : p[h];
          t = mfma4(qf[h][j], kf[x][j], t);
          u = mfma4(of[h][j], vf[x][j], u);
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s[h] += s1[h];
      p[h] += p1[h];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4 lse2 = *reinterpret_cast<const f32x4*>(stat + 64 + 16 * h + 4 * G);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = fast_exp2(__builtin_fmaf(s[h][i], c2, -lse2[i]));
        p[h][i] *= e;  // dS
        s[h][i] = e;   // P
      }
      if (cut) {
        const f32x4 pm = *reinterpret_cast<const f32x4*>(stat + 128 + 16 * h + 4 * G);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int qr = q0 + 16 * h + 4 * G + i, d = key - qr;
          const bool out = a.masked && (d < a.band_lo || d > a.band_hi);
          if (out || qr >= a.t) p[h][i] = 0.f;
          if (out) s[h][i] = pm[i];
          if (qr >= a.t) s[h][i] = 0.f;
        }
      }
    }
#pragma unroll
    for (int f0 = 0; f0 < NS; f0 += FG) {
      f32x4 tv[FG], tk[FG];
#pragma unroll
      for (int f = 0; f < FG; ++f) tv[f] = tk[f] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int f = 0; f < FG; ++f) {
            tv[f] = mfma4(off.feature(ot_, h, f0 + f, j), s[h][j], tv[f]);
            tk[f] = mfma4(off.feature(qt_, h, f0 + f, j), p[h][j], tk[f]);
          }
#pragma unroll
      for (int f = 0; f < FG; ++f) {
        dv[f0 + f] += tv[f];
        dk[f0 + f] += tk[f];
      }
      if constexpr (D == 128) __builtin_amdgcn_sched_barrier(0);  // keeps the next group's reads out: else 73 spills
    }
  };

  // items (query head of the group, tile), head-major; the staging cursor runs one item ahead
  const int n = hi > lo ? hi - lo : 0, total = n * a.group;
  int sg = 0, st = lo, ct = lo;
  auto advance = [&]() __attribute__((always_inline)) {
    if (++st == hi) {
      st = lo;
      ++sg;
    }
  };
  auto step = [&](int it, auto bufc) __attribute__((always_inline)) {
    wait_vmcnt0();
    __syncthreads();
    if (it + 1 < total) {
      stage(1 - decltype(bufc)::value, sg, st);
      advance();
    }
    compute(ct, bufc);
    if (++ct == hi) ct = lo;
  };
  if (total > 0) {
    stage(0, sg, st);
    advance();
  }
  for (int it = 0; it < total; it += 2) {
    step(it, std::integral_constant<int, 0>{});
    if (it + 1 < total) step(it + 1, std::integral_constant<int, 1>{});
  }
  if (key >= a.s) return;
  float* ko = a.dk + b * a.k_sb + hk * a.k_sh + static_cast<int64_t>(key) * a.k_st + 4 * G;
  float* vo = a.dv + b * a.v_sb + hk * a.v_sh + static_cast<int64_t>(key) * a.v_st + 4 * G;
#pragma unroll
  for (int f = 0; f < NS; ++f) {
    *reinterpret_cast<f32x4u*>(ko + 16 * f) = dk[f] * a.scale;
    *reinterpret_cast<f32x4u*>(vo + 16 * f) = dv[f];
  }
}

// dQ of 64 query rows: a wave keeps its 16 rows' Q and dO as B operands and
// sweeps key tiles (K, V in LDS):
//   S^T = K Q^T, dP^T = V dO^T - delta, dS^T as above, dQ^T += K^T dS^T
template <int D, bool AL>
__device__ __forceinline__ void bwd_dq(const AttnF32Args& a, int inst, int qb, unsigned char* smem) {
  constexpr int NS = D / 16;
  using T = Tile<D, 32, kBW, AL>;
  using L = BwdLds<D>;
  const int lane = threadIdx.x & 63, w = wave_id(), c = lane & 15, G = lane >> 4;
  const int64_t b = inst / a.heads, hq = inst % a.heads, hk = hq / a.group;
  const float* kp = a.k + b * a.k_sb + hk * a.k_sh;
  const float* vp = a.v + b * a.v_sb + hk * a.v_sh;
  const int q0 = qb * kBO, qw = q0 + 16 * w, qr = qw + c;
  const float c2 = a.scale * kLog2e;
  f32x4 qf[NS], of[NS], dq[NS];
  load_cols<D>(qf, a.q + b * a.q_sb + hq * a.q_sh, a.q_st, qw, a.t, lane);
  load_cols<D>(of, a.dout + b * a.o_sb + hq * a.o_sh, a.o_st, qw, a.t, lane);
#pragma unroll
  for (int f = 0; f < NS; ++f) dq[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int64_t row = static_cast<int64_t>(inst) * a.t + (qr < a.t ? qr : a.t - 1);
  const float ndelta = a.ws[row], lse2 = a.ws[a.rows + row];
  LaneOff<D> off;
  off.init(lane);
  int lo, hi;
  sweep_range<kBO, 32>(a, q0, a.s, true, lo, hi);

  auto stage = [&](int buf, int kt) __attribute__((always_inline)) {
    unsigned char* t = smem + buf * 2 * L::TB;
    T::stage(kp, a.k_st, kt * 32, a.s, t, lane, w);
    T::stage(vp, a.v_st, kt * 32, a.s, t + L::TB, lane, w);
  };
  auto compute = [&](int kt, auto bufc) __attribute__((always_inline)) {
    constexpr int buf = decltype(bufc)::value;
    const int k0 = kt * 32;
    bool cut = k0 + 32 > a.s;
    if (a.masked) {
      const int dmin = k0 - (qw + 15), dmax = k0 + 31 - qw;
      if (a.prune && (dmin > a.band_hi || dmax < a.band_lo)) return;
      cut = cut || dmin < a.band_lo || dmax > a.band_hi;
    }
    const unsigned char* kt_ = smem + buf * 2 * L::TB;
    const unsigned char* vt_ = kt_ + L::TB;
    f32x4 s[2], p[2], s1[2], p1[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s[h] = s1[h] = p1[h] = f32x4{0.f, 0.f, 0.f, 0.f};
      p[h] = f32x4{ndelta, ndelta, ndelta, ndelta};
    }
#pragma unroll
    for (int x = 0; x < NS; ++x) {
      f32x4 kf[2], vf[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        kf[h] = off.row(kt_, h, x);
        vf[h] = off.row(vt_, h, x);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          f32x4 &t = x & 1 ? s1[h] : s[h], &u = x & 1 ? p1[h] : p[h];
          t = mfma4(kf[h][j], qf[x][j], t);
          u = mfma4(vf[h][j], of[x][j], u);
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s[h] += s1[h];
      p[h] += p1[h];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) p[h][i] *= fast_exp2(__builtin_fmaf(s[h][i], c2, -lse2));
    if (cut) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = k0 + 16 * h + 4 * G + i, d = key - qr;
          if (key >= a.s || (a.masked && (d < a.band_lo || d > a.band_hi))) p[h][i] = 0.f;
        }
    }
#pragma unroll
    for (int f0 = 0; f0 < NS; f0 += 4) {
      f32x4 tq[4];
#pragma unroll
      for (int f = 0; f < 4; ++f) tq[f] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int f = 0; f < 4; ++f) tq[f] = mfma4(off.feature(kt_, h, f0 + f, j), p[h][j], tq[f]);
#pragma unroll
      for (int f = 0; f < 4; ++f) dq[f0 + f] += tq[f];
    }
  };
  auto step = [&](int kt, auto bufc) __attribute__((always_inline)) {
    wait_vmcnt0();
    __syncthreads();
    if (kt + 1 < hi) stage(1 - decltype(bufc)::value, kt + 1);
    compute(kt, bufc);
  };
  if (lo < hi) stage(0, lo);
  for (int kt = lo; kt < hi; kt += 2) {
    step(kt, std::integral_constant<int, 0>{});
    if (kt + 1 < hi) step(kt + 1, std::integral_constant<int, 1>{});
  }
  if (qr >= a.t) return;
  float* out = a.dq + b * a.q_sb + hq * a.q_sh + static_cast<int64_t>(qr) * a.q_st + 4 * G;
#pragma unroll
  for (int f = 0; f < NS; ++f) *reinterpret_cast<f32x4u*>(out + 16 * f) = dq[f] * a.scale;
}

// The backward on grids that cannot fill the chip: 16 owned rows a workgroup
// (a quarter of the blocks above), its four waves taking the swept 16-row
// tiles in turn, each through an LDS ring of its own (two buffers, no barrier
// in the sweep), and their partial gradients summed through LDS in wave order.
// Same roles, formulas and block order.
constexpr int kSW = 4;

template <int D>
struct SmallBwdLds {
  static constexpr int TB = 16 * D * 4, WAVE = 4 * TB;  // a wave: two buffers of two tiles
  static constexpr int BYTES = kSW * WAVE;
  static_assert(kSW * 2 * (D / 16) * 1024 <= BYTES, "the partial gradients fit the rings");
};

template <int D, bool AL>
__device__ __forceinline__ void small_dkdv(const AttnF32Args& a, int inst_kv, int kb, unsigned char* smem) {
  constexpr int NS = D / 16;
  using T = Tile<D, 16, 1, AL>;
  using L = SmallBwdLds<D>;
  const int lane = threadIdx.x & 63, w = wave_id(), c = lane & 15, G = lane >> 4;
  const int64_t b = inst_kv / a.heads_kv, hk = inst_kv % a.heads_kv;
  const int k0 = kb * 16, key = k0 + c;
  const float c2 = a.scale * kLog2e;
  unsigned char* ring = smem + w * L::WAVE;
  LaneOff<D> off;
  off.init(lane);
  int lo, hi;
  sweep_range<16, 16>(a, k0, a.t, false, lo, hi);
  const int n = hi > lo ? hi - lo : 0, total = n * a.group;
  f32x4 nd, l2, pm;  // the next tile's statistics (its rows 4 G + i)
  auto stage = [&](int buf, int it) __attribute__((always_inline)) {  // item: (query head of the group, tile), head-major
    const int gq = __builtin_amdgcn_readfirstlane(it / n);
    const int64_t hq = hk * a.group + gq;
    const int q0 = (lo + it - gq * n) * 16;
    T::stage(a.q + b * a.q_sb + hq * a.q_sh, a.q_st, q0, a.t, ring + buf * 2 * L::TB, lane, 0);
    T::stage(a.dout + b * a.o_sb + hq * a.o_sh, a.o_st, q0, a.t, ring + buf * 2 * L::TB + L::TB, lane, 0);
    const float* st = a.ws + (b * a.heads + hq) * a.t;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = q0 + 4 * G + i < a.t ? q0 + 4 * G + i : a.t - 1;
      nd[i] = st[r];
      l2[i] = st[a.rows + r];
      if (a.masked) pm[i] = st[2 * a.rows + r];
    }
  };
  if (w < total) stage(0, w);
  f32x4 kf[NS], vf[NS], dk[NS], dv[NS];
  load_cols<D>(kf, a.k + b * a.k_sb + hk * a.k_sh, a.k_st, k0, a.s, lane);
  load_cols<D>(vf, a.v + b * a.v_sb + hk * a.v_sh, a.v_st, k0, a.s, lane);
#pragma unroll
  for (int f = 0; f < NS; ++f) dk[f] = dv[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int it, auto bufc) __attribute__((always_inline)) {
    constexpr int buf = decltype(bufc)::value;
    const int q0 = (lo + it % n) * 16;
    wait_own_tile();
    f32x4 p = nd, s = f32x4{0.f, 0.f, 0.f, 0.f}, s1 = s, p1 = s;
    const f32x4 lse2 = l2, pmc = pm;
    if (it + kSW < total) stage(1 - buf, it + kSW);
    const unsigned char* qt = ring + buf * 2 * L::TB;
    const unsigned char* ot = qt + L::TB;
#pragma unroll
    for (int x = 0; x < NS; x += 2) {
      const f32x4 qa = off.row(qt, 0, x), qb = off.row(qt, 0, x + 1);
      const f32x4 oa = off.row(ot, 0, x), ob = off.row(ot, 0, x + 1);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s = mfma4(qa[j], kf[x][j], s);
        p = mfma4(oa[j], vf[x][j], p);
        s1 = mfma4(qb[j], kf[x + 1][j], s1);
        p1 = mfma4(ob[j], vf[x + 1][j], p1);
      }
    }
    s += s1;
    p += p1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int qrow = q0 + 4 * G + i, d = key - qrow;
      const bool out = a.masked && (d < a.band_lo || d > a.band_hi);
      const float e = fast_exp2(__builtin_fmaf(s[i], c2, -lse2[i]));
      p[i] = out || qrow >= a.t ? 0.f : p[i] * e;  // dS
      s[i] = qrow >= a.t ? 0.f : (out ? pmc[i] : e);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int f = 0; f < NS; ++f) {
        dv[f] = mfma4(off.feature(ot, 0, f, j), s[j], dv[f]);
        dk[f] = mfma4(off.feature(qt, 0, f, j), p[j], dk[f]);
      }
  };
  for (int it = w; it < total; it += 2 * kSW) {
    step(it, std::integral_constant<int, 0>{});
    if (it + kSW < total) step(it + kSW, std::integral_constant<int, 1>{});
  }
  __syncthreads();  // the rings become the partial sums
  f32x4(*sum)[2 * NS][64] = reinterpret_cast<f32x4(*)[2 * NS][64]>(smem);
#pragma unroll
  for (int f = 0; f < NS; ++f) {
    sum[w][f][lane] = dk[f];
    sum[w][NS + f][lane] = dv[f];
  }
  __syncthreads();
  if (key >= a.s) return;
  float* ko = a.dk + b * a.k_sb + hk * a.k_sh + static_cast<int64_t>(key) * a.k_st + 4 * G;
  float* vo = a.dv + b * a.v_sb + hk * a.v_sh + static_cast<int64_t>(key) * a.v_st + 4 * G;
#pragma unroll
  for (int i = 0; i < 2 * NS / kSW; ++i) {
    const int f = w + i * kSW;
    f32x4 x = sum[0][f][lane];
#pragma unroll
    for (int y = 1; y < kSW; ++y) x += sum[y][f][lane];
    if (f < NS)
      *reinterpret_cast<f32x4u*>(ko + 16 * f) = x * a.scale;
    else
      *reinterpret_cast<f32x4u*>(vo + 16 * (f - NS)) = x;
  }
}

template <int D, bool AL>
__device__ __forceinline__ void small_dq(const AttnF32Args& a, int inst, int qb, unsigned char* smem) {
  constexpr int NS = D / 16;
  using T = Tile<D, 16, 1, AL>;
  using L = SmallBwdLds<D>;
  const int lane = threadIdx.x & 63, w = wave_id(), c = lane & 15, G = lane >> 4;
  const int64_t b = inst / a.heads, hq = inst % a.heads, hk = hq / a.group;
  const float* kp = a.k + b * a.k_sb + hk * a.k_sh;
  const float* vp = a.v + b * a.v_sb + hk * a.v_sh;
  const int q0 = qb * 16, qr = q0 + c;
  const float c2 = a.scale * kLog2e;
  unsigned char* ring = smem + w * L::WAVE;
  LaneOff<D> off;
  off.init(lane);
  int lo, hi;
  sweep_range<16, 16>(a, q0, a.s, true, lo, hi);
  auto stage = [&](int buf, int kt) __attribute__((always_inline)) {
    T::stage(kp, a.k_st, kt * 16, a.s, ring + buf * 2 * L::TB, lane, 0);
    T::stage(vp, a.v_st, kt * 16, a.s, ring + buf * 2 * L::TB + L::TB, lane, 0);
  };
  if (lo + w < hi) stage(0, lo + w);
  f32x4 qf[NS], of[NS], dq[NS];
  load_cols<D>(qf, a.q + b * a.q_sb + hq * a.q_sh, a.q_st, q0, a.t, lane);
  load_cols<D>(of, a.dout + b * a.o_sb + hq * a.o_sh, a.o_st, q0, a.t, lane);
#pragma unroll
  for (int f = 0; f < NS; ++f) dq[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int64_t row = static_cast<int64_t>(inst) * a.t + (qr < a.t ? qr : a.t - 1);
  const float ndelta = a.ws[row], lse2 = a.ws[a.rows + row];
  auto step = [&](int kt, auto bufc) __attribute__((always_inline)) {
    constexpr int buf = decltype(bufc)::value;
    const int k0 = kt * 16;
    wait_own_tile();
    if (kt + kSW < hi) stage(1 - buf, kt + kSW);
    const unsigned char* kt_ = ring + buf * 2 * L::TB;
    const unsigned char* vt_ = kt_ + L::TB;
    f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f}, s1 = s, p1 = s, p = f32x4{ndelta, ndelta, ndelta, ndelta};
#pragma unroll
    for (int x = 0; x < NS; x += 2) {
      const f32x4 ka = off.row(kt_, 0, x), kb = off.row(kt_, 0, x + 1);
      const f32x4 va = off.row(vt_, 0, x), vb = off.row(vt_, 0, x + 1);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s = mfma4(ka[j], qf[x][j], s);
        p = mfma4(va[j], of[x][j], p);
        s1 = mfma4(kb[j], qf[x + 1][j], s1);
        p1 = mfma4(vb[j], of[x + 1][j], p1);
      }
    }
    s += s1;
    p += p1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = k0 + 4 * G + i, d = key - qr;
      const float e = fast_exp2(__builtin_fmaf(s[i], c2, -lse2));
      p[i] = key >= a.s || (a.masked && (d < a.band_lo || d > a.band_hi)) ? 0.f : p[i] * e;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int f = 0; f < NS; ++f) dq[f] = mfma4(off.feature(kt_, 0, f, j), p[j], dq[f]);
  };
  for (int kt = lo + w; kt < hi; kt += 2 * kSW) {
    step(kt, std::integral_constant<int, 0>{});
    if (kt + kSW < hi) step(kt + kSW, std::integral_constant<int, 1>{});
  }
  __syncthreads();
  f32x4(*sum)[NS][64] = reinterpret_cast<f32x4(*)[NS][64]>(smem);
#pragma unroll
  for (int f = 0; f < NS; ++f) sum[w][f][lane] = dq[f];
  __syncthreads();
  if (qr >= a.t) return;
  float* out = a.dq + b * a.q_sb + hq * a.q_sh + static_cast<int64_t>(qr) * a.q_st + 4 * G;
#pragma unroll
  for (int i = 0; i < NS / kSW; ++i) {
    const int f = w + i * kSW;
    f32x4 x = sum[0][f][lane];
#pragma unroll
    for (int y = 1; y < kSW; ++y) x += sum[y][f][lane];
    *reinterpret_cast<f32x4u*>(out + 16 * f) = x * a.scale;
  }
}

// Both roles in one launch (they depend only on the row statistics): a K / V
// instance's blocks alternate in proportion, heaviest first on a causal band
// (early keys, late queries). role(is_key_block, instance, block).
template <typename F>
__device__ __forceinline__ void bwd_role(const AttnF32Args& a, F&& role) {
  const int nq = a.group * a.nqb, nb = a.nkb + nq;
  int inst_kv, pos;
  instance_rank(xcd_position(), a.ninst_kv, nb, inst_kv, pos);
  const int before = __builtin_amdgcn_readfirstlane(
      static_cast<int>(static_cast<int64_t>(pos) * a.nkb / nb));  // key blocks in [0, pos)
  const bool is_k = static_cast<int64_t>(pos + 1) * a.nkb / nb > before;
  if (is_k) {
    role(std::true_type{}, inst_kv, before);
  } else {
    const int i = pos - before, b = inst_kv / a.heads_kv, hk = inst_kv % a.heads_kv;
    role(std::false_type{}, __builtin_amdgcn_readfirstlane(b * a.heads + hk * a.group + i % a.group),
         __builtin_amdgcn_readfirstlane(a.nqb - 1 - i / a.group));
  }
}

template <int D, bool AL>
__global__ __launch_bounds__(64 * kBW, 2) void attn_f32_bwd(AttnF32Args a) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[BwdLds<D>::BYTES];
  bwd_role(a, [&](auto is_k, int inst, int blk) __attribute__((always_inline)) {
    if constexpr (decltype(is_k)::value)
      bwd_dkdv<D, AL>(a, inst, blk, smem);
    else
      bwd_dq<D, AL>(a, inst, blk, smem);
  });
}

template <int D, bool AL>
__global__ __launch_bounds__(64 * kSW, D == 64 ? 2 : 1) void attn_f32_bwd_small(AttnF32Args a) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[SmallBwdLds<D>::BYTES];
  bwd_role(a, [&](auto is_k, int inst, int blk) __attribute__((always_inline)) {
    if constexpr (decltype(is_k)::value)
      small_dkdv<D, AL>(a, inst, blk, smem);
    else
      small_dq<D, AL>(a, inst, blk, smem);
  });
}

bool rows_aligned(const void* p, int64_t sb, int64_t sh, int64_t st) {
  return aligned16(p) && sb % 4 == 0 && sh % 4 == 0 && st % 4 == 0;
}

template <int D, bool AL>
int launch_fwd(AttnF32Args a, int64_t ninst, hipStream_t st) {
  static const int cus = pdh_device_cus() > 0 ? pdh_device_cus() : 256;
  auto blocks = [&](int bm) { return ninst * ((a.t + bm - 1) / bm); };
  auto go = [&](auto kern, int bm, int threads) {
    a.nqb = (a.t + bm - 1) / bm;
    PDH_REQUIRE(ninst * a.nqb <= INT32_MAX, PDH_EINVAL, "pdh_flash_fwd: too many rows");
    kern<<<dim3(static_cast<unsigned>(ninst * a.nqb)), threads, 0, st>>>(a);
    return check_launch("pdh_flash_fwd");
  };
  constexpr int SW = D == 64 ? 8 : 4;  // waves whose rings fill 128 KB of LDS
  constexpr int KS = D == 64 ? 2 : 1;  // 16-key runs per wave and step where two waves split the keys
  // The largest block that still fills the chip: larger ones read K and V less
  // often, smaller ones balance a causal band. 32 heads x 2048, D = 128 causal:
  // 128 rows 296 us, 64 rows 310, 32 rows 326; 24 heads x 1000, D = 64 causal:
  // 82, 70, 57 us (16 rows: 80); 4 heads x 300 rows of 2000 keys, D = 128: 266,
  // 160, 101 us, and 54 with 16 rows and the keys over four waves.
  if (blocks(128) >= 2 * cus) return go(attn_f32_fwd<D, 8, 1, 2, AL>, 128, 512);
  if (blocks(64) >= 2 * cus) return go(attn_f32_fwd<D, 4, 1, 2, AL>, 64, 256);
  if (blocks(32) >= cus) return go(attn_f32_fwd<D, 2, 2, KS, AL>, 32, 256);
  return go(attn_f32_fwd_small<D, SW, AL>, 16, 64 * SW);
}

template <int D, bool AL>
int launch_bwd(AttnF32Args a, int64_t ninst, hipStream_t st) {
  constexpr int RPB = 4 * (64 / (D / 4));
  const int64_t sb = (a.rows + RPB - 1) / RPB;
  static const int cus = pdh_device_cus() > 0 ? pdh_device_cus() : 256;
  auto blocks = [&](int bo) {
    a.nqb = (a.t + bo - 1) / bo;
    a.nkb = (a.s + bo - 1) / bo;
    return static_cast<int64_t>(a.ninst_kv) * a.nkb + ninst * a.nqb;
  };
  // Under two 64-row blocks per compute unit the longest block sets the time:
  // 16-row blocks are four times as many and a quarter as long (forward +
  // backward, causal, D = 64: 4 heads x 1024 rows, 128 blocks, 102 -> 67 us; 12 x
  // 512, 192 blocks, 64 -> 56; 12 x 1024, 384 blocks, 163 -> 154; but 16 x 1024, 512
  // blocks, 165 -> 176 and 24 x 1000, 768 blocks, 206 -> 212). At D = 128 their
  // rings leave one wave per SIMD, so the line is lower (8 heads x 512, 128 blocks,
  // 98 -> 74; 12 x 512, 192 blocks, 110 -> 106; 16 x 512, 256 blocks, 114 -> 125)
  // unless a group's heads make the key blocks long (heads over 4: 16 x 738, 240
  // blocks, 495 -> 327; 32 over 8 x 738, 480 blocks, 546 -> 461; x 1024, 640 blocks,
  // 853 -> 866).
  int64_t nblk = blocks(kBO);
  const bool small = nblk < (D == 64 || a.group > 1 ? 2 * cus : 3 * cus / 4);
  if (small) nblk = blocks(16);
  PDH_REQUIRE(sb <= INT32_MAX && nblk <= INT32_MAX, PDH_EINVAL, "pdh_flash_bwd: too many rows");
  attn_f32_bwd_stats<D><<<dim3(static_cast<unsigned>(sb)), 256, 0, st>>>(a);
  const int rc = check_launch("pdh_flash_bwd (fp32 row stats)");
  if (rc) return rc;
  if (small)
    attn_f32_bwd_small<D, AL><<<dim3(static_cast<unsigned>(nblk)), 64 * kSW, 0, st>>>(a);
  else
    attn_f32_bwd<D, AL><<<dim3(static_cast<unsigned>(nblk)), 64 * kBW, 0, st>>>(a);
  return check_launch("pdh_flash_bwd (fp32 dk, dv, dq)");
}

}  // namespace

bool attn_f32_takes(const pdh_attn_geom& g) {
  auto ok = [&](int64_t st) { return st >= 0 && st < max_stride(g.e); };
  return g.e == g.od && (g.e == 64 || g.e == 128) && g.t <= kMaxRows32 && g.s <= kMaxRows32 && ok(g.q_st) &&
         ok(g.k_st) && ok(g.v_st) && ok(g.o_st) && g.batch * g.heads_q < INT32_MAX / 8;
}

AttnF32Args attn_f32_args(const pdh_attn_geom& g, float scale, float fill, int masked, int64_t band_lo,
                          int64_t band_hi, int prune) {
  constexpr int64_t kBand32 = kMaxRows32 + 64;
  auto clamp32 = [](int64_t x) { return static_cast<int>(x < -kBand32 ? -kBand32 : (x > kBand32 ? kBand32 : x)); };
  AttnF32Args a{};
  a.rows = g.batch * g.heads_q * g.t;
  a.heads = static_cast<int>(g.heads_q);
  a.heads_kv = static_cast<int>(g.heads_kv);
  a.group = a.heads / a.heads_kv;
  a.t = static_cast<int>(g.t);
  a.s = static_cast<int>(g.s);
  a.q_sb = g.q_sb, a.q_sh = g.q_sh, a.q_st = g.q_st;
  a.k_sb = g.k_sb, a.k_sh = g.k_sh, a.k_st = g.k_st;
  a.v_sb = g.v_sb, a.v_sh = g.v_sh, a.v_st = g.v_st;
  a.o_sb = g.o_sb, a.o_sh = g.o_sh, a.o_st = g.o_st;
  a.scale = scale;
  a.fill = fill;
  a.masked = masked;
  a.band_lo = clamp32(band_lo);
  a.band_hi = clamp32(band_hi);
  a.prune = prune;
  a.ninst_kv = static_cast<int>(g.batch * g.heads_kv);
  return a;
}

int attn_f32_forward(AttnF32Args a, const pdh_attn_geom& g, hipStream_t st) {
  const int64_t ninst = g.batch * g.heads_q;
  const bool al = rows_aligned(a.k, g.k_sb, g.k_sh, g.k_st) && rows_aligned(a.v, g.v_sb, g.v_sh, g.v_st);
  if (g.e == 64) return al ? launch_fwd<64, true>(a, ninst, st) : launch_fwd<64, false>(a, ninst, st);
  return al ? launch_fwd<128, true>(a, ninst, st) : launch_fwd<128, false>(a, ninst, st);
}

int attn_f32_backward(AttnF32Args a, const pdh_attn_geom& g, hipStream_t st) {
  const int64_t ninst = g.batch * g.heads_q;
  const bool al = rows_aligned(a.k, g.k_sb, g.k_sh, g.k_st) && rows_aligned(a.v, g.v_sb, g.v_sh, g.v_st) &&
                  rows_aligned(a.q, g.q_sb, g.q_sh, g.q_st) && rows_aligned(a.dout, g.o_sb, g.o_sh, g.o_st);
  if (g.e == 64) return al ? launch_bwd<64, true>(a, ninst, st) : launch_bwd<64, false>(a, ninst, st);
  return al ? launch_bwd<128, true>(a, ninst, st) : launch_bwd<128, false>(a, ninst, st);
}

}  // namespace pdh
