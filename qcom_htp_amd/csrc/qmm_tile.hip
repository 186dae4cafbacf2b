// Quantized matmul on small output tiles with K split over the waves of a workgroup, i8 MFMA
// (v_mfma_i32_32x32x32_i8).  It serves the shapes whose 128 x 512 tiles (qmm_gemm.hip) would leave
// most compute units idle, the schemas whose dot product is not one int8 product times one
// per-channel constant, and the exact integer dot products:
//   * per-channel and LPBQ weights, requantised, with few output tiles (launch_qmm_gemm's rule);
//   * per-group (K64) scales (generate_qnn_matmul_python_cases.py:392-423), requantised;
//   * the integer contracts (gen_quant_chain.py:963-996, HmxU8I4ToU8MatMulOp.cpp:210-233,
//     HmxU16I4ToU16MatMulOp.cpp:514-568) of every prepared weight;
//   * int16 weights as two byte planes (docs/w16a16_is_two_w8a16.md:13-45): q16 = 256 hi +
//     (lo - 128) + 128, planes hi and lo - 128 plus 128 times the activation row sum;
//   * the int64 accumulators of the per-group and int16 formats.
//
// Workgroup: 512 threads = 8 waves = KS groups of 8 / KS waves.  A group takes one KS-th of K, and
// its waves stand side by side over the tile's columns; the groups' sums meet in LDS, where
// integer sums are exact whatever their order.  A tile is 64 rows (32 of 16-bit activations, whose
// high and low bytes are the two 32-row operand blocks) x 8 / KS waves x 32 or 64 channels, so
// that a product of a few hundred rows still gives every compute unit a tile, and the serial part
// of a tile is K / KS deep.  What bounds such products is memory latency, not the matrix cores:
// the split both shortens the loop and keeps 8 waves' loads in flight per compute unit.
//
// Activations go through registers into LDS (shared by the group's waves), shifted to int8 on the
// way (a - 128; a - 32896 = 256 hi + lo' for 16 bits: two byte planes), so the loop's fragment
// reads need no conversion.  Weights come in MFMA fragment order (qmm_internal.h) straight into
// registers.  Both are requested one 128-k step before they are needed.
//
// Per-group requantisation: with s_g = M_g 2^E_g the oracle's float32 weight fl32(q s_g) is
// 2^E_g (q M_g + r) for a small integer residue r, so the dot product is
// sum_g 2^E_g (M_g S_g + R_g), S_g = sum_{k in g} (a - zp) q and R_g the same sum over r.  Prepare
// writes M_g 2^E_g as int32 multiples of one unit per channel (mult; rounded to it where the
// channel's scales span too far), and every 64 k the exact int32 S_g goes into an int64 sum by one
// 32 x 32 + 64-bit multiply-add per output: the loop is bound by those (at two waves per SIMD an
// instruction issues every 2.4 to 2.7 ns; a float64 sum took two, an int64 multiplier about ten).
// 8-bit activations leave R_g out and bound it while few outputs are uncertain for it, and else form it
// as a second product (prepare_exact's rule); 16-bit ones form the high byte's part as a third product
// and bound the low byte's.  An output closer to a rounding boundary than that bound and
// the roundings is listed and recomputed as the oracle forms its dot product (float64 products of
// fl64((a - zp) sA) and fl32(q s_g)).
// Per-channel requantisation is the same with one group: 8-bit activations keep the code products
// alone, 16-bit ones add the high byte's residue products (sum M S + 256 R in int64), and a listed
// output first gets its missing residue sum exactly (a dot product over the residue plane or
// column), then the float64 recomputation if it still lies within the oracle's own noise.

#include <algorithm>
#include <type_traits>

#include "qmm_contract.h"

namespace qh {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

constexpr int kTlThreads = 512;
constexpr int kTlWaves = kTlThreads / 64;
constexpr int kTlStage = 64 * kBK;  // bytes of one group's activation tile: 64 operand rows x 128 k

enum TileMode : int { kGroup = 0, kContract = 1, kAccumulate = 2, kRequant = 3 };

__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) {
  return __builtin_amdgcn_perm(hi, lo, sel);
}

// 16 bytes per lane through a buffer resource: the lane's offset is one register for the whole loop
// and the step's a scalar, so a load costs no address arithmetic; past the end it returns zeros.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, static_cast<int>(bytes), 0x00020000);
}
__device__ __forceinline__ uint4 buf_load16(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t step_off) {
  const v4u v = __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(lane_off), static_cast<int>(step_off), 0);
  return make_uint4(v[0], v[1], v[2], v[3]);
}

// Workgroup barrier that waits for this wave's LDS operations but not for its loads in flight.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// 16 consecutive weights of operand column c (plane p of channel n: plane_col), depth k.
__device__ __forceinline__ int plane_col(int p, int n, int lp) { return (n >> 5) * (32 * lp) + p * 32 + (n & 31); }
__device__ __forceinline__ uint4 load_w16(const TileArgs &g, int c, int k) {
  const size_t tile = static_cast<size_t>(c / kBN) * g.KT + k / kBK;
  return *reinterpret_cast<const uint4 *>(g.tiles + tile * (kBN * kBK) + tile_off_i8(c % kBN, k));
}

__device__ __forceinline__ void store_out(const TileArgs &g, size_t idx, int v) {
  if (g.out16)
    static_cast<uint16_t *>(g.out)[idx] = static_cast<uint16_t>(v);
  else
    static_cast<uint8_t *>(g.out)[idx] = static_cast<uint8_t>(v);
}

// The oracle's float64 dot product for output (m, n), by one wave (per-channel weights: one group):
// sum_k fl64((a_k - zp) sA) * fl32(q_k s_g), then + bias, / sO, + zp, rint, clip.
template <bool A16>
__device__ void emulate_one(const TileArgs &g, int m, int n, int lane) {
  double s = 0.0;
  const int c0 = plane_col(0, n, g.lp);
  for (int kc = lane; kc < g.K / 16; kc += 64) {
    const int k = kc * 16;
    const uint4 wv = load_w16(g, c0, k);
    const float sc = g.s32g[static_cast<size_t>(n) * g.G + (k >> g.gshift)];
    uint4 av[2];
    if (A16) {
      const uint4 *ap = reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(g.act) + static_cast<size_t>(m) * g.K + k);
      av[0] = ap[0];
      av[1] = ap[1];
    } else {
      av[0] = *reinterpret_cast<const uint4 *>(g.act + static_cast<size_t>(m) * g.K + k);
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int a = A16 ? static_cast<int>(reinterpret_cast<const uint16_t *>(av)[j])
                        : static_cast<int>(reinterpret_cast<const uint8_t *>(av)[j]);
      const int w = reinterpret_cast<const int8_t *>(&wv)[j];
      const float wd = static_cast<float>(w) * sc;
      s = fma(static_cast<double>(a - g.act_zp) * g.sA, static_cast<double>(wd), s);
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
  if (lane == 0) {
    const double t = (s + g.bias_deq[n]) / g.sO + static_cast<double>(g.out_zp);
    const double o = fmin(fmax(rint(t), 0.0), static_cast<double>(g.out_qmax));
    store_out(g, static_cast<size_t>(m) * g.N + n, static_cast<int>(o));
  }
}

// A listed output of a per-channel weight, by one wave: S is its sum from the tile (8-bit acts
// sum (a - 128) w; 16-bit acts M sum (a - 32896) w + 256 sum hi' r).  The missing residue products
// (8-bit: sum (a - 128) r over the residue plane; 16-bit: sum lo' r over the residue column) make
// the dot product D exact in units of 2^E, and t = D alpha_e + beta rounds like the oracle unless it
// lies within the oracle's own float64 noise of a boundary.
template <bool A16>
__device__ void complete_one(const TileArgs &g, long long S, int m, int n, int lane) {
  const long long mant = g.mant[n], csum = g.colsum[n], csum_r = g.colsum_r[n];
  const double alpha_e = g.alpha_e[n], beta = g.beta[n], margin = g.margin_exact[n], absb = g.absb[n];
  int part = 0;  // |part| <= 128 * 64 * K / 64 per lane, 2^29 over the wave at K = 65536
  for (int kc = lane; kc < g.K / 16; kc += 64) {
    if (!A16) {
      const uint4 a = reinterpret_cast<const uint4 *>(g.act + static_cast<size_t>(m) * g.K)[kc];
      const uint4 r = reinterpret_cast<const uint4 *>(g.resid + static_cast<size_t>(n) * g.K)[kc];
      part = __builtin_amdgcn_sdot4(static_cast<int>(a.x ^ 0x80808080u), static_cast<int>(r.x), part, false);
      part = __builtin_amdgcn_sdot4(static_cast<int>(a.y ^ 0x80808080u), static_cast<int>(r.y), part, false);
      part = __builtin_amdgcn_sdot4(static_cast<int>(a.z ^ 0x80808080u), static_cast<int>(r.z), part, false);
      part = __builtin_amdgcn_sdot4(static_cast<int>(a.w ^ 0x80808080u), static_cast<int>(r.w), part, false);
    } else {
      const uint4 *ap = reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(g.act) + static_cast<size_t>(m) * g.K + kc * 16);
      const uint4 a0 = ap[0], a1 = ap[1], r = load_w16(g, plane_col(1, n, g.lp), kc * 16);
      part = __builtin_amdgcn_sdot4(static_cast<int>(perm(a0.y, a0.x, 0x06040200u) ^ 0x80808080u), static_cast<int>(r.x), part, false);
      part = __builtin_amdgcn_sdot4(static_cast<int>(perm(a0.w, a0.z, 0x06040200u) ^ 0x80808080u), static_cast<int>(r.y), part, false);
      part = __builtin_amdgcn_sdot4(static_cast<int>(perm(a1.y, a1.x, 0x06040200u) ^ 0x80808080u), static_cast<int>(r.z), part, false);
      part = __builtin_amdgcn_sdot4(static_cast<int>(perm(a1.w, a1.z, 0x06040200u) ^ 0x80808080u), static_cast<int>(r.w), part, false);
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) part += __shfl_xor(part, off, 64);
  // |D| < 2^63; partial terms may wrap, so the sum is formed modulo 2^64
  const unsigned long long M64 = static_cast<unsigned long long>(mant);
  const unsigned long long sw = M64 * static_cast<unsigned long long>(csum) + static_cast<unsigned long long>(csum_r);
  const unsigned long long Du = (A16 ? 1ull : M64) * static_cast<unsigned long long>(S) +
                                static_cast<unsigned long long>(static_cast<long long>(part)) +
                                static_cast<unsigned long long>(static_cast<long long>((A16 ? 32896 : 128) - g.act_zp)) * sw;
  const double u = static_cast<double>(static_cast<long long>(Du)) * alpha_e;
  const double tv = u + beta, rd = rint(tv);
  const double slack = margin + 0x1p-48 * (fabs(u) + fabs(tv) + absb);
  if (!(fabs(tv - rd) <= 0.5 - slack)) {  // uniform: every lane holds the same sums
    emulate_one<A16>(g, m, n, lane);
  } else if (lane == 0) {
    store_out(g, static_cast<size_t>(m) * g.N + n, static_cast<int>(fmin(fmax(rd, 0.0), static_cast<double>(g.out_qmax))));
  }
}

// Compile-time shape of one instantiation.  A16: 16-bit activations.  NT: weight fragments per wave
// and 32-k step.  PL2: those are the two planes of the same 32 channels (int16 bytes, or per-group
// codes and residues); otherwise NT blocks of 32 channels.  KS: K groups of the workgroup.
template <bool A16, int NT, bool PL2, int MODE, int KS>
struct TileCfg {
  static constexpr int kCols = PL2 ? 32 : 32 * NT;        // channels per wave
  static constexpr int kWavesN = kTlWaves / KS;           // waves of a group
  static constexpr int TC = kCols * kWavesN;              // channels of the tile
  static constexpr int RB = A16 ? 32 : 64;                // rows of the tile
  static constexpr bool kRound = MODE == kGroup || MODE == kRequant;  // requantised, with a list
  static constexpr bool kW16 = PL2 && !kRound;            // int16 weights
  // 16-bit activations: the low byte's residue products are left out (bounded instead)
  static constexpr bool kSkipLoRes = A16 && PL2 && kRound;
  // the sums in LDS: int64 where two digits or planes or the groups combine, else int32
  using Val = std::conditional_t<MODE == kGroup || A16 || kW16, long long, int>;
  static constexpr int kPlanes = MODE == kGroup ? (PL2 ? 2 : 1) : 0;  // group multipliers per channel
  static constexpr int kStages = 2 * KS * kTlStage;
  static constexpr int kSums = RB * TC * static_cast<int>(sizeof(Val));
  static constexpr int kList = kRound ? RB * TC * 2 : 0;  // every output fits: no overflow
  static constexpr int kSmem = kStages > kSums + kList ? kStages : kSums + kList;
  static constexpr int kUnits = 512 / (64 * kWavesN);     // 16-byte activation chunks per thread per 128-k step
};

// MODE kGroup: requantised per-group output; kRequant: requantised per-channel output; kContract:
// integer contract; kAccumulate: int64.
template <bool A16, int NT, bool PL2, int MODE, int KS>
__global__ __launch_bounds__(kTlThreads, 1) void qmm_tile_kernel(const TileArgs g) {
  using C = TileCfg<A16, NT, PL2, MODE, KS>;
  using Val = typename C::Val;
  constexpr int TC = C::TC, RB = C::RB, NW = C::kWavesN;
  __shared__ __attribute__((aligned(16))) uint8_t smem[C::kSmem];
  // per column: scale, offset and certified threshold (per-group), else the shift term and the bias
  __shared__ double ctab[C::kRound ? 3 * TC : 1];
  __shared__ long long itab[C::kRound ? 1 : 2 * TC];
  __shared__ int rsum[C::kW16 ? 64 : 1];                // row sums of the shifted operand rows
  __shared__ int fix_cnt;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int kg = wave / NW, wc = wave % NW;

  // Tile of this workgroup.  Workgroups go round-robin over the 8 XCDs; each XCD takes a run of
  // tiles, walked in groups of up to 8 row tiles, so that its concurrent tiles share weight columns.
  const int T = g.TM * g.TN, per_x = (T + 7) / 8;
  const int lin = (blockIdx.x & 7) * per_x + (blockIdx.x >> 3);
  if (static_cast<int>(blockIdx.x >> 3) >= per_x || lin >= T) return;  // uniform
  const int gid = lin / (8 * g.TN), first = gid * 8;
  const int gm = min(8, g.TM - first), in = lin - gid * 8 * g.TN;
  const int m0 = (first + in % gm) * RB, n0 = (in / gm) * TC;

  if (t == 0) fix_cnt = 0;
  if (C::kW16 && t < 64) rsum[t] = 0;
  // the epilogue's per-column constants are requested first, so that their latency is the loop's
  double calpha = 0.0, cbeta = 0.0, cthr = 0.0, cmargin = 0.0, cabsb = 0.0;
  long long ccorr = 0, cbias = 0, cmant = 0;
  if (t < TC) {
    if constexpr (MODE == kGroup) {
      calpha = g.alpha[n0 + t];
      cbeta = g.beta[n0 + t];
      cthr = g.thr[n0 + t];
    } else if constexpr (MODE == kRequant) {
      calpha = g.alpha[n0 + t];
      cbeta = g.beta[n0 + t];
      cmargin = g.margin[n0 + t] + (A16 ? g.margin_lo[n0 + t] : 0.0);
      cabsb = g.absb[n0 + t];
      ccorr = g.corr[n0 + t];
      if (A16) cmant = g.mant[n0 + t];
    } else {
      ccorr = g.corr[n0 + t];
      if (MODE == kContract && g.bias_q) cbias = g.bias_q[n0 + t];
    }
  }

  // This group's 128-k tiles kt0 .. kend - 1; every group runs `per` steps (the barriers are the
  // workgroup's), its weights past kend reading as zeros.
  const int per = (g.KT + KS - 1) / KS;
  const int kt0 = kg * per, kend = max(kt0, min(kt0 + per, g.KT));

  // Activation chunks: 8-bit rows 16 values = 16 bytes, 16-bit rows 16 values = 32 bytes (one unit
  // covers both halves of its two byte planes).  Rows past M read as zeros; k past K is other
  // rows' data, which meets zero weights.
  constexpr int kU = A16 ? C::kUnits / 2 : C::kUnits;
  constexpr uint32_t E = A16 ? 2 : 1;
  const int tg = t - kg * 64 * NW;
  struct ARegs {
    uint4 v[kU][A16 ? 2 : 1];
  };
  const uint32_t pitch = static_cast<uint32_t>(g.K) * E;  // bytes of an activation row
  const auto arsrc = buf_rsrc(g.act + static_cast<size_t>(m0) * pitch, static_cast<uint32_t>(min(g.M - m0, RB)) * pitch);
  uint32_t aoff[kU];
#pragma unroll
  for (int i = 0; i < kU; ++i) aoff[i] = static_cast<uint32_t>((i * 64 * NW + tg) >> 3) * pitch + (tg & 7) * 16 * E;
  auto load_a = [&](int kt, ARegs &r) __attribute__((always_inline)) {
    const uint32_t k = static_cast<uint32_t>(kt) * kBK * E;
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      r.v[i][0] = buf_load16(arsrc, aoff[i], k);
      if (A16) r.v[i][A16 ? 1 : 0] = buf_load16(arsrc, aoff[i], k + 16);
    }
  };
  // ... into LDS: operand row r, chunk c (16 bytes) at r * 128 + 16 (c ^ swz8(r)); 16-bit
  // activations: rows 0..31 the high bytes, 32..63 the low bytes.
  auto store_a = [&](uint8_t *st, const ARegs &a) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      const int r = (i * 64 * NW + tg) >> 3;
      uint8_t *const d = st + r * 128 + ((tg & 7) ^ swz8(r)) * 16;
      uint4 v = a.v[i][0];
      v.x ^= 0x80808080u; v.y ^= 0x80808080u; v.z ^= 0x80808080u; v.w ^= 0x80808080u;
      if (!A16) {
        *reinterpret_cast<uint4 *>(d) = v;
      } else {
        uint4 u = a.v[i][A16 ? 1 : 0];
        u.x ^= 0x80808080u; u.y ^= 0x80808080u; u.z ^= 0x80808080u; u.w ^= 0x80808080u;
        *reinterpret_cast<uint4 *>(d) = make_uint4(perm(v.y, v.x, 0x07050301u), perm(v.w, v.z, 0x07050301u),
                                                   perm(u.y, u.x, 0x07050301u), perm(u.w, u.z, 0x07050301u));
        *reinterpret_cast<uint4 *>(d + 32 * 128) = make_uint4(perm(v.y, v.x, 0x06040200u), perm(v.w, v.z, 0x06040200u),
                                                              perm(u.y, u.x, 0x06040200u), perm(u.w, u.z, 0x06040200u));
      }
    }
  };
  // Weight fragments of one 128-k tile: operand column block ob[nt], 32-k step s at
  // 1 KiB * (16 s + ob % 16) of the tile; per-group: the multipliers of its two 64-k halves.
  struct BRegs {
    v4i b[4][NT];
    int c[2][C::kPlanes > 0 ? C::kPlanes : 1];
  };
  // (a tile's operand columns lie in one 512-column panel)
  const int cb = (n0 + wc * C::kCols) / 32;
  const int ob = PL2 ? 2 * cb : g.lp * cb, onext = PL2 ? 1 : g.lp;
  const uint32_t panel = static_cast<uint32_t>(g.KT) * (kBN * kBK);
  const auto brsrc = buf_rsrc(g.tiles + static_cast<size_t>(ob / (kBN / 32)) * panel, static_cast<uint32_t>(kend) * (kBN * kBK));
  const uint32_t boff = static_cast<uint32_t>(ob % (kBN / 32)) * 1024;
  const uint32_t ncol = n0 + wc * C::kCols + (lane & 31);  // < Np: padding columns hold zero weights
  auto load_b = [&](int kt, BRegs &r) __attribute__((always_inline)) {
    const uint32_t k = boff + static_cast<uint32_t>(kt) * (kBN * kBK);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        r.b[s][nt] = __builtin_bit_cast(v4i, buf_load16(brsrc, lane * 16, k + s * (kBN / 32) * 1024 + nt * onext * 1024));
    if constexpr (MODE == kGroup) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int grp = min((kt * kBK + 64 * h) >> g.gshift, g.G - 1);
#pragma unroll
        for (int p = 0; p < C::kPlanes; ++p) {
          const int32_t *const row = g.mult + (static_cast<size_t>(p) * g.G + grp) * g.Np;  // uniform
          r.c[h][p] = row[ncol];
        }
      }
    }
  };

  v16i acc[2][NT];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = v16i{};
  // per-group sums: 8-bit activations two row blocks, 16-bit one (both digits and planes combine)
  constexpr int kGB = MODE == kGroup ? (A16 ? 1 : 2) : 1;
  long long dacc[kGB][MODE == kGroup ? 16 : 1];
#pragma unroll
  for (int i = 0; i < kGB; ++i)
#pragma unroll
    for (int j = 0; j < (MODE == kGroup ? 16 : 1); ++j) dacc[i][j] = 0;
  int rs[2] = {0, 0};
  const int wmant = A16 && MODE == kRequant ? static_cast<int>(g.mant[ncol]) : 0;  // 24 bits

  uint8_t *const stage0 = smem + kg * 2 * kTlStage;
  const int frow = lane & 31, fswz = swz8(frow);
  auto compute = [&](int kt, const uint8_t *st, const BRegs &r) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      v4i a[2];
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
        a[mt] = *reinterpret_cast<const v4i *>(st + (mt * 32 + frow) * 128 + 16 * ((2 * s + (lane >> 5)) ^ fswz));
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          if (C::kSkipLoRes && mt == 1 && nt == 1) continue;
          const v16i zero = {};
          acc[mt][nt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[mt], r.b[s][nt],
                                                              MODE == kGroup && (s & 1) == 0 ? zero : acc[mt][nt], 0, 0, 0);
        }
        if (C::kW16) {
          const int one = kt < kend && kt * kBK + 32 * s < g.K ? 0x01010101 : 0;  // past them only the weights are zero
#pragma unroll
          for (int x = 0; x < 4; ++x) rs[mt] = __builtin_amdgcn_sdot4(a[mt][x], one, rs[mt], false);
        }
      }
      if constexpr (MODE == kGroup) {
        if (s & 1) {  // 64 k done: |S| < 2^28
          const long long c0 = r.c[s >> 1][0];
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            if constexpr (!A16) {
              dacc[0][j] += acc[0][0][j] * c0;
              dacc[kGB - 1][j] += acc[1][0][j] * c0;
              if constexpr (PL2) {
                const long long c1 = r.c[s >> 1][C::kPlanes - 1];
                dacc[0][j] += acc[0][NT - 1][j] * c1;
                dacc[kGB - 1][j] += acc[1][NT - 1][j] * c1;
              }
            } else {
              // c1 carries the residue plane's multiplier times 256 (the high byte's weight)
              const long long c1 = r.c[s >> 1][C::kPlanes - 1];
              dacc[0][j] += (256 * acc[0][0][j] + acc[1][0][j]) * c0;
              dacc[0][j] += acc[0][NT - 1][j] * c1;
            }
          }
        }
      }
    }
  };

  // Step it: tile it + 1's weights are requested, tile it's products run (its weights were requested
  // a step ago), tile it + 1's activations (requested a step ago) go to the other stage, whose reads
  // ended at the last barrier, and tile it + 2's are requested.  Requests are answered in order and
  // the steps are straight-line code, so each wait leaves the younger requests in flight (behind a
  // branch the compiler waits for all of them); past a group's tiles the weights read as zeros.
  BRegs b0, b1;
  ARegs ar;
  load_a(kt0, ar);
  load_b(kt0, b0);
  store_a(stage0, ar);
  load_a(kt0 + 1, ar);
  if (t < TC) {
    if constexpr (MODE == kGroup) {
      ctab[t] = calpha;
      ctab[TC + t] = cbeta;
      ctab[2 * TC + t] = cthr;
    } else if constexpr (MODE == kRequant) {
      // the shift term folded into the offset; the threshold keeps the residue bound and the float
      // slack for |t| <= qmax + 2 (16-bit acts: |sum (a - 32896) w| <= K 33024 127)
      const double shift = static_cast<double>(ccorr) * calpha;
      const double umax = A16 ? fabs(calpha * static_cast<double>(cmant)) * static_cast<double>(g.K) * (33024.0 * 127.0) : 0.0;
      ctab[t] = calpha;
      ctab[TC + t] = cbeta + shift;
      ctab[2 * TC + t] = 0.5 - cmargin - 0x1p-48 * (cabsb + 2.0 * fabs(shift) + umax + static_cast<double>(g.out_qmax) + 2.0);
    } else {
      itab[t] = ccorr;
      itab[TC + t] = cbias;
    }
  }
  lds_barrier();
  auto step = [&](int it, const BRegs &cur, BRegs &nxt) __attribute__((always_inline)) {
    load_b(kt0 + it + 1, nxt);
    compute(kt0 + it, stage0 + (it & 1) * kTlStage, cur);
    store_a(stage0 + ((it + 1) & 1) * kTlStage, ar);
    load_a(kt0 + it + 2, ar);
    lds_barrier();
  };
  int it = 0;
  for (; it + 2 <= per; it += 2) {
    step(it, b0, b1);
    step(it + 1, b1, b0);
  }
  if (it < per) step(it, b0, b1);

  // ---- the groups' sums meet in LDS (over the activation stages, which are all read) ------------
  Val *const sums = reinterpret_cast<Val *>(smem);  // [RB][TC]
  auto each = [&](auto &&f) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int r = 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3), c = wc * C::kCols + (lane & 31);
      if constexpr (MODE == kGroup) {
#pragma unroll
        for (int i = 0; i < kGB; ++i) f(32 * i + r, c, dacc[i][j]);
      } else if constexpr (A16 && MODE == kRequant) {
        f(r, c, (256LL * acc[0][0][j] + acc[1][0][j]) * wmant + 256LL * acc[0][NT - 1][j]);
      } else if constexpr (A16 && C::kW16) {
        f(r, c, 65536LL * acc[0][0][j] + 256LL * (static_cast<long long>(acc[0][NT - 1][j]) + acc[1][0][j]) + acc[1][NT - 1][j]);
      } else if constexpr (A16) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) f(r, c + 32 * nt, 256LL * acc[0][nt][j] + acc[1][nt][j]);
      } else if constexpr (C::kW16) {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) f(32 * mt + r, c, 256LL * acc[mt][0][j] + acc[mt][NT - 1][j]);
      } else {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) f(32 * mt + r, c + 32 * nt, acc[mt][nt][j]);
      }
    }
  };
  if (kg == 0) each([&](int r, int c, Val v) { sums[r * TC + c] = v; });
  if (C::kW16 && wc == 0) {
    atomicAdd(&rsum[frow], rs[0]);
    atomicAdd(&rsum[32 + frow], rs[1]);
  }
  lds_barrier();
  if (KS > 1 && kg > 0 && kend > kt0) {
    each([&](int r, int c, Val v) {
      if constexpr (sizeof(Val) == 8)
        atomicAdd(reinterpret_cast<unsigned long long *>(&sums[r * TC + c]), static_cast<unsigned long long>(v));
      else
        atomicAdd(&sums[r * TC + c], v);
    });
  }
  if (KS > 1) lds_barrier();

  // ---- epilogue: 4 adjacent outputs of one row per thread and pass -------------------------------
  uint16_t *const list = reinterpret_cast<uint16_t *>(smem + C::kSums);
  constexpr int kQuads = TC / 4;
  static_assert(kTlThreads % kQuads == 0, "a thread keeps its columns");
  const int c4 = 4 * (t % kQuads), n = n0 + c4;
  const bool col_ok = n < g.N;  // N is a multiple of 32
  // op(row, o): the thread's four outputs of a row (kAccumulate: the int64 sums)
  auto outputs = [&](auto &&op) __attribute__((always_inline)) {
#pragma unroll
    for (int rr = 0; rr < (RB * kQuads + kTlThreads - 1) / kTlThreads; ++rr) {
      const int r = t / kQuads + rr * (kTlThreads / kQuads);
      const int m = m0 + r;
      if (r >= RB || m >= g.M || !col_ok) continue;  // (a tile of 32 rows x 32 columns has fewer quads than threads)
      const size_t idx = static_cast<size_t>(m) * g.N + n;
      if constexpr (MODE == kAccumulate) {
        long long o[4];
        op(r, o);
#pragma unroll
        for (int e = 0; e < 4; ++e) static_cast<long long *>(g.out)[idx + e] = o[e];
      } else {
        int o[4];
        op(r, o);
        if (!g.vec_out) {
#pragma unroll
          for (int e = 0; e < 4; ++e) store_out(g, idx + e, o[e]);
        } else if (g.out16) {
          *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(g.out) + idx) =
              make_uint2(static_cast<uint32_t>(o[0]) | (static_cast<uint32_t>(o[1]) << 16),
                         static_cast<uint32_t>(o[2]) | (static_cast<uint32_t>(o[3]) << 16));
        } else {
          *reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(g.out) + idx) =
              static_cast<uint32_t>(o[0]) | (static_cast<uint32_t>(o[1]) << 8) | (static_cast<uint32_t>(o[2]) << 16) |
              (static_cast<uint32_t>(o[3]) << 24);
        }
      }
    }
  };
  // the exact dot product sum_k (a - zp) w_int
  auto dot = [&](int r, int e) __attribute__((always_inline)) {
    long long D = static_cast<long long>(sums[r * TC + c4 + e]) + itab[c4 + e];
    if constexpr (C::kW16)
      D += 128LL * (A16 ? 256LL * rsum[r] + rsum[32 + (r & 31)] : static_cast<long long>(rsum[r]));
    return D;
  };
  if constexpr (C::kRound) {
    // rint by adding 1.5 * 2^52 after a clamp to [-1, qmax + 1].  An output that is not certain is
    // listed unless it clips to the same end over the whole error bound 0.5 - th, which can be any
    // number of steps: below t = th (above qmax - th) it does, and from 2 th - 1 on also with the
    // rounding of t itself.
    constexpr double kMagic = 6755399441055744.0;
    const double qmaxd = static_cast<double>(g.out_qmax);
    double al[4], be[4], th[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      al[e] = ctab[c4 + e];
      be[e] = ctab[TC + c4 + e];
      th[e] = ctab[2 * TC + c4 + e];
    }
    outputs([&](int r, int (&o)[4]) __attribute__((always_inline)) {
      double u[4];
      bool sure[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        u[e] = fma(static_cast<double>(sums[r * TC + c4 + e]), al[e], be[e]);
        const double tv = fmin(fmax(u[e], -1.0), qmaxd + 1.0);
        const double y = tv + kMagic;
        sure[e] = fabs(tv - (y - kMagic)) <= th[e];  // (a threshold that is not a number lists the output)
        o[e] = min(max(__double2loint(y), 0), g.out_qmax);
      }
      if (!(sure[0] & sure[1] & sure[2] & sure[3])) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const double end = 2.0 * th[e] - 1.0;
          if (!sure[e] && !(u[e] < end) && !(u[e] > qmaxd - end)) list[atomicAdd(&fix_cnt, 1)] = static_cast<uint16_t>(r * TC + c4 + e);
        }
      }
    });
  } else if constexpr (MODE == kAccumulate) {
    outputs([&](int r, long long (&o)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = dot(r, e);
    });
  } else {
    // one switch per thread, not one per output
    const double rcp = 1.0 / static_cast<double>(g.divisor > 0 ? g.divisor : 1);
    auto run = [&](auto ct) __attribute__((always_inline)) {
      constexpr int CT = decltype(ct)::value;
      outputs([&](int r, int (&o)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (contract_divides(CT))
            o[e] = contract_f64<CT>(g, static_cast<double>(dot(r, e)), rcp);
          else
            o[e] = contract_int<CT>(g, dot(r, e), itab[TC + c4 + e]);
        }
      });
    };
    switch (g.contract) {
      case QH_CONTRACT_CLIP_I32: run(std::integral_constant<int, QH_CONTRACT_CLIP_I32>{}); break;
      case QH_CONTRACT_CLIP_I64: run(std::integral_constant<int, QH_CONTRACT_CLIP_I64>{}); break;
      case QH_CONTRACT_DIV_RINT: run(std::integral_constant<int, QH_CONTRACT_DIV_RINT>{}); break;
      case QH_CONTRACT_FLOOR256_DIV_RINT: run(std::integral_constant<int, QH_CONTRACT_FLOOR256_DIV_RINT>{}); break;
      case QH_CONTRACT_ROUND_DIV: run(std::integral_constant<int, QH_CONTRACT_ROUND_DIV>{}); break;
      default: run(std::integral_constant<int, QH_CONTRACT_U8_DRAIN>{}); break;
    }
  }
  if constexpr (C::kRound) {
    lds_barrier();
    const int cnt = fix_cnt;
    if (cnt == 0) return;
    __syncthreads();  // every provisional output is stored before any is rewritten
    for (int e = wave; e < cnt; e += kTlWaves) {
      const int v = __builtin_amdgcn_readfirstlane(static_cast<int>(list[e]));
      if constexpr (MODE == kGroup)
        emulate_one<A16>(g, m0 + v / TC, n0 + v % TC, lane);
      else
        complete_one<A16>(g, sums[v], m0 + v / TC, n0 + v % TC, lane);
    }
  }
}

// Most workgroups of one launch: its threads are counted in 32 bits (a larger grid is cut short without
// an error), in whole rounds over the XCDs.
constexpr long long kMaxBlocks = 0xFFFFFFFFLL / kTlThreads / 8 * 8;

template <bool A16, int NT, bool PL2, int MODE, int KS>
qh_status launch(const TileArgs &whole, hipStream_t stream) {
  using C = TileCfg<A16, NT, PL2, MODE, KS>;
  const long long tn = (whole.N + C::TC - 1) / C::TC, rows = kMaxBlocks / tn * C::RB;  // rows of one launch
  const size_t out_row = static_cast<size_t>(whole.N) * (MODE == kAccumulate ? 8 : whole.out16 ? 2 : 1);
  for (long long m0 = 0; m0 < whole.M; m0 += rows) {
    TileArgs g = whole;
    g.M = static_cast<int>(std::min(rows, whole.M - m0));
    g.act += static_cast<size_t>(m0) * whole.K * (A16 ? 2 : 1);
    g.out = static_cast<uint8_t *>(whole.out) + static_cast<size_t>(m0) * out_row;
    g.TM = (g.M + C::RB - 1) / C::RB;
    g.TN = static_cast<int>(tn);
    const long long blocks = (static_cast<long long>(g.TM) * tn + 7) / 8 * 8;  // whole rounds over the XCDs
    hipLaunchKernelGGL((qmm_tile_kernel<A16, NT, PL2, MODE, KS>), dim3(static_cast<unsigned>(blocks)), dim3(kTlThreads), 0, stream, g);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return hip_fail(err, "qmm_tile_kernel launch");
  }
  return QH_STATUS_OK;
}

// Tiles of a launch with ks K groups per workgroup (cols: channels per wave).
long long tile_count(int m, int n, bool a16, int cols, int ks) {
  const long long tm = (m + (a16 ? 31LL : 63LL)) / (a16 ? 32 : 64), tc = cols * (kTlWaves / ks);
  return tm * ((n + tc - 1) / tc);
}

// K groups of a workgroup: as many as leave every tile a compute unit of its own.  More groups make
// a shorter loop and less to requantise per tile, but one tile more than compute units is a second
// round.  u8 x int4 500 x 4096 x 4096 (128 / 256 / 512 tiles for 2 / 4 / 8 groups): 24.2 / 18.8 / 27.9
// us; 200 x 4096 x 4096 (64 / 128 / 256): 23.0 / 16.9 / 15.0; 1000 x 2048 x 4096 (256 / 512 / 1024):
// 18.0 / 22.7 / 35.3; u16 x int4 500 x 4096 x 1024 (128 / 256 / 512): 22.8 / 20.2 / 28.1.  Eight
// groups also need eight 128-k steps to be worth their sums: int16 weights 200 x 512 x 1024 take 6.1
// us with 4 groups and 6.7 us with 8.
template <bool A16, int NT, bool PL2, int MODE>
qh_status pick_split(const TileArgs &g, hipStream_t stream) {
  const int cus = device_cu_count(), cols = PL2 ? 32 : 32 * NT;
  // (8-bit activations with both planes' group sums: eight groups spill 60 registers)
  if constexpr (!(!A16 && PL2 && MODE == kGroup)) {
    if (g.KT >= 8 && tile_count(g.M, g.N, A16, cols, 8) <= cus) return launch<A16, NT, PL2, MODE, 8>(g, stream);
  }
  if (tile_count(g.M, g.N, A16, cols, 4) <= cus) return launch<A16, NT, PL2, MODE, 4>(g, stream);
  return launch<A16, NT, PL2, MODE, 2>(g, stream);
}

}  // namespace

// One round of the widest tiles covers the product: then its time is one tile's, below the GEMM's,
// whose 128 x 512 tiles (64 x 256 outputs for 16-bit activations) are a quarter as many and deeper.
// Past that the GEMM wins: u8 x int4 1000 x 2048 x 4096 (256 tiles) 18.0 against 28.3 us, 500 x 2048 x
// 12000 (376) 31.1 against 29.7 us; u16 x int4 256 x 1024 x 4096 (256) 10.3 against 14.9 us, 500 x 1024
// x 4096 (512) 19.3 against 16.7 us.
bool tile_pays(const qh_qmm_prepared *p, int m) {
  const bool a16 = p->shape.act_bits == 16;
  return tile_count(m, p->shape.N, a16, a16 ? 32 : 64, 2) <= device_cu_count();
}

qh_status launch_qmm_tile(const qh_qmm_prepared *p, int m, const void *act, void *out, int mode, int contract,
                          int divisor, hipStream_t stream) {
  if (m > 65535 * 64) return fail(QH_STATUS_SHAPE_UNSUPPORTED, "M=%d too large for one launch", m);
  const QmmShape &sh = p->shape;
  const QmmDevice &D = p->dev;
  TileArgs g{};
  g.act = static_cast<const uint8_t *>(act);
  g.out = out;
  g.tiles = D.tiles;
  g.M = m;
  g.N = sh.N;
  g.K = sh.K;
  g.KT = sh.Kp / kBK;
  g.Np = sh.Np;
  g.lp = sh.layout_planes;
  g.act_zp = sh.act_zp;
  g.out_zp = sh.out_zp;
  g.out_qmax = (1 << sh.out_bits) - 1;
  g.out16 = sh.out_bits == 16;
  // 4 outputs per store; a buffer that is not aligned to that takes one output per store
  g.vec_out = reinterpret_cast<uintptr_t>(out) % (g.out16 ? 8 : 4) == 0;
  g.sA = sh.act_scale;
  g.sO = sh.out_scale;
  g.contract = contract;
  g.divisor = divisor;
  g.bias_q = D.bias_q;
  g.corr = D.corr_int;
  g.mult = D.mult;
  g.alpha = D.alpha_e;
  g.beta = D.beta;
  g.thr = D.thr;
  g.s32g = D.s32g;
  g.bias_deq = D.bias_deq;
  g.G = sh.groups;
  g.gshift = sh.group_shift;
  if (mode == kTileRequant) {
    g.alpha = D.alpha;
    g.corr = D.corr;
    g.margin = D.margin;
    g.margin_lo = D.margin_lo;
    g.absb = D.absb;
    g.mant = D.mant;
    g.colsum = D.colsum;
    g.colsum_r = D.colsum_r;
    g.alpha_e = D.alpha_e;
    g.margin_exact = D.margin_exact;
    g.resid = D.resid;
    g.s32g = D.s32;  // one group
    g.G = 1;
    g.gshift = 30;
  }
  const bool a16 = sh.act_bits == 16, w16 = sh.int_planes == 2;
  if (mode == kTileRequant) return a16 ? pick_split<true, 2, true, kRequant>(g, stream) : pick_split<false, 2, false, kRequant>(g, stream);
  if (mode == kTileGroup) {
    if (a16) return pick_split<true, 2, true, kGroup>(g, stream);
    return sh.group_resid ? pick_split<false, 2, true, kGroup>(g, stream) : pick_split<false, 1, false, kGroup>(g, stream);
  }
  if (mode == kTileAccumulate) {
    if (w16) return a16 ? pick_split<true, 2, true, kAccumulate>(g, stream) : pick_split<false, 2, true, kAccumulate>(g, stream);
    return a16 ? pick_split<true, 2, false, kAccumulate>(g, stream) : pick_split<false, 2, false, kAccumulate>(g, stream);
  }
  if (w16) return a16 ? pick_split<true, 2, true, kContract>(g, stream) : pick_split<false, 2, true, kContract>(g, stream);
  return a16 ? pick_split<true, 2, false, kContract>(g, stream) : pick_split<false, 2, false, kContract>(g, stream);
}

}  // namespace qh
