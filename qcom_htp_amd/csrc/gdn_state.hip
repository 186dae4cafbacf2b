// GDN chunk recurrence (stage B of the chunked gated delta rule), C = 64, D = 128:
// for every chunk of a (batch, head) sequence, in order, with the state S (D x D) carried,
//     q^ = l2norm(q) / sqrt(D),  k^ = l2norm(k),  g = cumsum(gc) inside the chunk,
//     P     = (q^ k^T) * e^{g_i - g_j}   (j <= i, else 0)
//     v_new = U - W S
//     o     = (q^ * e^g) S + P v_new
//     S     = S e^{g_last} + (k^ * e^{g_last - g})^T v_new
// from the stage-A outputs U = T (beta v) and W = T (beta k^ e^g)
// (scripts/gdn_ref_kernel.py:66-69,91-101; the chunk loop :104-131).
//
// One workgroup (8 waves) per sequence walks its chunks.  S lives in registers for the whole
// sequence: wave w owns S's value columns 16w .. 16w+15 as eight 16 x 16 MFMA result tiles,
// which is also the layout the MFMA reads as a B operand over pairs of key blocks (pair layout,
// bf16_split.h), so W S and q S take S straight from the accumulators.  q and k stay the bf16
// values they arrive as (exact MFMA operands); their l2norm factors scale the products' rows and
// columns instead.  Per chunk, between two barriers each:
//   M. each wave: W S and q S for its 16 value columns (4 token tiles), v_new = U - W S with U
//      from registers, o's first term e^g q^ S; the 10 lower 16 x 16 tiles of q k^T over the
//      waves, scaled by the norms and decays, into LDS as P;
//   N. S = e^{g_last} S + k^T ((e^{g_last - g} / |k|) v_new), k^T read from the k rows by LDS
//      transpose reads; o = e^g q^ S + P v_new for the wave's columns (causal tiles only), stored;
//      then the next chunk's rows into LDS: W and q, which are free after M, and k into the other
//      of two buffers, with the row norms (8-lane DPP sums), g's prefix sum (64-lane DPP scan),
//      e^g and e^{g_last - g} (one wave).  Their global loads were issued a whole chunk before.
// W, q and P lie in LDS in operand order (kpos): each half of a 32-deep product step's A operand is
// one 16-byte read, with nothing to repack.  The kernel is bound by what its two waves per SIMD
// issue and wait for; with W and P as hi | lo words (two reads and eight byte permutes an operand)
// and a staging phase of its own between two more barriers the median launch took 529 / 367 us (fp32 /
// bf16), now 524 / 363 (B = 8, T = 4096, H = 32; the bytes it moves take 365 / 257 us at the 5.2 TB/s of
// a large copy).
//
// Prefill of many sequences (FROM_T) needs no W and U: they are T (beta e^g k^) and T (beta v), so
//     v_new = T (beta v - beta e^g k^ S),
// where k^ S takes k from the rows that are in LDS anyway (exact, one operand half instead of W's two)
// and T times the result is one more lower triangular product of a wave's own columns.  gdn_t_kernel
// forms T (16 KB a chunk as hi / lo parts) from k, g and beta alone.  Stage A is bound by the 64 KB of W
// and U that it writes per chunk in float32 (1.6 GB, 312 us), which stage B then reads again: B = 8,
// T = 4096, H = 32 takes 136 + 560 us with T against 314 + 524 us (bf16: 111 + 399 against 228 + 363),
// median launches of 30 in a row.
//
// Precision: QH_GDN_FP32 carries W, S, P and v_new as bf16 hi/lo splits (hi*hi + hi*lo + lo*hi,
// fp32 accumulation; products with the exact q, k take two terms); QH_GDN_BF16 uses the hi
// parts only; T's own products and its right-hand side's parts are split in both.  Norms, decays and
// the prefix sum are fp32.  (With the right-hand side rounded to bf16 as well, BF16's o from T was further
// from 64 bits than from W and U, which round v_new once: 2.92e-3 against 2.54e-3 .. 2.90e-3; now 2.41e-3,
// for 7 us of the 399 above.  FP32 is at 5.1e-6 from T, 3.4e-4 from stage A's bf16 products.)
//
// Few sequences (gdn_state_cols_kernel): the chunks of a sequence follow one another, so the launch
// lasts as long as one sequence however few there are, and what counts is a chunk's latency.  The work
// of a chunk is spread over 16 waves and, since v_new, o and S act on value columns independently, over
// 128 / (16 CT) workgroups of CT column tiles each.  A column tile's waves share its S by key blocks; S,
// v_new and the state update's operand go through LDS as the records that the next products read as
// they are.  The next chunk's rows go into LDS behind the state update (q and W are free after the
// products, k has two buffers), and their global loads are issued a whole chunk ahead.  With a
// workspace, what a chunk needs besides the state (gdn_state_pre_kernel) is formed for all chunks first,
// and the recurrence only copies it.  A chunk of 16 sequences then takes 1.6 / 2.2 us (bf16 / fp32)
// against 3.1 / 3.8 us, and some 6 us before the first; its bounds are the LDS reads of a workgroup
// (16 CT columns of S by 8 waves each) and the chain of products behind two barriers.
// Stages A and B of T = 4096 x 16 sequences: bf16 212 -> 120 us, fp32 252 -> 158 us.

#include <type_traits>

#include "bf16_split.h"
#include "lane_ops.h"
#include "qmm_internal.h"

namespace qh {
namespace {

using namespace bf16s;

constexpr int kC = 64;          // chunk (tokens)
constexpr int kD = 128;         // head dimension
constexpr int kThreads = 512;   // 8 waves
constexpr int kQs = kD + 8;     // LDS row stride of the q / k stores, bf16 (16-byte aligned rows)
constexpr int kWs = kD + 16;    // LDS row stride of operand-ordered W and q, bf16 (72 words: 16-byte reads conflict-free)
constexpr int kPs = kC + 16;    // LDS row stride of operand-ordered P, bf16 (40 words)

struct StateArgs {
  const uint16_t *q, *k;  // bf16 [B][T][H][D]
  const float *g;         // [B][T][H] per-token log decays
  const void *w, *u;      // [B][T][H][D] bf16 or fp32 (stage-A outputs, W in the e^g form)
  const float *s_in;      // [B][H][D][D] or nullptr (zero state)
  float *s_out;           // [B][H][D][D]
  void *o;                // [B][T][H][D] bf16 or fp32
  int B, T, H, nchunks;
  // what gdn_state_pre_kernel formed of every (sequence, chunk), in order: P as [64][64] bf16 hi parts
  // (then lo parts with SPLIT), and kPreF floats (the factors of q^ S's and v_new's rows, e^{g_last})
  uint16_t *pre_p;
  float *pre_f;
  // FROM_T: T = (I - A)^-1 of every (sequence, chunk), [64][64] bf16 hi parts in operand order (then lo
  // parts with SPLIT), and beta; u holds v
  uint16_t *t;
  const float *beta;
};
constexpr int kPreF = 2 * kC + 4;

__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ float bf16f(uint32_t h) { return __uint_as_float(h << 16); }

// RAGGED: T need not be a multiple of the chunk.  Rows past T repeat row T - 1 with gc = 0 and a zero
// decay factor in the state update; P is lower triangular, so they touch no row before them, and
// they are not stored.
// Rows by which the row `row` of chunk n is moved back to exist (0 unless RAGGED).
template <bool RAGGED>
__device__ __forceinline__ uint32_t past_end(const StateArgs &a, int n, int row) {
  return RAGGED ? static_cast<uint32_t>(max(n * kC + row - (a.T - 1), 0)) : 0u;
}

// Position of column c of a row in operand order: within 32 columns, the 4 that a lane quarter takes of
// the first 16 and the 4 it takes of the last 16 lie side by side (8 k of one lane, 16 bytes).
__device__ __forceinline__ constexpr int kpos(int c) { return (c & ~31) + 8 * ((c >> 2) & 3) + 4 * ((c >> 4) & 1) + (c & 3); }

// 8 bf16 values of a uint4 as floats.
__device__ __forceinline__ void unbf16x8(const uint4 v, float *f) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    f[2 * x] = bf16f(w[x] & 0xFFFFu);
    f[2 * x + 1] = bf16f(w[x] >> 16);
  }
}

// Sum of the squares of a row's 128 values, 16 in each of 8 adjacent lanes.
__device__ __forceinline__ float row_square(const uint4 (&v)[2]) {
  float f[16];
  unbf16x8(v[0], f);
  unbf16x8(v[1], f + 8);
  float ss = 0.0f;
#pragma unroll
  for (int x = 0; x < 16; ++x) ss = fmaf(f[x], f[x], ss);
  return sum8(ss);
}
// 1 / |q| / sqrt(D) and 1 / |k| of a sum of squares (eps 1e-6 inside the root).
__device__ __forceinline__ float inv_k(float ss) { return 1.0f / sqrtf(ss + 1e-6f); }
__device__ __forceinline__ float inv_q(float ss) { return inv_k(ss) * (1.0f / 11.313708498984761f); }

// The 10 lower 16 x 16 tiles of P (token tile i >= j).
__device__ __forceinline__ void p_tile(int idx, int &i, int &j) {
  i = idx < 1 ? 0 : idx < 3 ? 1 : idx < 6 ? 2 : 3;
  j = idx - i * (i + 1) / 2;
}

// Four consecutive bf16 of an LDS row (8-byte aligned) as an exact operand half.
__device__ __forceinline__ Half4 bf16x4(const uint16_t *p) {
  const uint2 v = *reinterpret_cast<const uint2 *>(p);
  return exact4(v.x, v.y);
}

// 4 bf16 of one column of a row-major LDS tile, by a transposing LDS read (ds_read_b64_tr_b16):
// in each group of 16 lanes, lane j receives element j % 4 of the 8 bytes addressed by lane
// 4 e + j / 4 as its element e.  So if lane 4 e + a of the group addresses row r0 + e, columns
// c0 + 4 a .. + 3, lane j receives rows r0 .. r0 + 3 of column c0 + j.
__device__ __forceinline__ Half4 bf16x4_tr(const uint16_t *p) {
  typedef short v4s __attribute__((ext_vector_type(4)));
  const v4s r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s *)(p));
  const uint2 v = __builtin_bit_cast(uint2, r);
  return exact4(v.x, v.y);
}
__device__ __forceinline__ v4f mfma(const v8bf a, const v8bf b, const v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// A operand half of one 32-deep step in operand order.
__device__ __forceinline__ v8bf op8(const uint16_t *p) { return __builtin_bit_cast(v8bf, *reinterpret_cast<const uint4 *>(p)); }

// Of four bf16 rows x 4 adjacent columns in a quad of lanes (P0 = rows 0, 1 and P1 = rows 2, 3 of the
// lane's column): row q's 4 columns in lane q of the quad, by DPP quad broadcasts.
__device__ __forceinline__ uint2 quad_rows(uint32_t P0, uint32_t P1, int qq) {
  const uint32_t a0 = __builtin_amdgcn_mov_dpp(P0, 0x00, 0xF, 0xF, false);
  const uint32_t a1 = __builtin_amdgcn_mov_dpp(P0, 0x55, 0xF, 0xF, false);
  const uint32_t a2 = __builtin_amdgcn_mov_dpp(P0, 0xAA, 0xF, 0xF, false);
  const uint32_t a3 = __builtin_amdgcn_mov_dpp(P0, 0xFF, 0xF, 0xF, false);
  const uint32_t b0 = __builtin_amdgcn_mov_dpp(P1, 0x00, 0xF, 0xF, false);
  const uint32_t b1 = __builtin_amdgcn_mov_dpp(P1, 0x55, 0xF, 0xF, false);
  const uint32_t b2 = __builtin_amdgcn_mov_dpp(P1, 0xAA, 0xF, 0xF, false);
  const uint32_t b3 = __builtin_amdgcn_mov_dpp(P1, 0xFF, 0xF, 0xF, false);
  const uint32_t sel = (qq & 1) ? 0x07060302u : 0x05040100u;
  return qq < 2 ? make_uint2(__builtin_amdgcn_perm(a1, a0, sel), __builtin_amdgcn_perm(a3, a2, sel))
                : make_uint2(__builtin_amdgcn_perm(b1, b0, sel), __builtin_amdgcn_perm(b3, b2, sel));
}

// One 16 x 16 result tile of o: `at` is the element offset of the lane's column in row 4 qd of the
// tile, tok the elements per token, qq the lane's place in its quad; rows: how many of the lane's 4
// rows exist (RAGGED).
template <bool OUT_F32, bool RAGGED>
__device__ __forceinline__ void store_o(void *o, uint32_t at, uint32_t tok, int qq, const v4f &acc, int rows) {
  if constexpr (OUT_F32) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (!RAGGED || e < rows) static_cast<float *>(o)[at + static_cast<uint32_t>(e) * tok] = acc[e];
  } else {
    // lane q of the quad stores row 4 qd + q, the quad's 4 columns, in one 8-byte store
    const uint2 w = quad_rows(pack_bf16(acc[0], acc[1]), pack_bf16(acc[2], acc[3]), qq);
    if (!RAGGED || qq < rows)
      *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(o) + (at - static_cast<uint32_t>(qq) + static_cast<uint32_t>(qq) * tok)) = w;
  }
}

// acc[i] (or zero, with `fresh`) += sum over the token tiles j <= i of L_ij X_j, L lower triangular in
// LDS in operand order (lo parts with SPLIT); XLO: with X's lo parts.
template <bool SPLIT, bool XLO, int NL>
__device__ __forceinline__ void lower_product(const uint16_t (&hi)[kC][kPs], const uint16_t (&lo)[NL][kPs], int r16, int qd,
                                              const Half4 (&x)[4], v4f (&acc)[4], bool fresh) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v4f s = fresh ? v4f{0.f, 0.f, 0.f, 0.f} : acc[i];
#pragma unroll
    for (int p = 0; p <= i / 2; ++p) {
      // (no later tile beside a diagonal one: an infinity there would reach these rows)
      const Half4 x1 = 2 * p + 1 <= i ? x[2 * p + 1] : kZero4;
      const v8bf l = op8(&hi[16 * i + r16][32 * p + 8 * qd]), xh = op_hi(x[2 * p], x1);
      s = mfma(l, xh, s);
      if constexpr (XLO) s = mfma(l, op_lo(x[2 * p], x1), s);
      if constexpr (SPLIT) s = mfma(op8(&lo[16 * i + r16][32 * p + 8 * qd]), xh, s);
    }
    acc[i] = s;
  }
}

// FROM_T: v_new = T (beta v - beta e^g K^ S) from gdn_t_kernel's T instead of U - W S.
// ONE: the sequence is one whole chunk, and nothing is loaded or staged for a next one (a uniform branch
// around that in the same kernel spills 20 to 100 registers).  Sequences past the compute units run in
// rounds of one workgroup per unit: 1280 of them 56 us against 66 (fp32) and 44 against 51 (bf16).
template <bool SPLIT, bool WU_F32, bool OUT_F32, bool RAGGED, bool FROM_T, bool ONE = false>
__global__ __launch_bounds__(kThreads) void gdn_state_kernel(StateArgs a) {
  static_assert(!(FROM_T && WU_F32), "v is bf16");
  constexpr bool kWlo = SPLIT && WU_F32;  // a bf16 W has no lo part
  // q, k rows as given (bf16, exact MFMA operands) with their l2norm factors; W and the lower
  // tiles of P as bf16 hi parts (and lo parts with SPLIT); g, e^g, e^{g_last - g}
  __shared__ __attribute__((aligned(16))) uint16_t Ql[kC][kWs];
  __shared__ __attribute__((aligned(16))) uint16_t Kl[2][kC][kQs];
  __shared__ __attribute__((aligned(16))) uint16_t Wh[FROM_T ? 1 : kC][kWs], Wo[kWlo ? kC : 1][kWs];
  __shared__ __attribute__((aligned(16))) uint16_t Th[FROM_T ? kC : 1][kPs], Tl[FROM_T && SPLIT ? kC : 1][kPs];
  __shared__ __attribute__((aligned(16))) uint16_t Ph[kC][kPs], Po[SPLIT ? kC : 1][kPs];
  // 1 / |q| / sqrt(D), 1 / |k| (eps 1e-6 inside the root); g, e^g, e^{g_last - g}
  __shared__ __attribute__((aligned(16))) float invq[2][kC], invk[2][kC], gl[2][kC], egl[2][kC], decl[2][kC], bet[2][kC];
  __shared__ float eglast[2];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r16 = lane & 15, qd = lane >> 4;
  const int b = __builtin_amdgcn_readfirstlane(blockIdx.x / a.H), h = blockIdx.x - b * a.H;

  // S: tile kb holds rows (keys) 16 kb + 4 qd + e, column (value) 16 wave + r16
  v4f S[8];
  const size_t sbase = (static_cast<size_t>(b) * a.H + h) * kD * kD;
#pragma unroll
  for (int kb = 0; kb < 8; ++kb) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      S[kb][e] = a.s_in ? a.s_in[sbase + static_cast<size_t>(16 * kb + 4 * qd + e) * kD + 16 * wave + r16] : 0.0f;
  }

  // A thread stages 16 columns of one row: of q and k columns 16 seg .., of W the 8 columns
  // 32 (seg / 2) + 8 (seg % 2) .. and the 8 that are 16 further on, which are adjacent in operand order.
  // Addresses are a chunk's uniform base and a lane's 32-bit offset in the chunk, so that the bases are
  // scalar and few registers hold offsets (RAGGED: the row is at most the last one that exists).  The
  // offsets are opaque in every chunk: left alone, the compiler keeps a 64-bit address for each of the
  // 30 accesses across the loop, and spills.
  const uint32_t tok = static_cast<uint32_t>(a.H) * kD;
  const uint32_t head = (static_cast<uint32_t>(b) * a.T * a.H + h) * kD;
  const int row = t >> 3, seg = t & 7, wcol = 32 * (seg >> 1) + 8 * (seg & 1);
  auto chunk_at = [&](int n) __attribute__((always_inline)) { return static_cast<size_t>(head + static_cast<uint32_t>(n) * kC * tok); };
  auto row_at = [&](int n, int r) __attribute__((always_inline)) {
    return static_cast<uint32_t>(RAGGED ? min(r, a.T - 1 - n * kC) : r) * tok;
  };
  const uint32_t col = 16 * wave + r16;
  const uint32_t of_g = static_cast<uint32_t>(b) * a.T * a.H + lane * a.H + h;

  uint4 iq[2], ik[2], iw[2][WU_F32 ? 2 : 1];
  float iu[4][4], igc, ibeta = 0.0f;
  typedef unsigned v4u __attribute__((ext_vector_type(4)));
  v4u it[2] = {};
  auto load = [&](int n) __attribute__((always_inline)) {
    const size_t c0 = chunk_at(n);
    uint32_t ro = row_at(n, row);
    asm volatile("" : "+v"(ro));
    const uint4 *qp = reinterpret_cast<const uint4 *>(a.q + c0 + (ro + 16 * seg));
    const uint4 *kp = reinterpret_cast<const uint4 *>(a.k + c0 + (ro + 16 * seg));
    iq[0] = qp[0];
    iq[1] = qp[1];
    ik[0] = kp[0];
    ik[1] = kp[1];
    if constexpr (FROM_T) {
      const v4u *tp = reinterpret_cast<const v4u *>(a.t + (static_cast<size_t>(blockIdx.x) * a.nchunks + n) * (SPLIT ? 2 : 1) * (kC * kC)) + t;
      it[0] = tp[0];
      if constexpr (SPLIT) it[1] = tp[kC * kC / 8];
    } else {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const uint32_t wi = ro + wcol + 16 * x;
        const uint4 *wp = WU_F32 ? reinterpret_cast<const uint4 *>(static_cast<const float *>(a.w) + c0 + wi)
                                 : reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(a.w) + c0 + wi);
        iw[x][0] = wp[0];
        if constexpr (WU_F32) iw[x][1] = wp[1];
      }
    }
    const uint32_t gb = past_end<RAGGED>(a, n, lane);
    const uint32_t gi = of_g + (static_cast<uint32_t>(n) * kC - gb) * static_cast<uint32_t>(a.H);
    igc = a.g[gi];
    if constexpr (FROM_T) ibeta = a.beta[gi];
    if (RAGGED && gb) igc = ibeta = 0.0f;
  };
  auto load_u = [&](int n) __attribute__((always_inline)) {
    const size_t c0 = chunk_at(n);
    uint32_t lo = 4 * qd * tok + col;
    asm volatile("" : "+v"(lo));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // the lane's row is 4 qd + (16 i + e): the second part in the base unless rows are clamped
        const size_t base = RAGGED ? c0 : c0 + static_cast<size_t>(static_cast<uint32_t>(16 * i + e) * tok);
        const uint32_t ui = RAGGED ? row_at(n, 16 * i + 4 * qd + e) + col : lo;
        iu[i][e] = WU_F32 ? (static_cast<const float *>(a.u) + base)[ui] : bf16f((static_cast<const uint16_t *>(a.u) + base)[ui]);
      }
    }
  };
  // chunk n's rows into LDS (buffer n & 1 of the double-buffered arrays), with the norms and decays
  auto stage = [&](int n) __attribute__((always_inline)) {
    const int bf = n & 1;
    uint16_t *const qd4 = &Ql[row][32 * (seg >> 1) + 4 * (seg & 1)];  // kpos(16 seg); 4 columns on: + 8
    *reinterpret_cast<uint2 *>(qd4) = make_uint2(iq[0].x, iq[0].y);
    *reinterpret_cast<uint2 *>(qd4 + 8) = make_uint2(iq[0].z, iq[0].w);
    *reinterpret_cast<uint2 *>(qd4 + 16) = make_uint2(iq[1].x, iq[1].y);
    *reinterpret_cast<uint2 *>(qd4 + 24) = make_uint2(iq[1].z, iq[1].w);
    *reinterpret_cast<uint4 *>(&Kl[bf][row][16 * seg]) = ik[0];
    *reinterpret_cast<uint4 *>(&Kl[bf][row][16 * seg + 8]) = ik[1];
    const float sq = row_square(iq), sk = row_square(ik);
    if (seg == 0) {
      invq[bf][row] = inv_q(sq);
      invk[bf][row] = inv_k(sk);
    }
    // W: two lane quarters' 8 values, 4 of each 16-column block
    uint16_t *const wd = &Wh[FROM_T ? 0 : row][kpos(wcol)];
    if constexpr (FROM_T) {
      *reinterpret_cast<v4u *>(&Th[FROM_T ? row : 0][8 * seg]) = it[0];
      if constexpr (SPLIT) *reinterpret_cast<v4u *>(&Tl[FROM_T && SPLIT ? row : 0][8 * seg]) = it[1];
    } else if constexpr (WU_F32) {
      Half4 x[2][2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
          x[i][j] = split4<SPLIT>(__uint_as_float(iw[i][j].x), __uint_as_float(iw[i][j].y), __uint_as_float(iw[i][j].z),
                                  __uint_as_float(iw[i][j].w));
      }
      *reinterpret_cast<uint4 *>(wd) = make_uint4(x[0][0].h01, x[0][0].h23, x[1][0].h01, x[1][0].h23);
      *reinterpret_cast<uint4 *>(wd + 8) = make_uint4(x[0][1].h01, x[0][1].h23, x[1][1].h01, x[1][1].h23);
      if constexpr (kWlo) {
        uint16_t *const wl = &Wo[row][kpos(wcol)];
        *reinterpret_cast<uint4 *>(wl) = make_uint4(x[0][0].l01, x[0][0].l23, x[1][0].l01, x[1][0].l23);
        *reinterpret_cast<uint4 *>(wl + 8) = make_uint4(x[0][1].l01, x[0][1].l23, x[1][1].l01, x[1][1].l23);
      }
    } else {
      *reinterpret_cast<uint4 *>(wd) = make_uint4(iw[0][0].x, iw[0][0].y, iw[1][0].x, iw[1][0].y);
      *reinterpret_cast<uint4 *>(wd + 8) = make_uint4(iw[0][0].z, iw[0][0].w, iw[1][0].z, iw[1][0].w);
    }
    if (wave == 0) {
      const float g = scan64(igc);
      const float glast = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g), 63));
      gl[bf][lane] = g;
      egl[bf][lane] = expf(g);
      decl[bf][lane] = RAGGED && n * kC + lane >= a.T ? 0.0f : expf(glast - g);
      if (lane == 0) eglast[bf] = expf(glast);
      if constexpr (FROM_T) bet[bf][lane] = ibeta;
    }
  };

  load(0);
  load_u(0);
  // the upper tiles of P that a 32-deep step reads beside a diagonal one stay zero
  for (int x = t; x < kC * kPs / 2; x += kThreads) {
    reinterpret_cast<uint32_t *>(Ph)[x] = 0u;
    if constexpr (SPLIT) reinterpret_cast<uint32_t *>(Po)[x] = 0u;
  }
  stage(0);
  if constexpr (!ONE) load(min(1, a.nchunks - 1));
  lds_barrier();

  auto chunk = [&](const int n) __attribute__((always_inline)) {
    const int bf = n & 1;
    // ---- M: W S, q^ S, v_new; P tiles ----------------------------------------------------------
    v4f ws[4], qs[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ws[i] = qs[i] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < 4; ++p) {  // key blocks 2p, 2p + 1: 8 independent accumulations
      const int c = 32 * p + 8 * qd;
      const Half4 s0 = split4<SPLIT>(S[2 * p]), s1 = split4<SPLIT>(S[2 * p + 1]);
      const v8bf sh = op_hi(s0, s1), sl = op_lo(s0, s1);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint16_t *const krow = &Kl[bf][16 * i + r16][32 * p + 4 * qd];
        const v8bf w = FROM_T ? op_hi(bf16x4(krow), bf16x4(krow + 16)) : op8(&Wh[FROM_T ? 0 : 16 * i + r16][c]);
        const v8bf q = op8(&Ql[16 * i + r16][c]);
        ws[i] = mfma(w, sh, ws[i]);
        qs[i] = mfma(q, sh, qs[i]);
        if constexpr (SPLIT) {
          ws[i] = mfma(w, sl, ws[i]);
          qs[i] = mfma(q, sl, qs[i]);
        }
        if constexpr (kWlo) ws[i] = mfma(op8(&Wo[16 * i + r16][c]), sh, ws[i]);
      }
      if constexpr (FROM_T) __builtin_amdgcn_sched_barrier(0);  // (reads of a later step moved up here spill)
    }
    v4f vnew[4], oacc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const v4f iq4 = *reinterpret_cast<const v4f *>(&invq[bf][16 * i + 4 * qd]);
      const v4f eg4 = *reinterpret_cast<const v4f *>(&egl[bf][16 * i + 4 * qd]);
      const v4f be4 = *reinterpret_cast<const v4f *>(&bet[bf][16 * i + 4 * qd]);
      const v4f ik4 = *reinterpret_cast<const v4f *>(&invk[bf][16 * i + 4 * qd]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        vnew[i][e] = FROM_T ? be4[e] * (iu[i][e] - (eg4[e] * ik4[e]) * ws[i][e]) : iu[i][e] - ws[i][e];
        oacc[i][e] = qs[i][e] * (iq4[e] * eg4[e]);
      }
    }
    if constexpr (FROM_T) {  // v_new = T R, R's tiles from the accumulators as they are
      __builtin_amdgcn_sched_barrier(0);
      Half4 rB[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) rB[j] = split4<true>(vnew[j]);  // (with lo parts in both precisions)
      lower_product<SPLIT, true>(Th, Tl, r16, qd, rB, vnew, true);
      // (formed here: moved behind the P loop, its 12 operand reads would stay in registers across it)
#pragma unroll
      for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(vnew[i]));
    }
    if constexpr (!ONE) load_u(min(n + 1, a.nchunks - 1));
    for (int idx = kThreads / 64 - 1 - wave; idx < 10; idx += kThreads / 64) {  // wave-uniform
      int ti, tj;
      p_tile(idx, ti, tj);
      v4f acc = {0.f, 0.f, 0.f, 0.f};
      const uint16_t *krow = Kl[bf][16 * tj + r16];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int c = 32 * p + 4 * qd;
        acc = mfma(op8(&Ql[16 * ti + r16][32 * p + 8 * qd]), op_hi(bf16x4(krow + c), bf16x4(krow + c + 16)), acc);
      }
      const int pcol = 16 * tj + r16;
      const float kf = invk[bf][pcol], gc = gl[bf][pcol];
      const v4f iq4 = *reinterpret_cast<const v4f *>(&invq[bf][16 * ti + 4 * qd]);
      const v4f gr4 = *reinterpret_cast<const v4f *>(&gl[bf][16 * ti + 4 * qd]);
      const int pc = kpos(pcol);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int rw = 16 * ti + 4 * qd + e;
        const uint32_t pv = hilo<SPLIT>(pcol <= rw ? acc[e] * (iq4[e] * kf) * expf(gr4[e] - gc) : 0.0f);
        Ph[rw][pc] = static_cast<uint16_t>(pv);
        if constexpr (SPLIT) Po[rw][pc] = static_cast<uint16_t>(pv >> 16);
      }
    }
    lds_barrier();

    // ---- N: S = e^{g_last} S + k^T ((e^{g_last - g} / |k|) v_new) --------------------------------
    Half4 dB[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const v4f de4 = *reinterpret_cast<const v4f *>(&decl[bf][16 * j + 4 * qd]);
      const v4f ik4 = *reinterpret_cast<const v4f *>(&invk[bf][16 * j + 4 * qd]);
      v4f d;
#pragma unroll
      for (int e = 0; e < 4; ++e) d[e] = vnew[j][e] * (de4[e] * ik4[e]);
      dB[j] = split4<SPLIT>(d);
    }
    const float el = eglast[bf];
#pragma unroll
    for (int kb = 0; kb < 8; ++kb) {
#pragma unroll
      for (int e = 0; e < 4; ++e) S[kb][e] *= el;
    }
    // k^T operand (key 16 kb + r16, tokens c .. c + 3 and c + 16 .. c + 19) read from the
    // row-major k tile by transposing reads: lane 4 e + a of each 16-lane group addresses token
    // c + e, keys 16 kb + 4 a .. + 3
    const int te = r16 >> 2, ka = r16 & 3;
#pragma unroll
    for (int p = 0; p < 2; ++p) {  // token blocks 2p, 2p + 1: 8 independent accumulations
      const int c = 32 * p + 4 * qd;
#pragma unroll
      for (int kb = 0; kb < 8; ++kb) {
        S[kb] = mma_exact_a<SPLIT>(bf16x4_tr(&Kl[bf][c + te][16 * kb + 4 * ka]), bf16x4_tr(&Kl[bf][c + 16 + te][16 * kb + 4 * ka]),
                                   dB[2 * p], dB[2 * p + 1], S[kb]);
      }
    }
    if constexpr (FROM_T) __builtin_amdgcn_sched_barrier(0);
    // ---- o = e^g q^ S + P v_new (causal pairs of token tiles) ------------------------------------
    Half4 vB[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) vB[j] = split4<SPLIT>(vnew[j]);
    lower_product<SPLIT, SPLIT>(Ph, Po, r16, qd, vB, oacc, false);
    if constexpr (FROM_T) __builtin_amdgcn_sched_barrier(0);
    uint32_t oo = 4 * qd * tok + col;
    asm volatile("" : "+v"(oo));
#pragma unroll
    for (int i = 0; i < 4; ++i)
      store_o<OUT_F32, RAGGED>(static_cast<char *>(a.o) + (chunk_at(n) + static_cast<uint32_t>(16 * i) * tok) * (OUT_F32 ? 4 : 2),
                               oo, tok, r16 & 3, oacc[i], a.T - (n * kC + 16 * i + 4 * qd));
    // ---- the next chunk's rows.  Unconditional (the last chunk stages and loads itself again,
    // unused): behind a branch the compiler would lose count of the loads in flight and wait for every
    // memory operation, the o stores included.
    if constexpr (!ONE) {
      stage(n + 1);
      load(min(n + 2, a.nchunks - 1));
      lds_barrier();
    }
  };
  // Chunk 0 runs on its own: then every path into the loop has the same memory operations in
  // flight, and the compiler's wait before the first use of the loads counts only them.
  chunk(0);
  if constexpr (!ONE) {
    for (int n = 1; n < a.nchunks; ++n) chunk(n);
  }

#pragma unroll
  for (int kb = 0; kb < 8; ++kb) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      a.s_out[sbase + static_cast<size_t>(16 * kb + 4 * qd + e) * kD + 16 * wave + r16] = S[kb][e];
  }
}

// One sequence's value columns 16 CT s .. 16 CT s + 16 CT - 1.  The 8 waves of a column tile own one key
// block of S each, and are two per token tile: one for W S (and v_new), the other for q S (and o).  All
// 16 waves stage; with one column tile the last 8 do nothing else.  The sums are formed in the order of
// gdn_state_kernel, so the results are the same bit for bit.
constexpr int kColThreads = 1024;
// Fewest chunks for which gdn_state_pre_kernel runs: stages A and B of 16 sequences of 4 chunks take 22.8
// us (fp32) with it and 26.4 without; at 3 chunks and 64 sequences both take as long.
constexpr int kPreChunks = 3;
//
// PRE: P, the norms and the decays come from gdn_state_pre_kernel.
template <bool SPLIT, bool WU_F32, bool OUT_F32, bool RAGGED, int CT, bool PRE>
__global__ __launch_bounds__(kColThreads) void gdn_state_cols_kernel(StateArgs a) {
  static_assert(CT == 1 || CT == 2, "8 waves per column tile");
  constexpr int kPB = PRE ? 2 : 1;         // buffers of P: formed and read in one chunk, or staged a chunk ahead
  constexpr bool kWlo = SPLIT && WU_F32;   // a bf16 W has no lo part
  constexpr int kPr = kC + 8;              // P row stride, bf16 (36 words: 8-byte reads conflict-free)
  using Rec = std::conditional_t<SPLIT, uint4, uint2>;  // 4 values as an operand: hi pairs (, lo pairs)
  __shared__ __attribute__((aligned(16))) uint16_t Ql[kC][kQs];
  __shared__ __attribute__((aligned(16))) uint16_t Kl[2][kC][kQs];
  __shared__ __attribute__((aligned(16))) uint16_t Wh[kC][kQs], Wo[kWlo ? kC : 1][kQs];
  __shared__ __attribute__((aligned(16))) uint16_t Ph[kPB][kC][kPr], Po[kPB][SPLIT ? kC : 1][kPr];
  __shared__ Rec Sr[CT][8][64], Vr[CT][4][64], Dr[CT][4][64];  // S, v_new, (e^{g_last - g} / |k|) v_new
  constexpr int kN = PRE ? 1 : kC;
  __shared__ float invq[2][kN], invk[2][kN], gl[2][kN], egl[2][kN], decl[2][kN], eglast[2];
  __shared__ __attribute__((aligned(16))) float pre[2][PRE ? kPreF : 4];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r16 = lane & 15, qd = lane >> 4;
  // the slices of a sequence on one XCD (block indexes of one residue mod 8): they read the same q, k, W
  constexpr int kSlices = kD / (16 * CT);
  const int k8 = blockIdx.x >> 3, slice = k8 % kSlices, seq = (blockIdx.x & 7) + 8 * (k8 / kSlices);
  if (seq >= a.B * a.H) return;  // uniform: before any barrier
  const int b = seq / a.H, h = seq % a.H;
  const bool owns = CT == 2 || wave < 8;  // has a key block and a token tile
  const int ct = CT == 2 ? wave >> 3 : 0, wc = wave & 7;
  const int ti = wc & 3;                           // the wave's token tile
  const bool do_w = owns && wc < 4, do_q = owns && wc >= 4;
  const int gcol = 16 * (CT * slice + ct) + r16;   // value column
  auto put = [](Rec &r, const Half4 &x) __attribute__((always_inline)) {
    if constexpr (SPLIT) r = make_uint4(x.h01, x.h23, x.l01, x.l23);
    else r = make_uint2(x.h01, x.h23);
  };
  auto get = [](const Rec &r) __attribute__((always_inline)) {
    if constexpr (SPLIT) return Half4{r.x, r.y, r.z, r.w};
    else return exact4(r.x, r.y);
  };

  v4f S = {0.f, 0.f, 0.f, 0.f};  // key block wc: rows 16 wc + 4 qd + e, column gcol
  const size_t sbase = static_cast<size_t>(seq) * kD * kD + static_cast<size_t>(16 * wc + 4 * qd) * kD + gcol;
  if (owns) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (a.s_in) S[e] = a.s_in[sbase + static_cast<size_t>(e) * kD];
    put(Sr[ct][wc][lane], split4<SPLIT>(S));
  }
  // element offsets of chunk 0 (a chunk adds 64 H D).  Waves 0..7 stage q, 8..15 k: 16 columns of a row
  // per thread; every wave W: 8 columns of a row per thread.
  const uint32_t tok = static_cast<uint32_t>(a.H) * kD;
  const uint32_t head = (static_cast<uint32_t>(b) * a.T * a.H + h) * kD;
  const bool is_q = wave < 8;
  const int row = (t & 511) >> 3, seg = t & 7, wrow = t >> 4, wseg = t & 15;
  const uint16_t *const qk = is_q ? a.q : a.k;
  const uint32_t of_row = head + row * tok + 16 * seg, of_w = head + wrow * tok + 8 * wseg;
  const uint32_t of_tile = head + (16 * ti + 4 * qd) * tok + gcol;
  const uint32_t of_g = static_cast<uint32_t>(b) * a.T * a.H + lane * a.H + h;

  typedef unsigned v4u __attribute__((ext_vector_type(4)));
  v4u in0, in1;  // (vectors, not uint4: copied to LDS as they are, a struct goes through the stack)
  uint4 iw[WU_F32 ? 2 : 1];
  float iu[4], igc;  // igc: a token's log decay; PRE: one of the chunk's kPreF floats
  v4u ip = {};       // PRE: 8 values of a row of P (waves 0..7 hi parts, 8..15 lo parts)
  auto load = [&](int n) __attribute__((always_inline)) {
    const uint32_t c0 = static_cast<uint32_t>(n) * kC * tok;
    const v4u *p = reinterpret_cast<const v4u *>(qk + (of_row + c0 - past_end<RAGGED>(a, n, row) * tok));
    in0 = p[0];
    in1 = p[1];
    const uint32_t wi = of_w + c0 - past_end<RAGGED>(a, n, wrow) * tok;
    const uint4 *wp = WU_F32 ? reinterpret_cast<const uint4 *>(static_cast<const float *>(a.w) + wi)
                             : reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(a.w) + wi);
    iw[0] = wp[0];
    if (WU_F32) iw[WU_F32 ? 1 : 0] = wp[1];
    if constexpr (PRE) {
      const size_t item = static_cast<size_t>(seq) * a.nchunks + n;
      ip = *reinterpret_cast<const v4u *>(a.pre_p + (item * (SPLIT ? 2 : 1) + (SPLIT ? t >> 9 : 0)) * (kC * kC) + 8 * (t & 511));
      igc = a.pre_f[item * kPreF + min(t, 2 * kC)];
    } else {
      const uint32_t back = past_end<RAGGED>(a, n, lane);
      igc = a.g[of_g + (static_cast<uint32_t>(n) * kC - back) * static_cast<uint32_t>(a.H)];
      if (RAGGED && back) igc = 0.0f;
    }
  };
  auto load_u = [&](int n) __attribute__((always_inline)) {
    const uint32_t c0 = static_cast<uint32_t>(n) * kC * tok;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t ui = of_tile + c0 + static_cast<uint32_t>(e) * tok - past_end<RAGGED>(a, n, 16 * ti + 4 * qd + e) * tok;
      iu[e] = WU_F32 ? static_cast<const float *>(a.u)[ui] : bf16f(static_cast<const uint16_t *>(a.u)[ui]);
    }
  };
  // chunk n's rows into LDS (buffer n & 1 of the double-buffered arrays), with the norms and decays
  auto stage = [&](int n) __attribute__((always_inline)) {
    const int bf = n & 1;
    uint16_t *const d = is_q ? &Ql[row][16 * seg] : &Kl[bf][row][16 * seg];
    *reinterpret_cast<v4u *>(d) = in0;
    *reinterpret_cast<v4u *>(d + 8) = in1;
    if constexpr (!PRE) {
      const float ss = row_square({__builtin_bit_cast(uint4, in0), __builtin_bit_cast(uint4, in1)});
      if (seg == 0) {
        if (is_q)
          invq[bf][row] = inv_q(ss);
        else
          invk[bf][row] = inv_k(ss);
      }
    }
    if constexpr (WU_F32) {
      const Half4 x = split4<SPLIT>(__uint_as_float(iw[0].x), __uint_as_float(iw[0].y), __uint_as_float(iw[0].z), __uint_as_float(iw[0].w));
      const uint4 w1 = iw[WU_F32 ? 1 : 0];
      const Half4 y = split4<SPLIT>(__uint_as_float(w1.x), __uint_as_float(w1.y), __uint_as_float(w1.z), __uint_as_float(w1.w));
      *reinterpret_cast<uint4 *>(&Wh[wrow][8 * wseg]) = make_uint4(x.h01, x.h23, y.h01, y.h23);
      if constexpr (kWlo) *reinterpret_cast<uint4 *>(&Wo[wrow][8 * wseg]) = make_uint4(x.l01, x.l23, y.l01, y.l23);
    } else {
      *reinterpret_cast<uint4 *>(&Wh[wrow][8 * wseg]) = iw[0];
    }
    if constexpr (PRE) {
      if (SPLIT || wave < 8) {  // wave-uniform
        const int pr = (t & 511) >> 3, pc = 8 * (t & 7);
        *reinterpret_cast<v4u *>(SPLIT && wave >= 8 ? &Po[PRE ? bf : 0][SPLIT ? pr : 0][pc] : &Ph[PRE ? bf : 0][pr][pc]) = ip;
      }
      if (t <= 2 * kC) pre[bf][PRE ? t : 0] = igc;
    } else if (wave == 0) {  // (its token tile has no o to form)
      const float g = scan64(igc);
      const float glast = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g), 63));
      gl[bf][lane] = g;
      egl[bf][lane] = expf(g);
      decl[bf][lane] = RAGGED && n * kC + lane >= a.T ? 0.0f : expf(glast - g);
      if (lane == 0) eglast[bf] = expf(glast);
    }
  };
  load(0);
  load_u(0);
  stage(0);
  load(min(1, a.nchunks - 1));
  lds_barrier();

  auto chunk = [&](const int n) __attribute__((always_inline)) {
    const int bf = n & 1;
    const int pb = PRE ? bf : 0;
    // ---- products: W S and q^ S of the wave's token tile, v_new; P tiles -------------------------
    Half4 sB[8];
    if (owns) {
#pragma unroll
      for (int kb = 0; kb < 8; ++kb) sB[kb] = get(Sr[ct][kb][lane]);
    }
    v4f oacc = {0.f, 0.f, 0.f, 0.f};
    if (do_w) {  // wave-uniform
      v4f ws = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int c = 32 * p + 4 * qd;
        Half4 w0 = bf16x4(&Wh[16 * ti + r16][c]), w1 = bf16x4(&Wh[16 * ti + r16][c + 16]);
        if constexpr (kWlo) {
          const Half4 l0 = bf16x4(&Wo[16 * ti + r16][c]), l1 = bf16x4(&Wo[16 * ti + r16][c + 16]);
          w0.l01 = l0.h01; w0.l23 = l0.h23; w1.l01 = l1.h01; w1.l23 = l1.h23;
        }
        ws = WU_F32 ? mma<SPLIT>(w0, w1, sB[2 * p], sB[2 * p + 1], ws) : mma_exact_a<SPLIT>(w0, w1, sB[2 * p], sB[2 * p + 1], ws);
      }
      v4f vn, d;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int rw = 16 * ti + 4 * qd + e;
        vn[e] = iu[e] - ws[e];
        d[e] = vn[e] * (PRE ? pre[bf][kC + rw] : decl[bf][rw] * invk[bf][rw]);
      }
      put(Vr[ct][ti][lane], split4<SPLIT>(vn));
      put(Dr[ct][ti][lane], split4<SPLIT>(d));
    }
    if (do_q) {
      v4f qs = {0.f, 0.f, 0.f, 0.f};
      const uint16_t *qrow = Ql[16 * ti + r16];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int c = 32 * p + 4 * qd;
        qs = mma_exact_a<SPLIT>(bf16x4(qrow + c), bf16x4(qrow + c + 16), sB[2 * p], sB[2 * p + 1], qs);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int rw = 16 * ti + 4 * qd + e;
        oacc[e] = qs[e] * (PRE ? pre[bf][rw] : invq[bf][rw] * egl[bf][rw]);
      }
    }
    // (a load moved up across its registers' last use would have to be waited for and copied)
    if constexpr (PRE) __builtin_amdgcn_sched_barrier(0);
    load_u(min(n + 1, a.nchunks - 1));
    if (!PRE && 15 - wave < 10) {  // wave-uniform: one P tile on each of 10 waves
      int pi, pj;
      p_tile(15 - wave, pi, pj);
      v4f acc = {0.f, 0.f, 0.f, 0.f};
      const uint16_t *qrow = Ql[16 * pi + r16];
      const uint16_t *krow = Kl[bf][16 * pj + r16];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int c = 32 * p + 4 * qd;
        acc = mma<false>(bf16x4(qrow + c), bf16x4(qrow + c + 16), bf16x4(krow + c), bf16x4(krow + c + 16), acc);
      }
      const int col = 16 * pj + r16;
      const float kf = invk[bf][col];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int rw = 16 * pi + 4 * qd + e;
        const float pv = col <= rw ? acc[e] * (invq[bf][rw] * kf) * expf(gl[bf][rw] - gl[bf][col]) : 0.0f;
        const uint32_t w = hilo<SPLIT>(pv);
        Ph[pb][rw][col] = static_cast<uint16_t>(w);
        if constexpr (SPLIT) Po[pb][rw][col] = static_cast<uint16_t>(w >> 16);
      }
    }
    lds_barrier();

    // ---- S = e^{g_last} S + k^T ((e^{g_last - g} / |k|) v_new), the wave's key block ---------------
    const float el = PRE ? pre[bf][2 * kC] : eglast[bf];
    const int te = r16 >> 2, ka = r16 & 3;
    if (owns) {
#pragma unroll
      for (int e = 0; e < 4; ++e) S[e] *= el;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int c = 32 * p + 4 * qd, kc = 16 * wc + 4 * ka;
        S = mma_exact_a<SPLIT>(bf16x4_tr(&Kl[bf][c + te][kc]), bf16x4_tr(&Kl[bf][c + 16 + te][kc]), get(Dr[ct][2 * p][lane]),
                               get(Dr[ct][2 * p + 1][lane]), S);
      }
      put(Sr[ct][wc][lane], split4<SPLIT>(S));
    }
    // ---- o = e^g q^ S + P v_new ------------------------------------------------------------------
    if (do_q) {
      v4f acc = oacc;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        if (p > ti / 2) continue;  // wave-uniform
        const bool two = 2 * p + 1 <= ti;
        const int c = 32 * p + 4 * qd;
        Half4 p0 = bf16x4(&Ph[pb][16 * ti + r16][c]), p1 = kZero4;
        if (two) p1 = bf16x4(&Ph[pb][16 * ti + r16][c + 16]);
        if constexpr (SPLIT) {
          const Half4 l0 = bf16x4(&Po[pb][16 * ti + r16][c]);
          p0.l01 = l0.h01; p0.l23 = l0.h23;
          if (two) {
            const Half4 l1 = bf16x4(&Po[pb][16 * ti + r16][c + 16]);
            p1.l01 = l1.h01; p1.l23 = l1.h23;
          }
        }
        acc = mma<SPLIT>(p0, p1, get(Vr[ct][2 * p][lane]), two ? get(Vr[ct][2 * p + 1][lane]) : kZero4, acc);
      }
      store_o<OUT_F32, RAGGED>(a.o, of_tile + static_cast<uint32_t>(n * kC) * tok, tok, r16 & 3, acc, a.T - (n * kC + 16 * ti + 4 * qd));
    }
    // ---- the next chunk's rows (the last chunk stages itself again, unused) -------------------------
    stage(n + 1);
    if constexpr (PRE) __builtin_amdgcn_sched_barrier(0);
    load(min(n + 2, a.nchunks - 1));
    lds_barrier();
  };
  if constexpr (PRE) chunk(0);  // on its own, for the wait counts (as in gdn_state_kernel)
  for (int n = PRE ? 1 : 0; n < a.nchunks; ++n) chunk(n);

  if (owns) {
#pragma unroll
    for (int e = 0; e < 4; ++e) a.s_out[sbase + static_cast<size_t>(e) * kD] = S[e];
  }
}

// T = (I - A)^-1 of every chunk of 64 tokens, A_ij = -beta_i (k^_i . k^_j) e^{g_i - g_j} for i > j, as
// gdn_state_kernel reads it (FROM_T).  One workgroup (4 waves) per (sequence, chunk): the 10 lower tiles
// of K K^T over the waves; T's diagonal blocks by forward substitution, one lane per column; then wave j
// the strip of block column j, its solved blocks in registers as the next products' B operands.
constexpr int kTThreads = 256;
constexpr int kTd = 260;  // floats per diagonal block (padded: four blocks are read at once)
constexpr int kTr = 20;   // row stride of a lower block, floats
template <bool SPLIT, bool RAGGED>
__global__ __launch_bounds__(kTThreads) void gdn_t_kernel(StateArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t Kl[kC][kQs];
  __shared__ __attribute__((aligned(16))) float diag[4 * kTd], low[6][16][kTr], invk[kC], gl[kC], bet[kC];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r16 = lane & 15, qd = lane >> 4;
  const int seq = blockIdx.x / a.nchunks, n = blockIdx.x % a.nchunks, b = seq / a.H, h = seq % a.H;
  const uint32_t tok = static_cast<uint32_t>(a.H) * kD;
  const uint32_t head = (static_cast<uint32_t>(b) * a.T * a.H + h) * kD;
  uint4 ik[2][2];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int row = 32 * r + (t >> 3);
    const uint4 *kp = reinterpret_cast<const uint4 *>(a.k + (head + 16 * (t & 7) + (static_cast<uint32_t>(n) * kC + row - past_end<RAGGED>(a, n, row)) * tok));
    ik[r][0] = kp[0];
    ik[r][1] = kp[1];
  }
  if (wave == 0) {
    const uint32_t back = past_end<RAGGED>(a, n, lane);
    const uint32_t gi = static_cast<uint32_t>(b) * a.T * a.H + h + (static_cast<uint32_t>(n) * kC + lane - back) * static_cast<uint32_t>(a.H);
    const bool past = RAGGED && back;
    gl[lane] = scan64(past ? 0.0f : a.g[gi]);
    bet[lane] = past ? 0.0f : a.beta[gi];
  }
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int row = 32 * r + (t >> 3), seg = t & 7;
    *reinterpret_cast<uint4 *>(&Kl[row][16 * seg]) = ik[r][0];
    *reinterpret_cast<uint4 *>(&Kl[row][16 * seg + 8]) = ik[r][1];
    const float ss = row_square(ik[r]);
    if (seg == 0) invk[row] = inv_k(ss);
  }
  lds_barrier();
  for (int idx = wave; idx < 10; idx += kTThreads / 64) {  // wave-uniform
    int ti, tj;
    p_tile(idx, ti, tj);
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    const uint16_t *irow = Kl[16 * ti + r16], *jrow = Kl[16 * tj + r16];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int c = 32 * p + 4 * qd;
      acc = mma<false>(bf16x4(irow + c), bf16x4(irow + c + 16), bf16x4(jrow + c), bf16x4(jrow + c + 16), acc);
    }
    const int col = 16 * tj + r16;
    const float kf = invk[col], gc = gl[col];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 4 * qd + e, rw = 16 * ti + r;
      const float av = col < rw ? -bet[rw] * acc[e] * (invk[rw] * kf) * expf(gl[rw] - gc) : 0.0f;
      if (ti > tj)
        low[ti * (ti - 1) / 2 + tj][r][r16] = av;
      else
        diag[ti * kTd + r16 * 16 + r] = av;  // by columns
    }
  }
  lds_barrier();
  if (wave == 0) {  // T_II, lane: block lane / 16, column lane % 16; in place, by rows
    float *const d = diag + qd * kTd;
    float x[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float s = r == r16 ? 1.0f : 0.0f;
#pragma unroll
      for (int c = 0; c < r; ++c) s = fmaf(d[c * 16 + r], x[c], s);
      x[r] = s;
    }
    asm volatile("" ::: "memory");  // every read of A is before the first store of T
#pragma unroll
    for (int r = 0; r < 16; ++r) d[r * 16 + r16] = x[r];
  }
  lds_barrier();
  uint16_t *const T = a.t + static_cast<size_t>(blockIdx.x) * (SPLIT ? 2 : 1) * (kC * kC);
  const int j = wave, qq = r16 & 3;
  auto store = [&](int i, const Half4 &x) __attribute__((always_inline)) {
    uint16_t *const d = T + (16 * i + 4 * qd + qq) * kC + kpos(16 * j + (r16 & ~3));
    *reinterpret_cast<uint2 *>(d) = quad_rows(x.h01, x.h23, qq);
    if constexpr (SPLIT) *reinterpret_cast<uint2 *>(d + kC * kC) = quad_rows(x.l01, x.l23, qq);
  };
  auto f4 = [](const float *p) __attribute__((always_inline)) { return split4<true>(*reinterpret_cast<const float4 *>(p)); };
  if (j & 1) store(j - 1, kZero4);  // read beside the diagonal tile
  Half4 xs[4];
  {
    const float *const d = diag + j * kTd + 64 * qd + r16;
    xs[0] = split4<true>(d[0], d[16], d[32], d[48]);
    store(j, xs[0]);
  }
#pragma unroll
  for (int s = 1; s < 4; ++s) {
    const int i = j + s;
    if (i < 4) {  // wave-uniform
      v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < s; u += 2) {
        const int blk = i * (i - 1) / 2 + j + u;
        const bool two = u + 1 < s;
        acc = mma<true>(f4(&low[blk][r16][4 * qd]), two ? f4(&low[two ? blk + 1 : blk][r16][4 * qd]) : kZero4, xs[u],
                        two ? xs[u + 1] : kZero4, acc);
      }
      const v4f x = mma<true>(f4(diag + i * kTd + 16 * r16 + 4 * qd), kZero4, split4<true>(acc), kZero4, v4f{0.f, 0.f, 0.f, 0.f});
      xs[s] = split4<true>(x);
      store(i, xs[s]);
    }
  }
}

// What a chunk needs besides the state, for every (sequence, chunk) at once: P, the row factors of q^ S
// (e^g / |q| / sqrt(D)) and of v_new in the state update (e^{g_last - g} / |k|), e^{g_last}.  Left to
// the recurrence, these are some 60 % of the instructions of a chunk of gdn_state_cols_kernel, repeated
// by each of a sequence's workgroups, one chunk after another.
template <bool SPLIT, bool RAGGED>
__global__ __launch_bounds__(kThreads) void gdn_state_pre_kernel(StateArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t Ql[kC][kQs], Kl[kC][kQs];
  __shared__ __attribute__((aligned(16))) float invq[kC], invk[kC], gl[kC];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r16 = lane & 15, qd = lane >> 4;
  const size_t item = blockIdx.x;
  const int seq = blockIdx.x / a.nchunks, n = blockIdx.x % a.nchunks, b = seq / a.H, h = seq % a.H;
  const uint32_t tok = static_cast<uint32_t>(a.H) * kD;
  const int row = t >> 3, seg = t & 7;
  const uint32_t at = (static_cast<uint32_t>(b) * a.T * a.H + h) * kD + 16 * seg +
                      (static_cast<uint32_t>(n) * kC + row - past_end<RAGGED>(a, n, row)) * tok;
  const uint4 *qp = reinterpret_cast<const uint4 *>(a.q + at), *kp = reinterpret_cast<const uint4 *>(a.k + at);
  const uint4 iq[2] = {qp[0], qp[1]}, ik[2] = {kp[0], kp[1]};
  float gc = 0.0f;
  if (wave == 0) {
    const uint32_t back = past_end<RAGGED>(a, n, lane);
    gc = a.g[static_cast<uint32_t>(b) * a.T * a.H + h + (static_cast<uint32_t>(n) * kC + lane - back) * static_cast<uint32_t>(a.H)];
    if (RAGGED && back) gc = 0.0f;
  }
  *reinterpret_cast<uint4 *>(&Ql[row][16 * seg]) = iq[0];
  *reinterpret_cast<uint4 *>(&Ql[row][16 * seg + 8]) = iq[1];
  *reinterpret_cast<uint4 *>(&Kl[row][16 * seg]) = ik[0];
  *reinterpret_cast<uint4 *>(&Kl[row][16 * seg + 8]) = ik[1];
  const float sq = row_square(iq), sk = row_square(ik);
  if (seg == 0) {
    invq[row] = inv_q(sq);
    invk[row] = inv_k(sk);
  }
  const float g = scan64(gc);  // wave 0's counts
  if (wave == 0) gl[lane] = g;
  lds_barrier();
  if (wave == 0) {
    const float glast = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g), 63));
    float *const f = a.pre_f + item * kPreF;
    f[lane] = invq[lane] * expf(g);
    f[kC + lane] = (RAGGED && n * kC + lane >= a.T ? 0.0f : expf(glast - g)) * invk[lane];
    if (lane == 0) f[2 * kC] = expf(glast);
  }
  uint16_t *const P = a.pre_p + item * (SPLIT ? 2 : 1) * (kC * kC);
  for (int idx = kThreads / 64 - 1 - wave; idx < 10; idx += kThreads / 64) {  // wave-uniform
    int ti, tj;
    p_tile(idx, ti, tj);
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    const uint16_t *qrow = Ql[16 * ti + r16], *krow = Kl[16 * tj + r16];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int c = 32 * p + 4 * qd;
      acc = mma<false>(bf16x4(qrow + c), bf16x4(qrow + c + 16), bf16x4(krow + c), bf16x4(krow + c + 16), acc);
    }
    const int col = 16 * tj + r16;
    const float kf = invk[col];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int rw = 16 * ti + 4 * qd + e;
      const uint32_t w = hilo<SPLIT>(col <= rw ? acc[e] * (invq[rw] * kf) * expf(gl[rw] - gl[col]) : 0.0f);
      P[rw * kC + col] = static_cast<uint16_t>(w);
      if constexpr (SPLIT) P[kC * kC + rw * kC + col] = static_cast<uint16_t>(w >> 16);
    }
  }
}

// Workgroups of the column-sliced kernel with CT column tiles each, or 0 where they would not all have a
// compute unit of their own.  One tile where that fits (up to 32 sequences): 16 sequences of 4096 tokens
// take 120 / 158 us (bf16 / fp32) with one tile, 153 / 191 with two.
int cols_grid(int seqs, int ct) {
  const int per8 = (seqs + 7) / 8 * 8, grid = per8 * (kD / (16 * ct));
  return grid <= device_cu_count() ? grid : 0;
}

template <bool SPLIT, bool WU_F32, bool OUT_F32, bool RAGGED>
qh_status launch4(const StateArgs &a, hipStream_t stream) {
  const int seqs = a.B * a.H, grid1 = cols_grid(seqs, 1), grid2 = cols_grid(seqs, 2);
  if (grid2 && a.pre_p) {
    hipLaunchKernelGGL((gdn_state_pre_kernel<SPLIT, RAGGED>), dim3(seqs * a.nchunks), dim3(kThreads), 0, stream, a);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return hip_fail(err, "gdn_state_pre_kernel launch");
    if (grid1)
      hipLaunchKernelGGL((gdn_state_cols_kernel<SPLIT, WU_F32, OUT_F32, RAGGED, 1, true>), dim3(grid1), dim3(kColThreads), 0, stream, a);
    else
      hipLaunchKernelGGL((gdn_state_cols_kernel<SPLIT, WU_F32, OUT_F32, RAGGED, 2, true>), dim3(grid2), dim3(kColThreads), 0, stream, a);
  } else if (grid2)
    hipLaunchKernelGGL((gdn_state_cols_kernel<SPLIT, WU_F32, OUT_F32, RAGGED, 2, false>), dim3(grid2), dim3(kColThreads), 0, stream, a);
  else if (!RAGGED && a.nchunks == 1)
    hipLaunchKernelGGL((gdn_state_kernel<SPLIT, WU_F32, OUT_F32, false, false, true>), dim3(seqs), dim3(kThreads), 0, stream, a);
  else
    hipLaunchKernelGGL((gdn_state_kernel<SPLIT, WU_F32, OUT_F32, RAGGED, false>), dim3(seqs), dim3(kThreads), 0, stream, a);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return hip_fail(err, "gdn_state_kernel launch");
  return QH_STATUS_OK;
}

template <bool SPLIT, bool WU_F32, bool OUT_F32>
qh_status launch3(const StateArgs &a, hipStream_t stream) {
  return a.T % kC ? launch4<SPLIT, WU_F32, OUT_F32, true>(a, stream) : launch4<SPLIT, WU_F32, OUT_F32, false>(a, stream);
}

// Prefill of many sequences: T, then the recurrence from T and v.
template <bool SPLIT, bool RAGGED>
qh_status launch_prefill2(const StateArgs &a, bool out_f32, hipStream_t stream) {
  const int seqs = a.B * a.H;
  hipLaunchKernelGGL((gdn_t_kernel<SPLIT, RAGGED>), dim3(seqs * a.nchunks), dim3(kTThreads), 0, stream, a);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return hip_fail(err, "gdn_t_kernel launch");
  auto recurrence = [&](auto out32, auto one) {
    hipLaunchKernelGGL((gdn_state_kernel<SPLIT, false, decltype(out32)::value, RAGGED, true, decltype(one)::value>), dim3(seqs),
                       dim3(kThreads), 0, stream, a);
  };
  auto by_chunks = [&](auto out32) {
    if constexpr (!RAGGED) {
      if (a.nchunks == 1) return recurrence(out32, std::true_type{});
    }
    recurrence(out32, std::false_type{});
  };
  if (out_f32) by_chunks(std::true_type{});
  else by_chunks(std::false_type{});
  err = hipGetLastError();
  if (err != hipSuccess) return hip_fail(err, "gdn_state_kernel launch");
  return QH_STATUS_OK;
}

template <bool SPLIT>
qh_status launch2(const StateArgs &a, bool wu_f32, bool out_f32, hipStream_t stream) {
  if (wu_f32) return out_f32 ? launch3<SPLIT, true, true>(a, stream) : launch3<SPLIT, true, false>(a, stream);
  return out_f32 ? launch3<SPLIT, false, true>(a, stream) : launch3<SPLIT, false, false>(a, stream);
}

}  // namespace

// Bytes that gdn_state_pre_kernel writes: P, then the factors (both multiples of 16).
static size_t pre_p_bytes(size_t items, int precision) { return items * (precision == QH_GDN_BF16 ? 2 : 4) * kC * kC; }

size_t gdn_chunk_state_workspace(int B, int T, int H, int precision) {
  const int nchunks = (T + kC - 1) / kC;
  if (nchunks < kPreChunks || cols_grid(B * H, 2) == 0) return 0;
  const size_t items = static_cast<size_t>(B) * H * nchunks;
  return pre_p_bytes(items, precision) + items * kPreF * sizeof(float);
}

qh_status launch_gdn_chunk_state(const uint16_t *q, const uint16_t *k, const float *g, const void *w, const void *u,
                                 const float *s_in, float *s_out, void *o, int B, int T, int H, int precision,
                                 bool wu_f32, bool out_f32, void *ws, size_t ws_bytes, hipStream_t stream) {
  StateArgs a{q, k, g, w, u, s_in, s_out, o, B, T, H, (T + kC - 1) / kC, nullptr, nullptr, nullptr, nullptr};
  const size_t need = ws ? gdn_chunk_state_workspace(B, T, H, precision) : 0;
  if (need && ws_bytes >= need) {
    a.pre_p = static_cast<uint16_t *>(ws);
    a.pre_f = reinterpret_cast<float *>(static_cast<uint8_t *>(ws) + pre_p_bytes(static_cast<size_t>(B) * H * a.nchunks, precision));
  }
  return precision == QH_GDN_BF16 ? launch2<false>(a, wu_f32, out_f32, stream)
                                  : launch2<true>(a, wu_f32, out_f32, stream);
}

// Few sequences take the column-sliced recurrence, which reads W and U.
size_t gdn_prefill_workspace(int B, int T, int H, int precision) {
  if (cols_grid(B * H, 2) != 0) return 0;
  return pre_p_bytes(static_cast<size_t>(B) * H * ((T + kC - 1) / kC), precision);  // T is P's size
}

qh_status launch_gdn_prefill(const uint16_t *q, const uint16_t *k, const uint16_t *v, const float *g, const float *beta,
                             const float *s_in, float *s_out, void *o, int B, int T, int H, int precision, bool out_f32,
                             void *ws, hipStream_t stream) {
  StateArgs a{q, k, g, nullptr, v, s_in, s_out, o, B, T, H, (T + kC - 1) / kC, nullptr, nullptr, static_cast<uint16_t *>(ws), beta};
  const bool ragged = T % kC != 0;
  if (precision == QH_GDN_BF16)
    return ragged ? launch_prefill2<false, true>(a, out_f32, stream) : launch_prefill2<false, false>(a, out_f32, stream);
  return ragged ? launch_prefill2<true, true>(a, out_f32, stream) : launch_prefill2<true, false>(a, out_f32, stream);
}

}  // namespace qh
