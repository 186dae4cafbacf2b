// The reference's integer output contracts on an exact integer dot product D = sum_k (a - zp) w,
// shared by the tile kernel (qmm_tile.hip) and the one-launch chains (qmm_exact.hip).

#ifndef QHTP_QMM_CONTRACT_H_
#define QHTP_QMM_CONTRACT_H_

#include "qmm_internal.h"

namespace qh {
namespace {

constexpr bool contract_divides(int ct) {
  return ct == QH_CONTRACT_DIV_RINT || ct == QH_CONTRACT_FLOOR256_DIV_RINT || ct == QH_CONTRACT_ROUND_DIV;
}

// The contracts without a division.  bias: bias_q[n] (0 without a bias operand).
template <int CT, class Args>
__device__ __forceinline__ int contract_int(const Args &g, long long D, long long bias) {
  const long long qmax = g.out_qmax;
  if constexpr (CT == QH_CONTRACT_CLIP_I32) {  // int32 arithmetic of the reference (wraps modulo 2^32)
    const int v = static_cast<int>(static_cast<unsigned int>(static_cast<unsigned long long>(D + bias)));
    return v < 0 ? 0 : (v > qmax ? static_cast<int>(qmax) : v);
  } else if constexpr (CT == QH_CONTRACT_CLIP_I64) {
    const long long v = D + bias;
    return static_cast<int>(v < 0 ? 0 : (v > qmax ? qmax : v));
  } else {  // QH_CONTRACT_U8_DRAIN: (acc + bias) * s / 512 in float64, truncated, + b >> 7
    const uint32_t pk = static_cast<uint32_t>(g.divisor);
    const uint32_t e = (pk >> 10) & 31u, f = pk & 1023u;
    const double mag = e == 0 ? ldexp(static_cast<double>(f), -24) : ldexp(static_cast<double>(1024u + f), static_cast<int>(e) - 25);
    const double s = (pk & 0x8000u) ? -mag : mag;
    const long long drain = D + bias;
    const long long v = static_cast<long long>(trunc(static_cast<double>(drain) * s / 512.0)) + (pk >> 23);
    return static_cast<int>(v < 0 ? 0 : (v > qmax ? qmax : v));
  }
}

// The dividing contracts in float64 without a division, on D as an integer-valued double
// (|D| < 2^50; the largest, K = 65536 of 16-bit operands, is 2^47).
//  * rint(double(D) / d + zp): y = D rcp + zp (rcp = fl(1 / d), one fma) is within 2^-34 of
//    X = D / d + zp whenever rint(y) lies in [-1, qmax + 1] (then |D / d| < 2^18).
//    If y is also more than 2^-20 from the nearest half-integer, rint(y) = rint(X).  The
//    float64 division rounds the same X for every output that is not clipped: a quotient that
//    is not a tie lies at least 1 / (2 d) >= 2^-31 from a half-integer, and the division's two
//    roundings move it by less.  Outputs outside [-1, qmax + 1] clip the same either way.  The
//    few outputs near a half-integer (exact ties: only for even d) take the exact remainder
//    2 (D - (c - zp) d), which picks the neighbour the exact quotient rounds to (ties to even);
//    a wave enters that branch only when one of its lanes needs it.
//  * floor(n / d) (round_div, n >= 0): floor(n rcp) is within one; the remainder fixes it.
template <int CT, class Args>
__device__ __forceinline__ int contract_f64(const Args &g, double Dd, double rcp) {
  const double dd = static_cast<double>(g.divisor), zp = static_cast<double>(g.out_zp);
  const double qmax = static_cast<double>(g.out_qmax);
  if constexpr (CT == QH_CONTRACT_ROUND_DIV) {
    const double n = fabs(Dd) + static_cast<double>(g.divisor / 2);
    double q = floor(n * rcp);
    const double r = fma(-q, dd, n);
    q = r < 0.0 ? q - 1.0 : (r >= dd ? q + 1.0 : q);
    const double v = (Dd >= 0.0 ? q : -q) + zp;
    return static_cast<int>(fmin(fmax(v, 0.0), qmax));
  } else {
    if (CT == QH_CONTRACT_FLOOR256_DIV_RINT) Dd = floor(Dd * 0x1p-8) * 256.0;  // floor division, exact
    const double y = fma(Dd, rcp, zp);
    double c = rint(y);
    const bool near = fabs(y - c) > 0.5 - 0x1p-20 && c >= -1.0 && c <= qmax + 1.0;
    if (__builtin_amdgcn_ballot_w64(near) != 0) {  // wave-uniform: rare
      // exact for every lane: in range, c is within one of the rounded quotient (and lanes that
      // are not near stay put); out of range, c +- 1 clips like c
      const double r2 = 2.0 * fma(zp - c, dd, Dd);  // 2 (D - q d), q = c - zp
      const double h = c * 0.5;
      const bool odd = h != floor(h);
      c = (r2 > dd || (r2 == dd && odd)) ? c + 1.0 : ((r2 < -dd || (r2 == -dd && odd)) ? c - 1.0 : c);
    }
    return static_cast<int>(fmin(fmax(c, 0.0), qmax));
  }
}

}  // namespace
}  // namespace qh

#endif  // QHTP_QMM_CONTRACT_H_
