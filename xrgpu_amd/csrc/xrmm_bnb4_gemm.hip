// MatMulBnb4 with many rows on the matrix cores (xrmm_gemm_ks.h); the codebooks
// are complex_kernel.glsl:82's.
#include <cmath>

#include "xrmm_gemm_ks.h"
#include "xrmm_quant.h"

namespace xrmm {

namespace {

struct Planes {
  uint32_t t[16];
  float unscale;
};

// Factors of the codebooks. Two binary16 terms of one sign hold 22 bits of a value:
// at 2^15 the float32 codebooks' values were up to 1.6 units of 2^-24 off. A factor
// that is not a power of two moves all of them; of 32 million float32 factors in 2^14 ..
// 2^15 these leave 0.28 units at most for NF4, none for FP4 (nearly 192 times a power
// of two, FP4's common denominator), with every lo at least 2^-13 (a normal binary16
// value). What the factor's inverse and its product with a block's scale round is common
// to a block's weights.
constexpr double kNF4Factor = 0x1.8d1becp+14, kFP4Factor = 0x1.f80018p+14;

// The codebook, times the factor, as two binary16 terms of each value's own sign:
// hi the largest magnitude below the value, lo the rest (rounded to nearest,
// never zero unless the value is), split into their low and high bytes.
Planes planes(const float (&book)[16], double factor) {
  Planes p{};
  p.unscale = static_cast<float>(1.0 / factor);
  for (int c = 0; c < 16; ++c) {
    const double v = std::fabs(static_cast<double>(book[c])) * factor;
    double hi = 0.0;
    if (v > 0.0) {
      int e = 0;
      (void)std::frexp(v, &e);  // v in [2^(e - 1), 2^e): binary16 spacing 2^(e - 11)
      const double ulp = std::ldexp(1.0, e - 11);
      hi = std::floor(v / ulp) * ulp;
      if (hi == v) hi -= v == std::ldexp(1.0, e - 1) ? ulp / 2 : ulp;
    }
    const double sign = std::signbit(book[c]) ? -1.0 : 1.0;
    const uint16_t h = __builtin_bit_cast(uint16_t, static_cast<_Float16>(sign * hi));
    const uint16_t l = __builtin_bit_cast(uint16_t, static_cast<_Float16>(sign * (v - hi)));
    const uint32_t hu = h, lu = l, b[4] = {hu & 255u, hu >> 8, lu & 255u, lu >> 8};
    for (int q = 0; q < 4; ++q) p.t[4 * q + c / 4] |= b[q] << (8 * (c % 4));
  }
  return p;
}

}  // namespace

bool bnb4_gemm_ok(const Bnb4Args& a) {
  if (!a.f16 || !a.tb || (a.M < kBnb4GemmMinM && bnb4_fast_ok(a)) || a.K % 32 != 0 || a.bs < 32 || (a.bs & (a.bs - 1)) != 0 || a.K % a.bs != 0) return false;
  // 16-byte loads of A and B; a column's block scales load as 4- and 8-byte words,
  // which want absmax on a word (a view at an odd element stays with the GEMV, which
  // loads them one by one)
  if ((reinterpret_cast<uintptr_t>(a.B) & 15) != 0 || (reinterpret_cast<uintptr_t>(a.A) & 15) != 0 ||
      (reinterpret_cast<uintptr_t>(a.absmax) & 3) != 0)
    return false;
  // 32-bit buffer ranges, row and grid counts
  const int64_t lim = int64_t(1) << 31;
  return a.N * (a.K / 2) < lim && a.M * a.K * 2 < lim && a.M < lim / 2 && (a.M + 31) / 32 * ((a.N + 31) / 32) < lim;
}

hipError_t launch_bnb4_gemm(const Bnb4Args& a, const float (&nf4)[16], const float (&fp4)[16], hipStream_t st) {
  static const Planes nf = planes(nf4, kNF4Factor), fp = planes(fp4, kFP4Factor);
  ks::Args g{};
  g.A = a.A;
  g.B = a.B;
  g.S = a.absmax;
  g.Y = a.Y;
  g.M = static_cast<int>(a.M);
  g.K = static_cast<int>(a.K);
  g.N = static_cast<int>(a.N);
  g.bs = a.bs;
  g.lbs = __builtin_ctz(static_cast<unsigned>(a.bs));
  g.kb = static_cast<int>(a.K / a.bs);
  const Planes& p = a.qt == 1 ? nf : fp;
  for (int i = 0; i < 16; ++i) g.tbl[i] = p.t[i];
  g.unscale = p.unscale;
  const int cus = device_cus();
  const ks::Plan pl = ks::plan(a.M, a.N, a.K, cus > 0 ? cus : 256, 4);
  g.nrt = pl.nrt;
  return ks::launch_ks<f16, ks::KS_BNB>(g, pl, st);
}

}  // namespace xrmm
