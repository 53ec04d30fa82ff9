// int8-activation MatMulNBits with many rows on the matrix cores
// (xrmm_gemm_ks.h), on the activation codes of k_i8a_quant.
#include "xrmm_gemm_ks.h"
#include "xrmm_quant.h"

namespace xrmm {

bool i8a_gemm_ok(const Int8aArgs& a) {
  // scales load as words of 4 to 16 bytes, zero points as 2 bytes (the GEMV loads both
  // one by one and keeps views at odd elements)
  if ((reinterpret_cast<uintptr_t>(a.S) & 3) != 0 || (reinterpret_cast<uintptr_t>(a.Z) & 1) != 0) return false;
  const int64_t lim = int64_t(1) << 31;
  return a.M >= kI8aGemmMinM && a.M * a.N >= (kI8aGemmMinMacs + a.K - 1) / a.K && a.N * (a.K / 2) < lim && a.M * a.K < lim && (a.M + 31) / 32 * ((a.N + 31) / 32) < lim;
}

hipError_t launch_i8a_gemm(const Int8aArgs& a, hipStream_t st) {
  ks::Args g{};
  g.A = a.qa;
  g.as = a.as;
  g.B = a.B;
  g.S = a.S;
  g.Z = a.Z;
  g.bias = a.bias;
  g.Y = a.Y;
  g.M = static_cast<int>(a.M);
  g.K = static_cast<int>(a.K);
  g.N = static_cast<int>(a.N);
  g.bs = a.bs;
  g.lbs = __builtin_ctz(static_cast<unsigned>(a.bs));
  g.kb = static_cast<int>(a.K / a.bs);
  g.zrow = static_cast<int>(a.zrow);
  const int cus = device_cus();
  const ks::Plan pl = ks::plan(a.M, a.N, a.K, cus > 0 ? cus : 256, 3);
  g.nrt = pl.nrt;
  return a.f16 ? ks::launch_ks<f16, ks::KS_Q8>(g, pl, st) : ks::launch_ks<float, ks::KS_Q8>(g, pl, st);
}

}  // namespace xrmm
