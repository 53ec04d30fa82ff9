// GEMM for packed 4-bit weights whose value is (a function of the code) x (the
// block's scale), with every float32 the reference keeps kept: the codes'
// values enter v_mfma_f32_32x32x16_f16 as binary16 terms that hold them, each
// block's float32 sum is multiplied by the block's scale as it joins the
// column's running float32 sum. Two operators run on it:
//
//  * MatMulBnb4 (KS_BNB): float16 activations as they are; a codebook value is
//    the sum of two binary16 terms of its own sign (hi rounded towards zero and
//    below the value, lo the rest), so +-Inf activations meet no zero term that
//    the float32 product would not have; both terms go through the matrix cores.
//    Values are scaled (undone in the block scale) by a factor near 2^15, chosen
//    for each codebook so that the two terms hold its values to 0.3 of 2^-24.
//  * int8-activation MatMulNBits (KS_Q8): activation codes and code - zero
//    point are exact binary16 integers, so a block's sum is the exact integer
//    the int8 dot product gives (below 2^24); the block sums, times their weight
//    scales, add up over the 128 activations that share a scale, and that scale
//    multiplies the sum. Binary16 and not int8 matrix instructions: the int8 sum
//    needs a conversion besides the scaling for each output and block (two VALU
//    instructions against one), and those, not the MFMA rate, set the time.
//
// Shape. A workgroup of 8 waves owns 32 IM rows x (256 / KG) columns: KG groups
// of 8 / KG waves take contiguous ranges of K, each wave 32 columns and all rows
// of the tile, so each weight is decoded once per workgroup (a codebook pair
// costs 5 VALU instructions a code) and meets IM MFMA row tiles; the groups'
// sums meet in LDS at the end, in group order. Splitting K inside the workgroup
// fills the CUs where the output has few tiles, with no memory traffic. The
// weights go straight from memory into registers, the activations through a
// double-buffered LDS, both two steps of 64 ahead.
//
// Measured (one MI355X, among other passes): MatMulBnb4 NF4, 250 x 4096 x 11008,
// blocks of 64: 664 -> 63 us (the GEMV went over the weights once per four rows;
// floor 21 us at the dense fp16 library rate, 43 us for the two terms). int8
// activations, 384 x 4096 x 4096, blocks of 32: 223 -> 40.5 us (the GEMV's lanes
// read every activation code once per column). What bounds it: VALU issue (codebook
// decode, scaling of the block sums, staging) and the matrix cores, which two waves
// per SIMD overlap only in part. Counters over the kernel: NF4, 172 workgroups, on
// their CUs VALU issue 56 % and MFMA 38 % of the cycles; int8, 256 workgroups, 49 and 12 %.
#pragma once

#include <atomic>

#include "xrmm_device.h"

namespace xrmm {

int device_cus();

namespace ks {

enum Kind { KS_BNB = 0, KS_Q8 = 1 };

struct Args {
  const void* A;      // KS_BNB: float16 [M][K]; KS_Q8: int8 codes [M][K], 8-groups as k0 k2 k4 k6 k1 k3 k5 k7
  const float* as;    // KS_Q8: [M][K / 128] activation scales
  const uint8_t* B;   // [N][K / 2] codes
  const void* S;      // [N][kb] block scales
  const uint8_t* Z;   // KS_Q8: packed zero points [N][zrow], or null (8)
  const void* bias;   // [N] or null
  void* Y;            // [M][N]
  float unscale;      // KS_BNB: one over the codebook's factor
  uint32_t tbl[16];   // KS_BNB: the codebook as four byte planes of 16: hi low, hi high, lo low, lo high byte
  int M, K, N, kb, bs, lbs, zrow, nrt;  // bs = 2^lbs
};

constexpr int KSTEP = 64, LD = KSTEP + 8, THREADS = 512;

template <int IM, int KG>
constexpr size_t lds_bytes() {
  return 2 * static_cast<size_t>(KG) * 32 * IM * LD * sizeof(_Float16);
}

// Scale blocks per flush, BKM: 2 = every 32 codes, 4 = every 64, 8 = blocks of
// 128 or more (scaled where a block or the group's range ends).
// VEC: K is a multiple of 128 (a pair of steps' scales load as one vector); ZP:
// KS_Q8 with packed zero points.
template <typename T, int KIND, int IM, int KG, int BKM, bool VEC, bool ZP>
__global__ __launch_bounds__(THREADS, 2) void k_gemm_ks(Args a) {
  constexpr int NW = 8 / KG;        // waves of a group (32 columns each)
  constexpr int GT = 64 * NW;       // threads of a group
  constexpr int RT = 32 * IM, CT = 32 * NW;
  constexpr int AP = RT * 8 / GT;   // eight-value activation pieces a thread stages per step
  static_assert(AP * GT == RT * 8, "whole pieces per thread");
  constexpr int STAGE = RT * LD;    // halfs of one group's stage
  constexpr int NB = BKM == 2 ? 2 : 1;  // blocks of a step
  static_assert(KIND == KS_BNB || VEC, "KS_Q8: K is a multiple of 128");
  constexpr uint32_t OOB = 0x80000000u;
  constexpr bool Q8 = KIND == KS_Q8;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ __align__(16) float s_as[Q8 ? 2 : 1][Q8 ? KG : 1][Q8 ? RT : 1];  // activation scales of a step
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave / NW, wn = wave % NW, gt = tid - kg * GT;
  const int half = lane >> 5;
  f16* lds = reinterpret_cast<f16*>(smem) + kg * 2 * STAGE;
  // the row tiles of a column tile run side by side on one XCD (its L2 then
  // reads the weights once)
  const uint32_t bid = xcd_slot(blockIdx.x, gridDim.x);
  const int m0 = static_cast<int>(bid % static_cast<uint32_t>(a.nrt)) * RT;
  const int n0 = static_cast<int>(bid / static_cast<uint32_t>(a.nrt)) * CT;
  const int K = a.K, N = a.N;
  // K steps [k0, k0 + n) of this group; every group runs `per` steps (a step
  // past its range stages zeros), even counts so that 128 activations with one
  // scale stay in one group
  const int all = (K + KSTEP - 1) / KSTEP;
  const int per = ((all + KG - 1) / KG + 1) & ~1;
  const int k0 = kg * per, n = all - k0 < per ? all - k0 : per;

  // ---- activations: thread gt stages pieces gt + GT i (row p / 8, values 8 (p % 8) .. + 7)
  const rsrc_t rA = mk_rsrc(a.A, static_cast<uint32_t>(a.M) * static_cast<uint32_t>(K) * (Q8 ? 1u : 2u));
  const int grp = gt & 7;
  struct ARegs {
    u32x4 h[Q8 ? 1 : AP];
    u32x2 q[Q8 ? AP : 1];
    float as;
  };
  // Every load goes through a buffer resource with a 32-bit offset, past the
  // bound (which reads zero) where there is nothing to load, and stays raw bits
  // until its use: no branch and no conversion beside a load, so nothing waits
  // for it early.
  constexpr uint32_t ES = Q8 ? 1u : 2u;  // bytes of an activation
  uint32_t aoff[AP];
#pragma unroll
  for (int i = 0; i < AP; ++i) {
    const int m = m0 + (gt >> 3) + (GT / 8) * i;
    aoff[i] = m < a.M ? (static_cast<uint32_t>(m) * static_cast<uint32_t>(K) + static_cast<uint32_t>(grp) * 8u) * ES : OOB;
  }
  const uint32_t nas = static_cast<uint32_t>(K) / 128u;
  const rsrc_t rAs = mk_rsrc(Q8 ? static_cast<const void*>(a.as) : a.A, Q8 ? static_cast<uint32_t>(a.M) * nas * 4u : 0u);
  const uint32_t asoff = gt < RT && m0 + gt < a.M ? static_cast<uint32_t>(m0 + gt) * nas * 4u : OOB;
  // (the bound is set in the sum: set in the offset, a sum past 2^31 would wrap to the
  // first rows)
  auto aload = [&](ARegs& r, int s) {
    const uint32_t k = static_cast<uint32_t>(k0 + s) * KSTEP;
    const uint32_t past = s < n && k + static_cast<uint32_t>(grp) * 8u < static_cast<uint32_t>(K) ? 0u : OOB;  // K % 32 == 0: whole pieces
#pragma unroll
    for (int i = 0; i < AP; ++i) {
      if constexpr (Q8) r.q[i] = bld8(rA, (aoff[i] + k * ES) | past, 0);
      else r.h[i] = bld16(rA, (aoff[i] + k * ES) | past, 0);
    }
    if constexpr (Q8) r.as = __builtin_bit_cast(float, bld_u32(rAs, (asoff | (s < n ? 0u : OOB)) + k / 128u * 4u, 0));
  };
  auto astore = [&](const ARegs& r, int stage) {
    f16* A = lds + stage * STAGE;
#pragma unroll
    for (int i = 0; i < AP; ++i) {
      const int row = (gt >> 3) + (GT / 8) * i;
      u32x4 p;
      if constexpr (Q8) {
        // codes + 128 under the exponent of 1024, minus 1152: exact. Bytes
        // k0 k2 k4 k6 | k1 k3 k5 k7 to the weights' order 0 4 1 5 2 6 3 7
        const f16x2 m1152 = {static_cast<f16>(-1152.f), static_cast<f16>(-1152.f)};
        const uint32_t e = r.q[i].x ^ 0x80808080u, o = r.q[i].y ^ 0x80808080u, magic = 0x64646464u;
        p.x = as_u32(as_h2(__builtin_amdgcn_perm(magic, e, 0x04020400u)) + m1152);
        p.y = as_u32(as_h2(__builtin_amdgcn_perm(magic, o, 0x04020400u)) + m1152);
        p.z = as_u32(as_h2(__builtin_amdgcn_perm(magic, e, 0x04030401u)) + m1152);
        p.w = as_u32(as_h2(__builtin_amdgcn_perm(magic, o, 0x04030401u)) + m1152);
      } else {
        // the codebook's order 0 2 4 6 1 3 5 7
        const u32x4 w = r.h[i];
        p.x = __builtin_amdgcn_perm(w.y, w.x, 0x05040100u);
        p.y = __builtin_amdgcn_perm(w.w, w.z, 0x05040100u);
        p.z = __builtin_amdgcn_perm(w.y, w.x, 0x07060302u);
        p.w = __builtin_amdgcn_perm(w.w, w.z, 0x07060302u);
      }
      *reinterpret_cast<u32x4*>(A + row * LD + grp * 8) = p;
    }
    if constexpr (Q8) {
      if (gt < RT) s_as[stage][kg][gt] = r.as;
    }
  };

  // ---- weights: lane (c, half) holds column c's codes of a step. Blocks of
  // 64 and more: half h takes codes 32 h .. + 31 (MFMA kk: + 8 kk). Blocks of
  // 32: codes 16 h .. + 15 of each 32 (MFMA kk = 2 c + q: + 32 c + 8 q), so an
  // MFMA stays inside one block.
  const int col0 = n0 + wn * 32 + (lane & 31), col = col0 < N ? col0 : N - 1;
  const uint32_t rowb = static_cast<uint32_t>(K / 2);
  const rsrc_t rB = mk_rsrc(a.B, static_cast<uint32_t>(N) * rowb);
  // A pair of steps (128 codes, 64 bytes a column) is loaded at once, four lanes
  // side by side on a column: the address unit handles one line per column and
  // instruction, and 16 columns x 64 bytes take half of what 32 x 32 bytes do
  // (with each lane on its own column, and the scales loaded per step, it was the
  // address unit that set the time). Row swaps hand each lane its column's codes.
  uint32_t boff[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int c = n0 + wn * 32 + 16 * j + (lane & 15);
    boff[j] = static_cast<uint32_t>(c < N ? c : N - 1) * rowb + 16u * static_cast<uint32_t>(lane >> 4);
  }
  constexpr int SN = BKM == 2 ? 4 : BKM == 4 ? 2 : 1;  // scales of a pair
  struct WRegs {
    u32x4 w[2];
    uint32_t s[SN], z;  // raw scale bits (VEC: packed), the zero points' bytes
  };
  const rsrc_t rS = mk_rsrc(a.S, (static_cast<uint32_t>(N) * static_cast<uint32_t>(a.kb) * static_cast<uint32_t>(sizeof(T)) + 3u) & ~3u);
  const rsrc_t rZ = mk_rsrc(ZP ? a.Z : a.B, ZP ? (static_cast<uint32_t>(N) * static_cast<uint32_t>(a.zrow) + 3u) & ~3u : 0u);
  const uint32_t soff = static_cast<uint32_t>(col) * static_cast<uint32_t>(a.kb) * static_cast<uint32_t>(sizeof(T));
  const uint32_t zoff = static_cast<uint32_t>(col) * static_cast<uint32_t>(a.zrow);
  auto wload = [&](WRegs& r, int s) {  // steps s, s + 1 (s even)
    const uint32_t kbyte = static_cast<uint32_t>(k0 + s) * (KSTEP / 2);
    const uint32_t in = s < n ? 0u : OOB;
    const uint32_t past = kbyte + 16u * static_cast<uint32_t>(lane >> 4) < rowb ? in : OOB;  // the row may end inside the pair
#pragma unroll
    for (int j = 0; j < 2; ++j) r.w[j] = bld16(rB, (boff[j] | past) + kbyte, 0);
    const uint32_t b = BKM == 2 ? static_cast<uint32_t>(k0 + s) * 2u : BKM == 4 ? static_cast<uint32_t>(k0 + s)
                                                                      : (static_cast<uint32_t>(k0 + s) * KSTEP) >> a.lbs;
    const uint32_t so = (soff | in) + b * static_cast<uint32_t>(sizeof(T));
    if constexpr (VEC) {
      constexpr int bytes = SN * static_cast<int>(sizeof(T));
      if constexpr (bytes == 16) {
        const u32x4 v = bld16(rS, so, 0);
        r.s[0] = v.x, r.s[1] = v.y, r.s[2] = v.z, r.s[3] = v.w;
      } else if constexpr (bytes == 8) {
        const u32x2 v = bld8(rS, so, 0);
        r.s[0] = v.x, r.s[1] = v.y;
      } else if constexpr (bytes == 4) {
        r.s[0] = bld_u32(rS, so, 0);
      } else {
        r.s[0] = bld_u16(rS, so, 0);
      }
    } else {
#pragma unroll
      for (int f = 0; f < SN; ++f) {  // past the row: zero
        const uint32_t e = BKM == 8 || b + f < static_cast<uint32_t>(a.kb) ? 0u : OOB;
        r.s[f] = bld_u16(rS, (so | e) + 2u * f, 0);
      }
    }
    if constexpr (ZP) {  // two bytes of four blocks' zero points, or the byte of one or two
      if constexpr (BKM == 2) r.z = bld_u16(rZ, (zoff | in) + (b >> 1), 0);
      else r.z = bld_u8(rZ, (zoff | in) + (b >> 1), 0);
    }
  };
  // scale and zero point of block f of step t (0, 1) of the pair
  auto scale_of = [&](const WRegs& r, int t, int f) {
    const int i = BKM == 2 ? 2 * t + f : BKM == 4 ? t : 0;
    float v;
    if constexpr (sizeof(T) == 4) v = __builtin_bit_cast(float, r.s[i]);
    else if constexpr (VEC && SN > 1) v = static_cast<float>(__builtin_bit_cast(f16, static_cast<uint16_t>(r.s[i >> 1] >> (16 * (i & 1)))));
    else v = static_cast<float>(__builtin_bit_cast(f16, static_cast<uint16_t>(r.s[i])));
    return Q8 ? v : v * a.unscale;
  };
  auto zero_of = [&](const WRegs& r, int s, int t, int f) -> uint32_t {
    if constexpr (!ZP) return 8u;
    const int i = BKM == 2 ? 2 * t + f : BKM == 4 ? t : 0;
    if constexpr (BKM == 8) return (r.z >> (4u * (((static_cast<uint32_t>(k0 + s) * KSTEP) >> a.lbs) & 1u))) & 15u;
    return (r.z >> (4 * i)) & 15u;
  };
  // Lane (row r = lane / 16, c = lane % 16) loaded w[j] = column 16 j + c, codes
  // 32 r .. + 31. Step t wants column lane % 32, codes 64 t + 32 (lane / 32) .. + 31.
  // Blocks of 32: then each step's two blocks swap halves (see above).
  auto spread = [&](const WRegs& r, uint32_t (&w)[2][4]) {
    const u32x4 x = r.w[0], y = r.w[1];
    const uint32_t xv[4] = {x.x, x.y, x.z, x.w}, yv[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const auto p = __builtin_amdgcn_permlane16_swap(xv[d], yv[d], false, false);
      const auto q = __builtin_amdgcn_permlane32_swap(p[0], p[1], false, false);
      w[0][d] = q[0];
      w[1][d] = q[1];
    }
    if constexpr (BKM == 2) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const auto p = __builtin_amdgcn_permlane32_swap(w[t][0], w[t][2], false, false);
        const auto q = __builtin_amdgcn_permlane32_swap(w[t][1], w[t][3], false, false);
        w[t][0] = p[0], w[t][1] = q[0], w[t][2] = p[1], w[t][3] = q[1];
      }
    }
  };

  // ---- decode of eight codes
  uint32_t tb[Q8 ? 1 : 16];
  if constexpr (!Q8) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      tb[i] = a.tbl[i];
      if ((i & 1) == 0) asm volatile("" : "+v"(tb[i]));  // v_perm_b32 takes one scalar operand: half the table in vector registers
    }
  }
  // bytes looked up for four codes: sel their low three bits, m 0xFF where bit 3 is set
  auto look = [&](int plane, uint32_t sel, uint32_t m) {
    const uint32_t l = __builtin_amdgcn_perm(tb[4 * plane + 1], tb[4 * plane], sel);
    const uint32_t h = __builtin_amdgcn_perm(tb[4 * plane + 3], tb[4 * plane + 2], sel);
    return (h & m) | (l & ~m);
  };
  const f16x2 inv16 = {static_cast<f16>(0.0625f), static_cast<f16>(0.0625f)};
  auto dq_bnb = [&](uint32_t x, f16x8& hi, f16x8& lo) {
    // low nibbles: odd values, high nibbles: even ones. Selectors 8 .. 11 of
    // v_perm_b32 spread the sign bits of bytes 1, 3, 5, 7 of its operands.
    const uint32_t sl = x & 0x07070707u, sh = (x >> 4) & 0x07070707u;
    const uint32_t ml = __builtin_amdgcn_perm(x << 12, x << 4, 0x090B080Au);
    const uint32_t mh = __builtin_amdgcn_perm(x << 8, x, 0x090B080Au);
    u32x4 h, l;
    const uint32_t a0 = look(0, sh, mh), a1 = look(1, sh, mh), b0 = look(0, sl, ml), b1 = look(1, sl, ml);
    h.x = __builtin_amdgcn_perm(a1, a0, 0x05010400u);
    h.y = __builtin_amdgcn_perm(a1, a0, 0x07030602u);
    h.z = __builtin_amdgcn_perm(b1, b0, 0x05010400u);
    h.w = __builtin_amdgcn_perm(b1, b0, 0x07030602u);
    const uint32_t c0 = look(2, sh, mh), c1 = look(3, sh, mh), d0 = look(2, sl, ml), d1 = look(3, sl, ml);
    l.x = __builtin_amdgcn_perm(c1, c0, 0x05010400u);
    l.y = __builtin_amdgcn_perm(c1, c0, 0x07030602u);
    l.z = __builtin_amdgcn_perm(d1, d0, 0x05010400u);
    l.w = __builtin_amdgcn_perm(d1, d0, 0x07030602u);
    hi = __builtin_bit_cast(f16x8, h);
    lo = __builtin_bit_cast(f16x8, l);
  };
  auto dq_int = [&](uint32_t x, f16x2 n0v, f16x2 n1v) {  // pair order 0 4 1 5 2 6 3 7
    const uint32_t magic = 0x64006400u, x8 = x >> 8;
    const f16x2 d0 = as_h2(and_or(x, 0x000F000Fu, magic)) + n0v;
    const f16x2 d1 = __builtin_elementwise_fma(as_h2(and_or(x, 0x00F000F0u, magic)), inv16, n1v);
    const f16x2 d2 = as_h2(and_or(x8, 0x000F000Fu, magic)) + n0v;
    const f16x2 d3 = __builtin_elementwise_fma(as_h2(and_or(x8, 0x00F000F0u, magic)), inv16, n1v);
    return f16x8{d0[0], d0[1], d1[0], d1[1], d2[0], d2[1], d3[0], d3[1]};
  };

  // ---- sums: a block's (acc), KS_Q8 with blocks below 128 the scaled sums
  // over the activations that share a scale (tac), the output's (yacc)
  constexpr bool T2 = Q8 && BKM != 8;
  const f32x16 zero16 = {};
  f32x16 acc[IM];
  float yacc[IM][16], tac[T2 ? IM : 1][16];
#pragma unroll
  for (int i = 0; i < IM; ++i) {
    acc[i] = zero16;
#pragma unroll
    for (int q = 0; q < 16; ++q) yacc[i][q] = tac[T2 ? i : 0][q] = 0.f;
  }
  // rows 8 (q / 4) + 4 (lane / 32) + q % 4 of row tile i: their activation scales
  auto row_scales = [&](int stage, int i, float (&v)[16]) {
    const float* p = &s_as[Q8 ? stage : 0][Q8 ? kg : 0][Q8 ? 32 * i + 4 * half : 0];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 t = *reinterpret_cast<const f32x4*>(p + 8 * g);
      v[4 * g] = t.x, v[4 * g + 1] = t.y, v[4 * g + 2] = t.z, v[4 * g + 3] = t.w;
    }
  };
  // (kept in place by the empty asm and the scheduling barriers: sunk among the
  // next block's MFMAs it would hold two copies of the sums, and spill)
  auto flush = [&](float s, int stage, bool first128 = false) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < IM; ++i) {
      if constexpr (Q8 && BKM == 8) {
        float v[16];
        row_scales(stage, i, v);
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          yacc[i][q] = __builtin_fmaf(v[q], s * acc[i][q], yacc[i][q]);
          asm volatile("" : "+v"(yacc[i][q]));
        }
      } else {
        float (&t)[16] = T2 ? tac[T2 ? i : 0] : yacc[i];
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          t[q] = T2 && first128 ? s * acc[i][q] : __builtin_fmaf(s, acc[i][q], t[q]);
          asm volatile("" : "+v"(t[q]));
        }
      }
      if constexpr (BKM == 8) acc[i] = zero16;
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto flush128 = [&](int stage) {
    if constexpr (T2) {
#pragma unroll
      for (int i = 0; i < IM; ++i) {
        float v[16];
        row_scales(stage, i, v);
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          yacc[i][q] = __builtin_fmaf(v[q], tac[i][q], yacc[i][q]);
          asm volatile("" : "+v"(yacc[i][q]));
        }
      }
    }
  };
  // blocks of 128 and more end where (step + 1) % bsteps == 0; with activation
  // scales every 128
  const int bsteps = BKM == 8 ? (Q8 ? 2 : a.bs / KSTEP) : 1;

  auto compute = [&](const WRegs& w, const uint32_t (&wc)[4], int s, int t) {  // t = s % 2, also the stage
    const int stage = t;
    const f16* A = lds + stage * STAGE + (lane & 31) * LD;
    f16x2 nz0[NB], nz1[NB];
    if constexpr (Q8) {
#pragma unroll
      for (int f = 0; f < NB; ++f) {
        const uint32_t z = zero_of(w, s, t, f);
        const f16 z0 = static_cast<f16>(-1024.f - static_cast<float>(z)), z1 = static_cast<f16>(-64.f - static_cast<float>(z));
        nz0[f] = f16x2{z0, z0};
        nz1[f] = f16x2{z1, z1};
      }
    }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int ko = BKM == 2 ? 32 * (kk >> 1) + 16 * half + 8 * (kk & 1) : 32 * half + 8 * kk;
      f16x8 fa[IM];
#pragma unroll
      for (int i = 0; i < IM; ++i) fa[i] = *reinterpret_cast<const f16x8*>(A + i * 32 * LD + ko);
      const bool first = BKM == 2 ? (kk & 1) == 0 : BKM == 4 ? kk == 0 : false;
      if constexpr (Q8) {
        const f16x8 fb = dq_int(wc[kk], nz0[NB == 2 ? kk >> 1 : 0], nz1[NB == 2 ? kk >> 1 : 0]);
#pragma unroll
        for (int i = 0; i < IM; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[i], fb, first ? zero16 : acc[i], 0, 0, 0);
      } else {
        f16x8 hi, lo;
        dq_bnb(wc[kk], hi, lo);
#pragma unroll
        for (int i = 0; i < IM; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[i], hi, first ? zero16 : acc[i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < IM; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[i], lo, acc[i], 0, 0, 0);
      }
      if constexpr (BKM == 2) {
        if (kk & 1) flush(scale_of(w, t, kk >> 1), stage, t == 0 && kk == 1);
      }
    }
    if constexpr (BKM == 4) flush(scale_of(w, t, 0), stage, t == 0);
    if constexpr (BKM == 8) {
      if ((k0 + s + 1) % bsteps == 0 || s + 1 >= n) flush(scale_of(w, t, 0), stage);
    }
    if constexpr (T2) {
      if (t == 1) flush128(stage);
    }
  };

  // Step s on stage s % 2: `an` holds step s + 1's activations (to the other
  // stage at the end of the step), step s + 2's go to `af`; a pair's codes and scales
  // are loaded a pair ahead. No step has a branch: past the range, loads read zeros.
  auto step = [&](int s, int t, ARegs& an, ARegs& af, const WRegs& w, const uint32_t (&wc)[4]) {
    aload(af, s + 2);
    __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the matrix work
    compute(w, wc, s, t);
    astore(an, t ^ 1);
    __syncthreads();
  };
  auto pair = [&](int s, WRegs& w, WRegs& wn, ARegs& a0, ARegs& a1) {
    wload(wn, s + 2);
    uint32_t wc[2][4];
    spread(w, wc);
    step(s, 0, a1, a0, w, wc[0]);
    step(s + 1, 1, a0, a1, w, wc[1]);
  };
  ARegs a0, a1;
  WRegs w0, w1;
  wload(w0, 0);
  aload(a0, 0);
  aload(a1, 1);
  astore(a0, 0);
  __syncthreads();
  int s = 0;  // per is even
  for (; s + 2 < per; s += 4) {
    pair(s, w0, w1, a0, a1);
    pair(s + 2, w1, w0, a0, a1);
  }
  if (s < per) pair(s, w0, w1, a0, a1);

  // ---- the groups' sums, added in group order through LDS (the stages are free)
  float* red = reinterpret_cast<float*>(smem);
  static_assert((KG - 1) * NW * IM * 16 * 64 * sizeof(float) <= lds_bytes<IM, KG>(), "the sums fit the stages");
  if (kg > 0) {
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
      for (int q = 0; q < 16; ++q) red[((((kg - 1) * NW + wn) * IM + i) * 16 + q) * 64 + lane] = yacc[i][q];
  }
  __syncthreads();
  if (kg > 0) return;
  const float b = a.bias && col0 < N ? static_cast<float>(static_cast<const T*>(a.bias)[col0]) : 0.f;
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      float v = yacc[i][q];
#pragma unroll
      for (int g = 1; g < KG; ++g) v += red[((((g - 1) * NW + wn) * IM + i) * 16 + q) * 64 + lane];
      // lane holds D[8 (q / 4) + 4 (lane / 32) + q % 4][lane % 32]
      const int m = m0 + 32 * i + 8 * (q >> 2) + 4 * half + (q & 3);
      if (m < a.M && col0 < N) static_cast<T*>(a.Y)[static_cast<int64_t>(m) * N + col0] = static_cast<T>(v + b);
    }
}

// Row tile (32 im rows) and K groups of a launch.
struct Plan {
  int im, kg, nrt;
  int64_t grid;
};

// The cheapest of the tile shapes: rounds of workgroups on the CUs (two resident
// where 32 rows need half the registers, a step then taking 1.6 times as long, else
// one) x (a group's steps, and three
// steps' worth of start and end) x a step's time, which over the shapes fits
// 1 + im / 4 + 0.06 im kg (measured in units of 0.77 us, K = 4096: im, kg = 4, 2
// 1.9 us, 3, 2 1.6, 2, 2 1.2-1.3, 3, 4 2.1, 2, 4 1.55, 4, 4 2.6 (spills, not built)).
// 250 rows, N = 11008: 4, 2 in one round 63 us; 2, 4 75; 2, 2 84; 3, 4 100.
inline Plan plan(int64_t M, int64_t N, int64_t K, int cus, int most) {
  const int64_t all = (K + KSTEP - 1) / KSTEP;
  Plan best{};
  double best_t = 0.0;
  for (int im = 1; im <= most; ++im)
    for (int kg = 2; kg <= 8; kg *= 2) {
      if (im * kg > 12 && im != 2) continue;  // LDS, registers
      const int64_t nrt = (M + 32 * im - 1) / (32 * im), ct = 256 / kg, grid = nrt * ((N + ct - 1) / ct);
      const bool two = im == 1 && grid > cus;
      const int64_t cap = int64_t(cus) * (two ? 2 : 1), per = ((all + kg - 1) / kg + 1) / 2 * 2;
      const double t = static_cast<double>((grid + cap - 1) / cap * (per + 3)) * (1.0 + 0.25 * im + 0.06 * im * kg) * (two ? 1.6 : 1.0);
      if (best.kg == 0 || t < best_t) {
        best_t = t;
        best = Plan{im, kg, static_cast<int>(nrt), grid};
      }
    }
  return best;
}

template <typename T, int KIND, int IM, int KG, int BKM, bool VEC, bool ZP>
hipError_t launch_one(const Args& a, int64_t grid, hipStream_t st) {
  auto kern = k_gemm_ks<T, KIND, IM, KG, BKM, VEC, ZP>;
  constexpr size_t lds = lds_bytes<IM, KG>();
  if constexpr (lds > 64 * 1024) {
    static std::atomic<int> done[kMaxDevices];  // per instantiation and device
    if (hipError_t e = raise_lds_cap(reinterpret_cast<const void*>(kern), static_cast<int>(lds), done); e != hipSuccess)
      return e;
  }
  hipLaunchKernelGGL(kern, dim3(static_cast<uint32_t>(grid)), dim3(THREADS), lds, st, a);
  return hipGetLastError();
}

template <typename T, int KIND, int IM, int KG, bool VEC, bool ZP>
hipError_t launch_bkm(const Args& a, int64_t grid, hipStream_t st) {
  if (a.bs == 32) return launch_one<T, KIND, IM, KG, 2, VEC, ZP>(a, grid, st);
  if (a.bs == 64) return launch_one<T, KIND, IM, KG, 4, VEC, ZP>(a, grid, st);
  if constexpr (VEC) return launch_one<T, KIND, IM, KG, 8, VEC, ZP>(a, grid, st);
  return hipErrorInvalidValue;  // blocks of 128 and more divide K, which is then a multiple of 128
}

template <typename T, int KIND, int IM, int KG>
hipError_t launch_var(const Args& a, int64_t grid, hipStream_t st) {
  if constexpr (KIND == KS_Q8)
    return a.Z ? launch_bkm<T, KIND, IM, KG, true, true>(a, grid, st) : launch_bkm<T, KIND, IM, KG, true, false>(a, grid, st);
  else
    return a.K % 128 == 0 ? launch_bkm<T, KIND, IM, KG, true, false>(a, grid, st) : launch_bkm<T, KIND, IM, KG, false, false>(a, grid, st);
}

template <typename T, int KIND>
hipError_t launch_ks(const Args& a, const Plan& p, hipStream_t st) {
#define XRMM_KS(IM_, KG_) \
  if (p.im == IM_ && p.kg == KG_) return launch_var<T, KIND, IM_, KG_>(a, p.grid, st)
  XRMM_KS(1, 2);
  XRMM_KS(1, 4);
  XRMM_KS(1, 8);
  XRMM_KS(2, 2);
  XRMM_KS(2, 4);
  XRMM_KS(2, 8);
  XRMM_KS(3, 2);
  XRMM_KS(3, 4);
  if constexpr (KIND == KS_BNB) XRMM_KS(4, 2);
#undef XRMM_KS
  return hipErrorInvalidValue;
}

}  // namespace ks
}  // namespace xrmm
