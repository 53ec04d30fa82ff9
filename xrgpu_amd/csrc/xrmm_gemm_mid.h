// MatMulNBitsQkv / MatMulNBitsMlp prompts too short for the 256 x 256 pipeline
// (xrmm_gemm.h) to fill the chip: 128-row tiles on the same K loop (fp16
// activations already normalised, 4-bit weights dequantised on their way into
// LDS, v_mfma_f32_32x32x16_f16, float32 sums).
//
// Tiles. Narrow: 128 rows x 128 staged columns, two groups of 8 waves (4 x 2 of 32 x
// 64) that each take half of K on LDS stages of their own and meet in LDS at the end
// (one group alone leaves the CU waiting: 46 against 41 us at Qkv 65 x 4096 x 6144).
// Wide: 128 x 256, 8 waves (2 x 4 of 64 x 64), half the fragment reads per MFMA.
// Mlp interleaves the gate and up projections by 32 staged columns, so each wave's
// two MFMA column tiles are the two projections of the same outputs.
//
// Pipeline: double-buffered LDS, one barrier per K step of 64, global loads two
// steps ahead through buffer resources (no branch beside a load), the next step
// staged in parts between the MFMAs, fragments of the next K slice read before the
// current slice's MFMAs. The 128 x 128 kernel it replaces where the rows are
// normalised beforehand (k_gemm_fused: one stage, two barriers, loads in branches)
// took 4 us per K step. Measured, prologue included: Mlp 333 x 2048 x 5632 129 -> 40
// us, 65 x 4096 x 4096 120 -> 40, Qkv 128 x 4096 x (4096 + 2 x 4096) 111 -> 44, 200 x
// 14336 x (512 + 2 x 64) 369 -> 149. What bounds it at Mlp 333 x 2048 x 5632: the grid,
// 132 wide workgroups on 256 CUs (264 narrow ones would take two rounds: 50 us); on those
// CUs, by counters over the kernel, VALU issue 43 %, MFMA 29 % and LDS 26 % of the
// cycles, which two waves per SIMD overlap only in part.
#pragma once
#include <atomic>

#include "xrmm_device.h"

namespace xrmm {

int device_cus();

namespace mid {

constexpr int BM = 128, BK = 64, LD = BK + 8, THREADS = 512;
constexpr int cols(bool wide) { return wide ? 256 : 128; }  // staged columns of a tile
constexpr int kgroups(bool wide) { return wide ? 1 : 2; }
constexpr size_t lds_bytes(bool wide) { return 2 * static_cast<size_t>(BM + cols(wide)) * LD * sizeof(_Float16); }

// Column tiles of an operator's grid (outputs per tile: Qkv the staged columns,
// Mlp half of them).
inline int64_t col_tiles(const Launch& L, bool wide) {
  const int64_t w = cols(wide);
  if (L.op == OP_MLP) return (L.p[0].N + w / 2 - 1) / (w / 2);
  int64_t n = 0;
  for (int i = 0; i < 3; ++i) n += (L.p[i].N + w - 1) / w;
  return n;
}

template <int ZPK, int OPK, bool WIDE>
__global__ __launch_bounds__(THREADS * kgroups(WIDE), WIDE ? 2 : 4) void k_gemm_mid(Launch L, uint32_t mt) {
  constexpr int KG = kgroups(WIDE);
  constexpr bool MLP = OPK == OP_MLP;
  constexpr int BN = cols(WIDE), TM = WIDE ? 2 : 1, TN = 2, WN = WIDE ? 4 : 2;
  constexpr int STAGE = (BM + BN) * LD;
  constexpr int DP = BN / 64;  // weight dwords (8 codes) a thread stages per step: 4 (16 bytes) or 2
  constexpr uint32_t OOB = 0x80000000u;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x & (THREADS - 1), lane = tid & 63;  // inside the K group
  const int kg = KG == 2 ? __builtin_amdgcn_readfirstlane(threadIdx.x / THREADS) : 0;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  f16* lds = reinterpret_cast<f16*>(smem) + kg * 2 * STAGE;
  const int wm = wave / WN, wn = wave % WN;

  // this tile: the row tiles of a column tile run side by side on one XCD
  const uint32_t b = xcd_slot(blockIdx.x, gridDim.x);
  const int m0 = static_cast<int>(b % mt) * BM;
  int ct = static_cast<int>(b / mt), pi = 0;
  if constexpr (!MLP) {
    const int t0 = static_cast<int>((L.p[0].N + BN - 1) / BN), t1 = static_cast<int>((L.p[1].N + BN - 1) / BN);
    pi = ct < t0 ? 0 : ct < t0 + t1 ? 1 : 2;
    ct -= pi == 0 ? 0 : pi == 1 ? t0 : t0 + t1;
  }
  const int n0 = ct * (MLP ? BN / 2 : BN);
  const int M = static_cast<int>(L.M), K = static_cast<int>(L.K);
  const uint32_t rowb = static_cast<uint32_t>(L.kb * L.block_size / 2), kb = static_cast<uint32_t>(L.kb);
  // K steps of a group: [kg ksteps, + ksteps) of the row's (loads past its end read zeros)
  const int ksteps = (static_cast<int>((rowb + BK / 2 - 1) / (BK / 2)) + KG - 1) / KG;
  const int ks0 = kg * ksteps;

  // ---- activations: pieces tid + 512 i of the 128 x 64 tile
  const rsrc_t rA = mk_rsrc(L.A, static_cast<uint32_t>(M) * static_cast<uint32_t>(K) * 2u);
  const int grp = tid & 7;
  uint32_t aoff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = m0 + (tid >> 3) + 64 * i;
    aoff[i] = m < M ? (static_cast<uint32_t>(m) * static_cast<uint32_t>(K) + static_cast<uint32_t>(grp) * 8u) * 2u : OOB;
  }
  // ---- weights: 8 DP codes of staged column bc
  constexpr int TPC = 8 / DP;  // threads per staged column
  const int bc = tid / TPC, bq = tid % TPC;
  // Mlp: staged columns 32 g .. are the gate (g even) or up projection of outputs
  // n0 + 32 (g / 2) ..; a wave stages columns of one projection
  const int bpi = MLP ? __builtin_amdgcn_readfirstlane((bc >> 5) & 1) : pi;
  const Proj& P = L.p[bpi];
  const int N = static_cast<int>(P.N);
  const int bn = MLP ? n0 + 32 * (bc >> 6) + (bc & 31) : n0 + bc;
  const uint32_t zrow = ZPK == ZP_PACKED ? static_cast<uint32_t>(L.zrow) : kb * (L.zp_dtype == DT_F32 ? 4u : 2u);
  const rsrc_t rB = mk_rsrc(P.B, static_cast<uint32_t>(N) * rowb);
  // bounds rounded to 16 bytes: the range check zeroes a whole dword straddling
  // the bound, and 16-byte aligned tensors keep the rounded bound in their last block
  const rsrc_t rS = mk_rsrc(P.scales, (static_cast<uint32_t>(N) * kb * 2u + 15u) & ~15u);
  const rsrc_t rZ = mk_rsrc(P.zp ? P.zp : P.scales, (static_cast<uint32_t>(N) * zrow + 15u) & ~15u);
  const uint32_t none = bn < N ? 0u : OOB;
  const uint32_t bcol = static_cast<uint32_t>(bn) * rowb + static_cast<uint32_t>(bq * DP * 4);
  const uint32_t scol = static_cast<uint32_t>(bn) * kb * 2u, zcol = static_cast<uint32_t>(bn) * zrow;

  struct Regs {
    u32x4 a[2];
    uint32_t w[DP];
    uint32_t s, z;  // raw scale and zero-point bits
  };
  auto gload = [&](Regs& r, int ks) {
    const uint32_t k = static_cast<uint32_t>(ks0 + ks) * BK;
    const uint32_t apast = k + static_cast<uint32_t>(grp) * 8u < static_cast<uint32_t>(K) ? 0u : OOB;  // K % 8 == 0
#pragma unroll
    for (int i = 0; i < 2; ++i) r.a[i] = bld16(rA, (aoff[i] + k * 2u) | apast, 0);
    const uint32_t o = k / 2u;
    const uint32_t past = none | (o + static_cast<uint32_t>(bq * DP * 4) < rowb ? 0u : OOB);
    if constexpr (DP == 4) {
      const u32x4 v = bld16(rB, (bcol + o) | past, 0);
      r.w[0] = v.x, r.w[1] = v.y, r.w[2] = v.z, r.w[3] = v.w;
    } else {
      const u32x2 v = bld8(rB, (bcol + o) | past, 0);
      r.w[0] = v.x, r.w[1] = v.y;
    }
    const uint32_t blk = (k + static_cast<uint32_t>(bq * DP * 8)) >> L.bs_log2;  // blocks of 32 and more: one per thread
    r.s = bld_u16(rS, (scol + blk * 2u) | past, 0);
    r.z = 0u;
    if constexpr (ZPK == ZP_PACKED) r.z = bld_u8(rZ, (zcol + (blk >> 1)) | past, 0);
    else if constexpr (ZPK == ZP_FLOAT)
      r.z = L.zp_dtype == DT_F32 ? bld_u32(rZ, (zcol + blk * 4u) | past, 0) : bld_u16(rZ, (zcol + blk * 2u) | past, 0);
  };
  struct StepMeta {
    Dq c;
    float z, s;
  };
  auto meta = [&](const Regs& r, int ks) {
    StepMeta mt;
    const f16 sc = __builtin_bit_cast(f16, static_cast<uint16_t>(r.s));
    mt.s = static_cast<float>(sc);
    if constexpr (ZPK == ZP_NONE) {
      mt.z = 8.f;
    } else if constexpr (ZPK == ZP_PACKED) {
      const uint32_t blk = (static_cast<uint32_t>(ks0 + ks) * BK + static_cast<uint32_t>(bq * DP * 8)) >> L.bs_log2;
      mt.z = static_cast<float>((r.z >> ((blk & 1u) * 4u)) & 15u);
    } else {
      mt.z = L.zp_dtype == DT_F32 ? __builtin_bit_cast(float, r.z)
                                  : static_cast<float>(__builtin_bit_cast(f16, static_cast<uint16_t>(r.z)));
    }
    if constexpr (ZPK != ZP_FLOAT) mt.c = dq_consts(mt.z, sc);
    return mt;
  };
  // part d (0 .. 3) of writing a step's registers to a stage: weight dword d, and
  // activation piece d
  auto store_part = [&](const Regs& r, const StepMeta& mt, int stage, int d) {
    f16* As = lds + stage * STAGE;
    f16* Bs = As + BM * LD;
    if (d < 2)
      *reinterpret_cast<f16x8*>(As + ((tid >> 3) + 64 * d) * LD + grp * 8) = pair_order(__builtin_bit_cast(f16x8, r.a[d < 2 ? d : 0]));
    const int w = DP == 4 ? d : d - 2;
    if (w >= 0) {
      f16x8 v;
      if constexpr (ZPK == ZP_FLOAT) v = dq8_f32z(r.w[w < 0 ? 0 : w], mt.z, mt.s);
      else v = dq8(r.w[w < 0 ? 0 : w], mt.c);
      *reinterpret_cast<f16x8*>(Bs + bc * LD + bq * DP * 8 + (w < 0 ? 0 : w) * 8) = v;
    }
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  f16x8 fa[2][TM], fb[2][TN];
  auto read_frags = [&](int stage, int kk, int buf) {
    const int ko = kk * 16 + (lane >> 5) * 8;
    const f16* As = lds + stage * STAGE + (wm * 32 * TM + (lane & 31)) * LD + ko;
    const f16* Bs = lds + stage * STAGE + (BM + wn * 32 * TN + (lane & 31)) * LD + ko;
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[buf][i] = *reinterpret_cast<const f16x8*>(As + i * 32 * LD);
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[buf][j] = *reinterpret_cast<const f16x8*>(Bs + j * 32 * LD);
  };
  auto step = [&](int ks, int stage, Regs& nxt, Regs& fill) {
    gload(fill, ks + 2);
    __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the matrix work
    const StepMeta mt = meta(nxt, ks + 1);
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      if (kk + 1 < BK / 16) read_frags(stage, kk + 1, (kk + 1) & 1);
      store_part(nxt, mt, stage ^ 1, kk);
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[kk & 1][i], fb[kk & 1][j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
    read_frags(stage ^ 1, 0, 0);
  };
  Regs r0, r1;
  gload(r0, 0);
  gload(r1, 1);
  {
    const StepMeta mt = meta(r0, 0);
#pragma unroll
    for (int d = 0; d < 4; ++d) store_part(r0, mt, 0, d);
  }
  __syncthreads();
  read_frags(0, 0, 0);
  int ks = 0;
  for (; ks + 1 < ksteps; ks += 2) {
    step(ks, 0, r1, r0);
    step(ks + 1, 1, r0, r1);
  }
  if (ks < ksteps) step(ks, 0, r1, r0);

  // ---- epilogue through LDS: rows of whole 16-byte pieces
  constexpr int OUTW = MLP ? BN / 2 : BN, YLD = OUTW + 8;
  static_assert(BM * YLD * 2 <= static_cast<int>(lds_bytes(WIDE)), "the output tile fits the LDS");
  __syncthreads();
  if constexpr (KG == 2) {
    // group 1's sums to group 0 through LDS (its own stages); it then only keeps
    // the barriers company
    float* red = reinterpret_cast<float*>(reinterpret_cast<f16*>(smem) + 2 * STAGE);
    static_assert(TM * TN * 16 * THREADS * 4 <= static_cast<int>(lds_bytes(WIDE)), "the sums fit a group's stages");
    if (kg == 1) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) red[((i * TN + j) * 16 + e) * THREADS + tid] = acc[i][j][e];
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][j][e] += red[((i * TN + j) * 16 + e) * THREADS + tid];
    }
  }
  lds = reinterpret_cast<f16*>(smem);  // the output tile
  if (kg != 0) {
  } else if constexpr (MLP) {
    const f16* gbias = static_cast<const f16*>(L.p[0].bias);
    const f16* ubias = static_cast<const f16*>(L.p[1].bias);
    const int c = wn * 32 + (lane & 31);
    const float gb = (gbias != nullptr && n0 + c < N) ? static_cast<float>(gbias[n0 + c]) : 0.f;
    const float ub = (ubias != nullptr && n0 + c < N) ? static_cast<float>(ubias[n0 + c]) : 0.f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int r = wm * 32 * TM + i * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
        lds[r * YLD + c] = static_cast<f16>(activate(acc[i][0][e] + gb, L.act) * (acc[i][1][e] + ub));
      }
  } else {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int r = wm * 32 * TM + i * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
          lds[r * YLD + wn * 32 * TN + j * 32 + (lane & 31)] = static_cast<f16>(acc[i][j][e]);
        }
  }
  __syncthreads();
  f16* Y = static_cast<f16*>(L.p[pi].Y);
  constexpr int PPR = OUTW / 8;
  const bool vec = (N & 7) == 0 && (reinterpret_cast<uintptr_t>(Y) & 15u) == 0;
  for (int idx = threadIdx.x; idx < BM * PPR; idx += THREADS * KG) {
    const int r = idx / PPR, p = idx % PPR;
    const int m = m0 + r, n = n0 + 8 * p;
    if (m >= M || n >= N) continue;
    const f16* src = lds + r * YLD + 8 * p;
    f16* dst = Y + static_cast<int64_t>(m) * N + n;
    if (vec) *reinterpret_cast<u32x4*>(dst) = *reinterpret_cast<const u32x4*>(src);
    else
      for (int e = 0; e < 8 && n + e < N; ++e) dst[e] = src[e];
  }
}

template <int ZPK, int OPK, bool WIDE>
inline hipError_t launch_one(const Launch& L, hipStream_t st) {
  auto kern = k_gemm_mid<ZPK, OPK, WIDE>;
  constexpr int KG = kgroups(WIDE);
  constexpr size_t lds = KG * lds_bytes(WIDE);
  static std::atomic<int> done[kMaxDevices];  // per instantiation and device
  if (hipError_t e = raise_lds_cap(reinterpret_cast<const void*>(kern), static_cast<int>(lds), done); e != hipSuccess)
    return e;
  const int64_t mt = (L.M + BM - 1) / BM, tiles = mt * col_tiles(L, WIDE);
  if (tiles > 0x7FFFFFFF) return hipErrorInvalidValue;  // launch limit
  hipLaunchKernelGGL(kern, dim3(static_cast<uint32_t>(tiles)), dim3(THREADS * KG), lds, st, L, static_cast<uint32_t>(mt));
  return hipGetLastError();
}

template <int ZPK, int OPK>
inline hipError_t launch_op(const Launch& L, hipStream_t st) {
  // Narrow tiles while they fit one round of the CUs, else wide ones (fewer fragment
  // reads per MFMA). Narrow against wide: Mlp 128 x 4096 x 14336 (224 / 112 tiles)
  // 50 / 64 us, Qkv 65 x 4096 x (4096 + 2 x 1024) 41 / 64; Mlp 333 x 2048 x 5632
  // (264 / 132) 50 / 40, 256 x 4096 x 11008 (344 / 172) 88 / 70.
  const int cus = device_cus();
  const int64_t narrow = (L.M + BM - 1) / BM * col_tiles(L, false);
  return narrow <= (cus > 0 ? cus : 256) ? launch_one<ZPK, OPK, false>(L, st) : launch_one<ZPK, OPK, true>(L, st);
}

}  // namespace mid

// Blocks of 32 codes and more (a thread's codes then share one scale).
inline bool gemm_mid_ok(const Launch& L) { return L.block_size >= 32 && (L.xs != nullptr || !fused_prologue(L)) && L.residual == nullptr; }

template <int ZPK>
inline hipError_t launch_gemm_mid(const Launch& L, hipStream_t st) {
  return L.op == OP_MLP ? mid::launch_op<ZPK, OP_MLP>(L, st) : mid::launch_op<ZPK, OP_QKV>(L, st);
}

// Entry of one zero-point kind (defined in xrmm_gemm_fused_zp.hip).
template <int ZPK>
hipError_t launch_gemm_mid_for(const Launch& L, hipStream_t st);

}  // namespace xrmm
