// Grouped-expert QMoE for many tokens (included by xrmm_moe.hip): instead of
// one pass over an expert's rows per (token, slot) pair, the pairs routed to
// each expert are gathered into the rows of one GEMM per expert, so every
// expert matrix is read once per 128 (or 64) pairs.
//
// Launches:
//  1. k_moe_prep: per token the routing, the row exponent of x, and x split into
//     its binary16 terms (into yp, which nothing uses before FC2);
//  2. k_moe_group: per-expert pair counts, offsets, the two GEMMs' row-tile offsets and
//     the pair lists (one workgroup; the order of pairs inside a list does not
//     change any result, every GEMM row being independent);
//  3. k_moe_ggemm FC1: rows = an expert's pairs (their tokens' x), columns =
//     its FC1 rows, K = H; the epilogue applies the row scale, the activation
//     (SwiGLU rows 2j / 2j + 1 sit in neighbouring lanes) and writes h[pair],
//     folding each pair's largest |h| into an arrival-order-free atomic max;
//  4. k_moe_hsplit: h into its binary16 terms, in place;
//  5. k_moe_ggemm FC2: rows = the pairs' h, columns = the expert's FC2 rows,
//     K = I, split over a.ks workgroups when the tiles are few; writes each
//     split's yp[pair][split] (row scale applied);
//  6. k_moe_combine: y[t] = sum over slots (ascending expert index) of
//     w * (the slot's splits summed in split order), one fused multiply-add
//     per slot in slot order.
//
// Arithmetic. The codes enter v_mfma_f32_32x32x16_f16 as the exact binary16
// integers code - 8 (no scale), the row scale multiplies the float32 sum. The
// float32 activations are split into two binary16 terms per element: a row
// is first scaled by a power of two that puts its largest finite magnitude
// near 2^14 (exact), then hi = binary16(v) and lo = binary16(v - hi); the
// MFMA takes hi and lo against the same weights, so each product keeps about
// 22 bits of the activation, and the power of two is undone on the sum.
// Non-finite activations keep lo = 0, so +-Inf and NaN reach the sums as the
// reference's float32 products would. The terms take the place of the float32
// values: the 256 bytes of 64 values hold their 64 hi, then their 64 lo, eight by
// eight in the pair order of the dequantised codes, so the tiles stage them as they are
// (split in the tiles, every column tile of an expert split the same rows again:
// 40 of 180 VALU instructions a step).
//
// Tiles. 128 or 64 pairs x 256 columns, 8 waves of 2 x 4: a wave owns every other
// 32-pair MFMA tile (two or one) and 64 columns. At 128 pairs a dequantised weight
// fragment feeds two MFMA row tiles, and experts with 1 .. 128 pairs cost ceil(pairs /
// 32) MFMA tiles; a workgroup fills a CU (156 KB of LDS, 240 registers). At 64 pairs each
// weight is dequantised by two waves and staged by 64 bytes a column, but two
// workgroups share a CU (78 KB, 128 registers), and tiles that would leave CUs idle
// are twice as many. mg_tile_rows chooses for each of the two GEMMs.
//
// Measured (one MI355X; us with the 64-pair tiles that split float32 rows in the tile ->
// 128-pair tiles only -> both): Mixtral's experts (H = 4096, I = 14336, 8 experts, 2
// taken, blocks of 64) 16 tokens 621 -> 378 -> 324, 300 tokens 1036 -> 687 -> 686, 2048
// tokens 4760 -> 3344 -> 3356; row scales, ReLU, 8 experts: 1000 x 2048 x 4096, 2 taken,
// 239 -> 271 -> 233; 512 x 1024 x 4096, 4 taken, 150 -> 191 -> 161 (the passes that
// split x and h, 17 us, are not repaid by four FC2 column tiles); 200 x 1024 x 4096, 4
// taken, 96 -> 128 -> 94. Over 785 sizes 1.36 times as fast as the first, 13 of them 1.5
// to 8 % slower (55, up to 38 %, with 128-pair tiles alone). A step's time by wave (128 pairs): 1.7 - 2.0 k cycles of MFMAs
// and dequantisation, 0.4 k issuing loads, 0.3 k staging, the rest barrier: the two waves
// of a SIMD overlap only in part.
#pragma once

namespace xrmm {
namespace {

constexpr int MG_CT = 256;  // columns per tile
constexpr int MG_K = 64;    // K step
constexpr int MG_LD = MG_K + 8;
constexpr int MG_T = 512;   // threads: 8 waves, 2 (row tiles) x 4 (columns of 64)
// Weights are staged for several K steps at once, a super-step: RT bytes of every
// column (128: 256 codes of 4 bits, 128 of 8).
template <int BITS, int RT>
constexpr int mg_ss() {
  return (BITS == 4 ? 4 : 2) * RT / 128;
}
template <int RT>
constexpr int mg_astage() {  // halfs per A stage: hi, then lo (rows of MG_LD)
  return 2 * RT * MG_LD;
}
template <int RT>
constexpr int mg_wstage() {  // bytes of a super-step's codes
  return MG_CT * RT;
}
// scales of a column and super-step (block mode BKM: 2, 4, 8 = blocks of 32, 64, 128
// or more codes; longer blocks repeat one scale)
template <int BITS, int BKM, int RT>
constexpr int mg_sb() {
  return BKM == 0 ? 0 : BKM == 2 ? 2 * mg_ss<BITS, RT>() : BKM == 4 ? mg_ss<BITS, RT>() : (mg_ss<BITS, RT>() + 1) / 2;
}
template <int BITS, int BKM, int RT>
constexpr size_t mg_lds() {
  return 2 * (mg_astage<RT>() * sizeof(_Float16) + mg_wstage<RT>() + mg_sb<BITS, BKM, RT>() * MG_CT * sizeof(float));
}

// Block-scale modes of the GEMM: 0 = one scale per row (applied to the row's
// sum in the epilogue); 1, 2, 4 = blocks of 16, 32, 64 codes (a block's sum
// is scaled and added every 1, 2, 4 MFMA K slices); 8 = blocks of 128 or
// more (scaled at the end of every block_size / 64 K steps).
inline int mg_block_mode(int bs) { return bs == 0 ? 0 : bs == 16 ? 1 : bs == 32 ? 2 : bs == 64 ? 4 : 8; }

// Lists of the grouped path, inside the workspace's counter region.
struct MgLists {
  int32_t* off;    // [E + 1] first list entry of each expert
  int32_t* toff;   // [E + 1] first row tile of each expert, FC1
  int32_t* toff2;  // [E + 1] the same of FC2 (toff where both have one tile height)
  int32_t* list;   // [T k] pair indices grouped by expert
  uint32_t* hmax;  // [T k] bits of the largest finite |h| of each pair
  int32_t* ex;     // [T] row exponent of x
};

// Exponent e such that |v| * 2^-e is near 2^14 for the row maximum v (0 for an
// all-zero row), at least -126 so that 2^e and 2^-e are both normal float32
// values (rows below 2^-112 keep fewer bits).
__device__ __forceinline__ int mg_row_exp(float mx) {
  if (!(mx > 0.f) || !__builtin_isfinite(mx)) return 0;
  int e = 0;
  (void)__builtin_frexpf(mx, &e);  // mx = f * 2^e, f in [0.5, 1)
  return e - 15 < -126 ? -126 : e - 15;
}

// Eight values times 2^-e as their binary16 terms, hi then lo, in the codes' pair
// order (0 4 1 5 2 6 3 7).
__device__ __forceinline__ void mg_terms(const float (&x)[8], float scale, f16x8& hi, f16x8& lo) {
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const float v = x[(q >> 1) + 4 * (q & 1)] * scale;
    const f16 h = static_cast<f16>(v);
    hi[q] = h;
    lo[q] = __builtin_isfinite(v) ? static_cast<f16>(v - static_cast<float>(h)) : static_cast<f16>(0.f);
  }
}

__device__ __forceinline__ void mg_load8(const float* p, float (&x)[8]) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
  x[0] = a.x, x[1] = a.y, x[2] = a.z, x[3] = a.w, x[4] = b.x, x[5] = b.y, x[6] = b.z, x[7] = b.w;
}

// One workgroup per token: wave 0 routes it (k_moe_route's rule), every wave then
// finds the row's largest finite |x|, and the row's terms go to xs [T][H] (256
// bytes per 64 values). H % 64 == 0. P > 0: eight-value groups per thread in
// registers (H <= 2048 P), the row read once; P == 0: any H, read twice.
template <int P>
__global__ __launch_bounds__(256) void k_moe_prep(const float* __restrict__ router, const float* __restrict__ x,
                                                  int32_t* __restrict__ sel, float* __restrict__ wts, int E, int k,
                                                  int H, int32_t* __restrict__ ex, f16* __restrict__ xs) {
  __shared__ float red[4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t t = blockIdx.x;
  const float* row = x + t * H;
  const int ng = H / 8;
  float v[P > 0 ? P : 1][8];
  float m = 0.f;
  auto see = [&](const float (&a)[8]) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float u = __builtin_fabsf(a[q]);
      if (__builtin_isfinite(u)) m = fmaxf(m, u);
    }
  };
  if constexpr (P > 0) {
#pragma unroll
    for (int i = 0; i < P; ++i)
      if (tid + 256 * i < ng) mg_load8(row + (tid + 256 * i) * 8, v[i]);
#pragma unroll
    for (int i = 0; i < P; ++i)
      if (tid + 256 * i < ng) see(v[i]);
  } else {
    for (int g = tid; g < ng; g += 256) {
      mg_load8(row + g * 8, v[0]);
      see(v[0]);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  if (lane == 0) red[tid >> 6] = m;
  __syncthreads();
  const int e = mg_row_exp(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])));
  const float scale = __builtin_ldexpf(1.f, -e);
  if (tid == 0) ex[t] = e;
  f16x8* out = reinterpret_cast<f16x8*>(xs + t * H * 2);
  if constexpr (P > 0) {
#pragma unroll
    for (int i = 0; i < P; ++i)
      if (tid + 256 * i < ng) {
        f16x8 hi, lo;
        mg_terms(v[i], scale, hi, lo);
        const int g = tid + 256 * i, o = (g >> 3) * 16 + (g & 7);
        out[o] = hi;
        out[o + 8] = lo;
      }
  } else {
    for (int g = tid; g < ng; g += 256) {
      f16x8 hi, lo;
      mg_load8(row + g * 8, v[0]);
      mg_terms(v[0], scale, hi, lo);
      out[(g >> 3) * 16 + (g & 7)] = hi;
      out[(g >> 3) * 16 + (g & 7) + 8] = lo;
    }
  }
  if (tid < 64) route_token(router, sel, wts, static_cast<int>(t), E, k, lane);
}

// h [T k][I] into its terms in place, eight values per thread; the row exponent from
// the pair's largest |h| (FC1's atomic maximum). The eight threads that exchange
// places inside 256 bytes are lanes of one wave (I % 64 == 0): the fence and the wave
// barrier keep every lane's loads before the first lane's store.
__global__ __launch_bounds__(256) void k_moe_hsplit(float* __restrict__ h, const uint32_t* __restrict__ hmax, int64_t groups,
                                                    int gpr) {
  const int64_t g = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (g >= groups) return;
  const float scale = __builtin_ldexpf(1.f, -mg_row_exp(__builtin_bit_cast(float, hmax[g / gpr])));
  float x[8];
  f16x8 hi, lo;
  mg_load8(h + g * 8, x);
  mg_terms(x, scale, hi, lo);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  f16x8* out = reinterpret_cast<f16x8*>(h + (g >> 3) * 64) + (g & 7);
  out[0] = hi;
  out[8] = lo;
}

// Pair counts, offsets, lists and the row tiles of rt (FC1) and rt2 (FC2) pairs; also
// clears hmax. One workgroup of MG_T threads; E <= kMoeGroupMaxExperts (LDS counters).
__global__ __launch_bounds__(MG_T) void k_moe_group(const int32_t* __restrict__ sel, int npairs, int E, int rt, int rt2,
                                                    MgLists g) {
  __shared__ int cnt[kMoeGroupMaxExperts];
  __shared__ int part[3][MG_T];
  const int tid = threadIdx.x;
  for (int e = tid; e < E; e += MG_T) cnt[e] = 0;
  __syncthreads();
  for (int p = tid; p < npairs; p += MG_T) {
    const int e = min(max(sel[p], 0), E - 1);
    atomicAdd(&cnt[e], 1);
    g.hmax[p] = 0u;
  }
  __syncthreads();
  // exclusive scans of the counts and of the row tiles: each thread sums a
  // run of experts, the runs' totals are scanned in LDS
  const int per = (E + MG_T - 1) / MG_T, e0 = tid * per;
  int s[3] = {0, 0, 0};
  for (int e = e0; e < e0 + per && e < E; ++e) {
    s[0] += cnt[e];
    s[1] += (cnt[e] + rt - 1) / rt;
    s[2] += (cnt[e] + rt2 - 1) / rt2;
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) part[q][tid] = s[q];
  __syncthreads();
  for (int d = 1; d < MG_T; d <<= 1) {
    int v[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) v[q] = tid >= d ? part[q][tid - d] : 0;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 3; ++q) part[q][tid] += v[q];
    __syncthreads();
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) s[q] = part[q][tid] - s[q];
  for (int e = e0; e < e0 + per && e < E; ++e) {
    g.off[e] = s[0];
    g.toff[e] = s[1];
    g.toff2[e] = s[2];
    const int c = cnt[e];
    s[0] += c;
    s[1] += (c + rt - 1) / rt;
    s[2] += (c + rt2 - 1) / rt2;
  }
  if (tid == MG_T - 1) {  // the last thread's run ends at E
    g.off[E] = s[0];
    g.toff[E] = s[1];
    g.toff2[E] = s[2];
  }
  __syncthreads();
  // positions: a cursor per expert (the order inside a list is free)
  for (int e = tid; e < E; e += MG_T) cnt[e] = 0;
  __syncthreads();
  for (int p = tid; p < npairs; p += MG_T) {
    const int e = min(max(sel[p], 0), E - 1);
    const int pos = atomicAdd(&cnt[e], 1);
    g.list[g.off[e] + pos] = p;
  }
}

enum MgStage { MG_FC1_RELU = 0, MG_FC1_SWIGLU = 1, MG_FC2 = 2 };

// v of the lane N places on in its row of 16.
template <int N>
__device__ __forceinline__ float mg_ror(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x120 + N, 0xF, 0xF, true));
}

// One tile of RT pairs x 256 columns of an expert's matrix; BITS-bit codes, block
// mode BKM (mg_block_mode).
template <int ST, int BITS, int BKM, int RT>
__global__ __launch_bounds__(MG_T, RT == 64 ? 4 : 2) void k_moe_ggemm(MoeArgs a, MgLists g, int nct) {
  constexpr bool FC2 = ST == MG_FC2;
  constexpr int SS = mg_ss<BITS, RT>(), SB = mg_sb<BITS, BKM, RT>();
  constexpr int MG_ASTAGE = mg_astage<RT>(), MG_WSTAGE = mg_wstage<RT>();
  constexpr int NI = RT / 64;   // MFMA row tiles of a wave
  constexpr int CH = RT / 16;   // 16-byte chunks of a column's super-step
  constexpr int ROT = 64 / CH;  // places a chunk's columns are rotated by, times the chunk
  constexpr int BW = BITS / 4;  // dwords per fragment
  extern __shared__ __align__(16) unsigned char smem[];
  f16* lds = reinterpret_cast<f16*>(smem);                                   // [2] A stages
  uint32_t* wlds = reinterpret_cast<uint32_t*>(lds + 2 * MG_ASTAGE);         // [2] super-steps' codes
  float* slds = reinterpret_cast<float*>(wlds + 2 * (MG_WSTAGE / 4));        // [2][SB][column] scales
  __shared__ int s_pair[RT];
  __shared__ float s_ru[RT];  // 2^e per row (epilogue)
  constexpr uint32_t OOB = 0x80000000u;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int E = static_cast<int>(a.E);
  // FC2: workgroup b is split b % ks of tile b / ks
  const int ks2 = FC2 ? a.ks : 1;
  const int sp = static_cast<int>(blockIdx.x) % ks2, tb = static_cast<int>(blockIdx.x) / ks2;
  const int rt = tb / nct, ct = tb % nct;
  const int32_t* toff = FC2 ? g.toff2 : g.toff;
  const int total = toff[E];
  if (rt >= total) return;  // uniform: the grid is an upper bound of the row tiles
  // expert of this row tile: the last e with toff[e] <= rt
  int lo = 0, hi = E - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (toff[mid] <= rt) lo = mid;
    else hi = mid - 1;
  }
  const int e = lo;
  // the expert's pairs over its row tiles in equal whole 32s (260 pairs: 96, 96, 68)
  const int npe = g.off[e + 1] - g.off[e], nte = toff[e + 1] - toff[e];
  const int rpt = ((npe + nte - 1) / nte + 31) & ~31;
  const int lb = g.off[e] + (rt - toff[e]) * rpt;  // first list entry of the tile
  const int nrow = min(rpt, g.off[e + 1] - lb);
  const int Kd = static_cast<int>(FC2 ? a.I : a.H);   // reduction length
  const int Nd = static_cast<int>(FC2 ? a.H : a.F1);  // rows of the expert matrix
  const int n0 = ct * MG_CT;
  if (tid < RT) {
    const int p = tid < nrow ? g.list[lb + tid] : -1;
    s_pair[tid] = p;
    int ex = 0;
    if (p >= 0) {
      if constexpr (FC2) ex = mg_row_exp(__builtin_bit_cast(float, g.hmax[p]));
      else ex = g.ex[p / a.k];
    }
    s_ru[tid] = __builtin_ldexpf(1.f, ex);
  }
  __syncthreads();

  const uint32_t rowb = static_cast<uint32_t>(Kd) * BITS / 8u;  // bytes per expert row
  const uint8_t* Wb = FC2 ? a.fc2 + static_cast<int64_t>(e) * a.H * rowb : a.fc1 + static_cast<int64_t>(e) * a.F1 * rowb;
  const rsrc_t rB = mk_rsrc(Wb, static_cast<uint32_t>(Nd) * rowb);
  // this workgroup's K steps [kstep0, kstep0 + ksteps); splits of blocks of
  // 128 codes or more hold whole blocks (a split past the end holds none and
  // writes zero partials)
  const int kall = (Kd + MG_K - 1) / MG_K;
  const int bsteps = BKM == 8 ? a.bs / MG_K : 1;  // K steps per block
  const int kper = ((kall + ks2 - 1) / ks2 + bsteps - 1) / bsteps * bsteps;
  const int kstep0 = sp * kper;
  const int ksteps = kall - kstep0 < kper ? kall - kstep0 : kper;

  // ---- staging. A wave waits for its loads in the order it issued them, so the
  // long-latency weight stream and the activations (in the L2) have waves of their
  // own: with both in one wave every step waited for the weights loaded just before
  // its activations (16 KB in flight per CU, 1.6 TB/s however few the pairs).
  //  * waves 4 .. 7 (256 threads): A, one step ahead. Thread t: values 8 (t % 8) .. + 7
  //    of rows t / 8 + 32 i (32 bytes of terms each), through per-lane addresses (the
  //    rows belong to different tokens); rows past the tile's pairs repeat its first
  //    pair and their sums are never written.
  //  * waves 0 .. 3: the codes and scales, a super-step ahead. Thread t: chunk t % 8 (16
  //    bytes) of columns t / 8 + 32 i, whole lines of eight columns per load, and the
  //    scales of column t.
  const int st_t = tid & 255;
  struct ARegs {
    u32x4 v[2 * NI][2];
  };
  const float* Arow[2 * NI];
  {
    const float* Asrc = FC2 ? a.h : a.yp;  // FC1: x's terms
#pragma unroll
    for (int i = 0; i < 2 * NI; ++i) {
      const int r = (st_t >> 3) + 32 * i, p = s_pair[r] < 0 ? s_pair[0] : s_pair[r];
      Arow[i] = Asrc + (FC2 ? static_cast<int64_t>(p) * a.I : static_cast<int64_t>(p / a.k) * a.H) + (st_t & 7) * 4;
    }
  }
  // row tiles of 32 that hold pairs; the others are neither loaded nor read
  const int nsub = (nrow + 31) / 32;
  auto aload = [&](ARegs& r, int ks) {
#pragma unroll
    for (int i = 0; i < 2 * NI; ++i) {
      if (i >= nsub) break;
      const float* pa = Arow[i] + (kstep0 + ks) * MG_K;
      r.v[i][0] = *reinterpret_cast<const u32x4*>(pa);
      r.v[i][1] = *reinterpret_cast<const u32x4*>(pa + 32);
    }
  };
  auto astore = [&](const ARegs& r, int stage) {
    f16* Ah = lds + stage * MG_ASTAGE + (st_t >> 3) * MG_LD + (st_t & 7) * 8;
#pragma unroll
    for (int i = 0; i < 2 * NI; ++i) {
      if (i >= nsub) break;
      *reinterpret_cast<u32x4*>(Ah + 32 * i * MG_LD) = r.v[i][0];
      *reinterpret_cast<u32x4*>(Ah + (RT + 32 * i) * MG_LD) = r.v[i][1];
    }
  };
  // scales: [E, Nd] (row scales) or [E, Nd, Kd / block_size]
  const int nblk = BKM ? Kd / a.bs : 1;
  const float* S = FC2 ? a.s2 + static_cast<int64_t>(e) * a.H * nblk : a.s1 + static_cast<int64_t>(e) * a.F1 * nblk;
  const rsrc_t rS = mk_rsrc(S, static_cast<uint32_t>(Nd) * static_cast<uint32_t>(nblk) * 4u);
  struct WRegs {
    u32x4 v[CH];
    uint32_t s[SB ? SB : 1];
  };
  // chunks i0 .. i1 - 1 (of a thread's CH) of super-step u, with the first its scales;
  // past the row: zeros
  auto wload = [&](WRegs& r, int u, int i0, int i1) __attribute__((always_inline)) {
    const uint32_t o = static_cast<uint32_t>((kstep0 + u * SS) * MG_K * BITS / 8 + (st_t & (CH - 1)) * 16);
    const uint32_t past = u * SS < ksteps && o < rowb ? 0u : OOB;
#pragma unroll
    for (int i = i0; i < i1; ++i) {
      const int c = n0 + st_t / CH + 256 / CH * i;
      r.v[i] = bld16(rB, ((c < Nd ? static_cast<uint32_t>(c) * rowb : OOB) | past) + o, 0);
    }
    if (i0 > 0) return;
    if constexpr (SB > 0) {
      const int c = n0 + st_t < Nd ? n0 + st_t : Nd - 1;
      const uint32_t b = static_cast<uint32_t>((kstep0 + u * SS) * MG_K / a.bs);
      const uint32_t so = (static_cast<uint32_t>(c) * static_cast<uint32_t>(nblk) + b) * 4u;
      // blocks past the row's last belong to steps that are not run
#pragma unroll
      for (int f = 0; f < SB; f += 4) {
        if constexpr (SB >= 4) {
          const u32x4 v = bld16(rS, so + 4u * f, 0);
          r.s[f] = v.x, r.s[f + 1] = v.y, r.s[f + 2] = v.z, r.s[f + 3] = v.w;
        } else if constexpr (SB == 2) {
          const u32x2 v = bld8(rS, so, 0);
          r.s[0] = v.x, r.s[1] = v.y;
        } else {
          r.s[0] = bld_u32(rS, so, 0);
        }
      }
    }
  };
  // codes as [fragment of the super-step][column][BW dwords], a fragment being eight
  // codes; chunk c's columns are rotated by 8 c places, so the eight chunks a wave
  // writes at once fall in different banks
  auto wstore = [&](const WRegs& r, int buf) {
    uint32_t* W = wlds + buf * (MG_WSTAGE / 4);
    const int c = st_t & (CH - 1);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int col = (st_t / CH + 256 / CH * i + ROT * c) & (MG_CT - 1);
      const u32x4 v = r.v[i];
      if constexpr (BW == 1) {
        uint32_t* d = W + 4 * c * MG_CT + col;
        d[0] = v.x, d[MG_CT] = v.y, d[2 * MG_CT] = v.z, d[3 * MG_CT] = v.w;
      } else {
        uint32_t* d = W + (2 * c * MG_CT + col) * 2;
        *reinterpret_cast<u32x2*>(d) = u32x2{v.x, v.y};
        *reinterpret_cast<u32x2*>(d + 2 * MG_CT) = u32x2{v.z, v.w};
      }
    }
    if constexpr (SB > 0) {
#pragma unroll
      for (int f = 0; f < SB; ++f) slds[(buf * SB + f) * MG_CT + st_t] = __builtin_bit_cast(float, r.s[f]);
    }
  };
  // a fragment's eight codes -> c - 2^(bits - 1) as exact binary16, pair
  // order (c0 c4 c1 c5 c2 c6 c3 c7, the activations' staging order)
  const f16x2 n1032 = {static_cast<f16>(-1032.f), static_cast<f16>(-1032.f)};
  const f16x2 inv16 = {static_cast<f16>(0.0625f), static_cast<f16>(0.0625f)};
  const f16x2 n72 = {static_cast<f16>(-72.f), static_cast<f16>(-72.f)};
  const f16x2 n1152 = {static_cast<f16>(-1152.f), static_cast<f16>(-1152.f)};
  auto dq = [&](const uint32_t* w) __attribute__((always_inline)) {
    const uint32_t magic = 0x64006400u;
    if constexpr (BW == 1) {
      const uint32_t x = w[0], x8 = x >> 8;
      const f16x2 d0 = as_h2(and_or(x, 0x000F000Fu, magic)) + n1032;
      const f16x2 d1 = __builtin_elementwise_fma(as_h2(and_or(x, 0x00F000F0u, magic)), inv16, n72);
      const f16x2 d2 = as_h2(and_or(x8, 0x000F000Fu, magic)) + n1032;
      const f16x2 d3 = __builtin_elementwise_fma(as_h2(and_or(x8, 0x00F000F0u, magic)), inv16, n72);
      return f16x8{d0[0], d0[1], d1[0], d1[1], d2[0], d2[1], d3[0], d3[1]};
    } else {
      // bytes c0..c3 in w[0], c4..c7 in w[1]: (c_i, c_i+4) into the low bytes
      // of a half pair, then 0x64 above each: 1024 + c exactly
      const uint32_t x0 = w[0], x1 = w[1];
      const f16x2 d0 = as_h2(__builtin_amdgcn_perm(x1, x0, 0x0c040c00u) | magic) + n1152;
      const f16x2 d1 = as_h2(__builtin_amdgcn_perm(x1, x0, 0x0c050c01u) | magic) + n1152;
      const f16x2 d2 = as_h2(__builtin_amdgcn_perm(x1, x0, 0x0c060c02u) | magic) + n1152;
      const f16x2 d3 = as_h2(__builtin_amdgcn_perm(x1, x0, 0x0c070c03u) | magic) + n1152;
      return f16x8{d0[0], d0[1], d1[0], d1[1], d2[0], d2[1], d3[0], d3[1]};
    }
  };

  // block sums (acc) and, with block scales, the scaled running sums (yacc), of
  // the wave's row tiles wm, wm + 2
  f32x16 acc[NI][2];
  float yacc[BKM ? NI : 1][BKM ? 2 : 1][16];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        acc[i][j][q] = 0.f;
        yacc[BKM ? i : 0][BKM ? j : 0][q] = 0.f;
      }
  // (kept in place by the empty asm and the scheduling barriers: sunk among the
  // next block's MFMAs it would hold two copies of the accumulators)
  const f32x16 zero16 = {};
  auto flush = [&](auto na, const float (&sc)[2]) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < na; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          float& y = yacc[BKM ? i : 0][BKM ? j : 0][q];
          y = __builtin_fmaf(sc[j], acc[i][j][q], y);
          asm volatile("" : "+v"(y));
        }
        if constexpr (BKM == 8) acc[i][j] = zero16;
      }
    __builtin_amdgcn_sched_barrier(0);
  };
  const int lcol = wn * 64 + (lane & 31);  // the lane's columns: lcol, lcol + 32
  // step t of its super-step, on A stage `stage` and weight buffer `buf`
  auto mfmas = [&](auto na, int stage, int buf, int t) __attribute__((always_inline)) {
    const f16* Ah = lds + stage * MG_ASTAGE;
    const f16* Al = Ah + RT * MG_LD;
    const uint32_t* W = wlds + buf * (MG_WSTAGE / 4) + 8 * t * MG_CT * BW;
    const float* sc = slds + buf * SB * MG_CT + lcol;
#pragma unroll
    for (int kk = 0; kk < MG_K / 16; ++kk) {
      const int ko = kk * 16 + (lane >> 5) * 8;
      f16x8 fh[NI], fl[NI];
#pragma unroll
      for (int i = 0; i < na; ++i) {
        const int ar = (wm + 2 * i) * 32 + (lane & 31);
        fh[i] = *reinterpret_cast<const f16x8*>(Ah + ar * MG_LD + ko);
        fl[i] = *reinterpret_cast<const f16x8*>(Al + ar * MG_LD + ko);
      }
      const bool first = BKM >= 1 && BKM <= 4 && kk % (BKM ? BKM : 1) == 0;  // a block starts: from zero
      const int chunk = BW == 1 ? 2 * t + kk / 2 : 4 * t + kk;  // both lane halves' fragments lie in it
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        // codes k = ko .. ko + 7 of column lcol + 32 j: fragment ko / 8
        const f16x8 fb = dq(W + ((ko >> 3) * MG_CT + ((lcol + 32 * j + ROT * chunk) & (MG_CT - 1))) * BW);
#pragma unroll
        for (int i = 0; i < na; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fh[i], fb, first ? zero16 : acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < na; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fl[i], fb, acc[i][j], 0, 0, 0);
      }
      if constexpr (BKM == 2 || BKM == 4) {
        if ((kk + 1) % BKM == 0) {
          const float* p = sc + (t * (4 / BKM) + kk / BKM) * MG_CT;
          const float sl[2] = {p[0], p[32]};
          flush(na, sl);
        }
      }
    }
  };
  // Order of the K steps: column tile ct starts at super-step ct of its range and wraps
  // around. The tiles run side by side; all at the same k, they would read the same
  // 128 bytes of every row, whose stride of H / 2 bytes lands on few memory channels
  // (1.6 TB/s). The start is a whole number of scale blocks. Not so for 64-pair tiles of
  // experts with many pairs: the L2 then serves a row's activations to all column tiles
  // at once (block scales, 60 pairs an expert and more: 5 % faster without, up to 12).
  const int ru = BKM == 8 && bsteps > SS ? bsteps : SS;
  const int nru = ksteps / ru;
  const int first_step = nru > 1 && !(RT == 64 && npe > 16) ? ct % nru * ru : 0;
  // role 0 (waves 0 .. 3): weights; 1: activations. na: the wave's row tiles that hold
  // pairs, 2, 1 or none (it then only stages). All loops have the same barriers.
  auto loop = [&](auto role, auto na) __attribute__((always_inline)) {
    ARegs ar;
    WRegs wr;
    int p = first_step, buf = 0;  // the step, its weight buffer
    if constexpr (role == 0) {
      wload(wr, p / SS, 0, CH);
      wstore(wr, 0);
    } else {
      aload(ar, p);
      astore(ar, 0);
    }
    __syncthreads();
    for (int i = 0; i < ksteps; ++i) {
      const int t = p & (SS - 1), next = p + 1 < ksteps ? p + 1 : 0;
      const bool last = t == SS - 1 || next == 0;  // of its super-step
      if constexpr (role == 0) {
        // the super-step after this one (the row's first after its last), over its first
        // three steps (all eight at once hold up the activations' loads: 1.5 k cycles)
        const int u = (p / SS + 1) * SS < ksteps ? p / SS + 1 : 0;
        if constexpr (SS == 4 && CH == 8) {
          if (t == 0) wload(wr, u, 0, 3);
          if (t == 1 || (last && t < 1)) wload(wr, u, 3, 6);  // the row may end inside the super-step
          if (t == 2 || (last && t < 2)) wload(wr, u, 6, 8);
        } else {
          if (t == 0) wload(wr, u, 0, CH);
        }
      } else {
        aload(ar, next);
      }
      __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the matrix work
      if constexpr (na > 0) {
        mfmas(na, i & 1, buf, t);
        if constexpr (BKM == 8) {
          if ((kstep0 + p + 1) % bsteps == 0) {
            const float* sp = slds + (buf * SB + (bsteps < SS ? t / bsteps : 0)) * MG_CT + lcol;
            const float sl[2] = {sp[0], sp[32]};
            flush(na, sl);
          }
        }
      }
      if constexpr (role == 0) {
        if (last) wstore(wr, buf ^ 1);
      } else {
        astore(ar, (i + 1) & 1);
      }
      if (last) buf ^= 1;
      p = next;
      __syncthreads();
    }
  };
  if (ksteps > 0) {  // uniform: a split past the end keeps zero sums
    const int na = ((nrow + 31) / 32 - wm + 1) / 2;
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    if (wm == 0) {
      if (NI == 2 && na >= 2) loop(I0{}, std::integral_constant<int, NI>{});
      else loop(I0{}, I1{});  // a tile holds a pair
    } else {
      if (NI == 2 && na >= 2) loop(I1{}, std::integral_constant<int, NI>{});
      else if (na == 1) loop(I1{}, I1{});
      else loop(I1{}, I0{});
    }
  }

  // ---- epilogue: lane holds D[8 (q / 4) + 4 (lane / 32) + q % 4][lane % 32]
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    if (wm + 2 * i >= nsub) break;  // no pair in the row tile
    const int r0 = (wm + 2 * i) * 32 + 4 * (lane >> 5);
    auto value = [&](int j, int q, float sc) {
      return (BKM ? yacc[BKM ? i : 0][BKM ? j : 0][q] : acc[i][j][q] * sc) * s_ru[r0 + 8 * (q >> 2) + (q & 3)];
    };
    float rmax[16];  // SwiGLU: even lanes' rows q, odd lanes' rows q + 1, in q / 2
#pragma unroll
    for (int q = 0; q < 16; ++q) rmax[q] = 0.f;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int c = n0 + wn * 64 + j * 32 + (lane & 31);
      const float sc = BKM ? 1.f : (c < Nd ? S[c] : 0.f);
      if constexpr (ST == MG_FC1_SWIGLU) {
        // gate = FC1 row 2m (even lane), linear = row 2m + 1 (odd lane): of two output
        // rows the even lane forms the first, the odd lane the second
        const bool odd = lane & 1;
#pragma unroll
        for (int q = 0; q < 16; q += 2) {
          const float v0 = value(j, q, sc), v1 = value(j, q + 1, sc);
          const float other = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, odd ? v0 : v1), 0xB1, 0xF, 0xF, true));
          const float o = swiglu(odd ? other : v0, odd ? v1 : other, a);
          const int p = s_pair[r0 + 8 * (q >> 2) + (q & 3) + (odd ? 1 : 0)];
          if (p >= 0 && c < Nd) {
            a.h[static_cast<int64_t>(p) * a.I + c / 2] = o;
            if (__builtin_isfinite(o)) rmax[q >> 1] = fmaxf(rmax[q >> 1], __builtin_fabsf(o));
          }
        }
      } else {
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const int p = s_pair[r0 + 8 * (q >> 2) + (q & 3)];
          const float v = value(j, q, sc);
          if constexpr (FC2) {
            if (p >= 0 && c < Nd) a.yp[(static_cast<int64_t>(p) * ks2 + sp) * a.H + c] = v;
          } else {
            const float o = fmaxf(v, 0.f);
            if (p >= 0 && c < Nd) {
              a.h[static_cast<int64_t>(p) * a.I + c] = o;
              if (__builtin_isfinite(o)) rmax[q] = fmaxf(rmax[q], o);
            }
          }
        }
      }
    }
    if constexpr (!FC2) {
      // each row's largest |h| over this tile, into the pair's running maximum
      // (non-negative floats order like their bit patterns)
      constexpr bool SW = ST == MG_FC1_SWIGLU;
#pragma unroll
      for (int q = 0; q < (SW ? 8 : 16); ++q) {
        float m = rmax[q];
        if constexpr (!SW) m = fmaxf(m, mg_ror<1>(m));
        m = fmaxf(m, mg_ror<2>(m));
        m = fmaxf(m, mg_ror<4>(m));
        m = fmaxf(m, mg_ror<8>(m));
        m = fmaxf(m, __shfl_xor(m, 16, 64));
        const int qq = SW ? 2 * q + (lane & 1) : q;
        const int p = s_pair[r0 + 8 * (qq >> 2) + (qq & 3)];
        if ((lane & 31) < (SW ? 2 : 1) && p >= 0 && m > 0.f) atomicMax(g.hmax + p, __builtin_bit_cast(uint32_t, m));
      }
    }
  }
}

// y[t][n] = sum over slots s of w[t k + s] * yp[t k + s][n], in slot order,
// each slot's a.ks FC2 splits summed first in split order; four columns per
// thread (H % 64 == 0).
__global__ __launch_bounds__(256) void k_moe_combine(MoeArgs a) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t h4 = a.H / 4;
  if (i >= a.T * h4) return;
  const int64_t t = i / h4, n = i % h4 * 4;
  f32x4 y = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < a.k; ++s) {
    const int64_t pair = t * a.k + s;
    const float* part = a.yp + pair * a.ks * a.H + n;
    f32x4 v = *reinterpret_cast<const f32x4*>(part);
    for (int sp = 1; sp < a.ks; ++sp) v += *reinterpret_cast<const f32x4*>(part + static_cast<int64_t>(sp) * a.H);
    const float w = a.wts[pair];
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = __builtin_fmaf(w, v[e], y[e]);
  }
  typedef f32x4 f32x4_a4 __attribute__((aligned(4)));  // y need not be 16-byte aligned
  *reinterpret_cast<f32x4_a4*>(a.y + t * a.H + n) = y;
}

}  // namespace
}  // namespace xrmm
