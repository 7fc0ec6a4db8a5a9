// W4A4 SVDQuant GEMM on small block tiles, for shapes whose 256 x 128 tiles leave most of the 256
// CUs idle: prompt-sized row counts and narrow layers.
//
// Same operands and arithmetic as the large tiles (svdq_gemm.hip): exact group sums P on the FP6
// MFMA, S = sx (x) sw on the bf16 MFMA, acc += P * S in group order, then mid @ l1cat^T (hi plane,
// lo plane, 16 ranks at a time) and the bias.  Every output therefore has the same bits on every
// tile, and the choice of tile is free.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <utility>

#include "svdq_common.h"
#include "svdq_kernels.h"

namespace svdq {
namespace {

// f(integral_constant<int, 0>), f(integral_constant<int, 1>), ...
template <class F, int... B>
__device__ __forceinline__ void for_each_index(F&& f, std::integer_sequence<int, B...>) {
  (f(std::integral_constant<int, B>{}), ...);
}

// Whether a tile's stages are moved by waves of their own (as many as multiply).
template <int WM, int WN>
constexpr bool small_split() {
  return WM * WN <= 4;
}

// Block tile (32 WM) x (32 WN), WM x WN multiplying waves, wave tile 32 x 32.
//
// What bounds it: few rows mean few tiles, so a tile's own serial chain over K.  K is not split: the
// sum over groups runs in group order as in the large tiles.  A wave alone on its SIMD issues an
// instruction every 4-6 cycles and waits in order behind a second MFMA, so a group's step is one
// MFMA, 8 rescale FMAs, one MFMA, 8 FMAs, and up to 64 x 64 the stages are moved by waves of their
// own (as many as multiply): 32 x 32 tiles at M = 64, N = 1536, K = 6144 took 13.7 us with the
// multiplying waves issuing the DMA and both MFMAs first, 9.4 us so (the 256 x 128 tiles: 40.3 us).
//
// A stage is 256 columns of K (four k-steps) in a ring of four LDS buffers, moved by DMA.  A stage's
// LDS image is a list of 16-byte chunks: A Q planes [k-step][half][row][16], B Q planes, A P planes
// [k-step][half][row][8], B P planes, then the scale words [row][group], all groups of a row
// together so that one read per stage fetches them.  One DMA instruction moves 64 consecutive chunks
// (scale words); a region with fewer instructions than waves is moved by several of them (the same
// bytes to the same place), so that every wave has the same number in flight.
//
// Group step g of a wave: read the fragments of group g + DIST from LDS, issue the MFMAs of group
// g + 1, then the rescale FMAs of group g, so that in a wave alone on its SIMD the FMAs run under
// the next group's MFMAs and the reads have a step or two to land.  The one barrier per stage sits
// where the reads cross into the next stage: stage s + 1 has landed, and every wave has issued MFMAs
// of stage s, so its reads of stage s - 1 are complete and stage s + 3 may overwrite that.
template <int G, int WM, int WN, bool OUT_F32>
__device__ __forceinline__ void w4a4_e3m2_small_tile(const GemmParams& p, int bm, int bn) {
  constexpr int NW = WM * WN, TBM = 32 * WM, TBN = 32 * WN, NBUF = 4;
  constexpr int KT = 4, GPS = KT * 64 / G, KS = G / 64;    // k-steps and groups per stage, k-steps per group
  constexpr int NAQ = KT * TBM / 32, NBQ = KT * TBN / 32, NAP = NAQ / 2, NBP = NBQ / 2;   // DMA instructions
  constexpr int NX = GPS * TBM / 64, NWS = GPS * TBN / 64;
  constexpr int D = (NAQ + NW - 1) / NW + (NBQ + NW - 1) / NW + (NAP + NW - 1) / NW + (NBP + NW - 1) / NW +
                    (NX + NW - 1) / NW + (NWS + NW - 1) / NW;                              // per wave and stage
  constexpr int OBQ = NAQ * 1024, OAP = OBQ + NBQ * 1024, OBP = OAP + NAP * 1024, OX = OBP + NBP * 1024,
                OW = OX + 256 * NX, OZ = OW + 256 * NWS, BUF = OZ + 64;   // (zeros at OZ)
  constexpr int DIST = G == 64 && NW < 8 ? 3 : 2, NSET = DIST == 3 ? 4 : 2;   // read-ahead, fragment sets
  constexpr int PITCH = 64 + 16;                            // output staging: bytes per row
  constexpr bool SPLIT = small_split<WM, WN>();
  static_assert(NAP % NW == 0 || NW % NAP == 0, "whole instructions per wave, or whole waves per instruction");
  static_assert(GPS % NSET == 0 && DIST <= GPS && NX >= 1, "whole sets per stage, whole DMA instructions");
  static_assert(NBUF * BUF <= 160 * 1024 && NW * 32 * PITCH <= NBUF * BUF, "LDS");
  static_assert((NBUF - 2) * D <= 63, "vmcnt counts to 63");
  __shared__ __attribute__((aligned(1024))) uint8_t sm[NBUF * BUF];

  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, h = lane >> 5;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool mover = SPLIT && wid >= NW;                    // moves the stages; the other waves multiply
  const int wave = mover ? wid - NW : wid, wm = wave / WN, wn = wave % WN;
  const int m0 = bm * TBM, n0 = bn * TBN;
  const int nkt = p.K / 64, nstages = (nkt + KT - 1) / KT, ngroups = p.K / G;
  const long Mp = (p.M + 1) & ~1, Np = (p.N + 1) & ~1;
  const uint32_t lds0 = lds_offset(sm);

  // The low-rank operands of the first 32 ranks, loaded ahead of everything else.
  const uint16_t* arow = p.midp + (long)min(m0 + 32 * wm + lr, p.M - 1) * (2 * p.RTp) + 8 * h;
  const uint16_t* brow = p.l1cat + (long)min(n0 + 32 * wn + lr, p.N - 1) * p.RTp + 8 * h;
  u32x4 ehi[2], elo[2], eb[2];
  auto load_ranks = [&](int k) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      ehi[u] = *reinterpret_cast<const u32x4*>(arow + k + 16 * u);
      elo[u] = *reinterpret_cast<const u32x4*>(arow + p.RTp + k + 16 * u);
      eb[u] = *reinterpret_cast<const u32x4*>(brow + k + 16 * u);
    }
  };

  // The six regions of a stage: A Q, B Q, A P, B P planes, A and B scale words.  The wave's d-th
  // instruction of a region is the region's instruction wave + NW d (wave mod its count).  Per
  // region a source base, advanced one stage at a time; per instruction a per-lane offset.
  constexpr int NR[6] = {NAQ, NBQ, NAP, NBP, NX, NWS};
  constexpr int LO[6] = {0, OBQ, OAP, OBP, OX, OW};
  const uint8_t* src[6] = {p.qa,
                           p.qwe,
                           p.qa + (long)nkt * 2 * Mp * 16,
                           p.qwe + (long)nkt * 2 * Np * 16,
                           reinterpret_cast<const uint8_t*>(p.sxp),
                           reinterpret_cast<const uint8_t*>(p.swp)};
  // offset of lane ln in instruction i of region r, its k-step (group) in the stage lowered to `most`
  auto lane_off = [&](int r, int i, int ln, int most) -> uint32_t {
    const bool a = r % 2 == 0;
    const int tb = a ? TBM : TBN, r0 = a ? m0 : n0, rows = a ? p.M : p.N, rp = (rows + 1) & ~1;
    const int c = 64 * i + ln;
    if (r >= 4)
      return 4u * ((uint32_t)min(c % GPS, most) * (uint32_t)rows + (uint32_t)min(r0 + c / GPS, rows - 1));
    const int per = r < 2 ? tb : tb / 2, plane = c / per, e = c % per;
    const uint32_t pl = 2 * min(plane / 2, most) + plane % 2, w = r < 2 ? 16 : 8;
    return (pl * (uint32_t)rp + (uint32_t)(r < 2 ? min(r0 + e, rows - 1) : min(r0 + 2 * e, rp - 2))) * w;
  };
  constexpr int MAXC = (NBQ > NAQ ? NBQ : NAQ) / NW > 0 ? (NBQ > NAQ ? NBQ : NAQ) / NW : 1;
  uint32_t off[6][MAXC];
#pragma unroll
  for (int r = 0; r < 6; ++r)
#pragma unroll
    for (int d = 0; d < (NR[r] + NW - 1) / NW; ++d) off[r][d] = lane_off(r, (wave + NW * d) % NR[r], lane, KT);
  auto issue = [&](int s, int buf) {
    int wv = wave;
    asm volatile("" : "+s"(wv));   // (LDS addresses computed here, not held for every buffer across the loop)
    const uint32_t lb = lds0 + 1024 * wv, lb4 = lds0 + 256 * wv;
    auto lds_at = [&](int r, int d) -> uint32_t {
      const int sz = r < 4 ? 1024 : 256;
      if (NR[r] < NW) return lds0 + buf * BUF + LO[r] + sz * (wv % NR[r]);
      return (r < 4 ? lb : lb4) + buf * BUF + LO[r] + sz * NW * d;
    };
    if (s == nstages - 1 && nkt % KT) {
      // K ends inside the stage: the k-steps and groups past it re-read the last one (never multiplied)
      int ln = lane;
      asm volatile("" : "+v"(ln));                          // (computed here, not held across the loop)
#pragma unroll
      for (int r = 0; r < 6; ++r)
#pragma unroll
        for (int d = 0; d < (NR[r] + NW - 1) / NW; ++d) {
          const uint32_t o = lane_off(r, (wv + NW * d) % NR[r], ln, r < 4 ? (nkt - 1) % KT : (ngroups - 1) % GPS);
          if (r < 4) dma16(src[r], o, lds_at(r, d));
          else dma4(src[r], o, lds_at(r, d));
        }
    } else {
#pragma unroll
      for (int r = 0; r < 6; ++r) {
#pragma unroll
        for (int d = 0; d < (NR[r] + NW - 1) / NW; ++d) {
          if (r < 4) dma16(src[r], off[r][d], lds_at(r, d));
          else dma4(src[r], off[r][d], lds_at(r, d));
        }
        const long rows = r % 2 == 0 ? p.M : p.N, rp = r % 2 == 0 ? Mp : Np;
        src[r] += r < 2 ? 32L * KT * rp : r < 4 ? 16L * KT * rp : 4L * GPS * rows;
      }
    }
  };

  f32x16 acc = f32x16{};

  // Per-lane LDS read bases; a read adds buffer and k-step as an immediate offset.
  typedef uint32_t scales __attribute__((ext_vector_type(GPS)));
  typedef const __attribute__((address_space(3))) uint8_t* lds_u8;
  typedef const __attribute__((address_space(3))) u32x4* lds_u32x4;
  typedef const __attribute__((address_space(3))) u32x2* lds_u32x2;
  typedef const __attribute__((address_space(3))) scales* lds_scales;
  const lds_u8 rAQ = (lds_u8)&sm[(h * TBM + 32 * wm + lr) * 16], rAP = (lds_u8)&sm[OAP + (h * TBM + 32 * wm + lr) * 8];
  const lds_u8 rBQ = (lds_u8)&sm[OBQ + (h * TBN + 32 * wn + lr) * 16];
  const lds_u8 rBP = (lds_u8)&sm[OBP + (h * TBN + 32 * wn + lr) * 8];
  const lds_u8 rX = (lds_u8)&sm[OX + 4 * GPS * (32 * wm + scale_row_perm(lr))];   // rows permuted: see rescale_acc
  // lanes 32-63 of the scale MFMA's B operand are zero: they read the buffer's zero words
  const lds_u8 rW = (lds_u8)&sm[h ? OZ : OW + 4 * GPS * (32 * wn + lr)];

  // NSET register sets of fragments and two of products, group g in set g mod NSET (g mod 2), and two
  // of scales, stage s in set s mod 2: a compile-time index everywhere.
  u32x4 aq[NSET][KS], bq[NSET][KS];
  u32x2 ap[NSET][KS], bp[NSET][KS];
  scales xs[2], ws[2];
  f32x16 P[2], S[2];
  auto read_frags = [&](int buf, int g) {
    const int f = g % NSET, o = buf * BUF;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const int t = g * KS + k;
      aq[f][k] = *(lds_u32x4)(rAQ + o + t * 2 * TBM * 16);
      ap[f][k] = *(lds_u32x2)(rAP + o + t * 2 * TBM * 8);
      bq[f][k] = *(lds_u32x4)(rBQ + o + t * 2 * TBN * 16);
      bp[f][k] = *(lds_u32x2)(rBP + o + t * 2 * TBN * 8);
    }
  };
  auto read_scales = [&](int buf, int set) {
    xs[set] = *(lds_scales)(rX + buf * BUF);
    ws[set] = *(lds_scales)(rW + buf * BUF);
  };
  // (the empty asm statements pin the order: the compiler would sink MFMAs and FMAs to their last use)
  auto mfma_p = [&](int g) {
    const int s = g % NSET, f = g % 2;
    P[f] = mfma_fp6_32x32x64(aq[s][0], ap[s][0], bq[s][0], bp[s][0], f32x16{});
#pragma unroll
    for (int k = 1; k < KS; ++k) P[f] = mfma_fp6_32x32x64(aq[s][k], ap[s][k], bq[s][k], bp[s][k], P[f]);
    asm volatile("" : "+v"(P[f]));
  };
  auto mfma_s = [&](int g, int set) {
    S[g % 2] = mfma_bf16_32x32x8(u32x2{xs[set][g % GPS], 0u}, u32x2{ws[set][g % GPS], 0u}, f32x16{});
    asm volatile("" : "+v"(S[g % 2]));
  };
  // rows 0-7 (8-15) of the lane's 16 products
  auto rescale = [&](int f, int half) {
#pragma unroll
    for (int r = 8 * half; r < 8 * half + 8; ++r)
      acc[(r + 2) & 15] = __builtin_fmaf(P[f][r], S[f][(r + 1) & 15], acc[(r + 2) & 15]);   // as rescale_acc
    asm volatile("" : "+v"(acc));
  };

  // the zero words of every buffer, written before the first barrier
  if (tid < 16 * NBUF) *reinterpret_cast<uint32_t*>(sm + (tid / 16) * BUF + OZ + 4 * (tid % 16)) = 0u;
  if (!mover) load_ranks(0);
  if (!SPLIT || mover) {
#pragma unroll
    for (int s = 0; s < NBUF - 1; ++s)
      if (s < nstages) issue(s, s);
    // stage 0 landed
    if (nstages >= NBUF - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NBUF - 2) * D) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  // Stage s + 1 landed, NBUF - 3 younger ones in flight (near the end, none); then the next one's DMA
  // into the buffer of stage s - 1.
  auto landed = [&](int s) {
    if (s + NBUF - 1 <= nstages) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NBUF - 3) * D) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };
  if (mover) {
    for (int s = 0, pb = NBUF - 1; s + 1 < nstages; ++s, pb = pb + 1 == NBUF ? 0 : pb + 1) {
      landed(s);
      asm volatile("s_barrier" ::: "memory");
      if (s + NBUF - 1 < nstages) issue(s + NBUF - 1, pb);
    }
    if constexpr (!OUT_F32) __syncthreads();                // the barrier ahead of the output staging
    return;
  }
  read_scales(0, 0);
#pragma unroll
  for (int g = 0; g < DIST; ++g)
    if (g < ngroups) read_frags(0, g);
  mfma_p(0);
  mfma_s(0, 0);
  int s = 0;
  // A stage that is not the last one.
  auto stage = [&](auto bufc) {
    constexpr int buf = decltype(bufc)::value, nb = (buf + 1) % NBUF, pb = (buf + NBUF - 1) % NBUF;
#pragma unroll
    for (int g = 0; g < GPS; ++g) {
      if (g == GPS - DIST) {
        if constexpr (!SPLIT) landed(s);
        asm volatile("s_barrier" ::: "memory");
        if constexpr (!SPLIT)
          if (s + NBUF - 1 < nstages) issue(s + NBUF - 1, pb);
        read_scales(nb, nb % 2);
      }
      // (a last stage with fewer groups: what is read past them is not used)
      if (g < GPS - DIST) read_frags(buf, g + DIST);
      else read_frags(nb, g + DIST - GPS);
      // one MFMA, then FMAs: a second MFMA right behind would hold the wave until the first is done
      mfma_p(g + 1);
      __builtin_amdgcn_sched_barrier(0);
      rescale(g % 2, 0);
      __builtin_amdgcn_sched_barrier(0);
      mfma_s(g + 1, g + 1 < GPS ? buf % 2 : nb % 2);
      __builtin_amdgcn_sched_barrier(0);
      rescale(g % 2, 1);
    }
    ++s;
  };
  while (s + NBUF < nstages) for_each_index(stage, std::make_integer_sequence<int, NBUF>{});
  const int lbuf = nstages - 1 - s;                         // 0 .. NBUF - 1
  for_each_index([&](auto b) { if (lbuf > decltype(b)::value) stage(b); }, std::make_integer_sequence<int, NBUF - 1>{});
  // the last stage: lg groups
  const int lg = ngroups - (nstages - 1) * GPS;
  if (lbuf % 2) xs[0] = xs[1], ws[0] = ws[1];
#pragma unroll
  for (int g = 0; g < GPS; ++g) {
    if (g < lg) {
      if (g + DIST < GPS && g + DIST < lg) read_frags(lbuf, g + DIST);
      if (g + 1 < GPS && g + 1 < lg) {
        mfma_p(g + 1);
        mfma_s(g + 1, 0);
      }
      rescale(g % 2, 0);
      rescale(g % 2, 1);
    }
  }

  // ---- low-rank term, bias, store ----
  f32x16 t;
#pragma unroll
  for (int r = 0; r < 16; ++r) t[r] = acc[(r + 2) & 15];   // undo rescale_acc's rotation
  acc = t;
  for (int k = 0; k < p.RTp; k += 32) {
    if (k) load_ranks(k);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      acc = mfma_bf16_32x32x16(ehi[u], eb[u], acc);
      acc = mfma_bf16_32x32x16(elo[u], eb[u], acc);
    }
  }
  const int mw = m0 + 32 * wm, nw = n0 + 32 * wn;
  const float bv = p.bias && nw + lr < p.N ? bf16f(p.bias[nw + lr]) : 0.0f;
  if constexpr (OUT_F32) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = mw + 8 * (r >> 2) + 4 * h + (r & 3), n = nw + lr;
      if (m < p.M && n < p.N) reinterpret_cast<float*>(p.y)[(long)m * p.ldy + n] = acc[r] + bv;
    }
  } else {
    // No DMA is in flight (the last stage's arrival waited for all); past this barrier every wave has
    // read its last fragments and the ring holds the waves' staging regions.
    __syncthreads();
    uint8_t* out_stage = sm + wave * 32 * PITCH;
#pragma unroll
    for (int r = 0; r < 16; ++r)
      *reinterpret_cast<uint16_t*>(out_stage + (8 * (r >> 2) + 4 * h + (r & 3)) * PITCH + 2 * lr) =
          (uint16_t)(pack_bf16x2(acc[r] + bv, 0.0f) & 0xFFFFu);
    const bool vec = (reinterpret_cast<uintptr_t>(p.y) & 15) == 0 && p.ldy % 8 == 0;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const int row = 16 * it + lane / 4, c = lane % 4;
      const u32x4 v = *reinterpret_cast<const u32x4*>(out_stage + row * PITCH + 16 * c);
      const int m = mw + row, n = nw + 8 * c;
      if (m >= p.M) continue;
      uint16_t* out = reinterpret_cast<uint16_t*>(p.y) + (long)m * p.ldy + n;
      if (vec && n + 8 <= p.N) {
        *reinterpret_cast<u32x4*>(out) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (n + e < p.N) out[e] = (uint16_t)(v[e / 2] >> (16 * (e % 2)));
      }
    }
  }
}

// Up to MAX_SIBLINGS layers over the same rows (one for a single layer), tiles numbered back to
// back (layer i from tile0[i]).  Block b runs on XCD b mod 8: each XCD takes a contiguous range of
// tiles, row blocks innermost, so the tiles that share weight columns share an L2.
template <int G, int WM, int WN, bool OUT_F32>
__global__ void __launch_bounds__(512) w4a4_e3m2_small_kernel(GemmSiblings gs) {
  const int total = gs.tile0[gs.count], x = blockIdx.x % 8, q = total / 8, r = total % 8;
  const int lin = x * q + min(x, r) + blockIdx.x / 8;
  int i = 0;
#pragma unroll
  for (int c = 1; c < MAX_SIBLINGS; ++c) i += (c < gs.count && lin >= gs.tile0[c]) ? 1 : 0;
  i = __builtin_amdgcn_readfirstlane(i);
  const GemmParams& p = gs.layer[i];
  const int nbm = (p.M + 32 * WM - 1) / (32 * WM), t = lin - gs.tile0[i];
  w4a4_e3m2_small_tile<G, WM, WN, OUT_F32>(p, t % nbm, t / nbm);
}

// The tiles, how many of them share a CU (their LDS), and what a round takes with groups of 64 and of 128.
struct SmallTile {
  const char* name;
  int tm, tn, slots;
  RoundCost us[2][3];
};
// (The third 32x32 tile of a CU is priced 15% above its fit: where the rows outgrow the L2s, the operands that
// such tiles re-read the most come slower than in the fitted grids: M = 2381, N = 256, K = 16384, rank 256 34 us on 64x64, 49 on 32x32.)
constexpr SmallTile kSmallTiles[] = {
    {"32x32", 32, 32, 3,
     {{{1.85f, 1.09f, 0.38f, 1.50f, 1.00f, 0.35f}, {2.01f, 1.28f, 0.39f, 1.89f, 1.22f, 0.40f}, {1.96f, 2.10f, 0.60f, 2.22f, 1.79f, 0.62f}},
      {{1.58f, 0.99f, 0.36f, 1.22f, 0.88f, 0.36f}, {1.53f, 1.14f, 0.41f, 1.53f, 1.10f, 0.39f}, {1.77f, 1.92f, 0.55f, 1.93f, 1.59f, 0.58f}}}},
    {"64x64", 64, 64, 1, {{{2.09f, 1.63f, 0.70f, 1.82f, 1.34f, 0.64f}}, {{1.83f, 1.44f, 0.71f, 1.59f, 1.13f, 0.67f}}}},
    {"128x64", 128, 64, 1, {{{2.02f, 3.17f, 1.27f, 1.51f, 2.80f, 1.17f}}, {{1.97f, 2.73f, 1.30f, 1.46f, 2.34f, 1.23f}}}},
};
constexpr RoundCost kLarge[2] = {{3.70f, 8.59f, 1.08f, 3.10f, 5.95f, 0.64f}, {3.31f, 7.60f, 1.18f, 2.79f, 5.79f, 0.62f}};   // 256 x 128
constexpr float kLaunchUs = 2.0f;   // a further launch
struct W4A4Small {
  int tile;
  float us;
};
constexpr int kSmallCount = sizeof(kSmallTiles) / sizeof(kSmallTiles[0]);
constexpr int kMaxRows = 1 << 25;

long tile_count(int M, const int* N, int count, int tm, int tn) {
  long t = 0;
  for (int i = 0; i < count; ++i) t += ((long)M + tm - 1) / tm * (((long)N[i] + tn - 1) / tn);
  return t;
}

template <int G, int WM, int WN>
hipError_t launch_tile(const GemmSiblings& gs, unsigned tiles, bool out_f32, hipStream_t st) {
  constexpr int threads = 64 * WM * WN * (small_split<WM, WN>() ? 2 : 1);
  if (out_f32) w4a4_e3m2_small_kernel<G, WM, WN, true><<<dim3(tiles), threads, 0, st>>>(gs);
  else w4a4_e3m2_small_kernel<G, WM, WN, false><<<dim3(tiles), threads, 0, st>>>(gs);
  return hipGetLastError();
}

template <int G>
hipError_t launch_g(const GemmSiblings& gs, int tile, unsigned tiles, bool out_f32, hipStream_t st) {
  switch (tile) {
    case 0: return launch_tile<G, 1, 1>(gs, tiles, out_f32, st);
    case 1: return launch_tile<G, 2, 2>(gs, tiles, out_f32, st);
    case 2: return launch_tile<G, 4, 2>(gs, tiles, out_f32, st);
  }
  return hipErrorInvalidValue;
}

// The small tile that takes least, or -1 where the 256 x 128 tiles do; a launch per layer where those do not take
// siblings (K not a multiple of 512).  Rank 32, K = 6144, small / 256 x 128, us:  M = 64, N = 1536 9.4 / 40.3;
// M = 128, N = 6144 13.7 / 41.0; M = 256, N = 6144 23.4 / 41.6; M = 512, N = 6144 37.7 / 42.9; M = 1100,
// N = 1536 24 / 43; and not taken: M = 256, N = 16384 44.8 / 45.3, M = 1024, N = 6144 66 / 50.  Ranks cost a small
// tile more (128x64: 1.3 us per 32 ranks and round; 256 x 128, through LDS: 1.1 for four times the outputs), and a small K
// leaves little to gain: M = 512, N = 6144 (64x64 or 128x64 / 256 x 128) at K = 128, rank 256 25 / 12.5; 512, 128
// 19.6 / 11.7; 1536, 256 31 / 20; 6144, 256 53 / 47; 512, 32 13.1 / 9.4.
W4A4Small choose(int M, const int* N, int count, int K, int G, int RTp) {
  const int g = G == 64 ? 0 : 1;
  W4A4Small best{-1, 0.0f};
  if (count > 1 && K % 512)
    for (int i = 0; i < count; ++i) best.us += choose(M, &N[i], 1, K, G, RTp).us + (i ? kLaunchUs : 0.0f);
  else
    best.us = rounds_us(&kLarge[g], 1, 0.5f, tile_count(M, N, count, 256, 128), K, RTp);
  for (int t = 0; t < kSmallCount; ++t) {
    const SmallTile& k = kSmallTiles[t];
    const float us = rounds_us(k.us[g], k.slots, 0.5f, tile_count(M, N, count, k.tm, k.tn), K, RTp);
    if (us < best.us) best = {t, us};
  }
  return best;
}

}  // namespace

int w4a4_small_tile(int M, const int* N, int count, int K, int G, int RTp) {
  if ((G != 64 && G != 128) || K % G) return -1;
  if (const char* e = getenv("SVDQ_W4A4_TILES")) {   // a tile by name (tests run every tile on one shape)
    for (int t = 0; t < kSmallCount; ++t)
      if (!strcmp(e, kSmallTiles[t].name)) return t;
    if (!strcmp(e, "256x128") || !strcmp(e, "256x256")) return -1;
  }
  // a lane's offset within a stage spans 8 planes of 16 bytes per row, in 32 bits
  for (int i = 0; i < count; ++i)
    if (std::max(M, N[i]) > kMaxRows) return -1;
  return choose(M, N, count, K, G, RTp).tile;
}

void w4a4_small_tile_size(int tile, int& rows, int& cols) {
  rows = kSmallTiles[tile].tm;
  cols = kSmallTiles[tile].tn;
}

hipError_t launch_w4a4_small(const GemmSiblings& gs, int G, int tile, bool out_f32, hipStream_t st) {
  if (tile < 0 || tile >= kSmallCount || gs.count < 1 || gs.count > MAX_SIBLINGS) return hipErrorInvalidValue;
  GemmSiblings w = gs;
  long tiles = 0;
  for (int i = 0; i < w.count; ++i) {
    const GemmParams& p = w.layer[i];
    if (p.M != w.layer[0].M || p.K != w.layer[0].K || p.K % G || p.epi || p.RTp % 32 || std::max(p.M, p.N) > kMaxRows)
      return hipErrorInvalidValue;
    w.tile0[i] = (int)tiles;
    tiles += tile_count(p.M, &p.N, 1, kSmallTiles[tile].tm, kSmallTiles[tile].tn);
    if (tiles > 0x7FFFFFFF) return hipErrorInvalidValue;
  }
  w.tile0[w.count] = (int)tiles;
  if (G == 64) return launch_g<64>(w, tile, (unsigned)tiles, out_f32, st);
  if (G == 128) return launch_g<128>(w, tile, (unsigned)tiles, out_f32, st);
  return hipErrorInvalidValue;
}

}  // namespace svdq
