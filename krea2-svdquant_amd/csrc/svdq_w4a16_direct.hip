// W4A16 SVDQuant GEMM with the weights dequantized straight into MFMA operands.
//
//   y = x_hat @ W^T + mid @ l1cat^T + bias,  W = bf16(q * bf16(sw))     (quant/svd.py:119-163, pack.py:26-44)
//
// Same operands, arithmetic and order as the tiles that stage the dequantized weights through LDS
// (svdq_gemm.hip): 16 columns of K per bf16 MFMA in order, then hi and lo low-rank products 16 ranks at
// a time, bias, one rounding.  Every output has the same bits on every kernel.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <utility>

#include "svdq_common.h"
#include "svdq_kernels.h"

namespace svdq {
namespace {

template <class F, int... B>
__device__ __forceinline__ void for_each_index(F&& f, std::integer_sequence<int, B...>) {
  (f(std::integral_constant<int, B>{}), ...);
}

// bf16(q * s) of 8 packed codes (k0 in the low nibble), two per register in k order.  A nibble u under
// the exponent bits 0x6400 is the half 1024 + u; (1024 + u) s - 1032 s is exact in one mixed-precision
// FMA (19 bits, then 11) and is (u - 8) s; one rounding to bf16.  19 instructions: 3 shifts, 4 AND-ORs,
// 8 v_fma_mix_f32, 4 packs (28 with a byte conversion per code).  mask = 0x000F000F in a scalar and
// one = 0x64006400 in a vector register: as literals they would split each AND-OR in two.
__device__ __forceinline__ u32x4 dequant8(uint32_t v, float s, float ns, uint32_t mask, uint32_t one) {
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  float lo[4], hi[4];   // codes 0-3, 4-7
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const f16x2 u = __builtin_bit_cast(f16x2, ((v >> (4 * e)) & mask) | one);
    lo[e] = __builtin_fmaf((float)u[0], s, ns);
    hi[e] = __builtin_fmaf((float)u[1], s, ns);
  }
  return u32x4{pack_bf16x2(lo[0], lo[1]), pack_bf16x2(lo[2], lo[3]), pack_bf16x2(hi[0], hi[1]), pack_bf16x2(hi[2], hi[3])};
}

// Block tile (32 MI) x (128 NJ): waves 0-3 multiply, wave tile (32 MI) x (32 NJ), each dequantizing the
// weight columns it multiplies into registers, once per row block; waves 4-7 move x_hat and the packed
// codes into LDS by DMA, so that the multiplying waves issue no other memory instruction than the scales.
//
// x_hat: a ring of NBUF stages of 64 columns; rows of 128 bytes, 16-byte chunk c of row r at
// c ^ ((r >> 1) & 7): the 16 lanes of a read phase (16 rows, one chunk) hit 16 distinct bank groups.
// Codes: a ring of R slots of 256 columns of K, 128 bytes per weight column, chunks placed likewise.  A
// DMA instruction then touches 8 lines of 128 bytes; loads straight into the MFMA's lanes touch 32 for
// the same bytes (M = 1024, N = K = 6144 on 64 x 128 tiles: 128 us so, 99 by DMA).
//
// Per stage and multiplying wave: 4 MI NJ MFMAs, under them the dequantization of the next k-step's
// columns (19 VALU instructions per 8 codes) and its fragment reads.  Scales come 3 pairs of stages ahead
// in registers, lane half h loading the pair's stage h (one gather of 32 lines per 2 stages).
//
// Bound by what one wave per SIMD issues in order, about 5 cycles an instruction: at MI = 1 the ~140 of a
// stage (270 ns, 32 x 128, whether 12 or 256 CUs work); at 4 x 2, 32 MFMAs (1024 cycles) and ~250 others
// (680 ns; 930 ns with every CU at work, where the clock falls: 1150 TFLOP/s).  The 192 x 128 tile reads one
// fragment from LDS per MFMA, as fast as LDS delivers them (128 bytes per cycle).
template <int G, int MI, int NJ, int NBUF, bool OUT_F32>
__device__ __forceinline__ void w4a16_direct_tile(const GemmParams& p, int bm, int bn) {
  constexpr int NW = 4, U = 8, PU = U / 2, TBM = 32 * MI, TBN = 128 * NJ, BUF = TBM * 128;
  constexpr int D = MI;                        // x_hat DMA instructions per mover and stage (TBM / 8 over 4)
  constexpr int X = NBUF + 3;                  // stages that the movers' code instructions run ahead
  constexpr int R = (X + 1) / 4 + 1, WSLOT = TBN * 128, W0 = NBUF * BUF;
  constexpr int PITCH = 64 + 16;               // output staging: bytes per row of 32 bf16
  static_assert(U % NBUF == 0 && (NBUF - 2) * (D + NJ) + NJ <= 63, "ring");
  static_assert(NW * 32 * PITCH <= NBUF * BUF, "staging");
  __shared__ __attribute__((aligned(1024))) uint8_t sm[W0 + R * WSLOT];

  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, h = lane >> 5;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wid & 3;
  const int m0 = bm * TBM, n0 = bn * TBN + 32 * NJ * wave;
  const int K = p.K, nst = K / 64, ngroups = K / G;

  if (wid >= NW) {
    // Lane l moves chunk (l & 7) ^ ((r >> 1) & 7) of row r = 8 i + l / 8, i the instruction within the
    // operand's stage or slot: mover w takes i = w + 4 d (x_hat) and w + 4 q (codes, part q of a slot).
    const uint32_t lds0 = lds_offset(sm);
    const uint8_t* xsrc = reinterpret_cast<const uint8_t*>(p.xhat) + (long)m0 * p.ldxh * 2;
    const uint8_t* wsrc = p.qw + (long)bn * TBN * (K / 2);
    uint32_t aoff[D], woff[4 * NJ], wc[4 * NJ];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int r = 8 * (wave + 4 * d) + lane / 8, c = (lane & 7) ^ ((r >> 1) & 7);
      aoff[d] = (uint32_t)min(r, p.M - 1 - m0) * (uint32_t)(2 * p.ldxh) + 16u * c;
    }
#pragma unroll
    for (int q = 0; q < 4 * NJ; ++q) {
      const int r = 8 * (wave + 4 * q) + lane / 8;
      wc[q] = 16u * ((lane & 7) ^ ((r >> 1) & 7));
      woff[q] = (uint32_t)min(r, p.N - 1 - bn * TBN) * (uint32_t)(K / 2);
    }
    auto dma_x = [&](int s, int buf) {
#pragma unroll
      for (int d = 0; d < D; ++d) dma16(xsrc + 128L * s, aoff[d], lds0 + buf * BUF + 1024 * (wave + 4 * d));
    };
    // part q of the slot that holds stages 4 t .. 4 t + 3 (the last slot's chunks past K re-read the last)
    auto dma_w = [&](int t, int q, int slot) {
#pragma unroll
      for (int e = NJ * q; e < NJ * q + NJ; ++e)
        dma16(wsrc, woff[e] + min(128u * t + wc[e], (uint32_t)(K / 2 - 16)), lds0 + W0 + slot * WSLOT + 1024 * (wave + 4 * e));
    };
#pragma unroll
    for (int q = 0; q < 4; ++q) dma_w(0, q, 0);
#pragma unroll
    for (int s = 0; s < NBUF - 1; ++s) {
      if (s < nst) dma_x(s, s);
      if ((4 + s) / 4 * 4 < nst) dma_w((4 + s) / 4, (4 + s) % 4, (4 + s) / 4);
    }
    if (nst >= X) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NBUF - 2) * (D + NJ) + NJ) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    int pb = NBUF - 1, slot = (X / 4) % R;     // buffer of stage s + NBUF - 1, slot of stage s + X
    auto step = [&](int s, auto qc) {
      constexpr int q = decltype(qc)::value;   // (s + X) % 4
      // Stage s + 1 landed, and with it the codes up to the slot of stage s + 2, whose last part was issued
      // in the same step; the NBUF - 3 younger steps in flight.  Without codes left, without stages left: fewer.
      if ((s - 1 + X) / 4 * 4 < nst) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NBUF - 3) * (D + NJ)) : "memory");
      else if (s + NBUF - 1 <= nst) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NBUF - 3) * D) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
      if (s + NBUF - 1 < nst) dma_x(s + NBUF - 1, pb);
      if ((s + X) / 4 * 4 < nst) dma_w((s + X) / 4, q, slot);
      pb = pb + 1 == NBUF ? 0 : pb + 1;
      if (q == 3) slot = slot + 1 == R ? 0 : slot + 1;
    };
    for (int s = 0; s + 1 < nst; s += 4)
      for_each_index([&](auto i) { if (s + i + 1 < nst) step(s + i, std::integral_constant<int, (decltype(i)::value + X) % 4>{}); },
                     std::make_integer_sequence<int, 4>{});
    __syncthreads();                           // the barrier ahead of the output staging
    return;
  }

  const uint16_t* srow[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) srow[j] = p.sw + (long)min(n0 + 32 * j + lr, p.N - 1) * ngroups;
  uint16_t rsc[PU][NJ];
  auto load_scales = [&](int pair, int set) {   // past the end the last group again, not used
#pragma unroll
    for (int j = 0; j < NJ; ++j) rsc[set][j] = srow[j][min(G == 64 ? 2 * pair + h : pair, ngroups - 1)];
  };

  f32x16 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x16{};

  // B operand of the k-step being multiplied and of the next one.  Lane half h reads 16 bytes (32 codes)
  // of its column's 32 bytes of the stage and needs bytes 8 ks + 4 h of them: one v_permlane32_swap per
  // register pair.
  u32x4 b[2][NJ], raw[2][NJ];
  uint32_t mask = 0x000F000Fu, one = 0x64006400u;
  asm volatile("" : "+s"(mask), "+v"(one));
  float sc[NJ], nsc[NJ];
  uint32_t cw[4][NJ], sh[2][NJ];
  auto unpack = [&](auto uc) {
    constexpr int u = decltype(uc)::value;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      uint32_t d0 = raw[u % 2][j][0], d1 = raw[u % 2][j][1], d2 = raw[u % 2][j][2], d3 = raw[u % 2][j][3];
      permlane32_swap(d0, d1);   // d0: dwords 0 | 1 (k-step 0), d1: 4 | 5 (k-step 2)
      permlane32_swap(d2, d3);   // d2: dwords 2 | 3 (k-step 1), d3: 6 | 7 (k-step 3)
      cw[0][j] = d0;
      cw[1][j] = d2;
      cw[2][j] = d1;
      cw[3][j] = d3;
      if (u % 2 == 0) {
        sh[0][j] = sh[1][j] = rsc[u / 2][j];
        if (G == 64) permlane32_swap(sh[0][j], sh[1][j]);   // the lower half's, the upper half's scale in both
      }
      if (G == 64 || u % 2 == 0) {
        sc[j] = round_bf16(half_bits_to_float((uint16_t)sh[u % 2][j]));   // bf16 scale, as the sim
        nsc[j] = -1032.0f * sc[j];
      }
    }
  };
  auto dequant = [&](int ks) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) b[ks % 2][j] = dequant8(cw[ks][j], sc[j], nsc[j], mask, one);
  };
  typedef const __attribute__((address_space(3))) uint8_t* lds_u8;
  typedef const __attribute__((address_space(3))) u32x4* lds_u32x4;
  lds_u8 ra[4], rw[4];   // chunk 2 j + h of row lr: x_hat's k-step j, the code slot's stage j
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = 16 * ((2 * j + h) ^ ((lr >> 1) & 7));
    ra[j] = (lds_u8)&sm[lr * 128 + c];
    rw[j] = (lds_u8)&sm[W0 + (32 * NJ * wave + lr) * 128 + c];
  }
  u32x4 a[2][MI];
  auto read_a = [&](int buf, int ks, int set) {
#pragma unroll
    for (int i = 0; i < MI; ++i) a[set][i] = *(lds_u32x4)(ra[ks] + buf * BUF + 4096 * i);
  };
  int slot = 0;   // byte offset of the slot that raw reads next
  auto read_w = [&](int u, int set) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) raw[set][j] = *(lds_u32x4)(rw[u % 4] + slot + 4096 * j);
  };

#pragma unroll
  for (int i = 0; i < PU - 1; ++i) load_scales(i, i);
  asm volatile("s_barrier" ::: "memory");   // stage 0 and its slot landed
  read_w(0, 0);
  read_w(1, 1);
  read_a(0, 0, 0);
  unpack(std::integral_constant<int, 0>{});
  dequant(0);
  int s = 0;
  // Stage s, buffer and register sets by its index in the unrolled loop.
  auto stage = [&](auto uc, auto tail) {
    constexpr int u = decltype(uc)::value, buf = u % NBUF, nb = (u + 1) % NBUF;
    if (u % 2 == 0) load_scales(s / 2 + PU - 1, (u / 2 + PU - 1) % PU);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks == 3) {
        // Stage s + 1 landed, with the slot of stage s + 2.  Every wave has taken the fragments of stage
        // s - 1 and the codes of stage s + 1: the movers fill what held them next.
        if (!decltype(tail)::value || s + 1 < nst) asm volatile("s_barrier" ::: "memory");
        read_a(nb, 0, 0);
        unpack(std::integral_constant<int, (u + 1) % U>{});
        if ((u + 2) % 4 == 0) slot = slot + WSLOT == R * WSLOT ? 0 : slot + WSLOT;
        read_w(u + 2, u % 2);
      } else {
        read_a(buf, ks + 1, (ks + 1) % 2);
      }
      dequant((ks + 1) % 4);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = mfma_bf16_32x32x16(a[ks % 2][i], b[ks % 2][j], acc[i][j]);
      // the k-step's reads first, then the dequantization spread over its MFMAs
      if (ks == 3) __builtin_amdgcn_sched_group_barrier(0x100, MI + NJ, 0);
      else __builtin_amdgcn_sched_group_barrier(0x100, MI, 0);
#pragma unroll
      for (int i = 0; i < MI * NJ; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, (20 * NJ + MI * NJ - 1) / (MI * NJ), 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    ++s;
  };
  // (the last stage, which meets no barrier, is always left to the tail)
  while (s + U < nst) for_each_index([&](auto u) { stage(u, std::false_type{}); }, std::make_integer_sequence<int, U>{});
  for_each_index([&](auto u) { if (s < nst) stage(u, std::true_type{}); }, std::make_integer_sequence<int, U>{});
  __syncthreads();   // every DMA landed and every fragment read before LDS is used again

  // ---- low-rank term, bias, store ----
  for (int k = 0; k < p.RTp; k += 32) {
    u32x4 eb[NJ][2];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int v = 0; v < 2; ++v)
        eb[j][v] = *reinterpret_cast<const u32x4*>(p.l1cat + (long)min(n0 + 32 * j + lr, p.N - 1) * p.RTp + k + 16 * v + 8 * h);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const uint16_t* arow = p.midp + (long)min(m0 + 32 * i + lr, p.M - 1) * (2 * p.RTp) + k + 8 * h;
      u32x4 ehi[2], elo[2];
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        ehi[v] = *reinterpret_cast<const u32x4*>(arow + 16 * v);
        elo[v] = *reinterpret_cast<const u32x4*>(arow + p.RTp + 16 * v);
      }
#pragma unroll
      for (int v = 0; v < 2; ++v)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          acc[i][j] = mfma_bf16_32x32x16(ehi[v], eb[j][v], acc[i][j]);
          acc[i][j] = mfma_bf16_32x32x16(elo[v], eb[j][v], acc[i][j]);
        }
    }
  }
  uint8_t* stg = sm + wave * 32 * PITCH;
  const bool vec = (reinterpret_cast<uintptr_t>(p.y) & 15) == 0 && p.ldy % 8 == 0;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int nw = n0 + 32 * j;
    const float bv = p.bias && nw + lr < p.N ? bf16f(p.bias[nw + lr]) : 0.0f;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int mw = m0 + 32 * i;
      if constexpr (OUT_F32) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = mw + 8 * (r >> 2) + 4 * h + (r & 3), n = nw + lr;
          if (m < p.M && n < p.N) reinterpret_cast<float*>(p.y)[(long)m * p.ldy + n] = acc[i][j][r] + bv;
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          *reinterpret_cast<uint16_t*>(stg + (8 * (r >> 2) + 4 * h + (r & 3)) * PITCH + 2 * lr) =
              (uint16_t)(pack_bf16x2(acc[i][j][r] + bv, 0.0f) & 0xFFFFu);
#pragma unroll
        for (int it = 0; it < 2; ++it) {
          const int row = 16 * it + lane / 4, c = lane % 4;
          const u32x4 v = *reinterpret_cast<const u32x4*>(stg + row * PITCH + 16 * c);
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
  }
}

// Up to MAX_SIBLINGS layers over the same rows (one for a single layer), tiles numbered back to back;
// each XCD takes a contiguous range of tiles, row blocks innermost (they share weight columns).
template <int G, int MI, int NJ, int NBUF, bool OUT_F32>
__global__ void __launch_bounds__(512) w4a16_direct_kernel(GemmSiblings gs) {
  const int total = gs.tile0[gs.count], x = blockIdx.x % 8, q = total / 8, r = total % 8;
  const int lin = x * q + min(x, r) + blockIdx.x / 8;
  int i = 0;
#pragma unroll
  for (int c = 1; c < MAX_SIBLINGS; ++c) i += (c < gs.count && lin >= gs.tile0[c]) ? 1 : 0;
  i = __builtin_amdgcn_readfirstlane(i);
  const GemmParams& p = gs.layer[i];
  const int nbm = (p.M + 32 * MI - 1) / (32 * MI), t = lin - gs.tile0[i];
  w4a16_direct_tile<G, MI, NJ, NBUF, OUT_F32>(p, t % nbm, t / nbm);
}

struct Tile {
  const char* name;
  int tm, tn, slots;
  RoundCost us[2];   // within 3-5% of the measured times in the root mean square
  float flat = 0.5f;
};
constexpr Tile kTiles[] = {
    {"32x128", 32, 128, 1, {{1.81f, 3.92f, 0.70f, 1.71f, 3.70f, 0.68f}}},
    {"64x128", 64, 128, 2, {{2.19f, 5.15f, 1.12f, 2.00f, 4.58f, 1.11f}, {1.95f, 9.38f, 2.00f, 2.12f, 8.44f, 2.03f}}},
    {"128x128", 128, 128, 1, {{3.29f, 8.17f, 1.99f, 3.32f, 6.13f, 1.98f}}},
    {"192x128", 192, 128, 1, {{3.99f, 11.05f, 3.24f, 4.59f, 7.54f, 2.90f}}},
    {"128x256", 128, 256, 1, {{5.21f, 14.11f, 2.54f, 5.82f, 9.77f, 2.34f}}},
};
constexpr int kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);
// the older kernels (svdq_gemm.hip): specialized waves, and register-staged
constexpr Tile kWs = {"192x256", 192, 256, 1, {{6.58f, 22.08f, 1.39f, 7.22f, 15.51f, 0.98f}}};
constexpr Tile kWide = {"256x256", 256, 256, 1, {{6.81f, 31.46f, 4.67f, 8.87f, 6.00f, 4.97f}}, 0.0f};
constexpr Tile kStaged = {"128x128staged", 128, 128, 2, {{3.90f, 12.94f, 1.38f, 3.51f, 12.18f, 1.38f}, {4.00f, 21.24f, 2.31f, 5.09f, 18.24f, 2.39f}}};
constexpr float kLaunchUs = 2.0f;   // a further launch

long tile_count(const GemmSiblings& gs, const Tile& t) {
  long n = 0;
  for (int i = 0; i < gs.count; ++i)
    n += ((long)gs.layer[i].M + t.tm - 1) / t.tm * (((long)gs.layer[i].N + t.tn - 1) / t.tn);
  return n;
}
float tile_us(const GemmSiblings& gs, const Tile& t) {
  int rtp = 0;
  for (int i = 0; i < gs.count; ++i) rtp = std::max(rtp, gs.layer[i].RTp);
  return rounds_us(t.us, t.slots, t.flat, tile_count(gs, t), gs.layer[0].K, rtp);
}
// A direct tile: x_hat beyond what the L2s hold is read again for every column of tiles, at about 7 TB/s
// (M = 12288, N = 1536, K = 6144 on 192x128: 274 us for 1.8 GB, where its rounds alone would take 220).
float direct_us(const GemmSiblings& gs, const Tile& t) {
  float mb = 0.0f;
  for (int i = 0; i < gs.count; ++i)
    mb += ((long)gs.layer[i].N + t.tn - 1) / t.tn * (2e-6f * gs.layer[i].M * gs.layer[i].K);
  const float us = tile_us(gs, t);
  return 2e-6f * gs.layer[0].M * gs.layer[0].K > 32.0f ? std::max(us, mb / 7.0f) : us;
}

template <int G, int MI, int NJ, int NBUF>
hipError_t launch_tile(const GemmSiblings& gs, unsigned tiles, bool out_f32, hipStream_t st) {
  if (out_f32) w4a16_direct_kernel<G, MI, NJ, NBUF, true><<<dim3(tiles), 512, 0, st>>>(gs);
  else w4a16_direct_kernel<G, MI, NJ, NBUF, false><<<dim3(tiles), 512, 0, st>>>(gs);
  return hipGetLastError();
}
template <int G>
hipError_t launch_g(const GemmSiblings& gs, int tile, unsigned tiles, bool out_f32, hipStream_t st) {
  switch (tile) {
    case 0: return launch_tile<G, 1, 1, 8>(gs, tiles, out_f32, st);
    case 1: return launch_tile<G, 2, 1, 4>(gs, tiles, out_f32, st);   // (80 KB: two workgroups per CU)
    case 2: return launch_tile<G, 4, 1, 4>(gs, tiles, out_f32, st);
    case 3: return launch_tile<G, 6, 1, 4>(gs, tiles, out_f32, st);
    case 4: return launch_tile<G, 4, 2, 4>(gs, tiles, out_f32, st);
  }
  return hipErrorInvalidValue;
}

}  // namespace

// The kernel that takes least by its rounds of tiles; the older ones unless a direct tile gains 3% (10% on the
// 256 x 256 tiles, which re-read the least where there are many row blocks).  Measured,
// older / direct, us.  Rank 32, K = 6144:  M = 64, N = 1536: 80 / 26 (32x128);  M = 77, N = 16384: 84 / 39 (64x128);
// M = 256, N = 6144: 82 / 37 (64x128);  M = 512, N = 6144: 87 / 52 (128x128);  M = 768, N = 8192: 130 / 74 (192x128);
// M = 1024, N = 6144: 128 / 84, M = 4096, N = 6144: 353 / 283 (128x256).  A direct tile gathers its low-rank operands from 32
// lines per instruction (192x128: 3.2 us per 32 ranks; specialized waves, by DMA: 1.4), and a small K leaves little
// of what it gains elsewhere, so rank and K decide too (K, rank; 192x256 or 256x256 / direct): M = 1100, N = 16384: 128,
// 256 39 / 91; M = 3000, N = 6144: 512, 256 52 / 112; M = 1100, N = 16384: 1536, 128 79 / 98; M = 4352, N = 6144: 6144,
// 256 403 / 459; M = 4352, N = 16384: 6144, 256 849 / 950.
// These kernels take byte offsets from the tile's first row and column in 32 bits: rows of x_hat below
// 2^24 bytes, K below 2^25.  SVDQ_W4A16_TILES=<name> in the environment forces a kernel where it can run, so that
// tests can run all on one shape.
W4A16Route w4a16_route(const GemmSiblings& gs) {
  const char* e = getenv("SVDQ_W4A16_TILES");
  const char* ke = getenv("SVDQ_W4A16_KERNEL");
  bool ws = true, direct = true;
  for (int i = 0; i < gs.count; ++i) {
    ws = ws && w4a16_ws_fits(gs.layer[i]);
    direct = direct && gs.layer[i].ldxh < (1L << 23) && gs.layer[i].K < (1 << 25) && !gs.layer[i].epi;
  }
  W4A16Route best{W4A16_WIDE, 0.0f};
  if (gs.count > 1) {
    if (ke && !strcmp(ke, "wide")) return best;
    for (int i = 0; i < gs.count; ++i) {
      GemmSiblings one{};
      one.count = 1;
      one.layer[0] = gs.layer[i];
      best.us += w4a16_route(one).us + (i ? kLaunchUs : 0.0f);
    }
    if (const float c = tile_us(gs, kWs); ws && (c < best.us || (e && !strcmp(e, kWs.name)))) best = {W4A16_WS, c};
  } else {
    // 256 x 256 tiles where they fill half the chip, 192 rows where those need fewer rounds x rows
    const long wide = tile_count(gs, kWide), t192 = tile_count(gs, kWs);
    if (wide < 128) best = {W4A16_STAGED, tile_us(gs, kStaged)};
    else if (ws && (t192 + 255) / 256 * 192 < (wide + 255) / 256 * 256) best = {W4A16_WS, tile_us(gs, kWs)};
    else best = {W4A16_WIDE, tile_us(gs, kWide)};
    if (e && !strcmp(e, kStaged.name)) return {W4A16_STAGED, best.us};
    if (e && !strcmp(e, kWide.name)) return {W4A16_WIDE, best.us};
    if (e && ws && !strcmp(e, kWs.name)) return {W4A16_WS, best.us};
  }
  if (e && ws && !strcmp(e, kWs.name)) return best;
  float most = (best.tile == W4A16_WIDE && gs.count == 1 ? 0.90f : 0.97f) * best.us;
  for (int t = 0; t < kTileCount && direct; ++t) {
    const float c = direct_us(gs, kTiles[t]);
    if (e && !strcmp(e, kTiles[t].name)) return {t, c};
    if (c < most) best = {t, c}, most = c;
  }
  return best;
}

void w4a16_tile(int tile, int& rows, int& cols) {
  const Tile& t = tile >= 0 ? kTiles[tile] : tile == W4A16_WS ? kWs : tile == W4A16_STAGED ? kStaged : kWide;
  rows = t.tm;
  cols = t.tn;
}

hipError_t launch_w4a16_direct(const GemmSiblings& gs, int G, int tile, bool out_f32, hipStream_t st) {
  if (tile < 0 || tile >= kTileCount || gs.count < 1 || gs.count > MAX_SIBLINGS) return hipErrorInvalidValue;
  GemmSiblings w = gs;
  long tiles = 0;
  for (int i = 0; i < w.count; ++i) {
    const GemmParams& p = w.layer[i];
    if (p.M != w.layer[0].M || p.K != w.layer[0].K || p.K % G || p.epi || p.RTp % 32) return hipErrorInvalidValue;
    w.tile0[i] = (int)tiles;
    tiles += ((long)p.M + kTiles[tile].tm - 1) / kTiles[tile].tm * (((long)p.N + kTiles[tile].tn - 1) / kTiles[tile].tn);
    if (tiles > 0x7FFFFFFF) return hipErrorInvalidValue;
  }
  w.tile0[w.count] = (int)tiles;
  if (G == 64) return launch_g<64>(w, tile, (unsigned)tiles, out_f32, st);
  if (G == 128) return launch_g<128>(w, tile, (unsigned)tiles, out_f32, st);
  return hipErrorInvalidValue;
}

}  // namespace svdq
