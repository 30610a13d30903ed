// MFMA GEMM for every size, alignment and grid the direct-to-LDS kernel (gemm_lds.hip) is not made
// for: f32 operands (v_mfma_f32_32x32x2_f32, full f32 products and sums), 16-bit operands whose
// rows are not 16-byte aligned or whose K is not a multiple of 64, and products with so few tiles
// that K has to be split to fill the chip.
//   C[b][m][n] = alpha * colscale[n] * sum_k A[b][m][k] * B[b][k][n], f32 accumulation, one rounding.
// Semantics: kurumi_core/src/interp/contract.rs:26-64.
//
// Stages of 128 K-bytes travel global -> registers -> LDS, double-buffered with one barrier per
// stage; the loads of stage t + DEPTH are issued before stage t is multiplied. Loads of 16
// bytes need only element alignment (the hardware takes any; reading 16-bit rows at odd elements as aligned dwords shifted into place measured 8-30 % slower). The last
// stage of a ragged K loads its cut chunks element by element, zeros past K; rows past M or N
// repeat the last one, unstored.
// LDS layouts are those of gemm_lds.hip (128-byte rows with swizzled chunks; n-major B read with
// transposing reads), except for f32. There the upper half-wave of an MFMA holds the odd k of a
// pair, and pairs are taken in increasing k, so an unsplit sum is the plain fold over k (its bits
// are those of a chain of FMAs). Rows of k keep each 8 k as 0 2 4 6 1 3 5 7, which makes a
// half-wave's four values one 16-byte read; an n-major B is read one float per lane, rows k and
// k + 1 kept 32 floats apart in the banks.
// The tile is A rows x B columns, so a lane owns one column of C and its stores are 128-byte (f32)
// or 64-byte row segments at any N.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "gemm_mfma.h"
#include "kernels.h"
#include "numeric.h"

namespace ku::hipbk {

namespace {

constexpr int E_F32 = 3;

struct FlexArgs {
  GemmArgs g;
  float* part;     // [splits][batch][m][n] partial sums, splits > 1
  int splits;
  int per;         // K stages per split
  // QB: B is a packed weight [n, k * QB / 8], low field first, with an f16 scale (and min) per group
  // of k columns (a multiple of 16)
  const uint8_t* qw;
  const uint16_t* scales;
  const uint16_t* mins;
  int ng;            // groups per row
  uint32_t by_group; // ceil(2^32 / group): k / group is the high half of k * by_group
};

// 16 bytes at any element alignment
template <int EB>
__device__ __forceinline__ u32x4 ld16(const unsigned char* p) {
  typedef u32x4 __attribute__((aligned(2))) u32x4_2;
  typedef u32x4 __attribute__((aligned(4))) u32x4_4;
  if constexpr (EB == 1) return *reinterpret_cast<const u32x4*>(p);  // e4m3 rows are 16-byte aligned
  else if constexpr (EB == 4) return *reinterpret_cast<const u32x4_4*>(p);
  else return *reinterpret_cast<const u32x4_2*>(p);
}
// The first `n` elements of a chunk, zeros after them (n <= 0: all zeros). Every load is made, at
// an element clamped into the chunk's valid part, or at `safe` where it has none: branches here
// would put each chunk's loads behind a wait of its own.
template <int EB>
__device__ __forceinline__ u32x4 ld16_cut(const unsigned char* p, int64_t n, const unsigned char* safe) {
  constexpr int VE = 16 / EB;
  if constexpr (EB == 1) return n > 0 ? ld16<EB>(p) : u32x4{0, 0, 0, 0};  // K a multiple of 128: never cut
  const unsigned char* q = n > 0 ? p : safe;
  const int last = n > 0 ? (int)(n < VE ? n : VE) - 1 : 0;
  u32x4 v = {0, 0, 0, 0};
#pragma unroll
  for (int e = 0; e < VE; ++e) {
    const int at = e < last ? e : last;
    if constexpr (EB == 4) {
      const uint32_t x = reinterpret_cast<const uint32_t*>(q)[at];
      v[e] = e < n ? x : 0u;
    } else {
      const uint32_t x = reinterpret_cast<const uint16_t*>(q)[at];
      v[e >> 1] |= (e < n ? x : 0u) << ((e & 1) * 16);
    }
  }
  return v;
}

// two f32 -> one dword of two operand-type values, rounded to nearest even
template <int E>
__device__ __forceinline__ uint32_t pack16(float lo, float hi) {
  const f32x2 v = {lo, hi};
  if constexpr (E == E_BF16) return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  else return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
}

__device__ __forceinline__ void store_any(void* c, int64_t i, int out_type, float v) {
  if (out_type == GT_F32) static_cast<float*>(c)[i] = v;
  else if (out_type == GT_BF16) static_cast<uint16_t*>(c)[i] = d_bf16_st(v);
  else static_cast<uint16_t*>(c)[i] = d_f16_st(v);
}

// QB: 0, or the bits of a quantised B (k-contiguous rows), dequantised on its way to LDS: each value
// q * scale (+ min) in f32, rounded once to a 16-bit operand type (the values the separate
// dequantisation writes). A unit is 16 values of a row.
template <int E, bool BNMAJ, int BM, int BN, int WM, int WN, int QB = 0, bool SYM = false>
__global__ void __launch_bounds__(WM* WN * 64, 2) gemm_flex_k(FlexArgs fa) {
  constexpr int NT = WM * WN * 64;
  constexpr int EB = E == E_F32 ? 4 : E == E_FP8 ? 1 : 2;
  constexpr int KE = KB / EB, VE = 16 / EB;     // K elements per stage, elements per 16-byte chunk
  constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 32, FN = TN / 32;
  constexpr int ABYTES = BM * KB, BBYTES = BN * KB;
  constexpr int AI = ABYTES / 16 / NT, BI = BBYTES / 16 / NT;  // chunks per thread and stage
  constexpr int NROW = BN * EB, NCH = NROW / 16;               // n-major B: bytes and chunks per k-row
  static_assert(AI * NT * 16 == ABYTES && BI * NT * 16 == BBYTES, "stage / thread mismatch");
  static_assert(FM >= 1 && FN >= 1 && (NCH >= 8 || !BNMAJ) && !(QB && BNMAJ) && !(E == E_FP8 && (BNMAJ || QB)), "tile");
  constexpr int UPR = KE / 16, UI = (BN * UPR + NT - 1) / NT, QW = QB / 2 > 0 ? QB / 2 : 1;  // units per row and thread, words
  __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[2 * (ABYTES + BBYTES)];
  KU_LDS unsigned char* lds = (KU_LDS unsigned char*)lds_raw;
  const GemmArgs& a = fa.g;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5,
            l32 = lane & 31;
  const int wm = wave / WN, wn = wave % WN;
  const int tm = (int)((a.m + BM - 1) / BM), tn = (int)((a.n + BN - 1) / BN);
  const int z = (int)(blockIdx.x / (unsigned)(tm * tn));
  int im, in;
  tile_of((int)(blockIdx.x % (unsigned)(tm * tn)), tm, tn, &im, &in);
  const int64_t m0 = (int64_t)im * BM, n0 = (int64_t)in * BN, bz = blockIdx.y;
  const unsigned char* A = static_cast<const unsigned char*>(a.a) + bz * a.sab * EB;
  const unsigned char* B = static_cast<const unsigned char*>(a.b) + bz * a.sbb * EB;
  const int64_t KT = (a.k + KE - 1) / KE, KF = a.k / KE;  // stages, whole stages
  const int64_t t0 = (int64_t)z * fa.per, t1 = min(KT, t0 + fa.per);

  // per-thread chunks: global source at stage 0
  const unsigned char* asrc[AI];
  const unsigned char* bsrc[BI];
#pragma unroll
  for (int i = 0; i < AI; ++i) {
    const int q = i * NT + tid, r = q / 8, c = q % 8;
    const int64_t gm = m0 + r < a.m ? m0 + r : a.m - 1;
    asrc[i] = A + gm * a.sam * EB + c * 16;
  }
  // swizzle of chunk c of n-major k-row r
  auto nswz = [](int c, int r) {
    if constexpr (EB == 4) return c ^ ((r & 1) * 8);
    else if constexpr (NCH >= 16) return c ^ (4 * (r & 3));
    else return c ^ (4 * ((r >> 1) & 1));
  };
#pragma unroll
  for (int i = 0; i < BI; ++i) {
    const int q = i * NT + tid;
    if constexpr (BNMAJ) {
      const int r = q / NCH, c = q % NCH;
      // chunks wholly past N repeat the one that holds column N - 1
      const int64_t gn = min(n0 + c * VE, n0 + (a.n - 1 - n0) / VE * VE);
      bsrc[i] = B + ((int64_t)r * a.sbk + gn) * EB;
    } else if constexpr (!QB) {
      const int r = q / 8, c = q % 8;
      const int64_t gn = n0 + r < a.n ? n0 + r : a.n - 1;
      bsrc[i] = B + gn * a.sbn * EB + c * 16;
    }
  }
  const int64_t bstep = BNMAJ ? (int64_t)KE * a.sbk * EB : KB;  // bytes between B's stages
  // A chunk that runs past N reads on into the next k-row (its columns past N are never stored);
  // only where there is none, in the last stage, or where rows are shorter than a chunk, is it cut.
  const bool nedge = BNMAJ && n0 + BN > a.n;
  const int64_t fast = nedge ? (a.sbk >= VE ? min(KF, KT - 1) : 0) : KF;  // B's stages of whole chunks
  // Stages in flight. Two for 16-bit 64 x 64 tiles, whose stages are shorter than the memory's
  // latency (1024 x 1024 x 1024: 13.5 -> 11.5 us; 64 x 4096 x 4096 unsplit: 54 -> 38 us); the
  // other tiles lose more to the registers than they gain (16 x 11008 x 4096 on 32 x 128 tiles:
  // 19.7 -> 22.1 us), and an f32 stage's products cover the latency by themselves.
  constexpr int DEPTH = E != E_F32 && BM == 64 ? 2 : 1;
  struct Unit { uint32_t w[QW]; uint16_t s, m; };
  struct Plain { u32x4 v[BI]; };
  struct Packed { Unit u[UI]; };
  using BRegs = std::conditional_t<QB != 0, Packed, Plain>;
  u32x4 ra[DEPTH][AI];
  BRegs rb[DEPTH];
  auto load = [&](u32x4 (&va)[AI], BRegs& vb, int64_t t) {
    if (t < KF) {
#pragma unroll
      for (int i = 0; i < AI; ++i) va[i] = ld16<EB>(asrc[i] + t * KB);
    } else {
#pragma unroll
      for (int i = 0; i < AI; ++i) va[i] = ld16_cut<EB>(asrc[i] + t * KB, a.k - t * KE - (i * NT + tid) % 8 * VE, A);
    }
    if constexpr (QB) {
#pragma unroll
      for (int i = 0; i < UI; ++i) {
        const int q = i * NT + tid, r = q / UPR;
        const int64_t gn = min(n0 + r, a.n - 1), k = t * KE + q % UPR * 16;
        const uint32_t kc = k < a.k ? (uint32_t)k : 0u;  // units past K: any, weighed zero
        Unit& u = vb.u[i];
        const uint8_t* p = fa.qw + gn * (a.k * QB / 8) + kc * QB / 8;
        if constexpr (QB == 8) {
          const u32x4 x = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
          for (int e = 0; e < 4; ++e) u.w[e] = x[e];
        } else if constexpr (QB == 4) {
          const u32x2 x = *reinterpret_cast<const u32x2*>(p);
          u.w[0] = x[0];
          u.w[1] = x[1];
        } else {
          u.w[0] = *reinterpret_cast<const uint32_t*>(p);
        }
        const int64_t gi = gn * fa.ng + __umulhi(kc, fa.by_group);
        u.s = fa.scales[gi];
        if constexpr (!SYM) u.m = fa.mins[gi];
      }
    } else if (t < fast) {
#pragma unroll
      for (int i = 0; i < BI; ++i) vb.v[i] = ld16<EB>(bsrc[i] + t * bstep);
    } else {
#pragma unroll
      for (int i = 0; i < BI; ++i) {
        const int q = i * NT + tid;
        int64_t left;  // elements of the chunk inside B
        if constexpr (BNMAJ) left = t * KE + q / NCH < a.k ? a.n - n0 - q % NCH * VE : 0;
        else left = a.k - t * KE - q % 8 * VE;
        vb.v[i] = ld16_cut<EB>(bsrc[i] + t * bstep, left, B);
      }
    }
  };
  // chunk c of a 128-byte row r
  auto put_row = [](KU_LDS unsigned char* L, int r, int c, const u32x4& v) {
    if constexpr (EB == 4) {  // k even to the first chunk of the pair, k odd to the second
      const int sw = (r >> 1) & 7, half = (c & 1) * 8;
      *(KU_LDS u32x2*)(L + r * KB + (((c & ~1) ^ sw) << 4) + half) = u32x2{v[0], v[2]};
      *(KU_LDS u32x2*)(L + r * KB + (((c | 1) ^ sw) << 4) + half) = u32x2{v[1], v[3]};
    } else {
      *(KU_LDS u32x4*)(L + r * KB + ((c ^ ((r >> 1) & 7)) << 4)) = v;
    }
  };
  auto put = [&](const u32x4 (&va)[AI], const BRegs& vb, int64_t t, int buf) {
    KU_LDS unsigned char* L = lds + buf * (ABYTES + BBYTES);
#pragma unroll
    for (int i = 0; i < AI; ++i) put_row(L, (i * NT + tid) / 8, (i * NT + tid) % 8, va[i]);
    if constexpr (QB) {
#pragma unroll
      for (int i = 0; i < UI; ++i) {
        const int q = i * NT + tid, r = q / UPR, u0 = q % UPR * (16 / VE);
        if (BN * UPR % NT != 0 && r >= BN) continue;
        const bool in = t * KE + q % UPR * 16 < a.k;
        const float s = in ? d_f16_ld(vb.u[i].s) : 0.f, m = in && !SYM ? d_f16_ld(vb.u[i].m) : 0.f;
        float w[16];
#pragma unroll
        for (int e = 0; e < 16; ++e)
          w[e] = d_dequant<QB, SYM>((vb.u[i].w[e * QB / 32] >> (e * QB % 32)) & ((1u << QB) - 1), s, m);
#pragma unroll
        for (int c = 0; c < 16 / VE; ++c) {
          u32x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            v[e] = E == E_F32 ? __float_as_uint(w[c * VE + e]) : pack16<E>(w[(c * VE + 2 * e) & 15], w[(c * VE + 2 * e + 1) & 15]);
          put_row(L + ABYTES, r, u0 + c, v);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < BI; ++i) {
        const int q = i * NT + tid;
        if constexpr (BNMAJ) *(KU_LDS u32x4*)(L + ABYTES + q / NCH * NROW + (nswz(q % NCH, q / NCH) << 4)) = vb.v[i];
        else put_row(L + ABYTES, q / 8, q % 8, vb.v[i]);
      }
    }
  };

  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // 16 bytes of row r of a 128-byte-row operand
  auto row16 = [&](const KU_LDS unsigned char* L, int r, int c) {
    return *(const KU_LDS u32x4*)(L + r * KB + ((c ^ ((r >> 1) & 7)) << 4));
  };
  auto compute = [&](int buf) {
    const KU_LDS unsigned char* LA = lds + buf * (ABYTES + BBYTES);
    const KU_LDS unsigned char* LB = LA + ABYTES;
    if constexpr (E == E_F32) {
      // 8 k per step: half-wave h takes k = 8s + 2e + h, one MFMA per e = 0..3
#pragma unroll
      for (int s = 0; s < KE / 8; ++s) {
        u32x4 af[FM], bf[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) af[i] = row16(LA, wm * TM + i * 32 + l32, 2 * s + h);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const int n = wn * TN + j * 32 + l32;
          if constexpr (BNMAJ) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int k = 8 * s + 2 * e + h;
              bf[j][e] = *(const KU_LDS uint32_t*)(LB + k * NROW + (nswz(n >> 2, k) << 4) + (n & 3) * 4);
            }
          } else {
            bf[j] = row16(LB, n, 2 * s + h);
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(af[i][e]), __uint_as_float(bf[j][e]),
                                                               acc[i][j], 0, 0, 0);
      }
    } else if constexpr (E == E_FP8) {
      // 64 k per MFMA: half-wave h takes 32 consecutive ones, two chunks
#pragma unroll
      for (int s = 0; s < KE / 64; ++s) {
        u32x4 af[FM][2], bf[FN][2];
#pragma unroll
        for (int v = 0; v < 2; ++v) {
#pragma unroll
          for (int i = 0; i < FM; ++i) af[i][v] = row16(LA, wm * TM + i * 32 + l32, 4 * s + 2 * h + v);
#pragma unroll
          for (int j = 0; j < FN; ++j) bf[j][v] = row16(LB, wn * TN + j * 32 + l32, 4 * s + 2 * h + v);
        }
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) Op<E>::run(acc[i][j], af[i], bf[j]);
      }
    } else {
#pragma unroll
      for (int s = 0; s < KE / 16; ++s) {
        u32x4 af[FM], bf[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) af[i] = row16(LA, wm * TM + i * 32 + l32, 2 * s + h);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          if constexpr (BNMAJ) {
            // transposing reads: in each 16-lane group, lane 4k' + q points at k-row k', columns
            // 4q..4q+3, and lane i receives rows 0..3 of column i
            const int g = lane >> 4, c16 = lane & 15;
            const int n = wn * TN + j * 32 + (g & 1) * 16 + (c16 & 3) * 4;
#pragma unroll
            for (int r2 = 0; r2 < 2; ++r2) {
              const int k = s * 16 + (g >> 1) * 8 + r2 * 4 + (c16 >> 2);
              const KU_LDS unsigned char* p = LB + k * NROW + (nswz(n >> 3, k) << 4) + (n & 7) * 2;
              const u32x2 half = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((KU_LDS s16x4*)p));
              bf[j][2 * r2] = half[0];
              bf[j][2 * r2 + 1] = half[1];
            }
          } else {
            bf[j] = row16(LB, wn * TN + j * 32 + l32, 2 * s + h);
          }
        }
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) Op<E>::run(acc[i][j], &af[i], &bf[j]);
      }
    }
  };

  if (DEPTH == 1 || t1 - t0 <= 1) {
    if (t0 < t1) {
      load(ra[0], rb[0], t0);
      put(ra[0], rb[0], t0, 0);
    }
    __syncthreads();
    for (int64_t t = t0; t < t1; ++t) {
      const int cur = (int)(t - t0) & 1;
      if (t + 1 < t1) load(ra[0], rb[0], t + 1);
      compute(cur);
      if (t + 1 < t1) put(ra[0], rb[0], t + 1, cur ^ 1);  // last read before the previous barrier
      __syncthreads();
    }
  } else if constexpr (DEPTH == 2) {
    // Stage t + 2 is requested before stage t is multiplied and put into LDS an iteration later.
    // Past the last stage the requests repeat the first one: with a branch around them the
    // compiler would wait for everything in flight at the next put.
    auto step = [&](int64_t t, auto par) __attribute__((always_inline)) {
      constexpr int P = decltype(par)::value;
      load(ra[P], rb[P], t + 2 < t1 ? t + 2 : t0);
      compute(P);
      put(ra[P ^ 1], rb[P ^ 1], t + 1, P ^ 1);  // stage t + 1; that buffer was last read before the barrier
      __syncthreads();
    };
    load(ra[0], rb[0], t0);
    load(ra[1], rb[1], t0 + 1);
    put(ra[0], rb[0], t0, 0);
    __syncthreads();
    int64_t t = t0;
    for (; t + 1 < t1; t += 2) {
      step(t, std::integral_constant<int, 0>{});
      step(t + 1, std::integral_constant<int, 1>{});
    }
    if (t < t1) compute(0);
  }

  // lane l32 owns column l32 of each 32 x 32 block; register 4g + e is row 8g + 4h + e
  const float alpha = a.alpha ? a.alpha[0] : 1.f;
  const int64_t rbase = m0 + wm * TM + 4 * h, cbase = n0 + wn * TN + l32;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int64_t col = cbase + j * 32;
    if (col >= a.n) continue;
    if (fa.splits > 1) {
      float* P = fa.part + ((int64_t)z * a.batch + bz) * a.m * a.n;
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int64_t row = rbase + i * 32 + 8 * (v >> 2) + (v & 3);
          if (row < a.m) P[row * a.n + col] = acc[i][j][v];
        }
    } else {
      const float cs = a.col_scale ? alpha * a.col_scale[col * a.col_scale_stride] : alpha;
      void* C = static_cast<unsigned char*>(a.c) + bz * a.m * a.n * (a.out_type == GT_F32 ? 4 : 2);
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int64_t row = rbase + i * 32 + 8 * (v >> 2) + (v & 3);
          if (row < a.m) store_any(C, row * a.n + col, a.out_type, d_round_through(a.round_type, acc[i][j][v] * cs));
        }
    }
  }
}

struct Tile { int bm, bn; };
constexpr Tile kTiles[] = {{128, 128}, {64, 64}, {32, 128}};

}  // namespace

// C from the partial sums of FlexArgs::part (gemm_flex.hip)
void launch_gemm_fold(const void* flex_args, hipStream_t s);
// Estimated microseconds of a tile and split of the kernel, `extra` of them per stage for work the
// plain products do not have; `b_bytes` of B to read
double gemm_flex_cost(const GemmArgs& a, int tile, int64_t splits, double extra, double b_bytes);

}  // namespace ku::hipbk
