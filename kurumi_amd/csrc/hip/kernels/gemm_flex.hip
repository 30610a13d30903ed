// MFMA GEMM for every size, alignment and grid the direct-to-LDS kernel (gemm_lds.hip) is not made
// for: f32 operands (v_mfma_f32_32x32x2_f32, full f32 products and sums), 16-bit operands whose
// rows are not 16-byte aligned or whose K is not a multiple of 64, and products with so few tiles
// that K has to be split to fill the chip.
//   C[b][m][n] = alpha * colscale[n] * sum_k A[b][m][k] * B[b][k][n], f32 accumulation, one rounding.
// Semantics: kurumi_core/src/interp/contract.rs:26-64.
//
// Stages of 128 K-bytes travel global -> registers -> LDS, double-buffered with one barrier per
// stage; the loads of stage t + DEPTH are issued before stage t is multiplied. Loads of 16 bytes need only element alignment (the hardware takes any; reading
// 16-bit rows at odd elements as aligned dwords shifted into place measured 8-30 % slower). The last
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
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <string>
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
};

// 16 bytes at any element alignment
template <int EB>
__device__ __forceinline__ u32x4 ld16(const unsigned char* p) {
  typedef u32x4 __attribute__((aligned(2))) u32x4_2;
  typedef u32x4 __attribute__((aligned(4))) u32x4_4;
  if constexpr (EB == 4) return *reinterpret_cast<const u32x4_4*>(p);
  else return *reinterpret_cast<const u32x4_2*>(p);
}
// The first `n` elements of a chunk, zeros after them (n <= 0: all zeros). Every load is made, at
// an element clamped into the chunk's valid part, or at `safe` where it has none: branches here
// would put each chunk's loads behind a wait of its own.
template <int EB>
__device__ __forceinline__ u32x4 ld16_cut(const unsigned char* p, int64_t n, const unsigned char* safe) {
  constexpr int VE = 16 / EB;
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

__device__ __forceinline__ void store_any(void* c, int64_t i, int out_type, float v) {
  if (out_type == GT_F32) static_cast<float*>(c)[i] = v;
  else if (out_type == GT_BF16) static_cast<uint16_t*>(c)[i] = d_bf16_st(v);
  else static_cast<uint16_t*>(c)[i] = d_f16_st(v);
}

template <int E, bool BNMAJ, int BM, int BN, int WM, int WN>
__global__ void __launch_bounds__(WM* WN * 64, 2) gemm_flex_k(FlexArgs fa) {
  constexpr int NT = WM * WN * 64;
  constexpr int EB = E == E_F32 ? 4 : 2;
  constexpr int KE = KB / EB, VE = 16 / EB;     // K elements per stage, elements per 16-byte chunk
  constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 32, FN = TN / 32;
  constexpr int ABYTES = BM * KB, BBYTES = BN * KB;
  constexpr int AI = ABYTES / 16 / NT, BI = BBYTES / 16 / NT;  // chunks per thread and stage
  constexpr int NROW = BN * EB, NCH = NROW / 16;               // n-major B: bytes and chunks per k-row
  static_assert(AI * NT * 16 == ABYTES && BI * NT * 16 == BBYTES, "stage / thread mismatch");
  static_assert(FM >= 1 && FN >= 1 && NCH >= 8, "tile");
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
    } else {
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
  u32x4 ra[DEPTH][AI], rb[DEPTH][BI];
  auto load = [&](u32x4 (&va)[AI], u32x4 (&vb)[BI], int64_t t) {
    if (t < KF) {
#pragma unroll
      for (int i = 0; i < AI; ++i) va[i] = ld16<EB>(asrc[i] + t * KB);
    } else {
#pragma unroll
      for (int i = 0; i < AI; ++i) va[i] = ld16_cut<EB>(asrc[i] + t * KB, a.k - t * KE - (i * NT + tid) % 8 * VE, A);
    }
    if (t < fast) {
#pragma unroll
      for (int i = 0; i < BI; ++i) vb[i] = ld16<EB>(bsrc[i] + t * bstep);
    } else {
#pragma unroll
      for (int i = 0; i < BI; ++i) {
        const int q = i * NT + tid;
        int64_t left;  // elements of the chunk inside B
        if constexpr (BNMAJ) left = t * KE + q / NCH < a.k ? a.n - n0 - q % NCH * VE : 0;
        else left = a.k - t * KE - q % 8 * VE;
        vb[i] = ld16_cut<EB>(bsrc[i] + t * bstep, left, B);
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
  auto put = [&](const u32x4 (&va)[AI], const u32x4 (&vb)[BI], int buf) {
    KU_LDS unsigned char* L = lds + buf * (ABYTES + BBYTES);
#pragma unroll
    for (int i = 0; i < AI; ++i) put_row(L, (i * NT + tid) / 8, (i * NT + tid) % 8, va[i]);
#pragma unroll
    for (int i = 0; i < BI; ++i) {
      const int q = i * NT + tid;
      if constexpr (BNMAJ) *(KU_LDS u32x4*)(L + ABYTES + q / NCH * NROW + (nswz(q % NCH, q / NCH) << 4)) = vb[i];
      else put_row(L + ABYTES, q / 8, q % 8, vb[i]);
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
      put(ra[0], rb[0], 0);
    }
    __syncthreads();
    for (int64_t t = t0; t < t1; ++t) {
      const int cur = (int)(t - t0) & 1;
      if (t + 1 < t1) load(ra[0], rb[0], t + 1);
      compute(cur);
      if (t + 1 < t1) put(ra[0], rb[0], cur ^ 1);  // last read before the previous barrier
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
      put(ra[P ^ 1], rb[P ^ 1], P ^ 1);  // stage t + 1; that buffer was last read before the barrier
      __syncthreads();
    };
    load(ra[0], rb[0], t0);
    load(ra[1], rb[1], t0 + 1);
    put(ra[0], rb[0], 0);
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

// C from the splits' partial sums, added in split order: V consecutive elements per thread.
template <int V>
__global__ void __launch_bounds__(256) gemm_fold_k(FlexArgs fa) {
  const GemmArgs& a = fa.g;
  const int64_t total = a.batch * a.m * a.n, i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
  if (i >= total) return;
  float v[V];
#pragma unroll
  for (int e = 0; e < V; ++e) v[e] = 0.f;
#pragma unroll 4
  for (int z = 0; z < fa.splits; ++z) {
    const float* p = fa.part + z * total + i;
    if constexpr (V == 4) {
      const float4 q = *reinterpret_cast<const float4*>(p);
      v[0] += q.x; v[1] += q.y; v[2] += q.z; v[3] += q.w;
    } else {
      v[0] += p[0];
    }
  }
  const float alpha = a.alpha ? a.alpha[0] : 1.f;
#pragma unroll
  for (int e = 0; e < V; ++e) {
    float cs = alpha;
    if (a.col_scale) cs *= a.col_scale[(i + e) % a.n * a.col_scale_stride];
    v[e] = d_round_through(a.round_type, v[e] * cs);
  }
  if (a.out_type == GT_F32 && V == 4) {
    *reinterpret_cast<float4*>(static_cast<float*>(a.c) + i) = make_float4(v[0], v[V > 1 ? 1 : 0], v[V > 2 ? 2 : 0], v[V > 3 ? 3 : 0]);
  } else {
#pragma unroll
    for (int e = 0; e < V; ++e) store_any(a.c, i + e, a.out_type, v[e]);
  }
}

struct Tile { int bm, bn; };
constexpr Tile kTiles[] = {{128, 128}, {64, 64}, {32, 128}};

template <int E, bool BNMAJ>
void launch_flex(const FlexArgs& f, int tile, hipStream_t s) {
  const GemmArgs& a = f.g;
  const Tile t = kTiles[tile];
  const dim3 grid((unsigned)((a.m + t.bm - 1) / t.bm * ((a.n + t.bn - 1) / t.bn) * f.splits), (unsigned)a.batch);
  switch (tile) {
    case 0: hipLaunchKernelGGL((gemm_flex_k<E, BNMAJ, 128, 128, 2, 2>), grid, dim3(256), 0, s, f); break;
    case 1: hipLaunchKernelGGL((gemm_flex_k<E, BNMAJ, 64, 64, 2, 2>), grid, dim3(256), 0, s, f); break;
    default: hipLaunchKernelGGL((gemm_flex_k<E, BNMAJ, 32, 128, 1, 4>), grid, dim3(256), 0, s, f); break;
  }
}

int64_t stages(const GemmArgs& a) { return (a.k * (a.in_type == GT_F32 ? 4 : 2) + KB - 1) / KB; }

// Estimated microseconds of a tile and split, from sweeps over 35 products (f32 and bf16, both
// layouts, 1 to 4096 rows, every tile and split): a stage takes `busy` us of a CU's time when
// enough work-groups share it and `alone` us of latency when one has it to itself (k-contiguous B
// reads one 128-byte line per row and stage, from rows often a power of two apart: slower alone);
// reading the operands takes bytes / 5 TB/s whatever the grid; a split adds the fold's launch and
// the partial sums' round trip. The choice was within 10 % of the best tile and split measured.
struct Rate { double busy, alone_nn, alone_nt; };

double flex_cost(const GemmArgs& a, int tile, int64_t splits) {
  static constexpr Rate f32[] = {{2.05, 2.3, 2.5}, {0.58, 0.76, 1.07}, {0.60, 0.80, 1.08}};
  static constexpr Rate b16[] = {{0.55, 1.1, 1.1}, {0.25, 0.47, 0.58}, {0.27, 0.66, 0.85}};
  static constexpr int resident[] = {2, 4, 4};  // work-groups that fit a CU's LDS
  const bool is32 = a.in_type == GT_F32;
  const Rate r = (is32 ? f32 : b16)[tile];
  const Tile& t = kTiles[tile];
  const int64_t wgs = (a.m + t.bm - 1) / t.bm * ((a.n + t.bn - 1) / t.bn) * a.batch * splits;
  const int64_t per = (stages(a) + splits - 1) / splits, w = (wgs + cu_count() - 1) / cu_count();
  // 16-bit rows that do not start at 16-byte boundaries load slower in narrow tiles (1111 x 2222 x
  // 3333: 0.36 us a 64 x 64 stage)
  const bool odd = !is32 && tile > 0 && ((a.sam | (a.sbk == 1 ? a.sbn : a.sbk)) & 7) != 0;
  const double bytes = (double)(a.m * a.k + a.k * a.n + a.m * a.n) * a.batch * (is32 ? 4 : 2);
  double us = (tile == 0 && is32 ? 14 : 4) + std::max({(double)(w * per) * r.busy * (odd ? 1.45 : 1.0),
                            (double)((w + resident[tile] - 1) / resident[tile] * per) * (a.sbk == 1 ? r.alone_nt : r.alone_nn),
                            bytes / 5e6});
  if (splits > 1) us += 2 + (double)(splits * a.batch * a.m * a.n) * 8 / 4.5e6;
  return us;
}

struct FlexPlan { int tile; int64_t splits; double us; };

FlexPlan flex_plan(const GemmArgs& a) {
  FlexPlan best{2, 1, 1e30};
  const int64_t kt = stages(a);
  for (int i = 0; i < 3; ++i) {
    if (i < 2 && kTiles[i].bm >= 2 * a.m) continue;  // more than half of the tile's rows past M
    for (int64_t s = 1; s <= 64 && (s == 1 || kt / s >= 2); s *= 2) {
      const double us = flex_cost(a, i, s);
      if (us < best.us) best = {i, s, us};
    }
  }
  return best;
}

}  // namespace

bool gemm_flex_ok(const GemmArgs& a) {
  if (const char* e = std::getenv("KURUMI_HIP_NO_MFMA"); e && *e && *e != '0') return false;
  if (!(a.in_type == GT_BF16 || a.in_type == GT_F16 || a.in_type == GT_F32)) return false;
  if (!(a.out_type == GT_BF16 || a.out_type == GT_F16 || a.out_type == GT_F32)) return false;
  if (a.k <= 0 || a.m <= 0 || a.n <= 0 || a.sak != 1 || !(a.sbk == 1 || a.sbn == 1)) return false;
  return a.batch <= 65535 && (a.m + 31) / 32 * ((a.n + 63) / 64) < ((int64_t)1 << 24);
}

// Estimated microseconds of the launch (gemm.hip compares it with the direct-to-LDS kernel's).
double gemm_flex_us(const GemmArgs& a) { return flex_plan(a).us; }

size_t gemm_flex_scratch_bytes(const GemmArgs& a) {
  const FlexPlan p = flex_plan(a);
  return p.splits > 1 ? (size_t)(p.splits * a.batch * a.m * a.n) * 4 : 0;
}

std::string gemm_flex_name(const GemmArgs& a) {
  const FlexPlan p = flex_plan(a);
  std::string n = a.in_type == GT_F32 ? "gemm_mfma_f32" : a.in_type == GT_F16 ? "gemm_mfma_f16" : "gemm_mfma_bf16";
  n += a.sbk == 1 ? "_nt_" : "_nn_";
  n += std::to_string(kTiles[p.tile].bm) + "x" + std::to_string(kTiles[p.tile].bn) + "_flex";
  if (p.splits > 1) n += "_split" + std::to_string(p.splits);
  return n;
}

// one tile shape and split (launch_gemm_flex picks them)
void launch_gemm_flex_as(const GemmArgs& a, int tile, int64_t splits, hipStream_t s) {
  FlexArgs f;
  f.g = a;
  f.part = static_cast<float*>(a.ws);
  const int64_t kt = stages(a);
  f.per = (int)((kt + splits - 1) / splits);
  f.splits = (int)splits;
  const bool nt = a.sbk == 1;
  if (a.in_type == GT_F32) nt ? launch_flex<E_F32, false>(f, tile, s) : launch_flex<E_F32, true>(f, tile, s);
  else if (a.in_type == GT_F16) nt ? launch_flex<E_F16, false>(f, tile, s) : launch_flex<E_F16, true>(f, tile, s);
  else nt ? launch_flex<E_BF16, false>(f, tile, s) : launch_flex<E_BF16, true>(f, tile, s);
  if (splits > 1) {
    const int64_t total = a.batch * a.m * a.n;
    if (total % 4 == 0) hipLaunchKernelGGL((gemm_fold_k<4>), dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0, s, f);
    else hipLaunchKernelGGL((gemm_fold_k<1>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, f);
  }
}

void launch_gemm_flex(const GemmArgs& a, hipStream_t s) {
  const FlexPlan p = flex_plan(a);
  const bool room = a.ws && a.ws_bytes >= (size_t)(p.splits * a.batch * a.m * a.n) * 4;
  launch_gemm_flex_as(a, p.tile, p.splits > 1 && room ? p.splits : 1, s);
}

}  // namespace ku::hipbk
