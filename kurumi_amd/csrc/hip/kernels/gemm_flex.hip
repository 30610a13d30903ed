// Host side of the register-staged MFMA GEMM (gemm_flex.h): tile and split choice, launches, and the
// fold of split products.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <string>

#include "gemm_flex.h"

namespace ku::hipbk {

namespace {

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

int64_t width(const GemmArgs& a) { return a.in_type == GT_F32 ? 4 : a.in_type == GT_F8E4M3 ? 1 : 2; }
int64_t stages(const GemmArgs& a) { return (a.k * width(a) + KB - 1) / KB; }

// Estimated microseconds of a tile and split, from sweeps over 35 products (f32 and bf16, both
// layouts, 1 to 4096 rows, every tile and split): a stage takes `busy` us of a CU's time when
// enough work-groups share it and `alone` us of latency when one has it to itself (k-contiguous B
// reads one 128-byte line per row and stage, from rows often a power of two apart: slower alone);
// reading the operands takes bytes / 5 TB/s, more where few work-groups keep loads in flight; a split
// adds the fold's launch (nearly 4 us where launches are what bounds the stream) and the partial
// sums' round trip. The choice was within 10 % of the best tile and split measured.
struct Rate { double busy, alone_nn, alone_nt; };

}  // namespace

double gemm_flex_cost(const GemmArgs& a, int tile, int64_t splits, double extra, double b_bytes) {
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
  const bool odd = width(a) == 2 && tile > 0 && ((a.sam | (a.sbk == 1 ? a.sbn : a.sbk)) & 7) != 0;
  const double bytes = (double)(a.m * a.k + a.m * a.n) * a.batch * width(a) + b_bytes;
  double us = (tile == 0 && is32 ? 14 : 4) + std::max({(double)(w * per) * (r.busy * (odd ? 1.45 : 1.0) + extra),
                            (double)((w + resident[tile] - 1) / resident[tile] * per) * (a.sbk == 1 ? r.alone_nt : r.alone_nn),
                            bytes / 5e6 * (1 + 0.3 * cu_count() / wgs)});
  if (splits > 1) us += 4 + (double)(splits * a.batch * a.m * a.n) * 8 / 4.5e6;
  return us;
}

GemmRoute gemm_flex_route(const GemmArgs& a) {
  GemmRoute best{GemmPath::FLEX, 2, 1, 1e30};
  const int64_t kt = stages(a);
  for (int i = 0; i < 3; ++i) {
    if (i < 2 && kTiles[i].bm >= 2 * a.m) continue;  // more than half of the tile's rows past M
    for (int64_t s = 1; s <= 64 && (s == 1 || kt / s >= 2); s *= 2) {
      // e4m3: the partial sums fit beside the quantised activation in the static scratch of the entry
      // point that does not allocate, so that one rule gives the same sums through every entry point
      if (a.in_type == GT_F8E4M3 && s > 1 &&
          (uint64_t)(a.batch * (s * a.m * a.n * 4 + a.m * a.k)) > kLinearE4m3ScratchBytes - 8192)
        break;
      const double us = gemm_flex_cost(a, i, s, 0, (double)(a.k * a.n) * a.batch * width(a));
      if (us < best.us) best = {GemmPath::FLEX, i, s, us};
    }
  }
  return best;
}

bool gemm_flex_ok(const GemmArgs& a) {
  if (const char* e = std::getenv("KURUMI_HIP_NO_MFMA"); e && *e && *e != '0') return false;
  if (!(a.in_type == GT_BF16 || a.in_type == GT_F16 || a.in_type == GT_F32 || a.in_type == GT_F8E4M3)) return false;
  if (a.in_type == GT_F8E4M3) {
    // whole stages of 16-byte aligned rows, k-contiguous; more than 1024 rows stay with the direct
    // kernel (its path's tests pin its tiles there, and at a layer's widths they fill the chip)
    const auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    if (a.sbk != 1 || a.k % 128 != 0 || ((a.sam | a.sbn | a.sab | a.sbb) & 15) || !al(a.a) || !al(a.b) || a.m > 1024) return false;
  }
  if (!(a.out_type == GT_BF16 || a.out_type == GT_F16 || a.out_type == GT_F32)) return false;
  if (a.k <= 0 || a.m <= 0 || a.n <= 0 || a.sak != 1 || !(a.sbk == 1 || a.sbn == 1)) return false;
  return a.batch <= 65535 && (a.m + 31) / 32 * ((a.n + 63) / 64) < ((int64_t)1 << 24);
}

// elements of C that the route's tiles cover, those past M and N included
double gemm_flex_tiles_elements(const GemmArgs& a, const GemmRoute& r) {
  const Tile& t = kTiles[r.tile];
  return (double)((a.m + t.bm - 1) / t.bm * t.bm) * (double)((a.n + t.bn - 1) / t.bn * t.bn) * (double)a.batch;
}

std::string gemm_flex_name(const GemmArgs& a, const GemmRoute& p) {
  std::string n = a.in_type == GT_F8E4M3 ? "gemm_mfma_e4m3" : a.in_type == GT_F32 ? "gemm_mfma_f32" : a.in_type == GT_F16 ? "gemm_mfma_f16" : "gemm_mfma_bf16";
  n += a.sbk == 1 ? "_nt_" : "_nn_";
  n += std::to_string(kTiles[p.tile].bm) + "x" + std::to_string(kTiles[p.tile].bn) + "_flex";
  if (p.splits > 1) n += "_split" + std::to_string(p.splits);
  return n;
}

void launch_gemm_flex(const GemmArgs& a, const GemmRoute& r, hipStream_t s) {
  const bool room = a.ws && a.ws_bytes >= gemm_scratch_bytes(a, r);
  const int tile = r.tile;
  const int64_t splits = room ? r.splits : 1;
  FlexArgs f{};
  f.g = a;
  f.part = static_cast<float*>(a.ws);
  const int64_t kt = stages(a);
  f.per = (int)((kt + splits - 1) / splits);
  f.splits = (int)splits;
  const bool nt = a.sbk == 1;
  if (a.in_type == GT_F8E4M3) launch_flex<E_FP8, false>(f, tile, s);
  else if (a.in_type == GT_F32) nt ? launch_flex<E_F32, false>(f, tile, s) : launch_flex<E_F32, true>(f, tile, s);
  else if (a.in_type == GT_F16) nt ? launch_flex<E_F16, false>(f, tile, s) : launch_flex<E_F16, true>(f, tile, s);
  else nt ? launch_flex<E_BF16, false>(f, tile, s) : launch_flex<E_BF16, true>(f, tile, s);
  if (splits > 1) launch_gemm_fold(&f, s);
}

void launch_gemm_fold(const void* flex_args, hipStream_t s) {
  const FlexArgs& f = *static_cast<const FlexArgs*>(flex_args);
  const int64_t total = f.g.batch * f.g.m * f.g.n;
  if (total % 4 == 0) hipLaunchKernelGGL((gemm_fold_k<4>), dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0, s, f);
  else hipLaunchKernelGGL((gemm_fold_k<1>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, f);
}

}  // namespace ku::hipbk
