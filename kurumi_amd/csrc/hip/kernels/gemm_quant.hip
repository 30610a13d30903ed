// Weight-only quantised products through the register-staged MFMA GEMM (gemm_flex.h): the packed
// weight is dequantised on its way into LDS, so it is read once at 2, 4 or 8 bits a value instead of
// being expanded into act's type in memory and read back (int4 [11008, 4096]: 23 MB instead of 23
// + 2 x 90). Every value and, for equal tiles and splits, every sum is that of the expanded weight's
// product. Semantics: kurumi_core/src/interp/contract.rs:69-99 over quant.rs:100-133.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdlib>

#include "gemm_flex.h"

namespace ku::hipbk {

namespace {

GemmArgs as_gemm(const QuantArgs& q) {
  GemmArgs a;
  a.a = q.act;
  a.b = q.qw;
  a.c = q.out;
  a.sam = q.k; a.sak = 1; a.sbn = q.k; a.sbk = 1;
  a.m = q.m; a.n = q.n; a.k = q.k;
  a.in_type = a.out_type = q.act_type;
  a.ws = q.mm_scratch;
  return a;
}

template <int E, int QB, bool SYM>
void launch(const FlexArgs& f, int tile, hipStream_t s) {
  const GemmArgs& a = f.g;
  const Tile t = kTiles[tile];
  const dim3 grid((unsigned)((a.m + t.bm - 1) / t.bm * ((a.n + t.bn - 1) / t.bn) * f.splits));
  switch (tile) {
    case 0: hipLaunchKernelGGL((gemm_flex_k<E, false, 128, 128, 2, 2, QB, SYM>), grid, dim3(256), 0, s, f); break;
    case 1: hipLaunchKernelGGL((gemm_flex_k<E, false, 64, 64, 2, 2, QB, SYM>), grid, dim3(256), 0, s, f); break;
    default: hipLaunchKernelGGL((gemm_flex_k<E, false, 32, 128, 1, 4, QB, SYM>), grid, dim3(256), 0, s, f); break;
  }
}

template <int E>
void launch_bits(const FlexArgs& f, int bits, bool sym, int tile, hipStream_t s) {
  switch (bits * 2 + (sym ? 1 : 0)) {
    case 5: launch<E, 2, true>(f, tile, s); return;
    case 4: launch<E, 2, false>(f, tile, s); return;
    case 9: launch<E, 4, true>(f, tile, s); return;
    case 8: launch<E, 4, false>(f, tile, s); return;
    case 17: launch<E, 8, true>(f, tile, s); return;
    default: launch<E, 8, false>(f, tile, s); return;
  }
}

}  // namespace

GemmRoute quant_flex_route(const QuantArgs& q) {
  const GemmArgs a = as_gemm(q);
  const bool is32 = q.act_type == GT_F32;
  const int64_t kt = (q.k * (is32 ? 4 : 2) + KB - 1) / KB;
  const double b_bytes = (double)q.n * q.k * q.bits / 8;
  GemmRoute best{GemmPath::FLEX, 2, 1, 1e30};
  for (int i = 0; i < 3; ++i) {
    if (i < 2 && kTiles[i].bm >= 2 * q.m) continue;
    // dequantising a stage of B: about 4.5 instructions a value on 64 lanes a clock, as much again
    // for f32 values, which go to LDS one by one
    const double extra = kTiles[i].bn * 64 * 4.5 / 64 / 2100;
    for (int64_t s = 1; s <= 64 && (s == 1 || kt / s >= 2); s *= 2) {
      // Few stages of the 128 x 128 tile in 16 bits take 11 us before the first pays (int4 520 x 4096 x
      // 192 14.0 us, on 64 x 64 tiles 7.8), not the 4 that gemm_flex_cost counts for all.
      const double us = gemm_flex_cost(a, i, s, extra, b_bytes) + (i == 0 && !is32 && kt <= 8 ? 7 : 0);
      if (us < best.us) best = {GemmPath::FLEX, i, s, us};
    }
  }
  return best;
}

bool quant_flex_ok(const QuantArgs& a) {
  if (const char* e = std::getenv("KURUMI_HIP_NO_MFMA"); e && *e && *e != '0') return false;
  if (!(a.act_type == GT_BF16 || a.act_type == GT_F16 || a.act_type == GT_F32)) return false;
  // whole units of 16 values of one group; k / group by a 32-bit multiplication
  if (a.m <= 0 || a.n <= 0 || a.k <= 0 || a.group % 16 != 0 || a.k * a.group >= ((int64_t)1 << 32)) return false;
  if ((reinterpret_cast<uintptr_t>(a.qw) & 15) || (reinterpret_cast<uintptr_t>(a.act) & 3)) return false;
  return (a.m + 31) / 32 * ((a.n + 63) / 64) < ((int64_t)1 << 24);
}

// Whether the product on the packed weight is estimated to take less than expanding it and
// multiplying: dequantising once per tile of rows beats the expanded weight's round trip up to a few
// hundred rows (int4 -> bf16 11008 x 4096: 16 rows 20 us against 49, 100 rows 35 against 60, 256
// rows of int8 61 against 80; 1024 rows 151 against 127, 2048 rows 253 against 182).
bool quant_flex_better(const QuantArgs& q, const GemmRoute& r) {
  if (!quant_flex_ok(q)) return false;
  GemmArgs g = as_gemm(q);
  g.a = g.b = nullptr;
  const double w = q.act_type == GT_F32 ? 4 : 2;
  const double expand = 2 + (double)q.n * q.k * (q.bits / 8.0 + w) / 5e6;  // 11008 x 4096 int4 -> bf16: 24.5 us
  double us = r.us;
  // One or two stages of 16 bits: C is what takes the time, which this kernel writes two bytes a lane
  // (int8 -> bf16 400 x 2048 x 128: 5.4 us against 6.9 expanded; int4 1000 x 4096 x 128: 13.4 against
  // 8.1; 2048 x 11008 x 128: 39.9 against 20.4).
  if (q.k * w <= 2 * KB && w == 2) us = std::max(us, 4 + (double)q.m * q.n * w / 0.9e6);
  return us < expand + gemm_route(g).us;
}

size_t quant_flex_scratch_bytes(const QuantArgs& q, const GemmRoute& r) { return gemm_scratch_bytes(as_gemm(q), r); }

void launch_quant_flex(const QuantArgs& q, const GemmRoute& r, hipStream_t s) {
  GemmRoute c = r;
  if (c.splits > 1 && !q.mm_scratch) c.splits = 1;
  FlexArgs f{};
  f.g = as_gemm(q);
  f.part = static_cast<float*>(q.mm_scratch);
  f.qw = q.qw;
  f.scales = q.scales;
  f.mins = q.mins;
  f.ng = (int)(q.k / q.group);
  f.by_group = (uint32_t)((((uint64_t)1 << 32) + (uint64_t)q.group - 1) / (uint64_t)q.group);
  f.splits = (int)c.splits;
  const int64_t kt = (q.k * (q.act_type == GT_F32 ? 4 : 2) + KB - 1) / KB;
  f.per = (int)((kt + c.splits - 1) / c.splits);
  switch (q.act_type) {
    case GT_F32: launch_bits<E_F32>(f, q.bits, q.sym, c.tile, s); break;
    case GT_F16: launch_bits<E_F16>(f, q.bits, q.sym, c.tile, s); break;
    default: launch_bits<E_BF16>(f, q.bits, q.sym, c.tile, s); break;
  }
  if (c.splits > 1) launch_gemm_fold(&f, s);
}

}  // namespace ku::hipbk
