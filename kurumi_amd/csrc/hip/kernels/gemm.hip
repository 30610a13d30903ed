// GEMM dispatch: the direct-to-LDS MFMA kernel (gemm_lds.hip) for the bf16 / f16 / e4m3
// layouts it covers and fills the chip with, the register-staged MFMA kernel (gemm_flex.hip) for the
// other products of these types and for f32, the generic tiled kernel (gemm_generic.hip) for
// everything else.
#include <hip/hip_runtime.h>

#include <stdexcept>

#include "kernels.h"
#include "numeric.h"

namespace ku::hipbk {

bool gemm_lds_ok(const GemmArgs& a);
std::string gemm_lds_name(const GemmArgs& a);
void launch_gemm_lds(const GemmArgs& a, hipStream_t s);
bool gemm_lds_keeps(const GemmArgs& a);
bool gemm_flex_ok(const GemmArgs& a);
GemmRoute gemm_flex_route(const GemmArgs& a);
std::string gemm_flex_name(const GemmArgs& a, const GemmRoute& r);
double gemm_flex_tiles_elements(const GemmArgs& a, const GemmRoute& r);
double gemm_lds_us(const GemmArgs& a);
void launch_gemm_flex(const GemmArgs& a, const GemmRoute& r, hipStream_t s);

GemmRoute gemm_route(const GemmArgs& a) {
  // Where both take the product, the direct-to-LDS kernel wins when its big tiles fill the chip and
  // loses when they do not (bf16, K x N = 4096 x 11008: 16 rows 63 against 20 us, 300 rows with
  // 2048 x 5504 42 against 25 us; 600 rows 58 against 73 us, 2048 rows 160 against 236 us), so the
  // two kernels' estimates are compared; within 10 % of each other the direct one is kept.
  GemmRoute lds;
  if (gemm_lds_ok(a)) {
    lds.path = GemmPath::LDS;
    lds.us = gemm_lds_us(a);
    if (gemm_lds_keeps(a)) return lds;
  }
  if (!gemm_flex_ok(a)) return lds;
  const GemmRoute flex = gemm_flex_route(a);
  // K within one 16-deep tile of the generic kernel, which a stage of the register-staged one, cut
  // and loaded element by element, does not beat at any size (f32 500 x 500 x 16: 5.1 against 6.0 us,
  // x 20: 6.9 against 6.0); up to twice that where writing C takes the time, which the generic kernel
  // does faster (bf16 3000 x 4001 x 24: 21.7 against 25.4 us; 1000 x 2001 x 24: 8.4 against 7.5).
  if (lds.path != GemmPath::LDS && (a.k <= 16 || (a.k < 32 && gemm_flex_tiles_elements(a, flex) >= 4e6))) return lds;
  return lds.path != GemmPath::LDS || 1.1 * flex.us < lds.us ? flex : lds;
}

std::string gemm_variant(const GemmArgs& a, const GemmRoute& r) {
  switch (r.path) {
    case GemmPath::LDS: return gemm_lds_name(a);
    case GemmPath::FLEX: return gemm_flex_name(a, r);
    default: return "gemm_generic";
  }
}

size_t gemm_scratch_bytes(const GemmArgs& a, const GemmRoute& r) {
  return r.splits > 1 ? (size_t)(r.splits * a.batch * a.m * a.n) * 4 : 0;
}

void launch_gemm(const GemmArgs& a, const GemmRoute& r, hipStream_t s) {
  if (a.batch * a.m * a.n == 0) return;
  // what the route was decided for: the direct kernel's and e4m3's 16-byte loads need the alignment
  if ((r.path == GemmPath::LDS || (r.path == GemmPath::FLEX && a.in_type == GT_F8E4M3)) &&
      ((reinterpret_cast<uintptr_t>(a.a) | reinterpret_cast<uintptr_t>(a.b)) & 15))
    throw std::runtime_error("kurumi_hip gemm: operands are not aligned as planned");
  switch (r.path) {
    case GemmPath::LDS: launch_gemm_lds(a, s); return;
    case GemmPath::FLEX: launch_gemm_flex(a, r, s); return;
    default: launch_gemm_generic(a, s);
  }
}

}  // namespace ku::hipbk
