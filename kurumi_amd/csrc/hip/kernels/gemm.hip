// GEMM dispatch: the direct-to-LDS MFMA kernel (gemm_lds.hip) for the bf16 / f16 / e4m3
// layouts it covers and fills the chip with, the register-staged MFMA kernel (gemm_flex.hip) for the
// other products of these types and for f32, the generic tiled kernel (gemm_generic.hip) for
// everything else.
#include <hip/hip_runtime.h>

#include "kernels.h"
#include "numeric.h"

namespace ku::hipbk {

bool gemm_lds_ok(const GemmArgs& a);
std::string gemm_lds_name(const GemmArgs& a);
void launch_gemm_lds(const GemmArgs& a, hipStream_t s);
bool gemm_lds_keeps(const GemmArgs& a);
bool gemm_flex_ok(const GemmArgs& a);
std::string gemm_flex_name(const GemmArgs& a);
size_t gemm_flex_scratch_bytes(const GemmArgs& a);
double gemm_flex_us(const GemmArgs& a);
double gemm_lds_us(const GemmArgs& a);
void launch_gemm_flex(const GemmArgs& a, hipStream_t s);

namespace {
enum class Path { LDS, FLEX, GENERIC };
Path path_of(const GemmArgs& a) {
  // Where both take the product, the direct-to-LDS kernel wins when its big tiles fill the chip and
  // loses when they do not (bf16, K x N = 4096 x 11008: 16 rows 63 against 20 us, 300 rows with
  // 2048 x 5504 42 against 25 us; 600 rows 58 against 73 us, 2048 rows 160 against 236 us), so the
  // two kernels' estimates are compared; within 10 % of each other the direct one is kept.
  if (gemm_lds_ok(a)) return !gemm_lds_keeps(a) && gemm_flex_ok(a) && 1.1 * gemm_flex_us(a) < gemm_lds_us(a) ? Path::FLEX : Path::LDS;
  return gemm_flex_ok(a) ? Path::FLEX : Path::GENERIC;
}
}  // namespace

std::string gemm_variant(const GemmArgs& a) {
  switch (path_of(a)) {
    case Path::LDS: return gemm_lds_name(a);
    case Path::FLEX: return gemm_flex_name(a);
    default: return "gemm_generic";
  }
}

size_t gemm_scratch_bytes(const GemmArgs& a) { return path_of(a) == Path::FLEX ? gemm_flex_scratch_bytes(a) : 0; }

double gemm_estimated_us(const GemmArgs& a) {
  switch (path_of(a)) {
    case Path::LDS: return gemm_lds_us(a);
    case Path::FLEX: return gemm_flex_us(a);
    default: return 1e9;
  }
}

void launch_gemm(const GemmArgs& a, hipStream_t s) {
  if (a.batch * a.m * a.n == 0) return;
  switch (path_of(a)) {
    case Path::LDS: launch_gemm_lds(a, s); return;
    case Path::FLEX: launch_gemm_flex(a, s); return;
    default: launch_gemm_generic(a, s);
  }
}

}  // namespace ku::hipbk
