// GEMM dispatch: the direct-to-LDS MFMA kernel (gemm_lds.hip) for the bf16 / f16 / e4m3
// layouts it covers, the register-staged MFMA kernel (gemm_flex.hip) for the other 16-bit products
// and for f32, the generic tiled kernel (gemm_generic.hip) for everything else.
#include <hip/hip_runtime.h>

#include "kernels.h"
#include "numeric.h"

namespace ku::hipbk {

bool gemm_lds_ok(const GemmArgs& a);
std::string gemm_lds_name(const GemmArgs& a);
void launch_gemm_lds(const GemmArgs& a, hipStream_t s);
bool gemm_flex_ok(const GemmArgs& a);
std::string gemm_flex_name(const GemmArgs& a);
size_t gemm_flex_scratch_bytes(const GemmArgs& a);
void launch_gemm_flex(const GemmArgs& a, hipStream_t s);

namespace {
enum class Path { LDS, FLEX, GENERIC };
Path path_of(const GemmArgs& a) {
  if (gemm_lds_ok(a)) return Path::LDS;
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

void launch_gemm(const GemmArgs& a, hipStream_t s) {
  if (a.batch * a.m * a.n == 0) return;
  switch (path_of(a)) {
    case Path::LDS: launch_gemm_lds(a, s); return;
    case Path::FLEX: launch_gemm_flex(a, s); return;
    default: launch_gemm_generic(a, s);
  }
}

}  // namespace ku::hipbk
