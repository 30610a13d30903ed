// Fused scaled-dot-product attention over [bh, s, d] (kernel family 4).
//
// Semantics: out = softmax(scale * q k^T [+ causal -inf above the diagonal]) v per head,
// the oracle of `Op::Sdpa` (kurumi_core/src/interp/nn.rs:125-172) and of the decomposed
// chain (graph/ops/nn/attention.rs:97-113). The kernel keeps scores and the running
// softmax in f32 (online softmax, never materialising [s, s]) and rounds the output once.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>

#include "attention_row.h"
#include "kernels.h"
#include "numeric.h"

namespace ku::hipbk {

void launch_attention_mfma(const AttnArgs& a, hipStream_t s);
bool attention_mfma_ok(const AttnArgs& a);
void launch_attention_f32(const AttnArgs& a, hipStream_t s);
bool attention_f32_ok(const AttnArgs& a);

namespace {

// Sequences of a few positions and unaligned buffers: one thread per query row.
template <int D, int DT, class T>
__global__ void __launch_bounds__(64) attn_rowwise_k(AttnArgs a) {
  const int64_t qi = (int64_t)blockIdx.x * 64 + threadIdx.x;
  if (qi < a.s) attn_row<D, DT, T>(a, blockIdx.y, qi);
}

template <int D>
void launch_rowwise(const AttnArgs& a, hipStream_t s) {
  dim3 grid((unsigned)((a.s + 63) / 64), (unsigned)a.bh);
  switch (a.dtype) {
    case GT_BF16: hipLaunchKernelGGL((attn_rowwise_k<D, GT_BF16, uint16_t>), grid, dim3(64), 0, s, a); return;
    case GT_F16: hipLaunchKernelGGL((attn_rowwise_k<D, GT_F16, uint16_t>), grid, dim3(64), 0, s, a); return;
    case GT_F32: hipLaunchKernelGGL((attn_rowwise_k<D, GT_F32, float>), grid, dim3(64), 0, s, a); return;
    default: throw std::runtime_error("kurumi_hip attention: unsupported dtype");
  }
}
// The tiled kernels' time is that of their one tile of 32 queries or more however few it holds, a
// query's chain costs 0.7 to 2.5 us a key. 25 heads, this kernel against the tiled one (us):
//   f32, d 32:   1 position 3.7 / 5.0, 4 positions 4.3 / 5.0, 5 positions 5.0 / 4.8
//   f32, d 64:   1: 3.7 / 6.6, 5: 6.1 / 6.3, 8: 8.6 / 6.6
//   f32, d 128:  1: 4.9 / 11.4, 3: 9.9 / 10.7, 4: 12.4 / 11.5
//   f16, d 32:   1: 3.6 / 5.2, 4: 4.9 / 5.2, 5: 5.8 / 5.2
// 16-bit heads of 64 and 128 stay with the tiled kernel at every length.
bool few_positions(const AttnArgs& a) {
  return (a.dtype == GT_F32 || a.d == 32) && a.s <= (a.d == 128 ? 3 : a.d == 64 ? 5 : 4) && a.bh <= 65535;
}

}  // namespace

bool attn_supported(const AttnArgs& a) {
  bool dt = a.dtype == GT_BF16 || a.dtype == GT_F16 || a.dtype == GT_F32;
  bool d = a.d == 32 || a.d == 64 || a.d == 128;
  return dt && d && a.s > 0 && a.bh > 0;
}

const char* attn_variant(const AttnArgs& a) {
  if (few_positions(a)) return "attn_rowwise";
  if (attention_mfma_ok(a)) return "attn_mfma";
  if (attention_f32_ok(a)) return "attn_mfma_f32";
  return "attn_rowwise";
}

void launch_attention(const AttnArgs& a, hipStream_t s) {
  if (!attn_supported(a)) throw std::runtime_error("kurumi_hip attention: unsupported shape");
  const bool few = few_positions(a);
  if (!few && attention_mfma_ok(a)) {
    launch_attention_mfma(a, s);
    return;
  }
  if (!few && attention_f32_ok(a)) {
    launch_attention_f32(a, s);
    return;
  }
  switch (a.d) {
    case 32: launch_rowwise<32>(a, s); return;
    case 64: launch_rowwise<64>(a, s); return;
    default: launch_rowwise<128>(a, s); return;
  }
}

}  // namespace ku::hipbk
