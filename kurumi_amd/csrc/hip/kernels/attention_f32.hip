// Flash attention forward in f32 on MFMA for gfx950: every product and sum in f32
// (v_mfma_f32_32x32x2_f32), the exponentials by expf.
//
// out[h] = softmax(scale * q[h] k[h]^T [+ causal -inf above the diagonal]) v[h] for each of the
// bh heads of contiguous [bh, s, d] tensors, d 32, 64 or 128 (kurumi_core/src/interp/nn.rs:125-172).
//
// Bound by the f32 matrix rate: a 32 x 32 x 2 product takes 64 cycles and its operands are one
// float per lane, so K and V come straight from the caches (16 bytes a clock and CU) and only Q
// goes through LDS. A work-group is one tile of 32 queries; its waves take blocks of 32 keys in
// turn, each with a running softmax of its own, combined through LDS at the end: the tiles are
// small, so that short sequences still fill the chip. One query per thread, as before, gave the
// [2, 8, 500, 64] tensors 128 waves, each a serial chain over the keys: 444 us.
//
// Computed transposed, so one lane owns one query:
//   S^T[key][q] = K . Q^T: A = K (lane l: key l % 32), B = Q; half-wave h takes dims 8s + 4h + e
//   O^T[d][q] += V^T . P^T: register v of S^T (key 8 (v / 4) + 4h + v % 4 of the block, query l % 32)
//     is the B operand of one product as it stands; A = V, lane l: dim l % 32 of that key.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdlib>

#include "kernels.h"

namespace ku::hipbk {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int NW = 4;  // waves per work-group

// the value of the lane that holds the same query in the other half of the wave
__device__ __forceinline__ float other_half(float v) { return __shfl_xor(v, 32, 64); }

template <int D>
__global__ void __launch_bounds__(NW * 64, 2) attn_f32_k(AttnArgs a) {
  constexpr int DT = D / 32, CH = D / 4;  // 32-dim tiles of O^T, 16-byte chunks per row
  constexpr int TP = DT < 2 ? DT : 2;     // tiles whose V is in registers at a time
  // Q, then (once every wave is done with it) each wave's O^T; rows of D floats, chunk c of query
  // row r at c ^ (r % CH)
  __shared__ __attribute__((aligned(16))) f32x4 rows[NW][32][CH];
  __shared__ float stat[2][NW][32];  // each wave's running max and sum
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5,
            l32 = lane & 31;
  const int64_t S = a.s, nqt = (S + 31) / 32;
  const int64_t head = blockIdx.x % a.bh, back = blockIdx.x / a.bh;
  const int64_t q0 = (a.causal ? nqt - 1 - back : back) * 32;  // causal: the longest tiles first
  const float* Q = static_cast<const float*>(a.q) + head * S * D;
  const float* K = static_cast<const float*>(a.k) + head * S * D;
  const float* V = static_cast<const float*>(a.v) + head * S * D;
  for (int i = tid; i < 32 * CH; i += NW * 64) {
    const int r = i / CH, c = i % CH;
    rows[0][r][c ^ (r % CH)] = *reinterpret_cast<const f32x4*>(Q + min(q0 + r, S - 1) * D + c * 4);
  }
  __syncthreads();

  const int64_t qi = q0 + l32;                              // this lane's query
  const int64_t last = a.causal ? min(qi, S - 1) : S - 1;   // its last visible key
  const int64_t kend = a.causal ? min(q0 + 32, S) : S;      // keys the tile needs
  f32x16 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[t][v] = 0.f;
  float m = -INFINITY, l = 0.f;  // l: this half-wave's keys
  for (int64_t k0 = wave * 32; k0 < kend; k0 += NW * 32) {
    const float* kr = K + min(k0 + l32, S - 1) * D + 4 * h;
    f32x16 sc;
#pragma unroll
    for (int v = 0; v < 16; ++v) sc[v] = 0.f;
#pragma unroll
    for (int s = 0; s < D / 8; ++s) {
      const f32x4 kf = *reinterpret_cast<const f32x4*>(kr + 8 * s), qf = rows[0][l32][(2 * s + h) ^ (l32 % CH)];
#pragma unroll
      for (int e = 0; e < 4; ++e) sc = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[e], qf[e], sc, 0, 0, 0);
    }
    // V of the block, TP tiles of dims at a time: zeros past the sequence, whose probabilities are
    // zero too; `odd` becomes true where there is an infinity or NaN among them
    auto load_v = [&](int t0, float (&vf)[TP][16], bool& odd) {
      odd = false;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int64_t key = k0 + 8 * (v >> 2) + 4 * h + (v & 3);
#pragma unroll
        for (int t = 0; t < TP; ++t) {
          const float x = V[min(key, S - 1) * D + 32 * (t0 + t) + l32];
          vf[t][v] = key < S ? x : 0.f;
        }
      }
#pragma unroll
      for (int t = 0; t < TP; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) odd = odd || !(fabsf(vf[t][v]) < INFINITY);
    };
    float vf[TP][16];
    bool odd;
    load_v(0, vf, odd);
    const int lim = (int)min(last - k0, (int64_t)32) - 4 * h;
    float bm = -INFINITY;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      sc[v] = 8 * (v >> 2) + (v & 3) > lim ? -INFINITY : sc[v] * a.scale;
      bm = fmaxf(bm, sc[v]);
    }
    const float mn = fmaxf(m, fmaxf(bm, other_half(bm)));
    // no key with a finite score yet: every probability is exp(-inf) = 0
    const float base = mn == -INFINITY ? 0.f : mn, corr = expf(m - base);
    m = mn;
    l *= corr;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      sc[v] = expf(sc[v] - base);
      l += sc[v];
    }
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) o[t][v] *= corr;
#pragma unroll
    for (int t0 = 0; t0 < DT; t0 += TP) {
      if (t0 > 0) load_v(t0, vf, odd);
      // Where the block crosses the diagonal a query must not meet the V of keys it does not see:
      // 0 * inf is NaN. Such values (rare) stay out of the product and are added one by one.
      const bool by_hand = a.causal && k0 + 31 > q0 && __builtin_amdgcn_ballot_w64(odd) != 0;
      if (by_hand) {
#pragma unroll
        for (int t = 0; t < TP; ++t)
#pragma unroll
          for (int v = 0; v < 16; ++v) vf[t][v] = fabsf(vf[t][v]) < INFINITY ? vf[t][v] : 0.f;
      }
#pragma unroll
      for (int v = 0; v < 16; ++v)
#pragma unroll
        for (int t = 0; t < TP; ++t)
          o[t0 + t] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[t][v], sc[v], o[t0 + t], 0, 0, 0);
      if (by_hand) {
        for (int64_t j = k0; j < min(k0 + 32, S); ++j) {
          const int jb = (int)(j - k0);
          float p = 0.f;
#pragma unroll
          for (int v = 0; v < 16; ++v)
            if (v == (jb >> 3) * 4 + (jb & 3)) p = sc[v];
          const float po = other_half(p);
          p = h == ((jb >> 2) & 1) ? p : po;
#pragma unroll
          for (int t = 0; t < TP; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
              const float x = V[j * D + 32 * (t0 + t) + 8 * (v >> 2) + 4 * h + (v & 3)];
              if (j <= last && !(fabsf(x) < INFINITY)) o[t0 + t][v] += p * x;
            }
        }
      }
    }
  }
  l += other_half(l);
  if (h == 0) {
    stat[0][wave][l32] = m;
    stat[1][wave][l32] = l;
  }
  __syncthreads();  // every wave has read Q for the last time and left its max and sum
  float M = stat[0][0][l32];
#pragma unroll
  for (int w = 1; w < NW; ++w) M = fmaxf(M, stat[0][w][l32]);
  // a wave without keys (or with scores of -inf alone) has nothing to add
  const float f = m == -INFINITY ? (M == -INFINITY ? 1.f : 0.f) : expf(m - M);
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = o[t][4 * g + e] * f;
      rows[wave][l32][(8 * t + 2 * g + h) ^ (l32 % CH)] = w;
    }
  __syncthreads();
  float* O = static_cast<float*>(a.o) + head * S * D;
  for (int i = tid; i < 32 * CH; i += NW * 64) {
    const int r = i / CH, c = i % CH;
    if (q0 + r >= S) continue;
    float top = stat[0][0][r];
#pragma unroll
    for (int w = 1; w < NW; ++w) top = fmaxf(top, stat[0][w][r]);
    float sum = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float mw = stat[0][w][r];
      sum += mw == -INFINITY ? 0.f : expf(mw - top) * stat[1][w][r];
      acc += rows[w][r][c ^ (r % CH)];
    }
    *reinterpret_cast<f32x4*>(O + (q0 + r) * D + c * 4) = acc / sum;  // no visible finite score: 0 / 0
  }
}

}  // namespace

bool attention_f32_ok(const AttnArgs& a) {
  if (const char* e = std::getenv("KURUMI_HIP_NO_MFMA"); e && *e && *e != '0') return false;
  auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  return a.dtype == GT_F32 && (a.d == 32 || a.d == 64 || a.d == 128) && a.s > 0 && a.bh > 0 &&
         a.bh * ((a.s + 31) / 32) < ((int64_t)1 << 31) && al(a.q) && al(a.k) && al(a.v) && al(a.o);
}

void launch_attention_f32(const AttnArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)((a.s + 31) / 32 * a.bh));
  switch (a.d) {
    case 32: hipLaunchKernelGGL((attn_f32_k<32>), grid, dim3(NW * 64), 0, s, a); return;
    case 64: hipLaunchKernelGGL((attn_f32_k<64>), grid, dim3(NW * 64), 0, s, a); return;
    default: hipLaunchKernelGGL((attn_f32_k<128>), grid, dim3(NW * 64), 0, s, a); return;
  }
}

}  // namespace ku::hipbk
