// Router: bf16 GEMV to fp32 logits and the top-k selectors.  Both are
// bit-exact against the CPU oracle: the logit summation order is fixed (see
// dot_bf16_row) and exp/divide are IEEE sequences shared with it.
#include "mf_device.h"
#include "mf_internal.h"
#include "mf_router.h"

#pragma clang fp contract(off)

namespace mf {

// One wave per (token, row), in dot_bf16_row's order.  A call of a few rows is one round trip to memory and what surrounds it, so a lane's
// first CPL chunks leave together (rows of up to 512 * CPL elements whole), and the waves are spread over the CUs (see the launch):
// 256 rows of 4096, one token, 4.0 -> 3.4 us (in two halves of four chunks, four waves to a workgroup, before).  FEW: no branch between
// the loads; the other form, for calls of many waves, which the requests themselves bound, asks for nothing past the row.
// (The pointers are not declared restrict: loads of memory that is never written may be moved behind the fence, next to their use.)
template <int CPL, bool ALIGNED, bool FEW>
__global__ __launch_bounds__(256) void router_logits_kernel(const uint16_t* w, const uint16_t* x,
                                                            uint32_t e, uint32_t d, uint32_t t,
                                                            uint32_t x_stride,
                                                            float* logits,
                                                            uint16_t* logits_bf16) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  if (wave >= e * t) return;
  const uint32_t tok = wave / e, row = wave % e, chunks = d / 8;
  const uint16_t* w_row = w + static_cast<size_t>(row) * d;
  const uint16_t* x_row = x + static_cast<size_t>(tok) * x_stride;
  float acc = 0.0f;
  for (uint32_t c0 = lane; c0 < chunks; c0 += CPL * kWave) {
    uint4 wv[CPL], xv[CPL];
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      const uint32_t c = FEW ? min(c0 + i * kWave, chunks - 1) : c0 + i * kWave;  // past the row: the last chunk again, dropped below
      if (FEW || c < chunks) {
        wv[i] = load_x8<ALIGNED>(w_row + c * 8);
        xv[i] = load_x8<ALIGNED>(x_row + c * 8);
      }
    }
    issue_fence();
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      if (c0 + i * kWave >= chunks) break;
      acc = fma_chunk_bf16(wv[i], xv[i], acc);
    }
  }
  const float v = wave_sum(acc);
  if (lane == 0) {
    if (logits) logits[static_cast<size_t>(tok) * e + row] = v;
    if (logits_bf16) logits_bf16[static_cast<size_t>(tok) * e + row] = f_to_bf16(v);
  }
}

// one wave per token
__global__ __launch_bounds__(64) void topk_kernel(const float* __restrict__ logits, uint32_t e,
                                                  uint32_t k, int mode,
                                                  uint32_t* __restrict__ idx,
                                                  float* __restrict__ w) {
  const uint32_t tok = blockIdx.x;
  if (mode == 0)
    topk_select_fast(logits + static_cast<size_t>(tok) * e, e, k, idx + static_cast<size_t>(tok) * k,
                     w + static_cast<size_t>(tok) * k, threadIdx.x);
  else {
    __shared__ float s_p[MF_MAX_EXPERTS];
    topk_full_softmax_fast(logits + static_cast<size_t>(tok) * e, s_p, e, k, idx + static_cast<size_t>(tok) * k,
                           w + static_cast<size_t>(tok) * k, threadIdx.x);
  }
}

hipError_t launch_router_logits(hipStream_t s, const uint16_t* w, const uint16_t* x, uint32_t e,
                                uint32_t d, uint32_t t, uint32_t x_stride, float* logits,
                                uint16_t* logits_bf16) {
  const uint32_t waves = e * t;
  if (!waves) return hipSuccess;
  const bool al = aligned16(w) && aligned16(x) && (x_stride % 8 == 0) && (d % 8 == 0);
  // The loads leave without a branch between them, by the width's number of chunks to a trip, while the waves are few; beyond, what lies
  // past the row is not asked for.  The line: 16 waves a CU where a row fills its trip, 2 where it leaves a quarter of it empty, 4 for
  // rows of more trips than one.  us with the selection, without / with branches: 256 rows of 2816, 1, 8, 15 tokens 5.70 / 5.83,
  // 6.27 / 6.37, 6.98 / 7.07; 64 rows of 5184, 1, 16, 64, 300, 1000 tokens 5.66 / 5.79, 6.34 / 6.38, 9.00 / 8.40, 22.3 / 17.8, 61.6 / 45.8;
  // 64 unaligned rows of 576, 8, 15, 64 tokens 5.25 / 5.25, 5.47 / 5.32, 6.24 / 6.04.
  const uint32_t cus = device_cu_count(), trip = d <= 1024 ? 2 : d <= 2048 ? 4 : d <= 3072 ? 6 : 8;
  const bool few = waves <= (d > 4096 ? 4 : d / 8 >= 3 * kWave / 4 * trip ? 16 : 2) * cus;
  const uint32_t block = waves <= 4 * cus ? 64u : 256u;  // a wave to a workgroup while that is at most four a CU
  const dim3 grid((waves + block / 64 - 1) / (block / 64));
#define MF_RL(CPL, FEW)                                                                                                               \
  do {                                                                                                                                \
    if (al) router_logits_kernel<CPL, true, FEW><<<grid, dim3(block), 0, s>>>(w, x, e, d, t, x_stride, logits, logits_bf16);          \
    else router_logits_kernel<CPL, false, FEW><<<grid, dim3(block), 0, s>>>(w, x, e, d, t, x_stride, logits, logits_bf16);            \
  } while (0)
  if (!few) MF_RL(4, false);
  else if (trip == 2) MF_RL(2, true);
  else if (trip == 4) MF_RL(4, true);
  else if (trip == 6) MF_RL(6, true);
  else MF_RL(8, true);
#undef MF_RL
  return hipGetLastError();
}

hipError_t launch_topk(hipStream_t s, const float* logits, uint32_t e, uint32_t k, uint32_t t,
                       int mode, uint32_t* idx, float* w) {
  if (!t) return hipSuccess;
  topk_kernel<<<dim3(t), dim3(64), 0, s>>>(logits, e, k, mode, idx, w);
  return hipGetLastError();
}

}  // namespace mf
