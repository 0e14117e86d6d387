// Family-specific routers: DeepSeek-V4 sqrtsoftplus selection and hash weighting, the Inkling
// sigmoid router with shared sinks, and Gemma's 8-bit affine router rows with per-expert scales.
// All share the tie rule of the plain top-k selector and are bit-exact against the CPU oracle:
// exp, log and the summation orders are fixed IEEE sequences, divide and sqrt are correctly rounded.
#include "mf_device.h"
#include "mf_internal.h"
#include "mf_router.h"

#include <algorithm>

#pragma clang fp contract(off)

namespace mf {

namespace {

// One wave per (token, expert) row of router_gemv_gemma4_body (moe.metal:102-139).  8-wide chunks
// are dealt to the 64 lanes; a chunk lies inside one group of 64, its sum q*x' and sum x' are built
// in ascending order from 0 and enter the lane's accumulator as fma(s, dot, acc), fma(b, sum, acc);
// x' = x * effective_scale is exact in fp32 for bf16 factors.  A lane's first CPL chunks are requested together
// (a row of 2816 is six chunks a lane: six trips to memory one after the other took 2 us of a one-token call), and the
// scales and biases of their groups come a group to a lane: two requests for all of them instead of two per chunk
// (128 rows of 2816, one token, with a wave to a workgroup: 3.9 -> 3.5 us).  FEW: as in router_logits_kernel.
// (The pointers are not declared restrict: loads of memory that is never written may be moved behind the fence, next to their use.)
template <int CPL, bool ALIGNED, bool FEW>
__global__ __launch_bounds__(256) void router_logits_int8_kernel(
    const uint8_t* codes, const uint16_t* scales,
    const uint16_t* biases, const uint16_t* x,
    const uint16_t* eff, uint32_t e, uint32_t d, uint32_t t, uint32_t x_stride,
    float* logits) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  if (wave >= e * t) return;
  const uint32_t tok = wave / e, row = wave % e;
  const uint8_t* q_row = codes + static_cast<size_t>(row) * d;
  const uint16_t* s_row = scales + static_cast<size_t>(row) * (d / MF_GROUP_SIZE);
  const uint16_t* b_row = biases + static_cast<size_t>(row) * (d / MF_GROUP_SIZE);
  const uint16_t* x_row = x + static_cast<size_t>(tok) * x_stride;
  float acc = 0.0f;
  const uint32_t chunks = d / 8;
  for (uint32_t base = 0; base < chunks; base += CPL * kWave) {
    const uint32_t c0 = base + lane, g = min(base / 8 + lane, chunks / 8 - 1);
    const uint32_t tab = b_row[g] | (static_cast<uint32_t>(s_row[g]) << 16);
    uint2 q[CPL];
    uint4 xv[CPL], ev[CPL];
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      const uint32_t c = FEW ? min(c0 + i * kWave, chunks - 1) : c0 + i * kWave;  // past the row: the last chunk again, dropped below
      if (!FEW && c >= chunks) continue;
      if constexpr (ALIGNED) q[i] = *reinterpret_cast<const uint2*>(q_row + c * 8);
      else q[i] = make_uint2(load_u32_bytes(q_row + c * 8), load_u32_bytes(q_row + c * 8 + 4));
      xv[i] = load_x8<ALIGNED>(x_row + c * 8);
      ev[i] = load_x8<ALIGNED>(eff + c * 8);
    }
    issue_fence();
    uint32_t sb[CPL];
#pragma unroll
    for (int i = 0; i < CPL; ++i) sb[i] = __builtin_amdgcn_ds_bpermute(4 * (8 * i + (lane >> 3)), tab);
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      if (c0 + i * kWave >= chunks) break;
      const uint32_t xs[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w}, es[4] = {ev[i].x, ev[i].y, ev[i].z, ev[i].w};
      float dot = 0.0f, sum = 0.0f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float x0 = bf16_lo(xs[j]) * bf16_lo(es[j]);
        const float x1 = bf16_hi(xs[j]) * bf16_hi(es[j]);
        const uint32_t word = (j < 2 ? q[i].x : q[i].y) >> ((j & 1) * 16);
        dot = __builtin_fmaf(static_cast<float>(word & 0xFFu), x0, dot);
        sum = sum + x0;
        dot = __builtin_fmaf(static_cast<float>((word >> 8) & 0xFFu), x1, dot);
        sum = sum + x1;
      }
      acc = __builtin_fmaf(bf16_hi(sb[i]), dot, acc);
      acc = __builtin_fmaf(bf16_lo(sb[i]), sum, acc);
    }
  }
  acc = wave_sum(acc);
  if (lane == 0) logits[static_cast<size_t>(tok) * e + row] = acc;
}

// The same rows for many tokens, bit-exact with the kernel above.  A wave keeps R expert rows in registers (lane l
// holds the chunks l, l+64, ... of each row as floats, with their group's scale and bias); the workgroup's threads make
// x' and the chunk sums of one token ahead, once for all its rows, in LDS (two buffers).  Bound by vector
// instructions: with x' made by every wave for its two rows it was 150 a row and token, here 90 (128 rows of 2816,
// 300 tokens: 29.6 -> 18.3 us).  Needs 16-byte aligned x and effective_scale, 8-byte aligned code rows.
template <int CPL, int R>
__global__ __launch_bounds__(256) void router_logits_int8_tiled_kernel(
    const uint8_t* __restrict__ codes, const uint16_t* __restrict__ scales,
    const uint16_t* __restrict__ biases, const uint16_t* __restrict__ x,
    const uint16_t* __restrict__ eff, uint32_t e, uint32_t d, uint32_t t, uint32_t x_stride,
    float* __restrict__ logits, uint32_t tokens_per_block) {
  constexpr uint32_t kChunks = 64 * CPL, kMine = (kChunks + 255) / 256;
  __shared__ float4 s_x[2][2][kChunks];  // [buffer][half of the chunk][chunk]
  __shared__ float s_sum[2][kChunks];
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint32_t row0 = (blockIdx.x * 4 + wv) * R;  // (a wave without a row still helps with x')
  const uint32_t chunks = d / 8, groups = d / MF_GROUP_SIZE;
  float qf[R][CPL][8], sf[R][CPL], bf[R][CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    const uint32_t ci = lane + 64 * c;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const bool live = ci < chunks && row0 + r < e;
      uint2 q = make_uint2(0, 0);
      if (live) q = *reinterpret_cast<const uint2*>(codes + static_cast<size_t>(row0 + r) * d + ci * 8);
#pragma unroll
      for (int j = 0; j < 8; ++j) qf[r][c][j] = static_cast<float>(((j < 4 ? q.x : q.y) >> (8 * (j & 3))) & 0xFFu);
      const size_t g = static_cast<size_t>(row0 + r) * groups + ci * 8 / MF_GROUP_SIZE;
      sf[r][c] = live ? bf16_to_f(scales[g]) : 0.0f;
      bf[r][c] = live ? bf16_to_f(biases[g]) : 0.0f;
    }
  }
  const uint32_t t0 = blockIdx.y * tokens_per_block;
  const uint32_t t1 = min(t, t0 + tokens_per_block);
  uint4 ev[kMine], xv[kMine];
  auto fetch = [&](uint32_t tok) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t i = 0; i < kMine; ++i)
      xv[i] = load_x8<true>(x + static_cast<size_t>(min(tok, t - 1)) * x_stride + min(threadIdx.x + 256 * i, chunks - 1) * 8);
  };
  auto put = [&](uint32_t buf) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t i = 0; i < kMine; ++i) {
      const uint32_t ci = threadIdx.x + 256 * i;
      if (ci < kChunks) {
        const uint32_t xw[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w}, ew[4] = {ev[i].x, ev[i].y, ev[i].z, ev[i].w};
        float p[8], sum = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          p[2 * j] = bf16_lo(xw[j]) * bf16_lo(ew[j]);
          p[2 * j + 1] = bf16_hi(xw[j]) * bf16_hi(ew[j]);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) sum = sum + p[j];
        s_x[buf][0][ci] = make_float4(p[0], p[1], p[2], p[3]);
        s_x[buf][1][ci] = make_float4(p[4], p[5], p[6], p[7]);
        s_sum[buf][ci] = sum;
      }
    }
  };
#pragma unroll
  for (uint32_t i = 0; i < kMine; ++i) ev[i] = load_x8<true>(eff + min(threadIdx.x + 256 * i, chunks - 1) * 8);
  fetch(t0);
  put(0);
  fetch(t0 + 1);
  for (uint32_t tok = t0; tok < t1; ++tok) {
    __syncthreads();  // this token's buffer is complete, the other one is no longer read
    const uint32_t buf = (tok - t0) & 1;
    put(buf ^ 1);
    fetch(tok + 2);
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.0f;
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      const uint32_t ci = lane + 64 * c;
      const float4 a = s_x[buf][0][ci], b = s_x[buf][1][ci];
      const float sum = s_sum[buf][ci], xs[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      if (ci < chunks) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          float dot = 0.0f;
#pragma unroll
          for (int j = 0; j < 8; ++j) dot = __builtin_fmaf(qf[r][c][j], xs[j], dot);
          acc[r] = __builtin_fmaf(sf[r][c], dot, acc[r]);
          acc[r] = __builtin_fmaf(bf[r][c], sum, acc[r]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float v = wave_sum(acc[r]);
      if (lane == 0 && row0 + r < e) logits[static_cast<size_t>(tok) * e + row0 + r] = v;
    }
  }
}

enum Family { kSqrtSoftplus = 0, kHash = 1, kInkling = 2, kScaledSoftmax = 3 };

struct FamilyArgs {
  const float* logits;            // [t, e + n_shared]
  const float* bias;              // [e] selection bias (sqrtsoftplus, Inkling)
  const float* global_scale;      // [1] (Inkling)
  const uint16_t* expert_scale;   // [e] bf16 (scaled softmax)
  const uint32_t* given;          // [t, k] (hash)
  uint32_t e, n_shared, k;
  float route_scale;
  uint32_t* idx;                  // [t, k]
  float* w;                       // [t, k]
  float* gammas;                  // [t, n_shared]
};

__device__ __forceinline__ void lds_settle() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_wave_barrier();
}

// sum of v over lanes 0..n-1 in ascending order, n <= 16 (the reference's serial tails)
__device__ __forceinline__ float ordered_sum(float v, uint32_t n) {
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; ++i)
    if (static_cast<uint32_t>(i) < n) sum += readlane_f(v, i);
  return sum;
}

// One wave per token selects.  A few tokens are all latency: there a workgroup of four waves takes a token, an expert
// per thread and no loop over them (four trips to memory one after the other otherwise: 5.4 -> 3.7 us for 256
// experts), and what the tail needs of the picked experts -- raw score, scale -- is kept in LDS instead of fetched
// again by index.
template <int FAMILY, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void family_select_kernel(FamilyArgs a) {
  __shared__ float s_sel[MF_MAX_EXPERTS];
  __shared__ float s_raw[MF_MAX_EXPERTS];
  __shared__ uint32_t s_idx[MF_MAX_TOPK];
  __shared__ float s_w[MF_MAX_TOPK];
  const uint32_t lane = threadIdx.x & 63, tok = blockIdx.x, k = a.k;
  constexpr uint32_t kThreads = 64 * WAVES;
  auto settle = [&]() {  // what the token's threads wrote to LDS is there
    if constexpr (WAVES > 1) __syncthreads();
    else lds_settle();
  };
  const float* lg = a.logits + static_cast<size_t>(tok) * (a.e + a.n_shared);
  uint32_t* idx = a.idx + static_cast<size_t>(tok) * k;
  float* w = a.w + static_cast<size_t>(tok) * k;

  if constexpr (FAMILY == kScaledSoftmax) {
    // router_topk_select_k8 (moe.metal:190-240): softmax over the selected, times per_expert_scale
    for (uint32_t x = threadIdx.x; x < a.e; x += kThreads) {
      s_sel[x] = lg[x];
      s_raw[x] = bf16_to_f(a.expert_scale[x]);
    }
    settle();
    if (threadIdx.x >= kWave) return;
    topk_select_fast(s_sel, a.e, k, s_idx, s_w, lane);
    lds_settle();
    if (lane < k) {
      const uint32_t my = s_idx[lane];
      idx[lane] = my;
      w[lane] = s_w[lane] * s_raw[my];
    }
    return;
  }

  uint32_t my = 0;
  float raw = 0.0f;  // the picked expert's raw score (sqrtsoftplus) or logit (Inkling)
  if constexpr (FAMILY == kHash) {
    if (lane < k) my = a.given[static_cast<size_t>(tok) * k + lane];
  } else {
    for (uint32_t x = threadIdx.x; x < a.e; x += kThreads) {
      const float l = lg[x], b = a.bias[x], sp = FAMILY == kSqrtSoftplus ? mf_sqrtsoftplus(l) : l;
      s_raw[x] = sp;
      s_sel[x] = (FAMILY == kSqrtSoftplus ? sp : 1.0f / (1.0f + mf_exp(-l))) + b;
    }
    settle();
    if (threadIdx.x >= kWave) return;
    topk_select_indices(s_sel, a.e, k, s_idx, lane);
    lds_settle();
    if (lane < k) {
      my = s_idx[lane];
      idx[lane] = my;
      raw = s_raw[my];
    }
  }

  if constexpr (FAMILY == kInkling) {
    // inkling.metal:540-565: softmax over logsigmoid of the raw logits of the selected experts and
    // the sinks, times route_scale * global_scale
    const uint32_t total = k + a.n_shared;
    float lp = -__builtin_inff();
    if (lane < total) {
      const float x = lane < k ? raw : lg[a.e + (lane - k)];
      lp = (x < 0.0f ? x : 0.0f) - mf_log_1to2(1.0f + mf_exp(-__builtin_fabsf(x)));
    }
    const float mx = wave_max(lp);
    const float ex = lane < total ? mf_exp(lp - mx) : 0.0f;
    const float denom = ordered_sum(ex, total);
    const float s_all = a.route_scale * a.global_scale[0] / denom;
    if (lane < k) w[lane] = ex * s_all;
    else if (lane < total) a.gammas[static_cast<size_t>(tok) * a.n_shared + (lane - k)] = ex * s_all;
  } else {
    // moe.metal:773-785 / :855-865: raw sqrtsoftplus scores of the chosen experts, renormalised.
    // An expert index past the table (possible only for given indices) weighs nothing.
    if constexpr (FAMILY == kHash) raw = (lane < k && my < a.e) ? mf_sqrtsoftplus(lg[my]) : 0.0f;
    const float inv = a.route_scale / (ordered_sum(raw, k) + 1e-20f);
    if (lane < k) w[lane] = raw * inv;
  }
}

template <int FAMILY>
hipError_t launch_family(hipStream_t s, const FamilyArgs& a, uint32_t t) {
  if (!t) return hipSuccess;
  // (given indices have nothing to select; from 512 tokens on the chip is full with a wave each)
  if (FAMILY != kHash && t < 512) family_select_kernel<FAMILY, 4><<<dim3(t), dim3(256), 0, s>>>(a);
  else family_select_kernel<FAMILY, 1><<<dim3(t), dim3(64), 0, s>>>(a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_router_logits_int8(hipStream_t s, const uint8_t* codes, const uint16_t* scales,
                                     const uint16_t* biases, const uint16_t* x, const uint16_t* eff,
                                     uint32_t e, uint32_t d, uint32_t t, uint32_t x_stride, float* logits) {
  const uint32_t waves = e * t;
  if (!waves) return hipSuccess;
  const bool al = (reinterpret_cast<uintptr_t>(codes) % 8 == 0) && aligned16(x) && aligned16(eff) &&
                 x_stride % 8 == 0 && d % 8 == 0;
  const uint32_t cpl = (d / 8 + 63) / 64;
  if (al && t >= 16 && cpl <= 8) {  // many tokens: rows stay in registers
    // about 600 workgroups of 8 rows (two to a CU), at least 4 tokens to a row load
    const uint32_t tpb = std::max(4u, std::min(64u, t * ((e + 7) / 8) / 600));
#define MF_R8(CPL, R)                                                                                \
  router_logits_int8_tiled_kernel<CPL, R><<<dim3((e + 4 * R - 1) / (4 * R), (t + tpb - 1) / tpb), dim3(256), 0, \
                                            s>>>(codes, scales, biases, x, eff, e, d, t, x_stride, logits, tpb)
    if (cpl <= 2) MF_R8(2, 4);
    else if (cpl <= 4) MF_R8(4, 2);
    else if (cpl <= 6) MF_R8(6, 2);
    else MF_R8(8, 1);
#undef MF_R8
    return hipGetLastError();
  }
  // A wave to a workgroup while that is at most four a CU: its loads have a CU's paths to themselves.  Few waves: nothing branches between
  // a row's loads; beyond, nothing past the row is asked for.  us with the selection, without / with branches: aligned, 128 rows of 2816, 15
  // tokens 6.83 / 7.04; of 5120, 16, 64, 300 tokens 7.8 / 7.95, 14.4 / 13.6, 46.1 / 40.8; unaligned, 64 rows of 1088, 15, 32, 300 tokens
  // 6.01 / 6.02, 6.48 / 6.28, 18.7 / 14.4.  Unaligned rows take two chunks a trip up to 2048 elements and six beyond (128 rows of 2816, 1, 64
  // tokens, two / six: 6.65 / 6.2, 14.3 / 13.4).
  const uint32_t cus = device_cu_count(), block = waves <= 4 * cus ? 64u : 256u;
  const bool few = waves <= (al ? 8 : 4) * cus;
  const dim3 grid((waves + block / 64 - 1) / (block / 64));
#define MF_R8(CPL, AL)                                                                                                                   \
  do {                                                                                                                                   \
    if (few) router_logits_int8_kernel<CPL, AL, true><<<grid, dim3(block), 0, s>>>(codes, scales, biases, x, eff, e, d, t, x_stride, logits); \
    else router_logits_int8_kernel<CPL, AL, false><<<grid, dim3(block), 0, s>>>(codes, scales, biases, x, eff, e, d, t, x_stride, logits);    \
  } while (0)
  if (!al && cpl <= 4) MF_R8(2, false);
  else if (!al) MF_R8(6, false);
  else if (cpl <= 2) MF_R8(2, true);
  else if (cpl <= 4) MF_R8(4, true);
  else MF_R8(6, true);
#undef MF_R8
  return hipGetLastError();
}

hipError_t launch_select_sqrtsoftplus(hipStream_t s, const float* logits, const float* bias, uint32_t e,
                                      uint32_t k, uint32_t t, float route_scale, uint32_t* idx, float* w) {
  FamilyArgs a{};
  a.logits = logits; a.bias = bias; a.e = e; a.k = k; a.route_scale = route_scale; a.idx = idx; a.w = w;
  return launch_family<kSqrtSoftplus>(s, a, t);
}

hipError_t launch_hash_weights(hipStream_t s, const float* logits, const uint32_t* given, uint32_t e,
                               uint32_t k, uint32_t t, float route_scale, float* w) {
  FamilyArgs a{};
  a.logits = logits; a.given = given; a.e = e; a.k = k; a.route_scale = route_scale; a.w = w;
  return launch_family<kHash>(s, a, t);
}

hipError_t launch_select_inkling(hipStream_t s, const float* logits, const float* bias,
                                 const float* global_scale, uint32_t n_routed, uint32_t n_shared, uint32_t k,
                                 uint32_t t, float route_scale, uint32_t* idx, float* w, float* gammas) {
  FamilyArgs a{};
  a.logits = logits; a.bias = bias; a.global_scale = global_scale; a.e = n_routed; a.n_shared = n_shared;
  a.k = k; a.route_scale = route_scale; a.idx = idx; a.w = w; a.gammas = gammas;
  return launch_family<kInkling>(s, a, t);
}

hipError_t launch_select_scaled_softmax(hipStream_t s, const float* logits, const uint16_t* expert_scale,
                                        uint32_t e, uint32_t k, uint32_t t, uint32_t* idx, float* w) {
  FamilyArgs a{};
  a.logits = logits; a.expert_scale = expert_scale; a.e = e; a.k = k; a.idx = idx; a.w = w;
  return launch_family<kScaledSoftmax>(s, a, t);
}

}  // namespace mf
