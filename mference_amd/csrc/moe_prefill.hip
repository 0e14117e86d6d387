// Ragged prefill: router for many tokens, device-side grouping of the
// (token, expert) routes, and the tokens-sorted-by-expert quantized matmul on
// the bf16 matrix cores.
//
// The matmul keeps the codes EXACT: a lane's packed uint32 is masked into bf16 subnormals (a 4-bit code in bits 4..7 of a
// 16-bit half is the number q * 2^-129, mf_device.h), which are a matrix-core operand as they stand -- no LDS
// staging of weights.  x rows are pre-permuted once per call to the same
// (j, j+4) pairing, times a power of two that the row's largest magnitude decides (2^64 for ordinary rows; what another
// lacks is made up for in the epilogue), and staged through LDS per 64-wide K group.  Per K group the
// matrix core yields 2^-65 sum(q * x) (bf16 x bf16 products are exact in
// fp32), and the group's bf16 scale is applied in fp32: acc += 2^65 s * tmp -- the
// reference's own factoring s*sum(q*x) + b*sum(x)
// (Metal/Quant/dequant_int4.metal:14-17), so no weight is ever rounded to bf16
// (rounding q*s+b to bf16 would cost ~1.6e-3 relative error per weight, above
// the layer tolerance).  The b*sum(x) term is one more small
// matmul over the group index (operands: the bf16 bias table, exact,
// and sum(x) split into three bf16 terms, exact).
//
// Replaces prefill_grouped_routed_moe_batched_{phase1,down}
// (Metal/Prefill/prefill.metal:748-820), prefill_moe_reduce_token_major
// (:631-652) and the staged-affine tensor-core QMM
// mpp_prefill_affine_threadgroup_f16 (Metal/TensorCore/tensorops.metal:13-105).
#include <algorithm>
#include <type_traits>
#include <vector>

#include "mf_device.h"
#include "mf_internal.h"
#include "mf_qmm.h"
#include "mf_router.h"

#pragma clang fp contract(off)

namespace mf {

// ------------------------------------------------------------------ router

// logits[t, e] for many tokens, bit-exact with dot_bf16_row: a wave keeps R
// expert rows in registers (lane l holds the chunks l, l+64, ... of each row)
// and streams token rows past them.
template <int CPL, int R>
__device__ __forceinline__ void router_rows(const uint16_t* __restrict__ W, const uint16_t* __restrict__ x,
                                            uint32_t E, uint32_t D, uint32_t T, uint32_t x_stride,
                                            float* __restrict__ logits, uint32_t tokens_per_block, uint32_t ld,
                                            uint32_t lane, uint32_t wv);

// What a short batch hangs on the router launch so that it needs no launch of its own: the x
// preparation (matmul order, group sums, scalar shared gate) in extra workgroup columns.  (The top-k of
// a token block by the last workgroup to finish that block's logits was tried and lost: the
// device-wide fence every workgroup needs for it costs more than the launch it saves.)
struct RouterTail {
  uint16_t* xp;          // null: none of this
  uint32_t router_cols;  // workgroup columns that compute logits; the columns behind them prepare x
  const uint16_t* w_sg;  // null: no scalar gate
  uint16_t* sums;
  float* row_max;
  uint16_t* gate;
};

__device__ __forceinline__ void prep_x_row(const uint16_t* __restrict__ x, uint16_t* __restrict__ xp,
                                           uint16_t* __restrict__ sums, float* __restrict__ row_max, const uint16_t* __restrict__ w_sg,
                                           uint16_t* __restrict__ gate, uint32_t row, uint32_t d, uint32_t lane);

template <int CPL, int R>
__global__ __launch_bounds__(256) void prefill_router_kernel(const uint16_t* __restrict__ W,
                                                             const uint16_t* __restrict__ x,
                                                             uint32_t E, uint32_t D, uint32_t T,
                                                             uint32_t x_stride,
                                                             float* __restrict__ logits,
                                                             uint32_t tokens_per_block, uint32_t ld,
                                                             const RouterTail tail) {
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (tail.xp && blockIdx.x >= tail.router_cols) {  // an x-preparation workgroup: one row per wave
    const uint32_t row = ((blockIdx.x - tail.router_cols) * gridDim.y + blockIdx.y) * 4 + wv;
    if (row < T) prep_x_row(x + static_cast<size_t>(row) * x_stride, tail.xp, tail.sums, tail.row_max, tail.w_sg, tail.gate, row, D, lane);
    return;
  }
  router_rows<CPL, R>(W, x, E, D, T, x_stride, logits, tokens_per_block, ld, lane, wv);
}

template <int CPL, int R>
__device__ __forceinline__ void router_rows(const uint16_t* __restrict__ W, const uint16_t* __restrict__ x,
                                            uint32_t E, uint32_t D, uint32_t T, uint32_t x_stride,
                                            float* __restrict__ logits, uint32_t tokens_per_block, uint32_t ld,
                                            uint32_t lane, uint32_t wv) {
  const uint32_t row0 = (blockIdx.x * 4 + wv) * R;
  if (row0 >= E) return;
  const uint32_t chunks = D / 8;
  float wf[R][CPL][8];
#pragma unroll
  for (int r = 0; r < R; ++r) {
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      const uint32_t ci = lane + 64 * c;
      uint4 v = make_uint4(0, 0, 0, 0);
      if (ci < chunks && row0 + r < E) v = load_x8<true>(W + static_cast<size_t>(row0 + r) * D + ci * 8);
      wf[r][c][0] = bf16_lo(v.x); wf[r][c][1] = bf16_hi(v.x);
      wf[r][c][2] = bf16_lo(v.y); wf[r][c][3] = bf16_hi(v.y);
      wf[r][c][4] = bf16_lo(v.z); wf[r][c][5] = bf16_hi(v.z);
      wf[r][c][6] = bf16_lo(v.w); wf[r][c][7] = bf16_hi(v.w);
    }
  }
  const uint32_t t0 = blockIdx.y * tokens_per_block;
  const uint32_t t1 = min(T, t0 + tokens_per_block);
  for (uint32_t t = t0; t < t1; ++t) {
    const uint16_t* xt = x + static_cast<size_t>(t) * x_stride;
    float xf[CPL][8];
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      const uint32_t ci = lane + 64 * c;
      uint4 v = make_uint4(0, 0, 0, 0);
      if (ci < chunks) v = load_x8<true>(xt + ci * 8);
      xf[c][0] = bf16_lo(v.x); xf[c][1] = bf16_hi(v.x);
      xf[c][2] = bf16_lo(v.y); xf[c][3] = bf16_hi(v.y);
      xf[c][4] = bf16_lo(v.z); xf[c][5] = bf16_hi(v.z);
      xf[c][6] = bf16_lo(v.w); xf[c][7] = bf16_hi(v.w);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float acc = 0.0f;
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        if (lane + 64 * c < chunks) {
#pragma unroll
          for (int j = 0; j < 8; ++j) acc = __builtin_fmaf(wf[r][c][j], xf[c][j], acc);
        }
      }
      const float v = wave_sum(acc);
      if (lane == 0 && row0 + r < E) logits[static_cast<size_t>(t) * ld + row0 + r] = v;
    }
  }
}

// The same logits on the fp32 matrix core, still bit for bit: a K=1 outer-product MFMA adds
// exactly one product to every accumulator element, c <- fl(c + x*w), and x*w is exact for
// bf16 inputs -- so a run of K=1 MFMAs is the per-lane fmaf chain of dot_bf16_row for a whole
// 32-token x 32-expert block at once.  "Lane l" of the reference order becomes chain l: the K
// values 8l..8l+7, then +512, +1024, ...  The two blocks of one instruction carry chains l and
// l+1; their accumulators are added (the stride-1 level of the butterfly), then combined with
// the later pairs as a binary counter, which reproduces the ascending-stride tree.  Each of the
// four waves of a workgroup owns 16 chains; the last two levels go through LDS.
// Needs D % 512 == 0 (all 64 chains the same length) and E % 32 == 0.
typedef __attribute__((ext_vector_type(32))) float f32x32_t;

// N_I = D / 512, 2 or 4, as a compile-time constant unrolls the whole walk (a wave's 8 chain pairs x N_I runs): the
// operand offsets, the ring slots and the levels of the binary counter are then literals, the operand ring
// needs no register moves and a chain's first instruction takes the constant 0 as its accumulator -- 3.9
// vector instructions per matrix instruction where a loop with operands in registers issued 10.6, and the
// matrix instructions of a SIMD wait for its vector instructions (T=2048: 38.6 -> 34.1 us, T=512: 18.5 ->
// 14.8 us).  (The unrolled form needs 123 registers; eight waves of 8 chains per block, four to a SIMD,
// measured no faster than these four of 16 chains: 34.7 / 15.8 us.)  Three waves per SIMD: the x-preparation
// workgroups behind the router's then share the CUs with them instead of waiting for a second round (-1.3 us).
template <int N_I>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3)))
void prefill_router_mfma_kernel(const uint16_t* __restrict__ W,
                                                                  const uint16_t* __restrict__ x,
                                                                  uint32_t E, uint32_t D, uint32_t T,
                                                                  uint32_t x_stride,
                                                                  float* __restrict__ logits, uint32_t ld,
                                                                  const RouterTail tail) {
  constexpr int WAVES = 4, kPairs = 32 / WAVES;  // waves of a workgroup, chain pairs of one wave
  __shared__ float s_part[WAVES - 1][16 * 64];
  __shared__ uint4 s_stage[WAVES][2][2 * 128];  // per wave: x and w, two buffers of 32 rows x 64 B
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (tail.xp && blockIdx.y >= tail.router_cols) {  // an x-preparation workgroup (rows behind the expert blocks)
    const uint32_t row = ((blockIdx.y - tail.router_cols) * gridDim.x + blockIdx.x) * WAVES + wv;
    if (row < T) prep_x_row(x + static_cast<size_t>(row) * x_stride, tail.xp, tail.sums, tail.row_max, tail.w_sg, tail.gate, row, D, lane);
    return;
  }
  const uint32_t m = lane & 31, b = lane >> 5;
  // token tiles vary fastest: workgroups go to the XCDs round-robin, so each XCD's L2 sees an
  // eighth of the token rows (and all of the small router matrix)
  const uint32_t t0 = blockIdx.x * 32, e0 = blockIdx.y * 32;

  float lev0[16], lev1[16], lev2[16], total[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) lev0[r] = lev1[r] = lev2[r] = total[r] = 0.0f;
  // A lane needs 16 bytes of its token row and of its expert row per step -- read straight from memory
  // that is 32 rows, 32 cache lines, per load instruction, and the L1's line rate, not the matrix core,
  // sets the pace.  So the wave fetches 64 contiguous bytes of every row at a time (the operands of two
  // chain pairs: four lanes side by side, 16 lines per instruction) and hands them to itself through a
  // wave-private LDS buffer.  A stage is (pair group pg, K run i): 2 steps, 16 matrix instructions.  The
  // two chain pairs of a group keep an accumulator each across the runs.
  constexpr int kGroups = kPairs / 2, kStages = kGroups * N_I;
  const uint32_t ld_row = lane >> 2, ld_chunk = lane & 3;  // fetch: rows ld_row, ld_row + 16; 16-byte chunk
  const uint16_t* xsrc[2];
  const uint16_t* wsrc[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    xsrc[j] = x + static_cast<size_t>(min(t0 + ld_row + 16 * j, T - 1)) * x_stride + 8 * (2 * kPairs * wv + ld_chunk);
    wsrc[j] = W + static_cast<size_t>(e0 + ld_row + 16 * j) * D + 8 * (2 * kPairs * wv + ld_chunk);
  }
  // LDS rows of 64 bytes; chunk c of row r sits in slot c ^ ((r >> 2) & 3): 16 lanes that read the same
  // chunk of 16 consecutive rows then cover 256 bytes of distinct banks
  uint4* stage_x = s_stage[wv][0];
  uint4* stage_w = s_stage[wv][1];
  uint32_t st_at[2], rd_at[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t r = ld_row + 16 * j;
    st_at[j] = r * 4 + (ld_chunk ^ ((r >> 2) & 3));
    rd_at[j] = m * 4 + ((2 * j + b) ^ ((m >> 2) & 3));  // pair j of the group, block b
  }
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
  u32x4_t fx0, fx1, fw0, fw1;  // the stage on its way from memory to LDS
#define MF_ROUTER_FETCH(ST)                                                                          \
  do {                                                                                               \
    const int f_off = 32 * ((ST) / N_I) + 512 * ((ST) % N_I);                                        \
    fx0 = *reinterpret_cast<const u32x4_t*>(xsrc[0] + f_off);                                        \
    fx1 = *reinterpret_cast<const u32x4_t*>(xsrc[1] + f_off);                                        \
    fw0 = *reinterpret_cast<const u32x4_t*>(wsrc[0] + f_off);                                        \
    fw1 = *reinterpret_cast<const u32x4_t*>(wsrc[1] + f_off);                                        \
  } while (0)
#define MF_ROUTER_PUT(BUF)                                                                           \
  do {                                                                                               \
    *reinterpret_cast<u32x4_t*>(stage_x + (BUF) * 128 + st_at[0]) = fx0;                             \
    *reinterpret_cast<u32x4_t*>(stage_x + (BUF) * 128 + st_at[1]) = fx1;                             \
    *reinterpret_cast<u32x4_t*>(stage_w + (BUF) * 128 + st_at[0]) = fw0;                             \
    *reinterpret_cast<u32x4_t*>(stage_w + (BUF) * 128 + st_at[1]) = fw1;                             \
  } while (0)
  MF_ROUTER_FETCH(0);
  MF_ROUTER_PUT(0);
  if (kStages > 1) MF_ROUTER_FETCH(1);
  f32x32_t acc[2];
#pragma unroll
  for (int st = 0; st < kStages; ++st) {
    const int pg = st / N_I, i = st % N_I;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint4 cxq = stage_x[(st & 1) * 128 + rd_at[j]], cwq = stage_w[(st & 1) * 128 + rd_at[j]];
      const uint32_t xw[4] = {cxq.x, cxq.y, cxq.z, cxq.w}, ww[4] = {cwq.x, cwq.y, cwq.z, cwq.w};
      float xa[8], wa[8];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        xa[2 * u] = bf16_lo(xw[u]); xa[2 * u + 1] = bf16_hi(xw[u]);
        wa[2 * u] = bf16_lo(ww[u]); wa[2 * u + 1] = bf16_hi(ww[u]);
      }
      // all 16 operands in registers of their own before the step's first matrix instruction
      asm volatile("" : "+v"(xa[0]), "+v"(xa[1]), "+v"(xa[2]), "+v"(xa[3]), "+v"(xa[4]), "+v"(xa[5]), "+v"(xa[6]), "+v"(xa[7]),
                        "+v"(wa[0]), "+v"(wa[1]), "+v"(wa[2]), "+v"(wa[3]), "+v"(wa[4]), "+v"(wa[5]), "+v"(wa[6]), "+v"(wa[7]));
      if (i == 0) {  // a chain's first product lands on 0
        f32x32_t zero;
#pragma unroll
        for (int r = 0; r < 32; ++r) zero[r] = 0.0f;
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x1f32(xa[0], wa[0], zero, 0, 0, 0);
      } else {
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x1f32(xa[0], wa[0], acc[j], 0, 0, 0);
      }
#pragma unroll
      for (int u = 1; u < 8; ++u) acc[j] = __builtin_amdgcn_mfma_f32_32x32x1f32(xa[u], wa[u], acc[j], 0, 0, 0);
    }
    if (st + 1 < kStages) {  // the next stage into the other buffer (read last a stage ago), the one after it on its way
      MF_ROUTER_PUT((st + 1) & 1);
      if (st + 2 < kStages) MF_ROUTER_FETCH(st + 2);
    }
    if (i == N_I - 1) {  // two pairs of chains are complete: stride-1 level, then the binary counter
      constexpr int kLevels = kPairs == 8 ? 3 : 2;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int pp = 2 * pg + j;
        float carry[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) carry[r] = acc[j][r] + acc[j][16 + r];
        int level = 0;
#pragma unroll
        for (; level < kLevels && ((pp >> level) & 1); ++level) {
          float* lv = level == 0 ? lev0 : level == 1 ? lev1 : lev2;
#pragma unroll
          for (int r = 0; r < 16; ++r) carry[r] = lv[r] + carry[r];
        }
        float* dst = level == kLevels ? total : level == 0 ? lev0 : level == 1 ? lev1 : lev2;
#pragma unroll
        for (int r = 0; r < 16; ++r) dst[r] = carry[r];
      }
    }
  }
#undef MF_ROUTER_FETCH
#undef MF_ROUTER_PUT
  if (wv > 0) {
#pragma unroll
    for (int r = 0; r < 16; ++r) s_part[wv - 1][r * 64 + lane] = total[r];
  }
  __syncthreads();
  if (wv == 0) {  // the last levels of the tree: neighbouring waves first
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float v[WAVES];
      v[0] = total[r];
#pragma unroll
      for (int u = 1; u < WAVES; ++u) v[u] = s_part[u - 1][r * 64 + lane];
#pragma unroll
      for (int stride = 1; stride < WAVES; stride *= 2)
#pragma unroll
        for (int u = 0; u < WAVES; u += 2 * stride) v[u] = v[u] + v[u + stride];
      const uint32_t t = t0 + 8 * (r / 4) + 4 * b + (r % 4);
      if (t < T) logits[static_cast<size_t>(t) * ld + e0 + m] = v[0];
    }
  }
}

// The same for rows of any number of runs of 512, in a loop of one stage (two chain pairs in one run).  What bounds it: a wave's matrix
// instructions, 64 cycles each, as long as everything else stays out of their way: rows go straight to LDS, three stages ahead.  Unrolled
// like the kernel above, the 32 stages of a row of 4096 are 32 KB of instructions that a wave runs once and, with a wave to a SIMD,
// waits for.  Router and selection, us, unrolled / as a loop: 256 rows of 4096, 200 tokens 30.0 / 26.8, 777 tokens 41.0 / 30.5, 2048
// 60.9 / 52.1, 4096 100.1 / 99.5; of 2048, 777 tokens 19.4 / 20.1, 4096 50.7 / 62.4; of 1024, 777 tokens 14.4 / 15.2.  A loop with operands
// four steps ahead in registers (16 bytes of a row a lane): 128 rows of 2560, 777 tokens 23.5 / 20.7, 64 rows of 5120 35.1 / 31.5.
constexpr int kRouterRing = 3;  // stages on their way
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3)))
void prefill_router_loop_kernel(const uint16_t* W, const uint16_t* x, uint32_t E, uint32_t D, uint32_t T, uint32_t x_stride,
                                float* logits, uint32_t ld, const RouterTail tail) {
  constexpr int WAVES = 4, kGroups = 4;  // waves of a workgroup; groups of two chain pairs of a wave
  __shared__ uint4 s_stage[WAVES][kRouterRing][2][128];  // per wave: a ring of stages of x and w, 32 rows x 64 bytes each
  const uint32_t lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (tail.xp && blockIdx.y >= tail.router_cols) {  // an x-preparation workgroup (rows behind the expert blocks)
    const uint32_t row = ((blockIdx.y - tail.router_cols) * gridDim.x + blockIdx.x) * WAVES + wv;
    if (row < T) prep_x_row(x + static_cast<size_t>(row) * x_stride, tail.xp, tail.sums, tail.row_max, tail.w_sg, tail.gate, row, D, lane);
    return;
  }
  const uint32_t m = lane & 31, b = lane >> 5;
  // token tiles vary fastest: workgroups go to the XCDs round-robin, so each XCD's L2 sees an
  // eighth of the token rows (and all of the small router matrix)
  const uint32_t t0 = blockIdx.x * 32, e0 = blockIdx.y * 32;
  const uint32_t n_i = D / 512, n_st = kGroups * n_i;
  // fetch: 16 rows an instruction, four lanes to a row; piece c of row r lies in place c ^ (r / 4 % 4), so that 16 lanes that read the
  // same piece of 16 consecutive rows cover 256 bytes of distinct banks
  const uint32_t ld_row = lane >> 2, ld_chunk = (lane & 3) ^ ((lane >> 4) & 3);
  const uint16_t* src[4];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    src[j] = x + static_cast<size_t>(min(t0 + ld_row + 16 * j, T - 1)) * x_stride + 8 * (16 * wv + ld_chunk);
    src[2 + j] = W + static_cast<size_t>(e0 + ld_row + 16 * j) * D + 8 * (16 * wv + ld_chunk);
  }
  const uint32_t lds = static_cast<uint32_t>(reinterpret_cast<size_t>((__attribute__((address_space(3))) uint4*)&s_stage[wv][0][0][0]));
  uint32_t rq_off = 0, rq_i = 0, rq = 0;  // the next stage to request: its first value, its run, its number
  auto request = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) load_to_lds(src[j] + rq_off, lds + (rq % kRouterRing) * 4096 + j * 1024);
    ++rq;
    rq_off += 512;
    if (++rq_i == n_i) {  // the next group's first run; behind the last stage: the first group's again, which nobody uses
      rq_i = 0;
      rq_off = rq < n_st ? 32 * (rq / n_i) : 0;
    }
  };
  uint32_t rd_at[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) rd_at[j] = m * 4 + ((2 * j + b) ^ ((m >> 2) & 3));  // pair j of the group, block b
  uint4 raw[2][2];  // [pair][x, w] of the stage at hand
  auto take = [&](uint32_t st) __attribute__((always_inline)) {
    const uint4* buf = &s_stage[wv][st % kRouterRing][0][0];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int o = 0; o < 2; ++o) raw[j][o] = buf[o * 128 + rd_at[j]];
  };
#pragma unroll
  for (int u = 0; u < kRouterRing; ++u) request();
  wait_loads<4 * (kRouterRing - 1)>();
  take(0);

  float lev1[16], lev2[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) lev1[r] = lev2[r] = 0.0f;
  uint32_t st = 0;
#pragma unroll 1
  for (uint32_t pg = 0; pg < kGroups; ++pg) {
    f32x32_t acc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 32; ++r) acc[j][r] = 0.0f;
#pragma unroll 1
    for (uint32_t i = 0; i < n_i; ++i, ++st) {
      // All operands of the stage in registers of their own before its first matrix instruction: a vector instruction that writes a
      // register an MFMA in flight still reads as A or B waits until that MFMA is done (64 cycles here), so operands made one at a
      // time in a recycled register pair cost 89 instead of 65 cycles per instruction.
      float op[2][2][8];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int o = 0; o < 2; ++o) {
          const uint32_t v[4] = {raw[j][o].x, raw[j][o].y, raw[j][o].z, raw[j][o].w};
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            op[j][o][2 * u] = bf16_lo(v[u]);
            op[j][o][2 * u + 1] = bf16_hi(v[u]);
          }
#pragma unroll
          for (int u = 0; u < 8; ++u) asm volatile("" : "+v"(op[j][o][u]));
        }
      request();  // into the stage just taken up
      wait_loads<4 * (kRouterRing - 1)>();
      take(st + 1);
      __builtin_amdgcn_sched_barrier(0);  // (left to itself the compiler reads them behind most of the matrix instructions)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int u = 0; u < 8; ++u) acc[j] = __builtin_amdgcn_mfma_f32_32x32x1f32(op[j][0][u], op[j][1][u], acc[j], 0, 0, 0);
    }
    // two pairs of chains are complete: the stride-1 level, the pairs' sum, then the binary counter
    float carry[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) carry[r] = (acc[0][r] + acc[0][16 + r]) + (acc[1][r] + acc[1][16 + r]);
    if (pg == 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) lev1[r] = carry[r];
    } else if (pg == 1) {
#pragma unroll
      for (int r = 0; r < 16; ++r) lev2[r] = lev1[r] + carry[r];
    } else if (pg == 2) {
#pragma unroll
      for (int r = 0; r < 16; ++r) lev1[r] = carry[r];
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) lev1[r] = lev2[r] + (lev1[r] + carry[r]);
    }
  }
  // the last levels of the tree, over the ring: neighbouring waves first
  wait_loads<0>();
  __syncthreads();
  float* s_part = reinterpret_cast<float*>(&s_stage[0][0][0][0]);  // [wave][16][64]
#pragma unroll
  for (int r = 0; r < 16; ++r) s_part[(wv * 16 + r) * 64 + lane] = lev1[r];
  __syncthreads();
#pragma unroll
  for (uint32_t q = 0; q < 4; ++q) {  // a wave stores a quarter: tokens 8 wv + 4b + q
    const uint32_t r = 4 * wv + q, t = t0 + 8 * wv + 4 * b + q;
    const float* v = s_part + r * 64 + lane;
    const float sum = (v[0] + v[1024]) + (v[2048] + v[3072]);
    if (t < T) logits[static_cast<size_t>(t) * ld + e0 + m] = sum;
  }
}

// ---------------------------------------------------------------- grouping
//
// PrefillMoEGrouping.groupTokenExpertPairs (PrefillMoEGrouping.swift:91-192) on
// device: pairs come token-major (token, rank), so "sorted by (expert, token,
// rank)" is a stable counting sort by expert.  The pair list is cut into at
// most kGroupChunks chunks; every chunk counts its routes per expert, one
// block turns the counts into per-(chunk, expert) start positions, and every
// chunk then places its routes in order.

constexpr uint32_t kGroupChunks = 256;   // rows of the per-chunk count matrix
constexpr uint32_t kGroupBlock = 256;    // pairs one workgroup handles per step

__global__ __launch_bounds__(256) void group_count_kernel(const uint32_t* __restrict__ idx,
                                                          uint32_t n_pairs, uint32_t E,
                                                          uint32_t chunk_pairs,
                                                          uint32_t* __restrict__ chunk_hist,
                                                          uint32_t* __restrict__ chunk_bad) {
  __shared__ uint32_t s_hist[MF_MAX_EXPERTS];
  for (uint32_t e = threadIdx.x; e < E; e += blockDim.x) s_hist[e] = 0;
  __syncthreads();
  const uint32_t p0 = blockIdx.x * chunk_pairs, p1 = min(n_pairs, p0 + chunk_pairs);
  bool bad = false;
  for (uint32_t p = p0 + threadIdx.x; p < p1; p += blockDim.x) {
    const uint32_t e = idx[p];
    if (e < E) atomicAdd(&s_hist[e], 1u);
    else bad = true;
  }
  // one flag per chunk, always written: nothing has to be cleared before the launch
  const int any_bad = __syncthreads_or(bad ? 1 : 0);
  if (threadIdx.x == 0) chunk_bad[blockIdx.x] = any_bad ? 1u : 0u;
  for (uint32_t e = threadIdx.x; e < E; e += blockDim.x) chunk_hist[blockIdx.x * E + e] = s_hist[e];
}

// From every expert's count (thread e holds c; threads past MF_MAX_EXPERTS only keep the barriers
// company): counts, offsets (0xFFFFFFFF for an empty expert), the start of every expert's run and
// the tile lists of the matmuls.
__device__ __forceinline__ void group_layout(uint32_t c, uint32_t E, uint32_t* __restrict__ counts,
                                             uint32_t* __restrict__ offsets, uint32_t* __restrict__ starts,
                                             const TileLists& tiles, uint32_t* s_cnt,
                                             bool publish = true) {
  const uint32_t e = threadIdx.x;
  const bool act = e < MF_MAX_EXPERTS;
  if (publish && e < E) counts[e] = c;
  // inclusive scans of the counts and of the two lists' tile counts over the MF_MAX_EXPERTS entries: inside a
  // wave by shuffles, the eight wave totals through the last slots of the two arrays' neighbours
  __shared__ uint32_t s_wave_cnt[MF_MAX_EXPERTS / 64], s_wave_tile[2][MF_MAX_EXPERTS / 64], s_total[2];
  uint32_t run_c = act ? c : 0u, mine[2] = {}, run_t[2];
#pragma unroll
  for (int l = 0; l < 2; ++l) {
    if (publish && act && tiles.list[l]) mine[l] = (c + tiles.tokens[l] - 1) / tiles.tokens[l];
    run_t[l] = mine[l];
  }
  const uint32_t lane = e & 63u;
  for (uint32_t o = 1; o < 64; o <<= 1) {
    const uint32_t a = static_cast<uint32_t>(__shfl_up(static_cast<int>(run_c), o, 64));
    const uint32_t b0 = static_cast<uint32_t>(__shfl_up(static_cast<int>(run_t[0]), o, 64));
    const uint32_t b1 = static_cast<uint32_t>(__shfl_up(static_cast<int>(run_t[1]), o, 64));
    if (lane >= o) {
      run_c += a;
      run_t[0] += b0;
      run_t[1] += b1;
    }
  }
  if (act && lane == 63) {
    s_wave_cnt[e >> 6] = run_c;
    s_wave_tile[0][e >> 6] = run_t[0];
    s_wave_tile[1][e >> 6] = run_t[1];
  }
  __syncthreads();
  if (act) {
    for (uint32_t v = 0; v < (e >> 6); ++v) {
      run_c += s_wave_cnt[v];
      run_t[0] += s_wave_tile[0][v];
      run_t[1] += s_wave_tile[1][v];
    }
    s_cnt[e] = run_c;
  }
  if (e == MF_MAX_EXPERTS - 1) {
    s_total[0] = run_t[0];
    s_total[1] = run_t[1];
  }
  __syncthreads();
  if (publish && e < E) {
    const uint32_t start = run_c - c;
    starts[e] = start;
    offsets[e] = c ? start : 0xFFFFFFFFu;
#pragma unroll
    for (int l = 0; l < 2; ++l) {
      if (!tiles.list[l]) continue;
      const uint32_t tokens = tiles.tokens[l], first = run_t[l] - mine[l], total = s_total[l];
      if (e == 0 && total == 0) tiles.list[l][0] = Tile{0, 0, 0, 0};
      for (uint32_t j = 0; j < mine[l]; ++j)
        tiles.list[l][first + j] = Tile{e, start + j * tokens, min(tokens, c - j * tokens), total};
    }
  }
}

// counts, offsets (0xFFFFFFFF for an empty expert), the start of every expert's
// run, chunk_hist turned into each chunk's first position inside its expert's
// run, and the tile lists of the matmuls.
__global__ __launch_bounds__(512) void group_scan_kernel(uint32_t* __restrict__ chunk_hist,
                                                         uint32_t n_chunks, uint32_t E,
                                                         uint32_t* __restrict__ counts,
                                                         uint32_t* __restrict__ offsets,
                                                         uint32_t* __restrict__ starts,
                                                         const TileLists tiles,
                                                         const uint32_t* __restrict__ chunk_bad,
                                                         uint32_t* __restrict__ status,
                                                         int drop_if_bad = 0) {
  __shared__ uint32_t s_cnt[MF_MAX_EXPERTS];
  const uint32_t e = threadIdx.x;
  // status word: 2 when any chunk met an expert index out of range (n_chunks <= blockDim)
  const int any_bad = __syncthreads_or(e < n_chunks && chunk_bad[e] ? 1 : 0);
  if (e == 0) *status = any_bad ? 2u : 0u;
  uint32_t c = 0;
  if (e < E && !(any_bad && drop_if_bad)) {  // a caller's grouping that failed its check yields no tiles
    uint32_t k = 0;
    for (; k + 32 <= n_chunks; k += 32) {  // 32 independent loads in flight: the loop is all latency
      uint32_t v[32];
#pragma unroll
      for (int u = 0; u < 32; ++u) v[u] = chunk_hist[(k + u) * E + e];
#pragma unroll
      for (int u = 0; u < 32; ++u) {
        chunk_hist[(k + u) * E + e] = c;
        c += v[u];
      }
    }
    for (; k < n_chunks; ++k) {
      const uint32_t v = chunk_hist[k * E + e];
      chunk_hist[k * E + e] = c;
      c += v;
    }
  }
  group_layout(c, E, counts, offsets, starts, tiles, s_cnt);
}

__global__ __launch_bounds__(256) void group_emit_kernel(const uint32_t* __restrict__ idx,
                                                         const float* __restrict__ w,
                                                         uint32_t n_pairs, uint32_t K, uint32_t E,
                                                         uint32_t chunk_pairs,
                                                         const uint32_t* __restrict__ chunk_base,
                                                         const uint32_t* __restrict__ starts,
                                                         mf_pair* __restrict__ sorted) {
  __shared__ uint32_t s_base[MF_MAX_EXPERTS];      // next free position of every expert's run
  __shared__ uint32_t s_wave[4][MF_MAX_EXPERTS];   // routes per expert of each wave in this step
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (uint32_t e = threadIdx.x; e < E; e += blockDim.x) {
    s_base[e] = starts[e] + chunk_base[blockIdx.x * E + e];
    s_wave[0][e] = s_wave[1][e] = s_wave[2][e] = s_wave[3][e] = 0;
  }
  __syncthreads();
  const uint32_t p0 = blockIdx.x * chunk_pairs, p1 = min(n_pairs, p0 + chunk_pairs);
  for (uint32_t q0 = p0; q0 < p1; q0 += kGroupBlock) {
    const uint32_t p = q0 + threadIdx.x;
    const bool valid = p < p1;
    const uint32_t e = valid ? idx[p] : 0xFFFFFFFFu;
    // rank of this route among the routes of its expert in this wave, in pair order
    bool open = valid && e < E;
    uint32_t rank = 0;
    unsigned long long todo = __ballot(open);
    while (todo) {
      const int leader = __ffsll(static_cast<long long>(todo)) - 1;
      const uint32_t e0 = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(e), leader));
      const unsigned long long same = __ballot(open && e == e0);
      if (open && e == e0) {
        rank = __popcll(same & ((1ull << lane) - 1ull));
        open = false;
      }
      if (lane == static_cast<uint32_t>(leader)) s_wave[wv][e0] = __popcll(same);
      todo &= ~same;
    }
    __syncthreads();
    if (valid && e < E) {
      uint32_t pos = s_base[e] + rank;
      for (uint32_t v = 0; v < wv; ++v) pos += s_wave[v][e];
      mf_pair r;
      r.token = p / K;
      r.expert = e;
      r.rank = p % K;
      r.weight_bits = __float_as_uint(w[p]);
      sorted[pos] = r;
    }
    __syncthreads();
    if (q0 + kGroupBlock < p1) {  // another step follows: advance the bases, clear the wave counts
      for (uint32_t x = threadIdx.x; x < E; x += blockDim.x) {
        s_base[x] += s_wave[0][x] + s_wave[1][x] + s_wave[2][x] + s_wave[3][x];
        s_wave[0][x] = s_wave[1][x] = s_wave[2][x] = s_wave[3][x] = 0;
      }
      __syncthreads();
    }
  }
}

// The stable counting sort by ballots, in one workgroup of 16 waves: each wave is a "chunk" (a contiguous
// run of the pair list) with its per-expert counts in LDS (s_hist: [16][MF_MAX_EXPERTS]).
__device__ __forceinline__ void group_serial(const uint32_t* __restrict__ idx, const float* __restrict__ w,
                                             uint32_t n_pairs, uint32_t K, uint32_t E,
                                             uint32_t* __restrict__ counts, uint32_t* __restrict__ offsets,
                                             uint32_t* __restrict__ starts, mf_pair* __restrict__ sorted,
                                             const TileLists tiles, uint32_t* s_hist_flat,
                                             uint32_t* s_cnt) {
  uint32_t (*s_hist)[MF_MAX_EXPERTS] = reinterpret_cast<uint32_t (*)[MF_MAX_EXPERTS]>(s_hist_flat);
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < 16 * MF_MAX_EXPERTS; i += blockDim.x) s_hist_flat[i] = 0;
  __syncthreads();
  const uint32_t chunk = ((n_pairs + 15) / 16 + 63) / 64 * 64;
  const uint32_t p0 = min(n_pairs, wv * chunk), p1 = min(n_pairs, p0 + chunk);
  for (uint32_t p = p0 + lane; p < p1; p += 64) {
    const uint32_t e = idx[p];
    if (e < E) atomicAdd(&s_hist[wv][e], 1u);
  }
  __syncthreads();
  uint32_t c = 0;
  if (threadIdx.x < E) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const uint32_t n = s_hist[v][threadIdx.x];
      s_hist[v][threadIdx.x] = c;
      c += n;
    }
  }
  group_layout(c, E, counts, offsets, starts, tiles, s_cnt);
  __syncthreads();
  // s_cnt holds the inclusive scan: an expert's run starts at s_cnt[e - 1]; the waves' bases are
  // relative to that start
  for (uint32_t q0 = p0; q0 < p1; q0 += 64) {
    const uint32_t p = q0 + lane;
    const bool valid = p < p1;
    const uint32_t e = valid ? idx[p] : 0xFFFFFFFFu;
    bool open = valid && e < E;
    const bool mine = open;
    uint32_t pos = 0;
    unsigned long long todo = __ballot(open);
    while (todo) {  // rank of this route among the routes of its expert in this step, in pair order
      const int leader = __ffsll(static_cast<long long>(todo)) - 1;
      const uint32_t e0 = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(e), leader));
      const unsigned long long same = __ballot(open && e == e0);
      const uint32_t base = s_hist[wv][e0];
      if (open && e == e0) {
        pos = base + __popcll(same & ((1ull << lane) - 1ull));
        open = false;
      }
      if (lane == static_cast<uint32_t>(leader)) s_hist[wv][e0] = base + __popcll(same);
      todo &= ~same;
    }
    if (mine) {
      const uint32_t run = (e ? s_cnt[e - 1] : 0u);
      mf_pair r;
      r.token = p / K;
      r.expert = e;
      r.rank = p % K;
      r.weight_bits = __float_as_uint(w[p]);
      sorted[run + pos] = r;
    }
  }
}

// The three steps above in one workgroup, for token counts whose (expert x token) bit matrix fits LDS.
// A token names an expert at most once (a top-k does), so "the routes of expert e in token order" is row
// e of that matrix: a route's place in its expert's run is the number of set bits before its token's, i.e.
// a per-word prefix count plus a popcount -- no serial ranking at all.  Every thread marks its routes
// (LDS atomic OR), the rows are prefix-counted (several threads per row), the expert counts go through the
// same layout step as the three-launch form, and every thread places its routes.  Input that does name
// an expert twice in one token (legal for the reference's grouping, never produced by a router) is
// noticed when the bit is already set; the workgroup then does the stable ranking the slow way (each of
// its 16 waves a chunk of the pair list, ballots per step) -- same result, same launch.
constexpr uint32_t kGroupOnePairs = 8192;  // beyond this the pair list is worth several workgroups (T=2048, K=8: 31 us in one, 20 us in three launches)
constexpr uint32_t kGroupOneMaxBytes = 112 * 1024;  // bit matrix + prefix counts the single workgroup may hold

__host__ __device__ __forceinline__ uint32_t group_one_row_words(uint32_t t) { return ((t + 31) / 32) | 1u; }  // odd: rows fall on different banks
__host__ __device__ __forceinline__ size_t group_one_lds_bytes(uint32_t t, uint32_t E) {
  const size_t bits = static_cast<size_t>(E) * group_one_row_words(t) * 6;  // u32 words + u16 prefix counts
  const size_t serial = 16 * MF_MAX_EXPERTS * 4;                            // the slow path's per-wave counts
  return (bits > serial ? bits : serial) + 16;
}

// Workgroups behind the first prepare x, a row per wave (the layer call with a router of its own has that done beside the router): one
// workgroup groups for 8 to 12 us while the chip is idle otherwise.  Given routing, us: 777 tokens of 4096 with the scalar gate, grouping
// 11.5 and a launch of 9.0 behind it -> 11.8; 300 tokens of 2816, 8.1 and 4.8 -> 8.3.  They carry the first one's threads and LDS, one or
// two to a CU, and gain where they are most, too.  The layer call, experts of 128, top 1, us, behind / beside: 16 experts of 2048, 8192 tokens
// 90.8 / 79.9; 64 experts of 2048, 512 tokens 38.0 / 34.7, 8192 90.0 / 79.4; of 4096, 8192 tokens 162.1 / 157.6 (shared expert of 128:
// 234.8 / 226.7); top 2, 128 experts of 5120, 4096 tokens 170.6 / 162.6.
__global__ __launch_bounds__(1024) void group_one_kernel(const uint32_t* __restrict__ idx,
                                                         const float* __restrict__ w, uint32_t n_pairs,
                                                         uint32_t K, uint32_t E, uint32_t tpe_log2,
                                                         uint32_t* __restrict__ counts,
                                                         uint32_t* __restrict__ offsets,
                                                         uint32_t* __restrict__ starts,
                                                         mf_pair* __restrict__ sorted, const TileLists tiles,
                                                         uint32_t* __restrict__ status, const uint16_t* __restrict__ x,
                                                         uint32_t D, const RouterTail prep) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ uint32_t s_cnt[MF_MAX_EXPERTS], s_row[MF_MAX_EXPERTS];
  const uint32_t T = n_pairs / K, W = group_one_row_words(T);
  if (blockIdx.x) {
    const uint32_t r = (blockIdx.x - 1) * 16 + (threadIdx.x >> 6);
    if (r < T) prep_x_row(x + static_cast<size_t>(r) * D, prep.xp, prep.sums, prep.row_max, prep.w_sg, prep.gate, r, D, threadIdx.x & 63);
    return;
  }
  uint32_t* bm = reinterpret_cast<uint32_t*>(smem);                 // [E][W] bits: token t of row e
  uint16_t* pref = reinterpret_cast<uint16_t*>(smem + static_cast<size_t>(E) * W * 4);  // [E][W] set bits before word
  // a thread's routes (at most kGroupOnePairs / 1024 = 8) stay in registers from the marking pass to the
  // placing pass: one round trip to memory instead of two
  constexpr uint32_t kMine = kGroupOnePairs / 1024;
  static_assert(kGroupOnePairs % 1024 == 0, "the launch has 1024 threads");
  uint32_t my_e[kMine], my_w[kMine];
#pragma unroll
  for (uint32_t u = 0; u < kMine; ++u) {
    const uint32_t p = threadIdx.x + u * 1024;
    my_e[u] = p < n_pairs ? idx[p] : 0xFFFFFFFFu;
    my_w[u] = p < n_pairs ? __float_as_uint(w[p]) : 0u;
  }
  for (uint32_t i = threadIdx.x; i < E * W; i += blockDim.x) bm[i] = 0;
  __syncthreads();
  bool bad = false, dup = false;
#pragma unroll
  for (uint32_t u = 0; u < kMine; ++u) {
    const uint32_t p = threadIdx.x + u * 1024;
    if (p >= n_pairs) break;
    const uint32_t e = my_e[u], t = p / K;
    if (e < E) {
      const uint32_t bit = 1u << (t & 31u);
      dup |= (atomicOr(&bm[e * W + (t >> 5)], bit) & bit) != 0u;
    } else {
      bad = true;
    }
  }
  const int any_bad = __syncthreads_or(bad ? 1 : 0);
  const int any_dup = __syncthreads_or(dup ? 1 : 0);
  if (threadIdx.x == 0) *status = any_bad ? 2u : 0u;
  if (any_dup) {
    group_serial(idx, w, n_pairs, K, E, counts, offsets, starts, sorted, tiles,
                 reinterpret_cast<uint32_t*>(smem), s_cnt);
    return;
  }
  // prefix counts of every row: 2^tpe_log2 threads per row, each a run of words
  const uint32_t tpe = 1u << tpe_log2, row = threadIdx.x >> tpe_log2, part = threadIdx.x & (tpe - 1u);
  const uint32_t per = (W + tpe - 1) / tpe, w0 = min(W, part * per), w1 = min(W, w0 + per);
  uint32_t mine = 0;
  if (row < E)
    for (uint32_t j = w0; j < w1; ++j) mine += __popc(bm[row * W + j]);
  // exclusive scan of `mine` over the row's threads (they are neighbours in one wave: tpe <= 16)
  uint32_t before = 0, total = mine;
  for (uint32_t o = 1; o < tpe; o <<= 1) {
    const uint32_t v = static_cast<uint32_t>(__shfl_up(static_cast<int>(total), o, 64));
    if (part >= o) total += v;
  }
  before = total - mine;
  const uint32_t row_total = static_cast<uint32_t>(__shfl(static_cast<int>(total), (threadIdx.x & 63u) | (tpe - 1u), 64));
  if (row < E) {
    uint32_t c = before;
    for (uint32_t j = w0; j < w1; ++j) {
      pref[row * W + j] = static_cast<uint16_t>(c);
      c += __popc(bm[row * W + j]);
    }
    if (part == 0) s_row[row] = row_total;  // parked for the layout step below
  }
  __syncthreads();
  const uint32_t c = threadIdx.x < E ? s_row[threadIdx.x] : 0u;
  __syncthreads();
  group_layout(c, E, counts, offsets, starts, tiles, s_cnt);
  __syncthreads();
#pragma unroll
  for (uint32_t u = 0; u < kMine; ++u) {
    const uint32_t p = threadIdx.x + u * 1024, e = my_e[u];
    if (p >= n_pairs || e >= E) continue;
    const uint32_t t = p / K, at = e * W + (t >> 5);
    const uint32_t pos = (e ? s_cnt[e - 1] : 0u) + pref[at] + __popc(bm[at] & ((1u << (t & 31u)) - 1u));
    mf_pair r;
    r.token = t;
    r.expert = e;
    r.rank = p - t * K;
    r.weight_bits = my_w[u];
    sorted[pos] = r;
  }
}

// The layer call selects the routes itself, so selection and grouping share launches: two instead of the
// selector's one plus the grouping's one or three.  A top-k names an expert at most once per token, so the
// routes of expert e inside a chunk of up to 64 consecutive tokens are a 64-bit word (bit i: token i of
// the chunk routes to e) and "how many routes of e come before mine" is a popcount.
//
// First launch: a workgroup selects the routes of one chunk (a wave a token at a time, the selectors of
// topk_kernel), stores them, and leaves the chunk's word per expert and, as a row of bytes, its number of
// routes per expert.
constexpr uint32_t kSelectWaves = 16;
constexpr uint32_t kChunkTokensMax = 64;
static_assert(kChunkTokensMax * MF_MAX_TOPK <= MF_MAX_EXPERTS, "a chunk's routes are placed by one workgroup in one step");

__global__ __launch_bounds__(kSelectWaves * 64) void topk_chunk_kernel(const float* __restrict__ logits, uint32_t T,
                                                                       uint32_t E, uint32_t K, int mode,
                                                                       uint32_t chunk_tokens,
                                                                       uint32_t* __restrict__ idx,
                                                                       float* __restrict__ w,
                                                                       unsigned long long* __restrict__ chunk_bits,
                                                                       uint8_t* __restrict__ chunk_cnt,
                                                                       uint32_t* __restrict__ chunk_bad) {
  __shared__ uint32_t s_bits[2][MF_MAX_EXPERTS];
  __shared__ float s_p[kSelectWaves][MF_MAX_EXPERTS];  // the full softmax's probabilities, a row per wave
  __shared__ uint32_t s_i[kSelectWaves][MF_MAX_TOPK];
  __shared__ float s_wt[kSelectWaves][MF_MAX_TOPK];
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (uint32_t e = threadIdx.x; e < E; e += blockDim.x) s_bits[0][e] = s_bits[1][e] = 0u;
  __syncthreads();
  const uint32_t t0 = blockIdx.x * chunk_tokens, t1 = min(T, t0 + chunk_tokens);
  bool bad = false;
  for (uint32_t t = t0 + wv; t < t1; t += kSelectWaves) {
    const float* lg = logits + static_cast<size_t>(t) * E;
    if (mode == 0) topk_select_fast(lg, E, K, s_i[wv], s_wt[wv], lane);
    else topk_full_softmax_fast(lg, s_p[wv], E, K, s_i[wv], s_wt[wv], lane);
    if (lane < K) {
      const uint32_t e = s_i[wv][lane];
      idx[static_cast<size_t>(t) * K + lane] = e;
      w[static_cast<size_t>(t) * K + lane] = s_wt[wv][lane];
      const uint32_t i = t - t0;
      if (e < E) atomicOr(&s_bits[i >> 5][e], 1u << (i & 31u));
      else bad = true;  // the full softmax's "routes nowhere"
    }
  }
  // one flag per chunk, always written: nothing has to be cleared before the launch
  const int any_bad = __syncthreads_or(bad ? 1 : 0);
  if (threadIdx.x == 0) chunk_bad[blockIdx.x] = any_bad ? 1u : 0u;
  for (uint32_t e = threadIdx.x; e < E; e += blockDim.x) {
    const uint32_t lo = s_bits[0][e], hi = s_bits[1][e];
    chunk_bits[static_cast<size_t>(blockIdx.x) * E + e] =
        static_cast<unsigned long long>(lo) | (static_cast<unsigned long long>(hi) << 32);
    chunk_cnt[static_cast<size_t>(blockIdx.x) * E + e] = static_cast<uint8_t>(__popc(lo) + __popc(hi));
  }
}

// Second launch: every workgroup adds up the chunks' counts per expert (an expert's total, and its routes
// in the chunks before the workgroup's own), repeats the layout scans for itself, and places the routes of
// its chunk; the first workgroup also publishes counts, offsets, starts, the tile list and the status word.
__global__ __launch_bounds__(MF_MAX_EXPERTS) void group_place_kernel(const uint32_t* __restrict__ idx,
                                                                    const float* __restrict__ w, uint32_t T,
                                                                    uint32_t K, uint32_t E, uint32_t chunk_tokens,
                                                                    uint32_t n_chunks,
                                                                    const unsigned long long* __restrict__ chunk_bits,
                                                                    const uint8_t* __restrict__ chunk_cnt,
                                                                    const uint32_t* __restrict__ chunk_bad,
                                                                    uint32_t* __restrict__ counts,
                                                                    uint32_t* __restrict__ offsets,
                                                                    uint32_t* __restrict__ starts,
                                                                    mf_pair* __restrict__ sorted,
                                                                    const TileLists tiles,
                                                                    uint32_t* __restrict__ status) {
  __shared__ uint32_t s_cnt[MF_MAX_EXPERTS], s_base[MF_MAX_EXPERTS];
  __shared__ unsigned long long s_mine[MF_MAX_EXPERTS];
  const uint32_t e = threadIdx.x, me = blockIdx.x;
  const bool first = me == 0;
  // this workgroup's routes, requested before anything is waited for
  const uint32_t t0 = me * chunk_tokens, t1 = min(T, t0 + chunk_tokens);
  const uint32_t n = (t1 - t0) * K;  // <= kChunkTokensMax * MF_MAX_TOPK <= blockDim
  const size_t p = static_cast<size_t>(t0) * K + threadIdx.x;
  uint32_t ex = 0xFFFFFFFFu, wbits = 0u;
  if (threadIdx.x < n) {
    ex = idx[p];
    wbits = __float_as_uint(w[p]);
  }
  uint32_t c = 0, before = 0;
  if (e < E) {
    s_mine[e] = chunk_bits[static_cast<size_t>(me) * E + e];
    uint32_t k = 0;
    for (; k + 32 <= n_chunks; k += 32) {  // 32 independent byte loads in flight
      uint32_t v[32];
#pragma unroll
      for (int u = 0; u < 32; ++u) v[u] = chunk_cnt[static_cast<size_t>(k + u) * E + e];
#pragma unroll
      for (int u = 0; u < 32; ++u) {
        c += v[u];
        before += k + u < me ? v[u] : 0u;
      }
    }
    for (; k < n_chunks; ++k) {
      const uint32_t v = chunk_cnt[static_cast<size_t>(k) * E + e];
      c += v;
      before += k < me ? v : 0u;
    }
  }
  const int any_bad = __syncthreads_or(e < n_chunks && chunk_bad[e] ? 1 : 0);  // n_chunks <= blockDim
  if (first && e == 0) *status = any_bad ? 2u : 0u;
  group_layout(c, E, counts, offsets, starts, tiles, s_cnt, first);
  if (e < E) s_base[e] = s_cnt[e] - c + before;  // s_cnt is the inclusive scan of the counts
  __syncthreads();
  if (ex < E) {
    const uint32_t i = threadIdx.x / K;
    mf_pair r;
    r.token = t0 + i;
    r.expert = ex;
    r.rank = threadIdx.x - i * K;
    r.weight_bits = wbits;
    sorted[s_base[ex] + __popcll(s_mine[ex] & ((1ull << i) - 1ull))] = r;
  }
}

// ---- the expert pool in the matmul's order
// Row by row a load instruction of the matmul touches 16 (4-bit) or 32 (2-bit) weight rows, a memory line each, and
// the L1's line rate is a part of what a work item costs.  In the
// tiled pool every sub-tensor keeps its place in the blob and its size; inside it, the 16-byte pieces of the 32 rows
// of a block sit side by side, so that a load instruction reads whole runs of consecutive bytes, every lane what it
// multiplies.  4-bit: one run of 1 KB per K group, piece l = m + 32 h = half h of the group of row 32 rb + m.
// 2-bit, ternary: one run of 1 KB per two groups, piece l = half h of both groups of that row.  Scale and bias tables
// stay row by row.  One thread per piece; sub-tensor w of every expert in one launch.
__global__ __launch_bounds__(256) void tile_codes_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                         size_t expert_stride, uint32_t w_off, uint32_t rows,
                                                         uint32_t ng, uint32_t group_bytes) {
  const uint32_t row_bytes = ng * group_bytes, runs = row_bytes / 32;  // (K is a multiple of 128)
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= static_cast<uint64_t>(rows) * (row_bytes / 16)) return;
  const uint32_t m = static_cast<uint32_t>(i & 31u), h = static_cast<uint32_t>(i >> 5) & 1u;
  const uint64_t run = i >> 6;
  const uint32_t r = static_cast<uint32_t>(run % runs), rb = static_cast<uint32_t>(run / runs);
  const size_t base = static_cast<size_t>(blockIdx.y) * expert_stride + w_off;
  const uint8_t* from = src + base + static_cast<size_t>(32u * rb + m) * row_bytes + r * 32;
  uint4 v;
  if (group_bytes == 32) {
    v = *reinterpret_cast<const uint4*>(from + h * 16);
  } else {
    const uint2 a = *reinterpret_cast<const uint2*>(from + h * 8), b = *reinterpret_cast<const uint2*>(from + 16 + h * 8);
    v = make_uint4(a.x, a.y, b.x, b.y);
  }
  *reinterpret_cast<uint4*>(dst + base + i * 16) = v;
}

// dst = the pool `src` (E blobs, expert_stride apart) with the three code sub-tensors of every blob tiled
hipError_t launch_tile_experts(hipStream_t s, const mf_moe_config& c, const void* src, size_t expert_stride,
                               const mf_expert_offsets& off, void* dst) {
  hipError_t e = hipMemcpyAsync(dst, src, expert_stride * c.num_experts, hipMemcpyDeviceToDevice, s);
  if (e != hipSuccess) return e;
  const uint32_t gb = c.bits == MF_BITS_4 ? 32u : 16u;
  const struct { uint32_t off, rows, k; } parts[3] = {{off.gate_w, c.f, c.d}, {off.up_w, c.f, c.d}, {off.down_w, c.d, c.f}};
  for (const auto& p : parts) {
    const uint64_t pieces = static_cast<uint64_t>(p.rows) * (p.k / kGroup) * gb / 16;
    tile_codes_kernel<<<dim3(static_cast<uint32_t>((pieces + 255) / 256), c.num_experts), dim3(256), 0, s>>>(
        static_cast<const uint8_t*>(src), static_cast<uint8_t*>(dst), expert_stride, p.off, p.rows, p.k / kGroup, gb);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// --------------------------------------------------------------- the matmul

// Activation rows as the matmul wants them: inside every run of 8 K values the
// order is (0,4,1,5,2,6,3,7) -- the pairing a packed code word expands to --, every value is times the row's scale,
// and the fp32 sum of every 64-wide K group is kept beside them.  One lane per run of 8.
__device__ __forceinline__ void prep_run(const uint4& v, float scale, uint32_t c, uint32_t chunks, bool live, uint16_t* __restrict__ dst,
                                         uint16_t* __restrict__ sums, float* largest) {
  float sum;
  const uint4 prepared = matmul_row8(v, scale, &sum, largest);
  sum = group_sum(sum, 8);
  if (!live) return;
  *reinterpret_cast<uint4*>(dst + static_cast<size_t>(c) * 8) = prepared;
  if ((c & 7) == 0) store_group_sum(sums, c >> 3, chunks / 8, sum * (scale * kRowUnscale));
}

// A workgroup a row, a thread a run of 8 (of longer rows several): the row's largest magnitude first, so that nothing is written before
// the barrier -- which would wait for it.  A thread's first run stays in registers.
constexpr uint32_t kPrepThreads = 1024;
__global__ __launch_bounds__(kPrepThreads) void prep_rows_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst,
                                                                 uint16_t* __restrict__ sums, float* __restrict__ row_max, uint32_t chunks) {
  __shared__ float s_max[kPrepThreads / kWave];
  const size_t row = blockIdx.x;
  src += row * chunks * 8;
  dst += row * chunks * 8;
  sums += row * group_sum_words(chunks / 8);
  auto run = [&](uint32_t c) { return c < chunks ? *reinterpret_cast<const uint4*>(src + static_cast<size_t>(c) * 8) : make_uint4(0, 0, 0, 0); };
  const uint4 first = run(threadIdx.x);
  float largest = 0.0f, sum;
  matmul_row8(first, kRowScale, &sum, &largest);
  for (uint32_t c = threadIdx.x + blockDim.x; c < chunks; c += blockDim.x) matmul_row8(run(c), kRowScale, &sum, &largest);
  largest = wave_max(largest);
  if ((threadIdx.x & 63u) == 0) s_max[threadIdx.x >> 6] = largest;
  __syncthreads();
  for (uint32_t w = 0; w < blockDim.x / kWave; ++w) largest = fmaxf(largest, s_max[w]);
  if (threadIdx.x == 0) row_max[row] = largest;
  const float scale = row_scale(largest);
  for (uint32_t c0 = 0; c0 < chunks; c0 += blockDim.x) {
    const uint32_t c = c0 + threadIdx.x;
    prep_run(c0 ? run(c) : first, scale, c, chunks, c < chunks, dst, sums, &largest);
  }
}

// The same for the layer's input rows and, in the same pass, the scalar shared gate's logit
// w_sg . x of every row (prefill_qwen_shared_scalar_gate, prefill.metal:42-80) in the router's lane
// order (dot_bf16_row: lane l takes the chunks l, l+64, ... of a row, neighbour-first butterfly), so
// the gate has the bits of the stand-alone router-row launch it replaces.  One wave per row, which is written at the ordinary
// scale, and a second time where its largest magnitude asks for another.
__device__ __forceinline__ void prep_x_row(const uint16_t* __restrict__ xr, uint16_t* __restrict__ xp,
                                           uint16_t* __restrict__ sums, float* __restrict__ row_max, const uint16_t* __restrict__ w_sg,
                                           uint16_t* __restrict__ gate, uint32_t row, uint32_t d, uint32_t lane) {
  const uint32_t chunks = d / 8;  // a multiple of 8: the 8 lanes of a K group are live together
  xp += static_cast<size_t>(row) * d;
  sums += row * group_sum_words(chunks / 8);
  float acc = 0.0f, largest = 0.0f;
  for (uint32_t c0 = 0; c0 < chunks; c0 += kWave) {
    const uint32_t c = c0 + lane;
    const bool live = c < chunks;
    uint4 v = make_uint4(0, 0, 0, 0), wv = make_uint4(0, 0, 0, 0);
    if (live) {
      v = *reinterpret_cast<const uint4*>(xr + static_cast<size_t>(c) * 8);
      if (w_sg) wv = *reinterpret_cast<const uint4*>(w_sg + static_cast<size_t>(c) * 8);
    }
    prep_run(v, kRowScale, c, chunks, live, xp, sums, &largest);
    if (live) {
      acc = __builtin_fmaf(bf16_lo(wv.x), bf16_lo(v.x), acc);
      acc = __builtin_fmaf(bf16_hi(wv.x), bf16_hi(v.x), acc);
      acc = __builtin_fmaf(bf16_lo(wv.y), bf16_lo(v.y), acc);
      acc = __builtin_fmaf(bf16_hi(wv.y), bf16_hi(v.y), acc);
      acc = __builtin_fmaf(bf16_lo(wv.z), bf16_lo(v.z), acc);
      acc = __builtin_fmaf(bf16_hi(wv.z), bf16_hi(v.z), acc);
      acc = __builtin_fmaf(bf16_lo(wv.w), bf16_lo(v.w), acc);
      acc = __builtin_fmaf(bf16_hi(wv.w), bf16_hi(v.w), acc);
    }
  }
  largest = wave_max(largest);
  if (lane == 0) row_max[row] = largest;
  const float scale = row_scale(largest);
  if (__builtin_expect(scale != kRowScale, 0)) {
    for (uint32_t c0 = 0; c0 < chunks; c0 += kWave) {
      const uint32_t c = c0 + lane;
      uint4 v = make_uint4(0, 0, 0, 0);
      if (c < chunks) v = *reinterpret_cast<const uint4*>(xr + static_cast<size_t>(c) * 8);
      prep_run(v, scale, c, chunks, c < chunks, xp, sums, &largest);
    }
  }
  acc = wave_sum(acc);
  if (w_sg && lane == 0) gate[row] = f_to_bf16(acc);
}

__global__ __launch_bounds__(256) void prep_x_gate_kernel(const uint16_t* __restrict__ x,
                                                          uint16_t* __restrict__ xp, uint16_t* __restrict__ sums,
                                                          float* __restrict__ row_max, const uint16_t* __restrict__ w_sg,
                                                          uint16_t* __restrict__ gate, uint32_t t, uint32_t d) {
  const uint32_t lane = threadIdx.x & 63, row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= t) return;
  prep_x_row(x + static_cast<size_t>(row) * d, xp, sums, row_max, w_sg, gate, row, d, lane);
}

// y[t,d] = bf16(h1[t,d] + sum_r w[t,r] * partial[t*K+r, d]), residual first, rank
// order, product then add (moe.metal:1262-1270; reduce of prefill.metal:631-652).
// h1 = bf16(hs / (1 + exp(-gate_t))) when a scalar gate is given (utility.metal:49-59).
template <bool NARROW>  // the per-route results are bf16 numbers (stored as such) instead of fp32
__global__ __launch_bounds__(256) void prefill_reduce_kernel(const float* __restrict__ partials,
                                                             const float* __restrict__ w,
                                                             const uint32_t* __restrict__ idx,
                                                             const uint16_t* __restrict__ hs,
                                                             const uint16_t* __restrict__ gate,
                                                             uint16_t* __restrict__ y, uint32_t T,
                                                             uint32_t K, uint32_t D, uint32_t E, int maple) {
  const size_t i4 = (static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x) * 4;
  if (i4 >= static_cast<size_t>(T) * D) return;
  const uint32_t t = static_cast<uint32_t>(i4 / D), d = static_cast<uint32_t>(i4 % D);
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  if (hs) {
    const uint2 hv = *reinterpret_cast<const uint2*>(hs + i4);
    acc[0] = bf16_lo(hv.x); acc[1] = bf16_hi(hv.x); acc[2] = bf16_lo(hv.y); acc[3] = bf16_hi(hv.y);
    if (gate) {
      const float den = 1.0f + mf_exp(-bf16_to_f(gate[t]));
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = round_bf16(acc[i] / den);
    }
  }
  // all of a token's routes are requested before the first is used (a short batch has few waves: a loop
  // that tests a route's expert before it asks for the route's row walks K round trips one after another);
  // the row of a route without an expert is read and dropped
  uint32_t ex[MF_MAX_TOPK];
  float wt[MF_MAX_TOPK];
  float4 v[MF_MAX_TOPK];
#pragma unroll
  for (uint32_t r = 0; r < MF_MAX_TOPK; ++r) {
    if (r < K) {
      ex[r] = idx ? idx[t * K + r] : 0u;
      wt[r] = w[t * K + r];
      if constexpr (NARROW) {
        const uint2 q = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(partials) +
                                                        (static_cast<size_t>(t) * K + r) * D + d);
        v[r] = make_float4(bf16_lo(q.x), bf16_hi(q.x), bf16_lo(q.y), bf16_hi(q.y));
      } else {
        v[r] = *reinterpret_cast<const float4*>(partials + (static_cast<size_t>(t) * K + r) * D + d);
      }
    }
  }
#pragma unroll
  for (uint32_t r = 0; r < MF_MAX_TOPK; ++r) {
    if (r < K && ex[r] < E) {  // a route without an expert adds nothing
      float4 q = v[r];
      if (maple && !NARROW) {  // maple_moe.metal:258: the down output is a bf16 number before its weight
        q.x = round_bf16(q.x); q.y = round_bf16(q.y); q.z = round_bf16(q.z); q.w = round_bf16(q.w);
      }
      const float p0 = wt[r] * q.x, p1 = wt[r] * q.y, p2 = wt[r] * q.z, p3 = wt[r] * q.w;
      acc[0] = acc[0] + p0; acc[1] = acc[1] + p1; acc[2] = acc[2] + p2; acc[3] = acc[3] + p3;
    }
  }
  uint2 o;
  o.x = static_cast<uint32_t>(f_to_bf16(acc[0])) | (static_cast<uint32_t>(f_to_bf16(acc[1])) << 16);
  o.y = static_cast<uint32_t>(f_to_bf16(acc[2])) | (static_cast<uint32_t>(f_to_bf16(acc[3])) << 16);
  *reinterpret_cast<uint2*>(y + i4) = o;
}

// The caller's counts as the one-chunk histogram of the scan, and the check's flag cleared (a kernel,
// not a memset or a copy node, so that the call can be captured into a graph).
__global__ __launch_bounds__(512) void ragged_begin_kernel(const uint32_t* __restrict__ counts, uint32_t E,
                                                           uint32_t* __restrict__ hist, uint32_t* __restrict__ bad) {
  if (threadIdx.x < E) hist[threadIdx.x] = counts[threadIdx.x];
  if (threadIdx.x == 0) *bad = 0;
}

// A caller's grouping before the matmuls trust it: the counts cover at most T*K routes, and every
// route the counts cover names a token below T and a rank below K.  Sets *bad otherwise.
__global__ __launch_bounds__(256) void ragged_check_kernel(const mf_pair* __restrict__ sorted,
                                                           const uint32_t* __restrict__ counts,
                                                           uint32_t E, uint32_t T, uint32_t K,
                                                           uint32_t* __restrict__ bad) {
  __shared__ unsigned long long s_total;
  if (threadIdx.x == 0) s_total = 0;
  __syncthreads();
  unsigned long long part = 0;
  for (uint32_t e = threadIdx.x; e < E; e += blockDim.x) part += counts[e];
  if (part) atomicAdd(&s_total, part);
  __syncthreads();
  const unsigned long long total = s_total, pairs = static_cast<unsigned long long>(T) * K;
  if (total > pairs) {
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(bad, 1u);
    return;
  }
  bool wrong = false;
  for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const mf_pair p = sorted[i];
    wrong |= p.token >= T || p.rank >= K;
  }
  if (wrong) atomicOr(bad, 1u);
}

// ------------------------------------------------------------------ launchers

// `tail` (optional): the x preparation a short batch wants done in the same launch; on return
// tail->xp is null when the launch did not take it on (the caller then launches it).
hipError_t launch_prefill_router(hipStream_t s, const uint16_t* W, const uint16_t* x, uint32_t E,
                                 uint32_t D, uint32_t T, uint32_t x_stride, float* logits, RouterTail* tail) {
  RouterTail fused{};
  if (tail) {
    fused = *tail;
    tail->xp = nullptr;
  }
  // Up to 192 tokens the matrix-core kernel has too few workgroups (T/32 x E/32) to cover the chip: the
  // register-tiled kernel is faster there (Qwen shape, layer time: 128 tokens 79 against 82 us, equal at 192,
  // 256 tokens 98.4 against 96.4 us; it holds rows of up to 4096 elements).  Both give the same bits.  The
  // matrix-core kernel takes whole blocks of 32 rows; rows left over (the two sink rows of a 258-row
  // Inkling router) go through the register-tiled kernel behind it.
  const uint32_t e32 = (T > 192 || D > 4096) && D % 512 == 0 && aligned16(W) && aligned16(x) && x_stride % 8 == 0
                           ? E & ~31u : 0u;
  // rows of more than 4096 elements that the matrix-core kernel does not take (a width that is no
  // multiple of 512, rows left over by the blocks of 32, unaligned operands): the register-tiled
  // kernel cannot hold them, so the whole call goes one wave per (token, row) -- the same bits
  if ((D / 8 + 63) / 64 > 8 && e32 != E) return launch_router_logits(s, W, x, E, D, T, x_stride, logits, nullptr);
  const bool tail_ok = fused.xp && x_stride == D && D % 64 == 0 && aligned16(x) && aligned16(fused.xp) &&
                       (!fused.w_sg || aligned16(fused.w_sg));
  if (e32) {
    RouterTail mt{};
    uint32_t prep_rows = 0;
    if (tail_ok) {  // the x preparation rides in this launch: workgroup rows behind the expert blocks
      mt = fused;
      mt.router_cols = e32 / 32;
      fused.xp = nullptr;  // done here: the register-tiled launch for left-over rows does not repeat it
      tail->xp = mt.xp;
    }
    if (tail_ok) prep_rows = ((T + 3) / 4 + (T + 31) / 32 - 1) / ((T + 31) / 32);
    const dim3 grid((T + 31) / 32, e32 / 32 + prep_rows);
    // (rows of 1024 and 2048 unrolled, all others as a loop: the times of both stand at the kernels)
    if (D == 1024) prefill_router_mfma_kernel<2><<<grid, dim3(256), 0, s>>>(W, x, e32, D, T, x_stride, logits, E, mt);
    else if (D == 2048) prefill_router_mfma_kernel<4><<<grid, dim3(256), 0, s>>>(W, x, e32, D, T, x_stride, logits, E, mt);
    else prefill_router_loop_kernel<<<grid, dim3(256), 0, s>>>(W, x, e32, D, T, x_stride, logits, E, mt);
    if (e32 == E) return hipGetLastError();
  }
  const uint32_t rest = E - e32;
  const uint16_t* Wr = W + static_cast<size_t>(e32) * D;
  float* lr = logits + e32;
  const uint32_t cpl = (D / 8 + 63) / 64;
  // about a thousand workgroups, >= 4 tokens per row load; the few rows left over by the matrix-core kernel
  // fill one workgroup column only, so they take the shortest token runs
  const uint32_t tpb = e32 ? 4u : std::max(4u, std::min(64u, T / 64));
  const uint32_t token_blocks = (T + tpb - 1) / tpb;
  // the whole call in this kernel, x rows as the preparation reads them: the launch takes the tail on
  const bool take_tail = tail_ok && fused.xp && !e32 && cpl <= 8;
  if (!take_tail) fused = RouterTail{};
  const uint32_t prep_cols = take_tail ? ((T + 3) / 4 + token_blocks - 1) / token_blocks : 0u;
#define MF_PR(CPL, R)                                                                              \
  do {                                                                                             \
    fused.router_cols = (rest + 4 * R - 1) / (4 * R);                                              \
    prefill_router_kernel<CPL, R><<<dim3(fused.router_cols + prep_cols, token_blocks), dim3(256), 0, s>>>( \
        Wr, x, rest, D, T, x_stride, lr, tpb, E, fused);                                           \
  } while (0)
  if (cpl <= 1) MF_PR(1, 4);
  else if (cpl <= 2) MF_PR(2, 4);
  else if (cpl <= 4) MF_PR(4, 4);
  else if (cpl <= 8) MF_PR(8, 2);
  else return hipErrorInvalidValue;
#undef MF_PR
  if (take_tail) tail->xp = fused.xp;
  return hipGetLastError();
}

hipError_t launch_prefill_router(hipStream_t s, const uint16_t* W, const uint16_t* x, uint32_t E,
                                 uint32_t D, uint32_t T, uint32_t x_stride, float* logits) {
  return launch_prefill_router(s, W, x, E, D, T, x_stride, logits, nullptr);
}

// `prep` (optional): the x preparation of rows of d values, for the grouping launch to take along; its xp is null on return when it did
hipError_t launch_group(hipStream_t s, const uint32_t* idx, const float* w, uint32_t t, uint32_t K,
                        uint32_t E, uint32_t* counts, uint32_t* offsets, uint32_t* starts,
                        mf_pair* sorted, const TileLists& tiles,
                        uint32_t* status, uint32_t* chunk_hist, const uint16_t* x, uint32_t d, RouterTail* prep) {
  const uint32_t n_pairs = t * K;
  if (n_pairs && n_pairs <= kGroupOnePairs && group_one_lds_bytes(t, E) <= kGroupOneMaxBytes) {
    const size_t lds = group_one_lds_bytes(t, E);
    uint32_t tpe_log2 = 0;  // threads per row of the bit matrix: as many as 1024 threads give, at most 16
    while (tpe_log2 < 4 && (E << (tpe_log2 + 1)) <= 1024) ++tpe_log2;
    const hipError_t e = allow_lds<group_one_kernel>(lds, static_cast<int>(kGroupOneMaxBytes));
    if (e != hipSuccess) return e;
    const bool take = prep && prep->xp;
    group_one_kernel<<<dim3(take ? 1 + (t + 15) / 16 : 1), dim3(1024), lds, s>>>(idx, w, n_pairs, K, E, tpe_log2, counts, offsets, starts,
                                                                                sorted, tiles, status, x, d, take ? *prep : RouterTail{});
    if (take) prep->xp = nullptr;
    return hipGetLastError();
  }
  if (n_pairs == 0) {  // no routes: the scan over no chunks writes empty experts and a clean status word
    group_scan_kernel<<<dim3(1), dim3(MF_MAX_EXPERTS), 0, s>>>(chunk_hist, 0, E, counts, offsets, starts,
                                                               tiles,
                                                               chunk_hist, status);
    return hipGetLastError();
  }
  // at most kGroupChunks chunks, each a whole number of kGroupBlock-pair steps
  const uint32_t steps = (n_pairs + kGroupBlock - 1) / kGroupBlock;
  const uint32_t chunk_pairs = (steps + kGroupChunks - 1) / kGroupChunks * kGroupBlock;
  const uint32_t n_chunks = (n_pairs + chunk_pairs - 1) / chunk_pairs;
  uint32_t* chunk_bad = chunk_hist + static_cast<size_t>(kGroupChunks) * MF_MAX_EXPERTS;
  group_count_kernel<<<dim3(n_chunks), dim3(256), 0, s>>>(idx, n_pairs, E, chunk_pairs, chunk_hist, chunk_bad);
  group_scan_kernel<<<dim3(1), dim3(MF_MAX_EXPERTS), 0, s>>>(chunk_hist, n_chunks, E, counts, offsets, starts,
                                                             tiles,
                                                             chunk_bad, status);
  group_emit_kernel<<<dim3(n_chunks), dim3(256), 0, s>>>(idx, w, n_pairs, K, E, chunk_pairs, chunk_hist, starts,
                                                         sorted);
  return hipGetLastError();
}

hipError_t launch_group(hipStream_t s, const uint32_t* idx, const float* w, uint32_t t, uint32_t K,
                        uint32_t E, uint32_t* counts, uint32_t* offsets, uint32_t* starts,
                        mf_pair* sorted, const TileLists& tiles,
                        uint32_t* status, uint32_t* chunk_hist) {
  return launch_group(s, idx, w, t, K, E, counts, offsets, starts, sorted, tiles, status, chunk_hist, nullptr, 0, nullptr);
}

// words of the handle's grouping scratch: 2048 of small tables, the per-chunk counts and flags of the
// three-launch grouping, and behind them the per-chunk 64-bit words and the [chunk][expert] count bytes of
// the layer call's own grouping
constexpr size_t kGroupBitsAt = 2048 + static_cast<size_t>(kGroupChunks) * MF_MAX_EXPERTS + kGroupChunks;  // even
constexpr size_t kGroupCntAt = kGroupBitsAt + 2 * static_cast<size_t>(kGroupChunks) * MF_MAX_EXPERTS;
size_t group_scratch_words() { return kGroupCntAt + static_cast<size_t>(kGroupChunks) * MF_MAX_EXPERTS / 4; }

// Selection and grouping of the layer call's own routes in two launches (topk_chunk_kernel,
// group_place_kernel); false when the batch is too long for chunks of 64 tokens.
bool topk_group_takes(uint32_t t) { return t != 0 && t <= kGroupChunks * kChunkTokensMax; }

hipError_t launch_topk_group(hipStream_t s, const float* logits, uint32_t t, uint32_t K, uint32_t E, int mode,
                             uint32_t* idx, float* w, uint32_t* counts, uint32_t* offsets, uint32_t* starts,
                             mf_pair* sorted, const TileLists& tiles, uint32_t* status,
                             uint32_t* group_tmp) {
  // a token per wave while that gives at most 128 chunks, then longer chunks, then more of them
  uint32_t chunk_tokens = ((t + 127) / 128 + kSelectWaves - 1) / kSelectWaves * kSelectWaves;
  chunk_tokens = std::min(std::max(chunk_tokens, kSelectWaves), kChunkTokensMax);
  const uint32_t n_chunks = (t + chunk_tokens - 1) / chunk_tokens;
  auto* bits = reinterpret_cast<unsigned long long*>(group_tmp + kGroupBitsAt);
  auto* cnt = reinterpret_cast<uint8_t*>(group_tmp + kGroupCntAt);
  uint32_t* bad = group_tmp + 2048 + static_cast<size_t>(kGroupChunks) * MF_MAX_EXPERTS;
  topk_chunk_kernel<<<dim3(n_chunks), dim3(kSelectWaves * 64), 0, s>>>(logits, t, E, K, mode, chunk_tokens, idx, w, bits,
                                                                       cnt, bad);
  group_place_kernel<<<dim3(n_chunks), dim3(MF_MAX_EXPERTS), 0, s>>>(idx, w, t, K, E, chunk_tokens, n_chunks, bits, cnt,
                                                                    bad, counts, offsets, starts, sorted,
                                                                    tiles,
                                                                    status);
  return hipGetLastError();
}

// `rows` rows of k values
hipError_t launch_prep_rows(hipStream_t s, const uint16_t* src, uint16_t* dst, uint16_t* sums, float* row_max, uint32_t rows, uint32_t k) {
  if (!rows || !k) return hipSuccess;
  const uint32_t chunks = k / 8, threads = std::min((chunks + kWave - 1) / kWave * kWave, kPrepThreads);
  prep_rows_kernel<<<dim3(rows), dim3(threads), 0, s>>>(src, dst, sums, row_max, chunks);
  return hipGetLastError();
}

static hipError_t launch_qmm(hipStream_t s, uint32_t tile, int bits, const QmmArgs& a, int nproj, uint32_t tile_slots,
                             const QmmArgs* b, uint32_t b_tile_slots, bool few = false) {
  return tile == kSmallTile ? launch_qmm_tiles<kSmallTile>(s, bits, a, nproj, tile_slots, b, b_tile_slots, few)
                            : launch_qmm_tiles<kTileTokens>(s, bits, a, nproj, tile_slots, b, b_tile_slots, few);
}
static hipError_t launch_qmm_kres(hipStream_t s, uint32_t tile, int bits, const QmmArgs& a, uint32_t tile_slots,
                                  const QmmArgs* b, uint32_t b_tile_slots) {
  return tile == kSmallTile ? launch_kres_tiles<kSmallTile>(s, bits, a, tile_slots, b, b_tile_slots)
                            : launch_kres_tiles<kTileTokens>(s, bits, a, tile_slots, b, b_tile_slots);
}

// Whether qmm_kres_kernel takes the problem: a down-projection epilogue, K of 128, 256 or 512, whole
// 256-row slices, tables aligned for vector loads.
bool kres_takes(const QmmArgs& q, size_t out_rows) {
  const uint32_t ng = q.kdim / kGroup;
  if (q.epi == 0 || q.gather || q.kdim % kGroup || !(ng == 2 || ng == 4 || ng == 8) || q.rows % 256) return false;
  if (static_cast<uint64_t>(out_rows) * q.rows * 4 >= (1ull << 32)) return false;  // 32-bit store offsets
  if (q.dense_mode) return aligned16(q.dense[0].scales) && aligned16(q.dense[0].biases) && aligned16(q.dense[0].weights);
  return aligned16(q.expert_base) && q.expert_stride % 16 == 0 && (q.w_off[0] | q.s_off[0] | q.b_off[0]) % 16 == 0;
}

namespace {
size_t up256(size_t v) { return (v + 255) / 256 * 256; }
}  // namespace

// ---- dense projections over many rows: MPPPrefillInt4QMM.encode (MPPPrefillInt4QMM.swift:34-78) and the
// block form of the shared expert / dense MLP (PrefillSharedExpert.encodeBlock, PrefillSharedExpert.swift:81-172)
//
// y[m, n] = x[m, k] . W[n, k]^T through qmm_kernel in dense mode.  A long K is cut into windows (multiples of 8 groups, the last
// takes the rest), which one launch computes side by side: each writes fp32 [m, n], and dense_combine_kernel adds the windows in
// order and narrows the sum.  A window is at most kDenseWindow groups, because a result's sum is one fp32 accumulator over its groups:
// error of the fp32 results against 64 bits, 512 x 17408, N(0, 1) and quantized N(0, 0.02): one window 3.9e-7, two 3.2e-7, five 2.6e-7;
// 512 x 8192: 3.1e-7, two 2.6e-7.  That bound has a price where the work items fill the chip without it (us, chosen / fewer windows:
// 5120 x 17408, 512 rows 134 / 122 (6, 3 windows); 17408 x 5120, 800 rows 200 / 173 (2, 1); 4096 x 12800, 1024 rows 156 / 138 (4, 2)).
// A gate / up pair is one launch up to kDenseFusedMax groups.  Beyond, both projections go in windows as fp32, which
// dense_swiglu_combine_kernel adds: again the shorter sums, and faster until a launch has a full round of work items.  The MLP, us,
// one launch / two windows: 7296 x 2048, 9 rows 77.3 / 54.3, 150 98.0 / 71.7, 1024 145 / 140, 2048 229 / 252; 8192 x 8192, 64 rows
// 107 / 83, 150 128 / 124, 1024 443 / 477; 12288 x 4096, 32 rows 111 / 76, 512 196 / 195, 2048 661 / 701.
constexpr uint32_t kDenseWindow = 64;   // K groups of a window (4096 values)
constexpr uint32_t kDenseFusedMax = 112;  // K groups of a gate/up + SwiGLU launch (7168 values)
__global__ __launch_bounds__(256) void dense_combine_kernel(const float* __restrict__ parts, uint32_t n_parts,
                                                            size_t part_stride, void* __restrict__ y, size_t count,
                                                            int out_f32) {
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= count) return;
  float acc = parts[i];
  for (uint32_t p = 1; p < n_parts; ++p) acc = acc + parts[p * part_stride + i];
  if (out_f32) static_cast<float*>(y)[i] = acc;
  else static_cast<uint16_t*>(y)[i] = f_to_bf16(acc);
}

// Windows of a contraction of length k for m rows of n results.  At least as many as kDenseWindow asks for; more where
// the work items (64 rows of x, 128 or 256 weight rows, one window) would leave the chip idle or its last round nearly
// empty.  A round is two items a CU, whose time follows the longest window: 4 us per 8 groups and 1.5; a last round of at
// most one item a CU has the CU to itself, 3 us per 8 groups and 1 less.  The windows' sums cost their bytes, written and read at 8 TB/s,
// and 2 us.  (16 shapes, n 1024 .. 17408, k 1024 .. 17408, 9 .. 2048 rows, up to 26 windows timed: 0.6 % from the best of those allowed
// on average, 9 % at worst (1024 x 17408, 64 rows: 34 windows 31.9, 17 29.3); the fewest windows 33 % and 113 %.  us for the projection, fewest /
// chosen: 5120 x 17408, 9 rows 41.7 / 30.3 (5, 12 windows), 150 rows 71.4 / 60.6 (7), 512 rows 144 / 134 (6); 1152 x 3200, 32 rows
// 28.6 / 15.4 (1, 6); 2048 x 8192, 64 rows 46.4 / 25.6 (2, 16); 4096 x 14336, 32 rows 40.8 / 27.7 (4, 14).)
// The choice follows the number of 64-row tiles, not m: a row's sums come out the same in every block of that many tiles.
// From kWholeRounds rounds of the fewest windows on an emptier last round is no longer worth the windows' bytes.
constexpr uint32_t kWholeRounds = 8;
static uint32_t dense_tile_items(uint32_t n) {
  const uint32_t slice_rows = n % (2 * kQmmRows) == 0 ? 2 * kQmmRows : kQmmRows;
  return (n + slice_rows - 1) / slice_rows;
}
static uint32_t dense_fewest_windows(uint32_t k) { return std::max(1u, (k / kGroup + kDenseWindow - 1) / kDenseWindow); }
// (none of the shapes timed wanted more than 25; the bound keeps the search short for any k)
static uint32_t dense_most_windows(uint32_t k) { return std::max(dense_fewest_windows(k), std::min(k / kGroup / 8, 64u)); }
// (as the differences of dense_window_start, which steps by ng / n_win, without a division a window)
static uint32_t dense_longest_window(uint32_t ng, uint32_t n_win) {
  const uint32_t whole = ng / n_win, part = ng % n_win;
  uint32_t longest = 0, at = 0, over = 0, start = 0;
  for (uint32_t w = 1; w < n_win; ++w) {
    at += whole;
    over += part;
    if (over >= n_win) { over -= n_win; ++at; }
    longest = std::max(longest, (at & ~7u) - start);
    start = at & ~7u;
  }
  return std::max(longest, ng - start);
}
// longest(w): groups of the longest of w windows
template <typename Longest>
static uint32_t dense_windows_of_tiles(uint32_t tiles, uint32_t n, uint32_t k, Longest longest) {
  const uint32_t lo = dense_fewest_windows(k), hi = dense_most_windows(k), num_cu = device_cu_count();
  const uint64_t items = static_cast<uint64_t>(tiles) * dense_tile_items(n);
  if (items * lo >= kWholeRounds * 2ull * num_cu) return lo;
  uint32_t best = lo;
  double best_us = 0.0;
  for (uint32_t w = lo; w <= hi; ++w) {
    const double steps = longest(w) / 8.0;
    const uint32_t all = static_cast<uint32_t>(items) * w, rounds = all / (2 * num_cu), rest = all % (2 * num_cu);
    double us = (rounds + (rest > num_cu)) * (4.0 * steps + 1.5);
    if (rest > 0 && rest <= num_cu) us += 3.0 * steps - 1.0;
    if (w > 1) us += 2.0 + static_cast<double>(w) * tiles * kTileTokens * n * 8.0 / 8.0e6;
    if (w == lo || us < best_us) { best = w; best_us = us; }
  }
  return best;
}
uint32_t dense_windows(uint32_t m, uint32_t n, uint32_t k) {
  return dense_windows_of_tiles((m + kTileTokens - 1) / kTileTokens, n, k, [&](uint32_t w) { return dense_longest_window(k / kGroup, w); });
}

// bytes of fp32 window results a projection of n rows over m tokens needs (0: one window, written directly)
static size_t dense_parts_bytes(uint32_t m, uint32_t n, uint32_t n_win) {
  return n_win > 1 ? up256(sizeof(float) * static_cast<size_t>(m) * n) * n_win : 0;
}
// ... and the most any call of up to m tokens needs: fewer tiles can take more windows, so the bytes of a single call do
// not grow with its rows (5120 x 17408: 27.5 MB of results for 192 rows, 24.6 for 200).  Only tile counts below kWholeRounds differ.
static size_t dense_parts_bytes_up_to(uint32_t m, uint32_t n, uint32_t k) {
  const uint32_t lo = dense_fewest_windows(k), hi = dense_most_windows(k);
  std::vector<uint32_t> longest(hi + 1);
  for (uint32_t w = lo; w <= hi; ++w) longest[w] = dense_longest_window(k / kGroup, w);
  const auto of_tiles = [&](uint32_t tiles) { return dense_windows_of_tiles(tiles, n, k, [&](uint32_t w) { return longest[w]; }); };
  size_t most = dense_parts_bytes(m, n, of_tiles((m + kTileTokens - 1) / kTileTokens));
  const uint64_t row = static_cast<uint64_t>(dense_tile_items(n)) * lo;
  const uint32_t tiles = static_cast<uint32_t>(std::min<uint64_t>((m - 1) / kTileTokens, kWholeRounds * 2ull * device_cu_count() / row + 1));
  for (uint32_t i = tiles; i > 0 && dense_parts_bytes(i * kTileTokens, n, hi) > most; --i)
    most = std::max(most, dense_parts_bytes(i * kTileTokens, n, of_tiles(i)));
  return most;
}
// ... and of the gate / up pair of an MLP (both projections of a work item: kQmmRows rows each)
static uint32_t dense_gate_up_windows(uint32_t d) {
  return std::max(1u, (d / kGroup + kDenseFusedMax - 1) / kDenseFusedMax);
}
static size_t dense_gate_up_parts_bytes(uint32_t t, uint32_t f, uint32_t d) {
  const uint32_t n_win = dense_gate_up_windows(d);
  return n_win > 1 ? 2 * up256(sizeof(float) * static_cast<size_t>(t) * f) * n_win : 0;
}

// The windows of a gate / up pair meet here: sums in window order, gate and up narrowed to bf16
// (dequant_int4.metal:240-245), act = bf16(silu(gate) * up) written in the matmul's order (0,4,1,5,2,6,3,7 inside
// every run of 8) with the fp32 sum of every 64-wide group beside it -- what the SwiGLU epilogue of the
// one-window launch and prep_rows_kernel produce together.  One thread per run of 8.
__global__ __launch_bounds__(256) void dense_swiglu_combine_kernel(const float* __restrict__ pg, const float* __restrict__ pu,
                                                                   uint32_t n_parts, size_t part_stride,
                                                                   uint16_t* __restrict__ act, uint16_t* __restrict__ sums,
                                                                   const float* __restrict__ row_max, size_t chunks, uint32_t ng, float limit) {
  const size_t c = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  float g[8], u[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) g[i] = u[i] = 0.0f;
  if (c < chunks) {
    for (uint32_t p = 0; p < n_parts; ++p) {
      const float4 g0 = *reinterpret_cast<const float4*>(pg + p * part_stride + c * 8);
      const float4 g1 = *reinterpret_cast<const float4*>(pg + p * part_stride + c * 8 + 4);
      const float4 u0 = *reinterpret_cast<const float4*>(pu + p * part_stride + c * 8);
      const float4 u1 = *reinterpret_cast<const float4*>(pu + p * part_stride + c * 8 + 4);
      const float gv[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
      const float uv[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        g[i] = p == 0 ? gv[i] : g[i] + gv[i];
        u[i] = p == 0 ? uv[i] : u[i] + uv[i];
      }
    }
  }
  uint32_t a[8];
  float v[8];
  const size_t grp = c >> 3, r = grp / ng;
  const float scale = act_scale(c < chunks ? row_max[r] : 0.0f);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float gr = round_bf16(g[i]), ur = round_bf16(u[i]);
    if (limit > 0.0f) {
      gr = fminf(gr, limit);
      ur = fminf(fmaxf(ur, -limit), limit);
    }
    a[i] = f_to_bf16(fast_silu(gr) * ur * scale);
    v[i] = bf16_to_f(static_cast<uint16_t>(a[i])) * kRowUnscale;
  }
  float sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
  sum = group_sum(sum, 8);
  if (c >= chunks) return;
  *reinterpret_cast<uint4*>(act + c * 8) = make_uint4(a[0] | (a[4] << 16), a[1] | (a[5] << 16), a[2] | (a[6] << 16),
                                                      a[3] | (a[7] << 16));
  if ((c & 7) == 0) store_group_sum(sums + r * group_sum_words(ng), static_cast<uint32_t>(grp - r * ng), ng, sum);
}

bool dense_qmm_takes(const mf_qtensor& w, int bits, const void* x, const void* y, uint32_t m, uint32_t n, uint32_t k) {
  if (n % kQmmRows || k % (2 * kGroup) || m == 0) return false;
  if (!aligned16(w.weights) || !aligned16(x) || !aligned16(y)) return false;
  if (static_cast<uint64_t>(m) * n >= (1ull << 31)) return false;
  return true;
}

// bytes of the group sums of `rows` rows of k values
static size_t sums_bytes(size_t rows, uint32_t k) { return sizeof(uint16_t) * rows * group_sum_words(k / kGroup); }
static size_t dense_qmm_rows_bytes(uint32_t m, uint32_t k) {
  return up256(sizeof(uint16_t) * static_cast<size_t>(m) * k) + up256(sums_bytes(m, k)) + up256(sizeof(float) * m);
}
size_t dense_qmm_needs(uint32_t m, uint32_t n, uint32_t k) { return dense_qmm_rows_bytes(m, k) + dense_parts_bytes(m, n, dense_windows(m, n, k)); }
size_t dense_qmm_workspace_bytes(uint32_t m, uint32_t n, uint32_t k) {
  return dense_qmm_rows_bytes(m, k) + dense_parts_bytes_up_to(m, n, k);
}

// xp: rows in the matmul's order, their group sums in sumx; act_rows: activations, row_max is that of the x in front
static hipError_t dense_project(hipStream_t s, const mf_qtensor& w, int bits, const uint16_t* xp, const uint16_t* sumx,
                                const float* row_max, bool act_rows, void* y, uint32_t m, uint32_t n, uint32_t k, uint32_t n_win, bool out_f32, void* parts) {
  const uint32_t ng = k / kGroup;
  const int code_bits = bits == MF_BITS_4 ? 4 : 2;
  QmmArgs d{};
  d.dense_mode = 1; d.dense_rows = m; d.top_k = 1;
  d.dense[0] = d.dense[1] = w;
  if (bits == MF_BITS_TERNARY) {  // bias = -scale: the kernel reads the scale table as bias table
    d.ternary = 1;
    d.dense[0].biases = d.dense[1].biases = w.scales;
  }
  d.x = xp; d.sumx = sumx; d.row_max = row_max; d.act_rows = act_rows; d.x_stride = k; d.rows = n;
  d.pair_rows = n % (2 * kQmmRows) == 0;
  const uint32_t tiles = (m + kTileTokens - 1) / kTileTokens;
  const size_t part_stride = up256(sizeof(float) * static_cast<size_t>(m) * n) / sizeof(float);
  d.ng_ld = ng;
  if (n_win == 1) {
    d.kdim = k; d.epi = out_f32 ? 1 : 2; d.out = y;
  } else {  // all windows in one launch, each writing fp32 into its own buffer
    d.kdim = dense_longest_window(ng, n_win) * kGroup; d.n_win = n_win; d.out_win_stride = part_stride; d.epi = 1; d.out = parts;
  }
  {
    const hipError_t e = launch_qmm(s, kTileTokens, code_bits, d, d.pair_rows ? 2 : 1, tiles, nullptr, 0);
    if (e != hipSuccess) return e;
  }
  if (n_win > 1) {
    const size_t count = static_cast<size_t>(m) * n;
    dense_combine_kernel<<<dim3(static_cast<uint32_t>((count + 255) / 256)), dim3(256), 0, s>>>(
        static_cast<const float*>(parts), n_win, part_stride, y, count, out_f32 ? 1 : 0);
    return hipGetLastError();
  }
  return hipSuccess;
}

hipError_t launch_dense_qmm(hipStream_t s, const mf_qtensor& w, int bits, const uint16_t* x, void* y, uint32_t m,
                            uint32_t n, uint32_t k, bool out_f32, void* workspace) {
  uint8_t* base = static_cast<uint8_t*>(workspace);
  uint16_t* xp = reinterpret_cast<uint16_t*>(base);
  uint16_t* sumx = reinterpret_cast<uint16_t*>(base + up256(sizeof(uint16_t) * static_cast<size_t>(m) * k));
  float* row_max = reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(sumx) + up256(sums_bytes(m, k)));
  void* parts = base + dense_qmm_rows_bytes(m, k);
  const hipError_t e = launch_prep_rows(s, x, xp, sumx, row_max, m, k);
  if (e != hipSuccess) return e;
  return dense_project(s, w, bits, xp, sumx, row_max, false, y, m, n, k, dense_windows(m, n, k), out_f32, parts);
}

// The block form of the shared expert / dense SwiGLU MLP: gate and up in one launch with the SwiGLU epilogue
// (gate and up narrowed first, dequant_int4.metal:240-245), then the down projection.
bool dense_mlp_takes(const mf_qtensor& gate, const mf_qtensor& up, const mf_qtensor& down, const void* x,
                     const void* y, const void* scratch, uint32_t d, uint32_t f, uint32_t t) {
  if (d % kGroup || f % kGroup || d < kQmmRows || f < kQmmRows || t == 0) return false;
  return aligned16(gate.weights) && aligned16(up.weights) && aligned16(down.weights) && aligned16(x) && aligned16(y) &&
         aligned16(scratch) && static_cast<uint64_t>(t) * std::max(d, f) < (1ull << 31);
}

static size_t dense_mlp_rows_bytes(uint32_t d, uint32_t f, uint32_t t) {
  return up256(sizeof(uint16_t) * static_cast<size_t>(t) * f) + up256(sizeof(uint16_t) * static_cast<size_t>(t) * d) +
         up256(sums_bytes(t, d)) + up256(sums_bytes(t, f)) + up256(sizeof(float) * t);
}
// (the window results of gate / up and of down follow one another in the same place)
size_t dense_mlp_needs(uint32_t d, uint32_t f, uint32_t t, uint32_t down_windows) {
  return dense_mlp_rows_bytes(d, f, t) + std::max(dense_parts_bytes(t, d, down_windows), dense_gate_up_parts_bytes(t, f, d));
}
size_t dense_mlp_scratch_bytes(uint32_t d, uint32_t f, uint32_t t) {
  return dense_mlp_rows_bytes(d, f, t) + std::max(dense_parts_bytes_up_to(t, d, f), dense_gate_up_parts_bytes(t, f, d));
}

hipError_t launch_dense_mlp(hipStream_t s, const mf_qtensor& gate, const mf_qtensor& up, const mf_qtensor& down,
                            int bits, const uint16_t* x, uint16_t* y, uint32_t d, uint32_t f, uint32_t t, uint32_t down_windows,
                            void* scratch) {
  uint8_t* base = static_cast<uint8_t*>(scratch);
  uint16_t* act = reinterpret_cast<uint16_t*>(base);
  base += up256(sizeof(uint16_t) * static_cast<size_t>(t) * f);
  uint16_t* xp = reinterpret_cast<uint16_t*>(base);
  base += up256(sizeof(uint16_t) * static_cast<size_t>(t) * d);
  uint16_t* sumx = reinterpret_cast<uint16_t*>(base);
  base += up256(sums_bytes(t, d));
  uint16_t* sum_act = reinterpret_cast<uint16_t*>(base);
  base += up256(sums_bytes(t, f));
  float* row_max = reinterpret_cast<float*>(base);
  base += up256(sizeof(float) * t);
  hipError_t e = launch_prep_rows(s, x, xp, sumx, row_max, t, d);
  if (e != hipSuccess) return e;
  const int code_bits = bits == MF_BITS_4 ? 4 : 2;
  QmmArgs q{};
  q.dense_mode = 1; q.dense_rows = t; q.top_k = 1; q.narrow = 1;
  q.dense[0] = gate; q.dense[1] = up;
  if (bits == MF_BITS_TERNARY) {
    q.ternary = 1;
    q.dense[0].biases = gate.scales;
    q.dense[1].biases = up.scales;
  }
  q.x = xp; q.sumx = sumx; q.row_max = row_max; q.x_stride = d; q.rows = f; q.kdim = d; q.epi = 0; q.out = act; q.out_sums = sum_act;
  const uint32_t gu_win = dense_gate_up_windows(d);
  // At most 32 rows over a long K: tiles of 32 in the form for few work items.  The MLP, us, tiles of 64 / this: 5120 x 17408, 9 rows
  // 77.3 / 74.5, 32 rows 79.5 / 77.8; 7168 x 2048, 9 rows 63.6 / 58.1; 4096 x 12800, 9 rows 53.3 / 50.7; at d of 2048 and less no gain.
  const uint32_t tile = t <= kSmallTile && d > 2048 && gu_win * ((f + kQmmRows - 1) / kQmmRows) <= 2 * device_cu_count() ? kSmallTile : kTileTokens;
  if (gu_win > 1) {
    // past kDenseFusedMax: the contraction in windows, both projections as fp32 per window, then one pass that adds the
    // windows, activates and sums the groups
    const uint32_t ng = d / kGroup;
    const size_t part_stride = up256(sizeof(float) * static_cast<size_t>(t) * f) / sizeof(float);
    float* pg = reinterpret_cast<float*>(base);
    float* pu = pg + part_stride * gu_win;
    q.ng_ld = ng; q.kdim = dense_longest_window(ng, gu_win) * kGroup; q.n_win = gu_win; q.out_win_stride = part_stride;
    q.epi = 1; q.out = pg; q.out2 = pu;
    e = launch_qmm(s, tile, code_bits, q, 2, (t + tile - 1) / tile, nullptr, 0, tile == kSmallTile);
    if (e != hipSuccess) return e;
    const size_t chunks = static_cast<size_t>(t) * f / 8;
    dense_swiglu_combine_kernel<<<dim3(static_cast<uint32_t>((chunks + 255) / 256)), dim3(256), 0, s>>>(
        pg, pu, gu_win, part_stride, act, sum_act, row_max, chunks, f / kGroup, 0.0f);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  } else {
    e = launch_qmm(s, tile, code_bits, q, 2, (t + tile - 1) / tile, nullptr, 0, tile == kSmallTile);
    if (e != hipSuccess) return e;
  }
  return dense_project(s, down, bits, act, sum_act, row_max, true, y, t, d, f, down_windows, false, base);
}

// entries of the tile list, a multiple of 8: an expert of c routes has ceil(c / tile) tiles, and at most min(experts, routes) have any
uint32_t prefill_tile_slots(const mf_moe_config& c, uint32_t t, uint32_t tile) {
  const size_t pairs = static_cast<size_t>(t) * c.top_k;
  const size_t n = std::max<size_t>((pairs + (tile - 1) * std::min<size_t>(c.num_experts, pairs)) / tile, 1);
  return static_cast<uint32_t>((n + 7) / 8 * 8);
}

// Routes of a tile of the layer call's two matmuls.  A tile of 32 leaves registers and LDS for three workgroups a CU where one
// of 64 leaves them for two, and wastes less where few tokens meet an expert; past 32 routes an expert (on average, over the
// layer's experts) more and more tiles of 64 are full, and expand a weight for 64 tokens at a time.  2-bit codes without a
// 4-bit shared expert beside them are read and expanded faster: past 128.  Layer call, tiles of 64 / 32 in both matmuls, us, pool as loaded
// (and tiled): 256 4-bit experts of 2048 x 512, shared 512: 93 tokens 79.5 / 68.9, 512 122.7 / 117.9, 1024 161 / 171 (153 / 153), 2048 244 / 277;
// 128 experts of 2816 x 704: 300 tokens 185 / 172, 500 216 / 225, 800 252 / 286; 256 2-bit experts of 4096 x 2048, shared 2048: 200 tokens
// 654 / 653 (587 / 551), 777 775 / 769 (698 / 672), 1365 987 / 1059 (916 / 955), 2048 1203 / 1368; 64 ternary experts of 2048 x 1024: 400 tokens
// 128 / 121, 1024 194 / 195 (193 / 185), 2048 303 / 328; 256 of 2048 x 512: 1500 tokens 185 / 182 (180 / 172), 3000 293 / 304, 4096 363 / 392.
// Around the lines no one number is right for every shape: the fewer work items a launch has, the longer tiles of 32 win.  At 32 routes an
// expert 128 2-bit experts of 4096 x 256, shared 512, 158 / 134; 64 of 2048 x 768 92.5 / 89.5; 128 of 4096 x 1024 294 / 312 (274 / 263); 32 of
// 5120 x 1536 199 / 224 (182 / 181).  At 64 of 2-bit codes 64 of 1536 x 128 71 / 63, 64 of 4096 x 2048 363 / 379 (348 / 349).
// The resident kernel on 4-bit rows of 512 has half the codes in flight each in its three workgroups a CU: tiles of 32 from a route
// an expert on and while their work items make up to 4.75 a CU.  Layer call, us, 64 / 32: 2048 x 512, 256 experts, top 8, shared 512, 16, 32, 64, 96, 192, 258, 280,
// 384, 768 tokens 54.2 / 55.2, 58.6 / 59.5, 71.2 / 69.3, 72.6 / 70.4, 81.6 / 77.5, 92.9 / 95.1, 93.6 / 95.1, 96.7 / 99.9, 144.4 / 149.0; 1024 x 512, 128 experts, 64, 192, 384 tokens
// 49.9 / 47.1, 55.7 / 53.6, 61.5 / 58.2; 4096 x 512, 64 experts, top 4, 96, 256, 384 tokens 72.4 / 69.5, 101.3 / 97.6, 120.0 / 120.8; 5120 x 512,
// 128 experts, shared 512, 9, 32, 96, 256 tokens 93.2 / 93.4, 114.3 / 116.7, 157.6 / 163.7, 211.6 / 218.4.
// resident: that kernel takes the down projections of the call.  Where it does not, the ring on tiles of 64 / 32, us a call: 2176 x 512,
// 128 experts, 93 tokens 67.5 / 65.3; 2048 x 512 beside a shared expert of 1024, 40 67.7 / 65.0, 93 74.4 / 70.2, 300 109.5 / 104.8;
// 1664 x 512, 64 experts, 93 56.6 / 54.1, 200 (25 routes an expert) 65.2 / 67.2.
struct PrefillTiles { uint32_t up, down; };
// Whether a matmul launch on tiles of 32 has few work items (`items`, at most) over a long contraction: the kernel's form for that, which
// keeps two workgroups on a CU.  Layer call, us, the form of three workgroups / that form.  Length: 1024 x 384, 48 experts, top 4, 64
// tokens 34.3 / 35.6; ternary 1536 x 128, 64 tokens 46.3 / 44.7; Qwen shape (2048), 9 tokens 44.5 / 42.6.  Items: 64 experts of 2048 x 1024,
// top 2, 300 tokens, 640 items 59.0 / 65.3; 32 of 5120 x 1536, top 1, 480 items, 193 tokens (6 routes an expert) 83.9 / 75.2, but
// 300 tokens (9), whose tiles have twice the results to scale, 105.8 / 109.3; 16 of 8192 x 512, top 2, 108 items, 193 tokens (24) 104.9 / 90.3.
static bool prefill_few(const mf_moe_config& c, uint32_t t, uint64_t items, uint32_t kdim) {
  return kdim > 1024 && (items <= device_cu_count() ||
                         (items <= 2 * device_cu_count() && static_cast<uint64_t>(t) * c.top_k <= 8ull * c.num_experts));
}
static PrefillTiles prefill_tiles(const mf_moe_config& c, uint32_t t, bool resident) {
  const bool two_bit = c.bits != MF_BITS_4 && !c.shared_f;
  const uint64_t few = static_cast<uint64_t>(two_bit ? 128 : 32) * c.num_experts;
  PrefillTiles p;
  p.up = static_cast<uint64_t>(t) * c.top_k <= few ? kSmallTile : kTileTokens;
  const bool few_or_many = static_cast<uint64_t>(t) * c.top_k <= c.num_experts ||
                           static_cast<uint64_t>(prefill_tile_slots(c, t, kSmallTile)) * c.d > 19ull * 128 * device_cu_count();  // (4.75 items of 512 rows)
  p.down = resident && c.bits == MF_BITS_4 && c.f == 512 && few_or_many ? kTileTokens : p.up;
  return p;
}

// workspace carve-up of one prefill layer call
struct PrefillWs {
  float* logits; uint32_t* idx; float* w; uint32_t* counts; uint32_t* offsets; uint32_t* starts;
  uint32_t* status; Tile* tiles[2]; mf_pair* sorted; uint16_t* acts; float* partials;
  uint16_t* sact; uint16_t* hs; uint16_t* gate;
  uint16_t* xp; uint16_t* sum_x; uint16_t* sum_acts; uint16_t* sum_sact; float* row_max;
  size_t bytes;
};

PrefillWs prefill_carve(const mf_moe_config& c, uint32_t t, void* base) {
  PrefillWs p{};
  size_t pos = 0;
  auto take = [&](size_t bytes) {
    uint8_t* at = static_cast<uint8_t*>(base) + pos;
    pos += up256(bytes);
    return static_cast<void*>(base ? at : nullptr);
  };
  const size_t pairs = static_cast<size_t>(t) * c.top_k;
  const size_t max_tiles = prefill_tile_slots(c, t, kSmallTile);  // (of either tile: bytes that grow with t)
  p.logits = static_cast<float*>(take(sizeof(float) * t * c.num_experts));
  p.idx = static_cast<uint32_t*>(take(sizeof(uint32_t) * pairs));
  p.w = static_cast<float*>(take(sizeof(float) * pairs));
  p.counts = static_cast<uint32_t*>(take(sizeof(uint32_t) * MF_MAX_EXPERTS));
  p.offsets = static_cast<uint32_t*>(take(sizeof(uint32_t) * MF_MAX_EXPERTS));
  p.starts = static_cast<uint32_t*>(take(sizeof(uint32_t) * MF_MAX_EXPERTS));
  p.status = static_cast<uint32_t*>(take(256));
  for (Tile*& list : p.tiles) list = static_cast<Tile*>(take(sizeof(Tile) * max_tiles));
  p.sorted = static_cast<mf_pair*>(take(sizeof(mf_pair) * pairs));
  p.acts = static_cast<uint16_t*>(take(sizeof(uint16_t) * pairs * c.f));
  p.partials = static_cast<float*>(take(sizeof(float) * pairs * c.d));
  p.sact = static_cast<uint16_t*>(take(sizeof(uint16_t) * static_cast<size_t>(t) * std::max<uint32_t>(c.shared_f, 64)));
  p.hs = static_cast<uint16_t*>(take(sizeof(uint16_t) * static_cast<size_t>(t) * c.d));
  p.gate = static_cast<uint16_t*>(take(sizeof(uint16_t) * t));
  p.xp = static_cast<uint16_t*>(take(sizeof(uint16_t) * static_cast<size_t>(t) * c.d));
  p.sum_x = static_cast<uint16_t*>(take(sums_bytes(t, c.d)));
  p.sum_acts = static_cast<uint16_t*>(take(sums_bytes(pairs, c.f)));
  p.sum_sact = static_cast<uint16_t*>(take(sums_bytes(t, std::max<uint32_t>(c.shared_f, 64))));
  p.row_max = static_cast<float*>(take(sizeof(float) * t));
  p.bytes = pos;
  return p;
}

size_t prefill_workspace_bytes(const mf_moe_config& c, uint32_t t) {
  return prefill_carve(c, t, nullptr).bytes;
}

// widths of whole 128-row workgroups: the configurations whose calls insist on a workspace (the others fall back to
// the decode launch without one) and whose pool can be tiled
bool prefill_whole_tiles(const mf_moe_config& c) {
  return prefill_supported(c) && c.d % kQmmRows == 0 && c.f % kQmmRows == 0 && c.shared_f % kQmmRows == 0;
}

bool prefill_supported(const mf_moe_config& c) {
  if (c.bits != MF_BITS_4 && c.bits != MF_BITS_2 && c.bits != MF_BITS_TERNARY) return false;
  if (c.shared_f && c.shared_bits != MF_BITS_4) return false;
  if (c.gate_group_size == 32) return false;  // the matmul's tables hold one entry per 64 weights
  // any multiple of the quantization group from 128 on; a width of 64 is one group, which the decode launch serves
  if (c.d % kGroup || c.f % kGroup || c.shared_f % kGroup) return false;
  if (c.d < kQmmRows || c.f < kQmmRows || (c.shared_f && c.shared_f < kQmmRows)) return false;
  if (c.d > 8192 || c.f > 8192 || c.shared_f > 8192) return false;
  return true;
}

struct RaggedOnly {
  const mf_pair* sorted;    // [t * top_k] by (expert, token, rank)
  const uint32_t* counts;   // [num_experts]
  float* partials;          // [t * top_k, d] fp32, row token * top_k + rank
};
hipError_t launch_prefill_layer(hipStream_t s, const mf_moe& h, const mf_moe_layer_weights& w,
                                const uint16_t* x, uint32_t t, uint16_t* y, void* workspace,
                                uint32_t* out_idx, float* out_w, const RaggedOnly* ragged);

// The routed experts alone over a grouping the caller holds (sorted pairs + per-expert counts):
// PrefillGroupedRoutedMoE.encodeStreamedBatched.  Runs the layer call's matmul launches and stops
// before the un-permute; the per-route results go to the caller's fp32 buffer.
hipError_t launch_ragged_qmm(hipStream_t s, const mf_moe& h, const void* expert_base, size_t expert_stride,
                             const mf_expert_offsets& off, const uint16_t* x, const mf_pair* sorted,
                             const uint32_t* counts, uint32_t t, float* partials, void* workspace) {
  RaggedOnly r{sorted, counts, partials};
  mf_moe_layer_weights w{};
  w.expert_base = expert_base;
  w.expert_stride = expert_stride;
  w.offsets = off;
  return launch_prefill_layer(s, h, w, x, t, nullptr, workspace, nullptr, nullptr, &r);
}

hipError_t launch_unpermute(hipStream_t s, const mf_moe_config& c, const float* partials, const float* w,
                            const uint32_t* idx, const uint16_t* residual, uint32_t t, uint16_t* y) {
  const size_t n4 = static_cast<size_t>(t) * c.d / 4;
  if (!n4) return hipSuccess;
  prefill_reduce_kernel<false><<<dim3(static_cast<uint32_t>((n4 + 255) / 256)), dim3(256), 0, s>>>(
      partials, w, idx, residual, nullptr, y, t, c.top_k, c.d, c.num_experts, static_cast<int>(c.maple_rounding));
  return hipGetLastError();
}

hipError_t launch_prefill_layer(hipStream_t s, const mf_moe& h, const mf_moe_layer_weights& w,
                                const uint16_t* x, uint32_t t, uint16_t* y, void* workspace,
                                uint32_t* out_idx, float* out_w, const RaggedOnly* ragged) {
  const mf_moe_config& cfg_in = h.cfg;
  mf_moe_config c = cfg_in;
  if (ragged) c.shared_f = 0;  // the routed experts only
  PrefillWs ws = prefill_carve(cfg_in, t, workspace);
  // the caller's routing outputs, when given, are the routing buffers of the whole call
  if (out_idx) ws.idx = out_idx;
  if (out_w) ws.w = out_w;
  hipError_t e;
#define MF_TRY(call) do { e = (call); if (e != hipSuccess) return e; } while (0)
  const size_t pairs = static_cast<size_t>(t) * c.top_k;
  QmmArgs q{};
  // the routed experts' blobs: the pool in the matmul's order when the caller built one (mf_moe_tile_experts)
  q.expert_base = static_cast<const uint8_t*>(w.expert_tiled ? w.expert_tiled : w.expert_base);
  q.tiled = w.expert_tiled != nullptr;
  q.expert_stride = w.expert_stride;
  q.top_k = c.top_k;
  q.limit = c.swiglu_limit;
  // ternary experts are 2-bit codes whose bias is -scale: the kernels take the scale table as bias table
  const int code_bits = c.bits == MF_BITS_4 ? 4 : 2;
  const bool ternary = c.bits == MF_BITS_TERNARY;
  q.ternary = ternary;
  q.maple = static_cast<int>(c.maple_rounding);
  // phase 2: routed down -> fp32 partials [token*K+rank, D]; shared down -> hs [token, D].
  // Per-route results as bf16 numbers where the rounding rule narrows them anyway before they meet their
  // weights -- MapleMoE's (maple_moe.metal:258), or on request (mf_moe_set_prefill_route_rounding; the
  // reference's prefill keeps 16-bit per-route results, prefill.metal:817-819, 644-651): half the bytes
  // written here and read by the reduce.  The caller's buffer of a ragged call stays fp32.
  const bool narrow_routes = !ragged && (c.maple_rounding || h.narrow_routes);
  QmmArgs q2 = q, d2{};
  q2.w_off[0] = w.offsets.down_w; q2.s_off[0] = w.offsets.down_s; q2.b_off[0] = ternary ? w.offsets.down_s : w.offsets.down_b;
  q2.x_stride = c.f; q2.rows = c.d; q2.kdim = c.f;
  q2.epi = narrow_routes ? 3 : 1;
  q2.limit = 0.0f;
  q2.act_rows = 1;
  q2.pair_rows = c.d % (2 * kQmmRows) == 0;
  if (c.shared_f) {
    d2.dense_mode = 1; d2.dense_rows = t; d2.top_k = c.top_k; d2.narrow = 1;
    d2.dense[0] = w.shared_down; d2.dense[1] = w.shared_up;
    d2.x_stride = c.shared_f; d2.rows = c.d; d2.kdim = c.shared_f; d2.epi = 2;
    d2.pair_rows = q2.pair_rows;
    d2.act_rows = 1;
  }
  const bool kres_q = kres_takes(q2, pairs), kres_d = c.shared_f && kres_takes(d2, t);
  // Both parts in one launch of one kernel: the resident one when it takes both (their K has to be the same), else the
  // ring.  Routed experts the resident kernel takes beside a shared expert of another width get it in a launch of their
  // own once its gain, which grows with the results it writes, outweighs the shared expert's launch, whose few items are then
  // alone on the chip: from 6 M results on, and of rows of 512, where the ring is nearly as good, from 24 M (2-bit layer, us, one launch /
  // two, same bits: 4096 x 256, shared 512, top 6: 100 tokens 93.5 / 93.0, 300 127.6 / 121.5, 2048 361 / 298; 2048 x 128, shared 512, top 8: 150
  // tokens 63.3 / 65.9, 400 79.3 / 79.4, 1000 111 / 103; 1024 x 128, shared 384, top 4: 1000 tokens 66.9 / 74.7, 2000 82.6 / 82.2, 4000 113 / 108;
  // 2048 x 256, shared 768, top 4: 600 tokens 86.5 / 89.0, 1000 105 / 106, 1500 123 / 114; 6144 x 256, shared 1536, top 2: 400 tokens 135 / 137,
  // 600 157 / 151.  Rows of 512: 2048, shared 1024, top 8: 300 tokens 93.5 / 103.3, 1024 162.1 / 162.3, 2048 263 / 261; shared 192, 1000 153 / 157,
  // 1500 194 / 186; 4096, shared 1024, top 4: 600 tokens 160 / 167, 2048 300 / 299, 3000 400 / 384.  4-bit experts alike: 2048 x 512, shared 1024,
  // 300 tokens 94 / 111; 1024 x 128, 1000 tokens 66 / 74.  Routed 1024 or 2048 beside a resident shared expert: one launch always, 375 / 385).
  const bool kres_both = kres_q && (!c.shared_f || (kres_d && d2.kdim == q2.kdim));
  const bool apart = c.shared_f && kres_q && !kres_both && pairs * c.d >= (c.f <= 256 ? 6u : 24u) << 20;
  const PrefillTiles tile = prefill_tiles(c, t, c.shared_f && !apart ? kres_both : kres_q);
  TileLists lists{{ws.tiles[0], tile.down != tile.up ? ws.tiles[1] : nullptr},
                  {prefill_tile_slots(c, t, tile.up), prefill_tile_slots(c, t, tile.down)}, {tile.up, tile.down}};
  bool x_prepared = false, fused_group = false;
  RouterTail tail{};  // what the router launch, or else the grouping launch, prepares on the side
  tail.xp = ws.xp;
  tail.w_sg = c.shared_f && !w.w_sg_q8.weights ? w.w_sg : nullptr;  // (an 8-bit gate row: its own launch below)
  tail.sums = ws.sum_x;
  tail.row_max = ws.row_max;
  tail.gate = ws.gate;
  if (ragged) {
    // the caller's grouping: its per-expert counts are a one-chunk histogram for the scan that lays
    // out the tile list (the runs start at 0 in expert order, as mf_moe_group writes them)
    uint32_t* hist = h.ws.group_tmp + 2048;
    uint32_t* bad = hist + static_cast<size_t>(kGroupChunks) * MF_MAX_EXPERTS;
    ws.status = h.ws.group_tmp + 3 * 512;  // the word mf_moe_group_status reads
    ragged_begin_kernel<<<dim3(1), dim3(MF_MAX_EXPERTS), 0, s>>>(ragged->counts, c.num_experts, hist, bad);
    const uint32_t check_wgs = static_cast<uint32_t>(std::min<size_t>((pairs + 255) / 256, 2048));
    ragged_check_kernel<<<dim3(std::max(check_wgs, 1u)), dim3(256), 0, s>>>(ragged->sorted, ragged->counts, c.num_experts,
                                                                           t, c.top_k, bad);
    MF_TRY(hipGetLastError());
    group_scan_kernel<<<dim3(1), dim3(MF_MAX_EXPERTS), 0, s>>>(hist, 1, c.num_experts, ws.counts, ws.offsets, ws.starts,
                                                               lists, bad, ws.status, 1);
    MF_TRY(hipGetLastError());
    ws.sorted = const_cast<mf_pair*>(ragged->sorted);
    ws.partials = ragged->partials;
  } else {
    if (w.router_w) {  // else the routing in out_idx / out_w is the caller's
      RouterTail routed = tail;
      MF_TRY(launch_prefill_router(s, w.router_w, x, c.num_experts, c.d, t, c.d, ws.logits, &routed));
      x_prepared = routed.xp != nullptr;
      fused_group = topk_group_takes(t) && pairs > kGroupOnePairs;
      if (fused_group)
        MF_TRY(launch_topk_group(s, ws.logits, t, c.top_k, c.num_experts, c.router_mode, ws.idx, ws.w, ws.counts,
                                 ws.offsets, ws.starts, ws.sorted, lists, ws.status,
                                 h.ws.group_tmp));
      else MF_TRY(launch_topk(s, ws.logits, c.num_experts, c.top_k, t, c.router_mode, ws.idx, ws.w));
    }
    if (!fused_group) {
      RouterTail grouped = tail;
      MF_TRY(launch_group(s, ws.idx, ws.w, t, c.top_k, c.num_experts, ws.counts, ws.offsets, ws.starts,
                          ws.sorted, lists, ws.status, h.ws.group_tmp + 2048, x, c.d, x_prepared ? nullptr : &grouped));
      x_prepared |= !x_prepared && !grouped.xp;
    }
  }

  const bool gate_q8 = c.shared_f && w.w_sg_q8.weights;
  const bool want_gate = c.shared_f && (w.w_sg || gate_q8);
  if (x_prepared) {
    // done on the side (the gate's logits, too)
  } else if (want_gate && !gate_q8) {  // one pass over x: matmul order, group sums and the shared gate's logits
    prep_x_gate_kernel<<<dim3((t + 3) / 4), dim3(256), 0, s>>>(x, ws.xp, ws.sum_x, ws.row_max, w.w_sg, ws.gate, t, c.d);
    MF_TRY(hipGetLastError());
  } else {
    MF_TRY(launch_prep_rows(s, x, ws.xp, ws.sum_x, ws.row_max, t, c.d));
  }
  // the scalar gate stored as an 8-bit row (RealForwardRunner.swift:2925-2941): one wave per token, the
  // bits of mf_gemv(MF_BITS_8) -- and of the decode launch
  if (gate_q8) MF_TRY(launch_gemv(s, w.w_sg_q8, MF_BITS_8, x, ws.gate, 1, c.d, t, false));

  q.sorted = ws.sorted;
  q.tiles = lists.list[0];
  // the (4-bit) shared expert rides in the routed launches of the same phase
  const bool shared_rides = c.shared_f != 0;
  const int launch_bits = c.shared_f && code_bits != 4 ? kMixedBits : code_bits;
  if (h.trace && h.trace_bytes >= 64) {  // stage stamps of the routed gate/up matmul
    q.trace = h.trace;
    q.trace_items = static_cast<uint32_t>(std::min<size_t>(h.trace_bytes / 64, 1u << 30));
  }
  // The shared expert's two matmuls ride in the routed launches of the same phase.
  QmmArgs d{};
  const uint32_t dense_up = c.shared_f ? (t + tile.up - 1) / tile.up : 0, dense_down = c.shared_f ? (t + tile.down - 1) / tile.down : 0;
  if (c.shared_f) {
    d.dense_mode = 1; d.dense_rows = t; d.top_k = c.top_k; d.narrow = 1;
    d.dense[0] = w.shared_gate; d.dense[1] = w.shared_up;
    d.x = ws.xp; d.sumx = ws.sum_x; d.x_stride = c.d; d.rows = c.shared_f; d.kdim = c.d; d.epi = 0; d.out = ws.sact;
    d.out_sums = ws.sum_sact;
    d.row_max = ws.row_max;
  }
  // phase 1: routed gate/up -> acts [pair, F]; shared gate/up -> sact [token, Fs]
  q.w_off[0] = w.offsets.gate_w; q.s_off[0] = w.offsets.gate_s; q.b_off[0] = ternary ? w.offsets.gate_s : w.offsets.gate_b;
  q.w_off[1] = w.offsets.up_w; q.s_off[1] = w.offsets.up_s; q.b_off[1] = ternary ? w.offsets.up_s : w.offsets.up_b;
  q.x = ws.xp; q.sumx = ws.sum_x; q.x_stride = c.d; q.gather = 1; q.rows = c.f; q.kdim = c.d; q.epi = 0;
  q.out = ws.acts;
  q.out_sums = ws.sum_acts;
  q.row_max = ws.row_max;
  // The shared expert's work items (whole 64-row tiles, the longest of the launch) go first: a short batch
  // leaves workgroup slots over, and up to about 4096 tokens the launch ends sooner with them out of the way
  // (Qwen shape, layer: 2048 tokens 280.5 -> 274.5 us, 1024 tokens 191 -> 187 us, 4096 tokens 506 -> 503 us;
  // at 16 384 tokens they are better last, 1763 against 1776 us, where they fill the holes of the last round).
  const bool dense_first = shared_rides && pairs <= 32768;
  const auto slices = [](uint32_t rows, uint32_t rows_per_item) -> uint64_t { return (rows + rows_per_item - 1) / rows_per_item; };
  const bool few_up = prefill_few(c, t, lists.slots[0] * slices(c.f, kQmmRows) + dense_up * slices(c.shared_f, kQmmRows), c.d);
  if (dense_first) MF_TRY(launch_qmm(s, tile.up, launch_bits, d, 2, dense_up, &q, lists.slots[0], few_up));
  else MF_TRY(launch_qmm(s, tile.up, launch_bits, q, 2, lists.slots[0], shared_rides ? &d : nullptr, dense_up, few_up));
  if (lists.list[1]) q.tiles = lists.list[1];
  q2.sorted = q.sorted; q2.tiles = q.tiles; q2.row_max = q.row_max;
  q2.x = ws.acts; q2.sumx = ws.sum_acts; q2.out = ws.partials;
  if (c.shared_f) {
    d2.x = ws.sact; d2.sumx = ws.sum_sact; d2.out = ws.hs; d2.row_max = d.row_max;
  }
  const int down_proj = q2.pair_rows ? 2 : 1;
  const uint64_t down_slices = slices(c.d, kQmmRows * down_proj);
  const bool few_down = prefill_few(c, t, (lists.slots[1] + (apart ? 0 : dense_down)) * down_slices, c.f);
  if (!shared_rides || apart) {
    if (kres_q) MF_TRY(launch_qmm_kres(s, tile.down, code_bits, q2, lists.slots[1], nullptr, 0));
    else MF_TRY(launch_qmm(s, tile.down, code_bits, q2, down_proj, lists.slots[1], nullptr, 0, few_down));
    if (apart && kres_d) MF_TRY(launch_qmm_kres(s, tile.down, 4, d2, dense_down, nullptr, 0));
    else if (apart) MF_TRY(launch_qmm(s, tile.down, 4, d2, down_proj, dense_down, nullptr, 0, prefill_few(c, t, dense_down * down_slices, c.shared_f)));
  } else if (kres_both) {
    if (dense_first) MF_TRY(launch_qmm_kres(s, tile.down, launch_bits, d2, dense_down, &q2, lists.slots[1]));
    else MF_TRY(launch_qmm_kres(s, tile.down, launch_bits, q2, lists.slots[1], &d2, dense_down));
  } else if (dense_first) MF_TRY(launch_qmm(s, tile.down, launch_bits, d2, down_proj, dense_down, &q2, lists.slots[1], few_down));
  else MF_TRY(launch_qmm(s, tile.down, launch_bits, q2, down_proj, lists.slots[1], &d2, dense_down, few_down));
  if (ragged) return hipSuccess;  // the per-route results are the caller's: mf_moe_unpermute reduces them
  const uint16_t* hs = nullptr;
  const uint16_t* gate = nullptr;
  if (c.shared_f) {
    hs = ws.hs;
    if (want_gate) gate = ws.gate;
  }
  const size_t n4 = static_cast<size_t>(t) * c.d / 4;
  const dim3 reduce_grid(static_cast<uint32_t>((n4 + 255) / 256));
  if (narrow_routes)
    prefill_reduce_kernel<true><<<reduce_grid, dim3(256), 0, s>>>(ws.partials, ws.w, ws.idx, hs, gate, y, t, c.top_k, c.d,
                                                                  c.num_experts, static_cast<int>(c.maple_rounding));
  else
    prefill_reduce_kernel<false><<<reduce_grid, dim3(256), 0, s>>>(ws.partials, ws.w, ws.idx, hs, gate, y, t, c.top_k, c.d,
                                                                   c.num_experts, static_cast<int>(c.maple_rounding));
  MF_TRY(hipGetLastError());
#undef MF_TRY
  return hipSuccess;
}

hipError_t launch_prefill_layer(hipStream_t s, const mf_moe& h, const mf_moe_layer_weights& w,
                                const uint16_t* x, uint32_t t, uint16_t* y, void* workspace,
                                uint32_t* out_idx, float* out_w) {
  return launch_prefill_layer(s, h, w, x, t, y, workspace, out_idx, out_w, nullptr);
}

}  // namespace mf
