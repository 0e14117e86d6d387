// 8-bit affine rows beyond the one-wave-per-(token, row) kernels of gemv.hip: a row kernel that requests a whole
// row before it uses any of it (few token rows, the bits of those kernels), and a matrix-core matmul (many).
//
// Replaces shared_int8_gate_up_act_simd and dequant_int8_gemv_simd (Metal/Quant/dequant_int8.metal:66-164).
#include <algorithm>

#include "mf_device.h"
#include "mf_internal.h"
#include "mf_router.h"

#pragma clang fp contract(off)

namespace mf {

struct Q8Args {
  const uint8_t* W[2];
  const uint16_t* S[2];
  const uint16_t* B[2];
  const uint16_t* x;  // [T, N]
  void* y;            // one projection: [T, M] bf16 or fp32; two: bf16 activations [T, M]
  uint32_t M, N, T;
  int out_f32, silu;
};

// narrowed gate and up, tanh-GELU or SiLU (int8_gelu_pytorch_tanh and FC_SHARED_INT8_ACT_SILU, dequant_int8.metal:44-57)
__device__ __forceinline__ uint16_t q8_activation(float g, float u, bool silu) {
  const float gh = round_bf16(g), uh = round_bf16(u);
  return f_to_bf16((silu ? mf_silu(gh) : mf_gelu_tanh(gh)) * uh);
}

// ---- few token rows: one wave per weight row (both projections), in dot_q8_row's order -- chunk c of 8 codes on lane
// c % 64, sums in ascending order, two fmas per chunk, neighbour-first butterfly -- so a token has the same bits in
// every kernel of this family.  Bound: a wave's life is one memory round trip plus its arithmetic.  Chunk by chunk
// (gemv_q8_kernel) a 2816-element row is six round trips in a row; here the codes, tables and the first token's x of
// the whole row leave together (CPL chunks per lane), and every further token reuses the codes.  Scales and biases come a group to a
// lane, a request per table, and are handed to the chunks' lanes (2816 x 2112 gate/up pair, one token: 7.2 -> 6.6 us against two
// requests per chunk; a wave to a workgroup, for an even load of the CUs, lost 1 % of eight layers).
// (The codes become numbers inside the token loop: kept as fp32 they take 180 registers for a gate / up pair of 2816,
// two waves to a SIMD, and 2112 rows are then a full round of waves plus a little.)
template <int NPROJ, int CPL>
__global__ __launch_bounds__(256) void rows_q8_kernel(const Q8Args a) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= a.M) return;
  const uint32_t chunks = a.N / 8, ng = a.N / kGroup;
  uint2 q[NPROJ][CPL];
  uint32_t tab[NPROJ];  // of group `lane` of the row: bias below scale
  uint4 xv[CPL], xn[CPL];
#pragma unroll
  for (int p = 0; p < NPROJ; ++p) {
    const size_t at = static_cast<size_t>(row) * ng + min(lane, ng - 1);
    tab[p] = a.B[p][at] | (static_cast<uint32_t>(a.S[p][at]) << 16);
  }
#pragma unroll
  for (int i = 0; i < CPL; ++i) {
    const uint32_t c = min(lane + 64 * i, chunks - 1);  // a chunk past the row repeats the last one and is dropped
    xv[i] = load_x8<true>(a.x + c * 8);
#pragma unroll
    for (int p = 0; p < NPROJ; ++p) q[p][i] = *reinterpret_cast<const uint2*>(a.W[p] + static_cast<size_t>(row) * a.N + c * 8);
  }
  issue_fence();
  uint32_t sb[NPROJ][CPL];  // of the group of chunk lane + 64 i: 8 i + lane / 8
#pragma unroll
  for (int p = 0; p < NPROJ; ++p)
#pragma unroll
    for (int i = 0; i < CPL; ++i) sb[p][i] = __builtin_amdgcn_ds_bpermute(4 * (8 * i + (lane >> 3)), tab[p]);
  for (uint32_t t = 0; t < a.T; ++t) {
    const uint16_t* nx = a.x + static_cast<size_t>(min(t + 1, a.T - 1)) * a.N;  // (the last token requests itself again)
#pragma unroll
    for (int i = 0; i < CPL; ++i) xn[i] = load_x8<true>(nx + min(lane + 64 * i, chunks - 1) * 8);
    issue_fence();
#pragma unroll
    for (int i = 0; i < CPL; ++i)
#pragma unroll
      for (int p = 0; p < NPROJ; ++p) asm volatile("" : "+v"(q[p][i].x), "+v"(q[p][i].y));
    float acc[NPROJ];
#pragma unroll
    for (int p = 0; p < NPROJ; ++p) acc[p] = 0.0f;
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      if (lane + 64 * i < chunks) {
        const uint32_t xs[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w};
        float dot[NPROJ], sum = 0.0f;
#pragma unroll
        for (int p = 0; p < NPROJ; ++p) dot[p] = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float x0 = bf16_lo(xs[j]), x1 = bf16_hi(xs[j]);
          sum = sum + x0;
          sum = sum + x1;
#pragma unroll
          for (int p = 0; p < NPROJ; ++p) {
            const uint32_t word = (j < 2 ? q[p][i].x : q[p][i].y) >> ((j & 1) * 16);
            dot[p] = __builtin_fmaf(static_cast<float>(word & 0xFFu), x0, dot[p]);
            dot[p] = __builtin_fmaf(static_cast<float>((word >> 8) & 0xFFu), x1, dot[p]);
          }
        }
#pragma unroll
        for (int p = 0; p < NPROJ; ++p) {
          acc[p] = __builtin_fmaf(bf16_hi(sb[p][i]), dot[p], acc[p]);
          acc[p] = __builtin_fmaf(bf16_lo(sb[p][i]), sum, acc[p]);
        }
      }
    }
#pragma unroll
    for (int p = 0; p < NPROJ; ++p) acc[p] = wave_sum(acc[p]);
    if (lane == 0) {
      const size_t at = static_cast<size_t>(t) * a.M + row;
      if constexpr (NPROJ == 2) static_cast<uint16_t*>(a.y)[at] = q8_activation(acc[0], acc[1], a.silu != 0);
      else if (a.out_f32) static_cast<float*>(a.y)[at] = acc[0];
      else static_cast<uint16_t*>(a.y)[at] = f_to_bf16(acc[0]);
    }
#pragma unroll
    for (int i = 0; i < CPL; ++i) xv[i] = xn[i];
  }
}

// ---- many token rows, on the bf16 matrix cores.  Codes 0..255 are bf16 numbers as they are, so a K group is
// sum(q x) from four 32x32x16 products, one fp32 multiply-add with the row's scale, and the biases enter as one more
// product per two groups: sum(x) of a group as three bf16 terms (all 24 bits) against the bias in three K slots.
// Tokens are the M side, weight rows the N side: a lane ends with one weight row, its scale is a per-lane scalar.
// (A code byte masked into the low half of a 16-bit word is the bf16 number q * 2^-133, as in mf_device.h, for half of the vector
// instructions; but codes below 128 then enter with the exponent of 128, the matrix core aligns products by the operands' exponents, and
// small codes beside large values of x lost bits: rms error over the size of the terms 2.4e-8 -> 7.8e-8 at 2112 x 2816, 300 rows, nine
// codes of ten below 16 and one value of 1000 in a row, 3.9e-8 -> 4.3e-7 at 256 x 128.  The 2- and 4-bit codes sit at the top of the byte.)
//
// A workgroup is 64 weight rows (of each projection) x 64 tokens.  Its four waves are 2 row blocks x 2 projections, or with one projection x
// the 2 groups of a stage, and each takes all 64 tokens: what bounds the kernel is vector instructions, above all those that make numbers of
// the codes, and so every code is converted once in a workgroup (waves of 2 row blocks x 2 token blocks did it twice).  A stage is 128 K values: x rows and
// code rows come in as whole 128-byte lines, three stages ahead of their use (two sets of registers and an LDS buffer: a stage's
// arithmetic is 0.5 us, a round trip to memory 1 to 2), and are handed out through LDS (16-byte
// pieces, XOR-swizzled so that 16 lanes reading one piece of 16 rows cover all banks): read straight from memory a
// lane's 16 bytes of its own row touch 32 lines per load instruction, and the line rate of the L1, not the matrix
// core, would set the pace.  Scales and biases come 8 groups (four stages) to a load.
// KS = 2: two such sets of four waves share the workgroup, each walks half of K in buffers of its own, and their sums
// meet in LDS at the end -- for problems of at most a workgroup per CU, where one wave to a SIMD neither hides its
// loads nor overlaps vector and matrix instructions (2816 x 2112, 300 tokens, waves of two token blocks: gate/up 47.6 -> 37.9 us).
// The MLP, us, waves of two token blocks with results stored by their lanes / now: 2816 x 2112, 16 rows 49.8 / 43.1, 300 53.8 / 47.1, 600
// 84.3 / 75.1, 2048 220.7 / 199.8; 704 x 8192, 16 rows 63.2 / 59.8, 300 87.3 / 81.5, 2048 240 / 220; 2048 x 2048, 16 rows 39.2 / 34.6, 1024
// 70.3 / 64.1; 192 x 128, 64 rows 12.3 / 10.6.  Nothing looks at a register where it is requested (the zeros for what lies past the row
// were put in there, and every stage waited for its own request, tables for all of them): 2816 x 2112, 16 rows 43.1 / 38.3, 300 47.1 / 43.5,
// 2048 199.8 / 179.9; 704 x 8192, 16 rows 59.8 / 51.0, 2048 220 / 192; 2048 x 2048, 16 rows 34.6 / 30.5.
// (128 tokens per workgroup, two accumulators a wave to one set of codes, lost at every size: 2816 x 2112, 2048 tokens 302
// against 224 us, 16384 tokens 1895 against 1492; 704 x 8192, 1500 tokens 227 against 195.)

// LONG: a set walks more than three stages.  A shorter walk ends before requests three ahead pay for themselves, and instructions that run
// once cost their fetch: it requests one stage ahead, its table entries by themselves.  us, long form / short: 128 x 192, 16 rows
// 13.9 / 10.0; 384 x 256, 64 rows 18.0 / 14.5; 768 x 384 (three stages a set), 200 rows 21.2 / 19.1; 1024 x 1024 (four), 16 rows 23.6 / 27.1.
template <int NPROJ, int KS, bool LONG>
__global__ __launch_bounds__(256 * KS) __attribute__((amdgpu_waves_per_eu(2, 2)))
void qmm8_kernel(const Q8Args a, uint32_t n_tiles, uint32_t n_work) {
  constexpr uint32_t kTok = 64;
  __shared__ uint4 s_x_all[KS][2][kTok * 16];      // [token][16 pieces of 8 values], piece ^ (token & 15)
  __shared__ uint4 s_w_all[KS][2][NPROJ][64 * 8];  // [row][8 pieces of 16 codes], piece ^ ((row >> 1) & 7)
  __shared__ float s_sum_all[KS][2][kTok][2];      // sum of x over the stage's two groups
  const uint32_t tid = threadIdx.x & 255u, kh = KS == 1 ? 0u : threadIdx.x >> 8;
  auto& s_x = s_x_all[kh];
  auto& s_w = s_w_all[kh];
  auto& s_sum = s_sum_all[kh];
  // consecutive work items (the token tiles of one row slice) on one XCD: its L2 serves the weight rows' re-reads
  const uint32_t per = (n_work + 7) / 8, work = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per || work >= n_work) return;
  const uint32_t t0 = (work % n_tiles) * kTok, r0 = (work / n_tiles) * 64;
  const uint32_t lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), m = lane & 31, h = lane >> 5;
  const uint32_t rb = wv & 1, z = wv >> 1;
  const uint32_t ng = a.N / kGroup, n_st = (ng + 1) / 2;
  const uint32_t n_walk = (n_st + KS - 1) / KS, st0 = kh * n_walk, st1 = min(n_st, st0 + n_walk);  // this set's stages

  // staging roles: x -- token t / 4, pieces 4q .. 4q + 3 (half a group); codes -- row t / 8 (+ 32), piece t % 8
  // (whole 256-byte token rows per 16 threads measured slower: 40.4 against 37.9 us, four row addresses a thread)
  const uint32_t xt = tid >> 2, xq = tid & 3, wr = tid >> 3, wc = tid & 7;
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
  u32x4_t xr[2][4], wreg[2][NPROJ][2];                  // stage st waits in set st & 1 (counted from st0)
  const uint32_t row = min(r0 + rb * 32 + m, a.M - 1);  // the lane's weight row (past the end: the last one, not stored)
  auto fetch = [&](uint32_t st, u32x4_t (&xs)[4], u32x4_t (&ws)[NPROJ][2]) __attribute__((always_inline)) {
    const uint32_t g = min(2 * st + (xq >> 1), ng - 1);  // (past the row: its last group, which `put` makes zeros of)
    const uint16_t* src = a.x + static_cast<size_t>(min(t0 + xt, a.T - 1)) * a.N + g * kGroup + (xq & 1) * 32;
#pragma unroll
    for (int i = 0; i < 4; ++i) xs[i] = *reinterpret_cast<const u32x4_t*>(src + 8 * i);
    const uint32_t k0 = min(st * 128 + wc * 16, a.N - 16);  // (codes past the row, or of a stage past the last, meet x = 0)
#pragma unroll
    for (int p = 0; p < NPROJ; ++p) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        ws[p][i] = *reinterpret_cast<const u32x4_t*>(a.W[p] + static_cast<size_t>(min(r0 + wr + 32 * i, a.M - 1)) * a.N + k0);
    }
  };
  // scales and biases of the wave's projection
  const uint16_t* tab_s = a.S[NPROJ == 2 ? z : 0];
  const uint16_t* tab_b = a.B[NPROJ == 2 ? z : 0];
  // Those of the eight groups from g (a group of the row) on.  A load past the row's last group reads on into the next row, the table's
  // last loads end with the table; what is not the row's is taken off, and groups past its last one become zeros, when the four stages
  // that use them begin.
  struct Tab { uint4 S, B; };
  auto fetch_tab = [&](uint32_t g) __attribute__((always_inline)) {
    const uint32_t base = min(row * ng + g, a.M * ng - 8);
    return Tab{load_16_bytes(tab_s + base), load_16_bytes(tab_b + base)};
  };
  auto settle_tab = [&](const Tab& t, uint32_t g) __attribute__((always_inline)) {
    const uint32_t at = row * ng + min(g, ng - 1), skip = at - min(at, a.M * ng - 8);
    uint4 S = drop_bf16(t.S, skip), B = drop_bf16(t.B, skip);
    if (g + 8 > ng) {
      uint32_t keep[4];
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) keep[i] = g + 2 * i + 1 < ng ? 0xFFFFFFFFu : g + 2 * i < ng ? 0xFFFFu : 0u;
      S = make_uint4(S.x & keep[0], S.y & keep[1], S.z & keep[2], S.w & keep[3]);
      B = make_uint4(B.x & keep[0], B.y & keep[1], B.z & keep[2], B.w & keep[3]);
    }
    return Tab{S, B};
  };
  // stage st into a buffer.  Half a stage behind an odd number of groups and a stage past this set's last are zeros, and become so here:
  // a look at the registers where they are requested would wait for them.
  auto put = [&](uint32_t buf, uint32_t st, const u32x4_t (&xs)[4], const u32x4_t (&ws)[NPROJ][2]) __attribute__((always_inline)) {
    const bool in = 2 * st + (xq >> 1) < ng && st < st1;
    float part = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u32x4_t v = in ? xs[i] : u32x4_t{0, 0, 0, 0};
      reinterpret_cast<u32x4_t*>(s_x[buf])[xt * 16 + ((4 * xq + i) ^ (xt & 15u))] = v;
      part += ((bf16_lo(v.x) + bf16_hi(v.x)) + (bf16_lo(v.y) + bf16_hi(v.y))) +
              ((bf16_lo(v.z) + bf16_hi(v.z)) + (bf16_lo(v.w) + bf16_hi(v.w)));
    }
    part = group_sum(part, 2);
    if ((xq & 1) == 0) s_sum[buf][xt][xq >> 1] = part;
#pragma unroll
    for (int p = 0; p < NPROJ; ++p)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t r = wr + 32 * i;
        reinterpret_cast<u32x4_t*>(s_w[buf][p])[r * 8 + (wc ^ ((r >> 1) & 7u))] = ws[p][i];
      }
  };
  f32x16_t acc[2];  // of the two blocks of 32 tokens
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[j][r] = 0.0f;
  const uint32_t tok_of[2] = {m, 32 + m};  // the tokens whose x operands this lane reads

  // one stage out of LDS; scale(g): of the stage's group g; bias: the bits of that of group h
  auto multiply = [&](uint32_t buf, auto scale, uint32_t bias) __attribute__((always_inline)) {
    // biases: K slots of half h = (hi, mid, lo) of sum(x) over the stage's group h (a group past the end sums to 0).  With one projection a
    // wave takes its own group's alone: q x and the bias term mostly cancel, so they belong into one sum (both groups' biases in one of
    // the two waves' sums: error against 64 bits 1.6e-7 -> 2.5e-7 at 2112 x 2816).  An infinite bias meets hi alone: mid, lo and what a
    // wave leaves to the other are zeros, and 0 times it would be NaN.
    const bool own = NPROJ == 2 || h == z;
    const uint32_t b_hi = own ? bias : 0u, b_rest = (b_hi & 0x7F80u) == 0x7F80u ? 0u : b_hi;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float v = own ? s_sum[buf][tok_of[j]][h] : 0.0f;
      const uint32_t hi = __float_as_uint(v) & 0xFFFF0000u;
      const float r1 = __builtin_isinf(v) ? 0.0f : v - __uint_as_float(hi);  // (an infinite sum has no rest: inf - inf would be NaN)
      const uint32_t mid = __float_as_uint(r1) & 0xFFFF0000u;
      const uint32_t lo = __float_as_uint(r1 - __uint_as_float(mid));
      acc[j] = mfma_bf16(make_uint4((hi >> 16) | mid, lo >> 16, 0, 0), make_uint4(b_hi | (b_rest << 16), b_rest, 0, 0), acc[j]);
    }
#pragma unroll
    for (int gi = 0; gi < NPROJ; ++gi) {
      const uint32_t g = NPROJ == 2 ? gi : z;
      uint4 bx[2][4];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int s = 0; s < 4; ++s) bx[j][s] = s_x[buf][tok_of[j] * 16 + ((8 * g + 4 * h + s) ^ (tok_of[j] & 15u))];
      const uint32_t r = rb * 32 + m;
      f32x16_t tmp[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i) tmp[j][i] = 0.0f;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const uint4 w = s_w[buf][NPROJ == 2 ? z : 0][r * 8 + ((4 * g + 2 * h + c) ^ ((r >> 1) & 7u))];
        const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int u = 0; u < 2; ++u) {  // eight codes -> eight bf16 numbers (a byte as fp32 has its bits in the upper half)
          uint32_t o[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const uint32_t word = ww[2 * u + (k >> 1)] >> (16 * (k & 1));
            o[k] = upper_halves(static_cast<float>(word & 0xFFu), static_cast<float>((word >> 8) & 0xFFu));
          }
#pragma unroll
          for (int j = 0; j < 2; ++j) tmp[j] = mfma_bf16(bx[j][2 * c + u], make_uint4(o[0], o[1], o[2], o[3]), tmp[j]);
        }
      }
      const float s = scale(g);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[j][i] = __builtin_fmaf(s, tmp[j][i], acc[j][i]);
    }
  };
  if constexpr (LONG) {
    // (no branch around a request: a wait for one stage's registers would cover the later stages' as well)
    fetch(st0, xr[0], wreg[0]);
    Tab next = fetch_tab(min(2 * st0, ng - 1));
    issue_fence();  // (in front of the stages' loads: the wait for the first table is not one for those)
    fetch(st0 + 1, xr[1], wreg[1]);
    put(0, st0, xr[0], wreg[0]);
    fetch(st0 + 2, xr[0], wreg[0]);
    for (uint32_t i0 = 0; i0 < n_walk; i0 += 4) {
      const Tab tab = settle_tab(next, 2 * (st0 + i0));
      next = fetch_tab(min(2 * (st0 + i0 + 4), ng - 1));
#pragma unroll
      for (int u4 = 0; u4 < 4; ++u4) {  // stage i0 + u4, in buffer u4 & 1
        if (i0 + u4 >= n_walk) break;
        __syncthreads();  // its buffer is complete, the other one is no longer read
        const int buf = u4 & 1, other = buf ^ 1;
        if (i0 + u4 + 1 < n_walk) put(other, st0 + i0 + u4 + 1, xr[other], wreg[other]);
        fetch(st0 + i0 + u4 + 3, xr[other], wreg[other]);
        const uint32_t s4[4] = {tab.S.x, tab.S.y, tab.S.z, tab.S.w}, b4[4] = {tab.B.x, tab.B.y, tab.B.z, tab.B.w};
        multiply(buf, [&](uint32_t g) { return g ? bf16_hi(s4[u4]) : bf16_lo(s4[u4]); }, h ? b4[u4] >> 16 : b4[u4] & 0xFFFFu);
      }
    }
  } else {
    uint16_t sc[2], bi;  // a stage's table entries
    auto fetch_entries = [&](uint32_t st) __attribute__((always_inline)) {
      const size_t at = static_cast<size_t>(row) * ng;
      sc[0] = tab_s[at + min(2 * st, ng - 1)];
      sc[1] = tab_s[at + min(2 * st + 1, ng - 1)];
      bi = tab_b[at + min(2 * st + h, ng - 1)];
    };
    if (st0 < st1) {
      fetch(st0, xr[0], wreg[0]);
      fetch_entries(st0);
      put(0, st0, xr[0], wreg[0]);
      if (st0 + 1 < st1) fetch(st0 + 1, xr[0], wreg[0]);
    }
#pragma unroll 1
    for (uint32_t i = 0; i < n_walk; ++i) {
      __syncthreads();
      if (st0 + i >= st1) continue;  // (the second set may have a stage less: it keeps the barriers company)
      // (half a stage behind an odd number of groups: zeros, like its x; the entry that came is the last group's)
      const bool whole = 2 * (st0 + i) + 1 < ng;
      const uint16_t sv[2] = {sc[0], whole ? sc[1] : uint16_t{0}}, bv = whole || h == 0 ? bi : uint16_t{0};
      if (st0 + i + 1 < st1) {
        put((i + 1) & 1u, st0 + i + 1, xr[0], wreg[0]);
        fetch_entries(st0 + i + 1);
        if (st0 + i + 2 < st1) fetch(st0 + i + 2, xr[0], wreg[0]);
      }
      multiply(i & 1u, [&](uint32_t g) { return bf16_to_f(g ? sv[1] : sv[0]); }, bv);
    }
  }
  // All sums go through LDS, over the x buffers, [set][part = wave's z][token][row], and the whole workgroup stores: 64 rows of a token per
  // wave and step, in a loop that stays short (straight-line code that runs once costs its fetch: with 16 results a lane of the first set's
  // waves it was 2400 instructions).
  static_assert(sizeof(s_x_all) >= KS * 2u * 64 * 64 * sizeof(float), "the sums fit the x buffers");
  float* s_acc = reinterpret_cast<float*>(&s_x_all[0][0][0]);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i)  // the lane holds weight row r0 + 32 rb + m for tokens 8 (i / 4) + 4h + i % 4 of a 32-token block
      s_acc[((kh * 2 + z) * 64 + j * 32 + 8 * (i >> 2) + 4 * h + (i & 3)) * 64 + rb * 32 + m] = acc[j][i];
  __syncthreads();
  const uint32_t out_row = r0 + lane, n_tok = min(kTok, a.T - t0);
  if (out_row >= a.M) return;
#pragma unroll 2
  for (uint32_t tok = kh * 4 + wv; tok < n_tok; tok += 4 * KS) {
    float v[2];
#pragma unroll
    for (uint32_t p = 0; p < 2; ++p) {
      v[p] = s_acc[(p * 64 + tok) * 64 + lane];
      if constexpr (KS == 2) v[p] = v[p] + s_acc[((2 + p) * 64 + tok) * 64 + lane];
    }
    const size_t at = static_cast<size_t>(t0 + tok) * a.M + out_row;
    if constexpr (NPROJ == 2) {
      static_cast<uint16_t*>(a.y)[at] = q8_activation(v[0], v[1], a.silu != 0);
    } else {
      const float sum = v[0] + v[1];
      if (a.out_f32) static_cast<float*>(a.y)[at] = sum;
      else static_cast<uint16_t*>(a.y)[at] = f_to_bf16(sum);
    }
  }
}

// Which kernel: from 16 token rows on the matmul (its workgroups take 64 tokens at the price of one), below that the row
// kernel while a row fits its registers and there are rows enough to cover the chip; false: neither takes the shape.
template <int NPROJ>
static bool q8_launch(hipStream_t s, const Q8Args& a, hipError_t& err) {
  for (int p = 0; p < NPROJ; ++p)
    if (!aligned16(a.W[p])) return false;
  if (!aligned16(a.x) || a.N % kGroup) return false;
  if (a.T >= 16 && a.M >= 64) {
    // K halved among two sets of waves while there is at most a workgroup per CU (2816 x 2112: 420 rows 69 us with, 75
    // without; 512 rows, 264 and 352 workgroups on 256 CUs, 101 and 88)
    const uint32_t tiles = (a.T + 63) / 64, n_work = (a.M + 63) / 64 * tiles;
    const dim3 grid((n_work + 7) / 8 * 8);
    const bool halved = n_work <= device_cu_count();
    const uint32_t stages = (a.N / kGroup + 1) / 2, walk = halved ? (stages + 1) / 2 : stages;
    if (!halved && walk > 3) qmm8_kernel<NPROJ, 1, true><<<grid, dim3(256), 0, s>>>(a, tiles, n_work);
    else if (!halved) qmm8_kernel<NPROJ, 1, false><<<grid, dim3(256), 0, s>>>(a, tiles, n_work);
    else if (walk > 3) qmm8_kernel<NPROJ, 2, true><<<grid, dim3(512), 0, s>>>(a, tiles, n_work);
    else qmm8_kernel<NPROJ, 2, false><<<grid, dim3(512), 0, s>>>(a, tiles, n_work);
    err = hipGetLastError();
    return true;
  }
  if (a.M < 256 || a.N > 8 * 512) return false;
  const uint32_t cpl = (a.N / 8 + 63) / 64;
  const dim3 grid((a.M + 3) / 4), block(256);
#define MF_Q8(C) rows_q8_kernel<NPROJ, C><<<grid, block, 0, s>>>(a)
  if (cpl <= 2) MF_Q8(2);
  else if (cpl <= 4) MF_Q8(4);
  else if (cpl <= 5) MF_Q8(5);
  else if (cpl <= 6) MF_Q8(6);
  else MF_Q8(8);
#undef MF_Q8
  err = hipGetLastError();
  return true;
}

bool launch_q8_gemv(hipStream_t s, const mf_qtensor& w, const uint16_t* x, void* y, uint32_t m, uint32_t n, uint32_t t,
                    bool out_f32, hipError_t& err) {
  Q8Args a{};
  a.W[0] = a.W[1] = static_cast<const uint8_t*>(w.weights);
  a.S[0] = a.S[1] = w.scales;
  a.B[0] = a.B[1] = w.biases;
  a.x = x; a.y = y; a.M = m; a.N = n; a.T = t; a.out_f32 = out_f32 ? 1 : 0;
  return q8_launch<1>(s, a, err);
}

bool launch_q8_gate_up(hipStream_t s, const mf_qtensor& gate, const mf_qtensor& up, const uint16_t* x, uint16_t* act,
                       uint32_t f, uint32_t d, uint32_t t, bool silu, hipError_t& err) {
  Q8Args a{};
  a.W[0] = static_cast<const uint8_t*>(gate.weights); a.W[1] = static_cast<const uint8_t*>(up.weights);
  a.S[0] = gate.scales; a.S[1] = up.scales;
  a.B[0] = gate.biases; a.B[1] = up.biases;
  a.x = x; a.y = act; a.M = f; a.N = d; a.T = t; a.silu = silu ? 1 : 0;
  return q8_launch<2>(s, a, err);
}

}  // namespace mf
