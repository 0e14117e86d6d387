// The quantized matmuls of the prefill path: device code and launches, for tiles of 64 and of 32 routes.  Instantiated by
// qmm_ring.hip, qmm_resident.hip and qmm_tile32.hip (a source each, so that they compile side by side).
#pragma once

#include <algorithm>
#include <type_traits>

#include "mf_qmm.h"

#pragma clang fp contract(off)

namespace mf {

// LDS of qmm_kernel: x tile ring (2 stages of 2 K groups, 4 of the form for few work items), the scales and the group sums of a step of 16 groups, 12 bytes a route
constexpr uint32_t kTabStep = 16;
__host__ __device__ constexpr uint32_t qmm_stages(bool few) { return few ? 4 : 2; }
__host__ __device__ constexpr uint32_t qmm_x_bytes(uint32_t tile, bool few) { return qmm_stages(few) * 2 * tile * 8 * 16; }
__host__ __device__ constexpr uint32_t qmm_scale_bytes(int nproj) { return nproj * kQmmWaves * kTabStep * 32 * 4; }
__host__ __device__ constexpr uint32_t qmm_sum_bytes(uint32_t tile) { return 3 * tile * 2 * 16; }
__host__ __device__ constexpr uint32_t qmm_lds_bytes(uint32_t tile, int nproj, bool few) {
  return qmm_x_bytes(tile, few) + qmm_scale_bytes(nproj) + qmm_sum_bytes(tile) + tile * 12;
}

// waves a SIMD (workgroups a CU) that the kernels' registers are budgeted for; few: the form for few work items
__host__ __device__ constexpr int qmm_waves(uint32_t tile, int nproj, bool few = false) {
  return !few && (tile == kSmallTile || nproj == 1) ? 3 : 2;
}

__device__ __forceinline__ void qmm_trace(const QmmArgs& a, uint32_t work, uint32_t k) {
  if (a.trace && threadIdx.x == 0 && work < a.trace_items) a.trace[work * 8 + k] = wall_clock64();
}

// Workgroups go to the 8 XCDs round-robin by blockIdx; consecutive work items (the row slices of one tile share its x rows, the
// tiles of one expert share its weights) are laid on ONE XCD so that its L2 serves the re-reads.  Every XCD gets an eighth of the
// routed part's live items, which are counted here (the first tile's record holds the number of tiles): with whole tiles dealt out
// by eighths seven XCDs had 66 items for 64 slots and the eighth 48 (2816 x 704, 300 tokens, 85 tiles of 6 items).
struct QmmPlace {
  uint32_t xcd, slot, per_xcd;
};
constexpr uint32_t kNoWork = 0xFFFFFFFFu;
__device__ __forceinline__ QmmPlace qmm_place(const uint32_t (&per_xcd)[2], bool& second) {
  const uint32_t xcd_slot = blockIdx.x >> 3;
  second = xcd_slot >= per_xcd[0];
  return {blockIdx.x & 7u, xcd_slot - (second ? per_xcd[0] : 0u), per_xcd[second ? 1 : 0]};
}
__device__ __forceinline__ uint32_t qmm_work(const QmmArgs& a, const QmmPlace& at, uint32_t items_per_tile) {
  if (a.dense_mode) return at.xcd * at.per_xcd + at.slot;
  const uint32_t live = a.tiles->list_tiles * items_per_tile, per = (live + 7) / 8, work = at.xcd * per + at.slot;
  return at.slot < per && work < live ? work : kNoWork;
}

// One workgroup: a tile of TT (64 or 32) routes of one expert x 128 weight rows (4 waves x 32) x
// NPROJ projections, the whole K.  The matrix core computes the TRANSPOSED
// product: the A operand is the x tile (tokens are the rows), the B operand is
// the expanded codes, so a lane ends up holding ONE weight row (its column
// m = lane % 32) for 16 tokens of each 32-token block, and the per-group scale
// is one scalar per lane.  Tiles of 64 keep two waves per SIMD (256 registers: the matrix-core results stay in ordinary
// registers, where the scale multiply reads them directly), three with one row block; tiles of 32 fit 168 registers, three waves.
// What bounds it: the vector and matrix instructions of the loop, at the clock that power leaves.  So whatever a work item waits
// for in front of its loop is time the SIMD is not full, and the loop takes everything along: x goes straight to LDS, a pair of
// groups ahead, and scales, biases and group sums come a step of 16 groups ahead (before, all of them in front of the loop, in
// sequence for tiles of 32).  Stage stamps of a routed gate / up item, us, before -> now: Qwen shape, 2048 tokens, in front of the
// loop 6.1 -> 3.5, whole item 33.1 -> 29.8.  Launches of both forms traced on one card, us: that one 127.5 -> 115; a 5120 x 17408 MLP of 150
// rows, gate / up 98.9 -> 89.6, down in windows 59.6 -> 54.5; tiles of 32, where the instructions of the loop are the bound: large 2-bit layer,
// 777 tokens, gate / up 354 -> 345, down 179 -> 181; 2816 x 704, 300 tokens, gate / up 67.2 -> 68.3, down (11 groups) 50.9 -> 44.5.
// LDS no longer grows with K, so every contraction keeps its two or three workgroups a CU.
// FEW (tiles of 32): a launch that leaves a CU at most two workgroups is bound by what each waits for, codes from HBM above all.  It has
// the registers of two waves and their LDS: codes run four pairs of groups ahead, x three, and units are not kept apart.  The layer call,
// us, x in registers and two pairs of codes (the kernel before) / one pair / this: 16 experts of 8192 x 512, top 2, 17 tokens 81.3 / 91.4 /
// 75.8, 150 tokens 95.6 / 100.9 / 86.5; 32 of 5120 x 1536, top 1, 17 tokens 66.3 / 70.5 / 61.2; Qwen shape, 9 tokens 53.2 / 55.6 / 52.6.
// LDS (dynamic): x tile ring, 2 stages (FEW: 4) x 2 K groups x [TT tokens][8 runs, turned] x 16 B; per wave the scales of a step
// [NPROJ][16][32 rows] fp32; group sums of a step; per route: out slot u32, what its results lack, scale of its activations.
// One launch can carry two independent problems of the same instantiation (the routed experts
// and the shared expert of the same phase): the second problem's work items follow the first's
// on every XCD, so they fill the slots the first problem's last round leaves empty instead of
// running as a launch of their own that covers a quarter of the chip.
struct QmmLaunch {
  QmmArgs part[2];
  uint32_t per_xcd[2];  // work items of each part on one XCD (grid = 8 * their sum)
};

// NG8: K is a whole number of steps of 8 groups and the rows a whole number of slices; the other form takes any number
// of groups and rows.
template <int TT, int BITS, int NPROJ, bool NG8, bool SWAPPED, bool FEW>
__device__ __forceinline__ void qmm_item(const QmmArgs& a, const QmmPlace& place, uint8_t* smem) {
  constexpr int NT = TT / 32;             // token blocks of a tile
  constexpr uint32_t kXGroup = TT * 8;    // 16-byte pieces of one K group of the x tile
  constexpr uint32_t kGB = QmmCodes<BITS>::kGroupBytes;  // bytes of one K group of one weight row
  const uint32_t lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t m = lane & 31, h = lane >> 5;
  const uint32_t wave_rows = a.pair_rows ? 32u * NPROJ : 32u;  // weight rows of one wave
  const uint32_t n_slices = NG8 ? a.rows / (kQmmWaves * wave_rows) : (a.rows + kQmmWaves * wave_rows - 1) / (kQmmWaves * wave_rows);
  const uint32_t work = qmm_work(a, place, n_slices);
  uint32_t tile_id = work / n_slices, slice = work % n_slices, win = 0;
  if (a.dense_mode) {
    if (work >= a.dense_items) return;
    const uint32_t inner = a.tile_major ? n_slices : a.dense_tiles, outer = a.tile_major ? a.dense_tiles : n_slices;
    const uint32_t lo = work % inner, rest = work / inner, hi = rest % outer;
    tile_id = a.tile_major ? hi : lo;
    slice = a.tile_major ? lo : hi;
    win = rest / outer;
    if (tile_id >= a.dense_tiles) return;
  }
  uint32_t ng = a.kdim / kGroup, g_off = a.g_off;
  uint8_t* out_base = static_cast<uint8_t*>(a.out);
  uint8_t* out2_base = static_cast<uint8_t*>(a.out2);
  if (a.n_win > 1) {  // this work item's window of the contraction
    g_off = dense_window_start(a.ng_ld, a.n_win, win);
    ng = dense_window_start(a.ng_ld, a.n_win, win + 1) - g_off;
    out_base += win * a.out_win_stride * sizeof(float);
    if (out2_base) out2_base += win * a.out_win_stride * sizeof(float);
  }
  qmm_trace(a, work, 0);

  uint32_t expert = 0, pair_start, count;
  if (a.dense_mode) {
    pair_start = tile_id * TT;
    count = min(static_cast<uint32_t>(TT), a.dense_rows - pair_start);
  } else {
    if (work == kNoWork) return;
    // (the whole 16-byte record in one load: read field by field, the count was fetched, tested, and the rest
    // fetched in a second round trip)
    const uint4 tv = *reinterpret_cast<const uint4*>(a.tiles + tile_id);
    count = __builtin_amdgcn_readfirstlane(tv.z);
    expert = __builtin_amdgcn_readfirstlane(tv.x);
    pair_start = __builtin_amdgcn_readfirstlane(tv.y);
  }

  uint4* s_x = reinterpret_cast<uint4*>(smem);                      // 2 stages x 2 groups x kXGroup uint4
  float* s_scale = reinterpret_cast<float*>(smem + qmm_x_bytes(TT, FEW)) + wv * (NPROJ * kTabStep * 32);  // this wave's [NPROJ][16 groups][32 rows]
  uint4* s_sum = reinterpret_cast<uint4*>(smem + qmm_x_bytes(TT, FEW) + qmm_scale_bytes(NPROJ));  // [NT][3 parts][64 lanes]
  uint32_t* s_slot = reinterpret_cast<uint32_t*>(smem + qmm_x_bytes(TT, FEW) + qmm_scale_bytes(NPROJ) + qmm_sum_bytes(TT));
  float* s_rel = reinterpret_cast<float*>(s_slot + TT);  // [TT]
  float* s_act = s_rel + TT;                              // [TT]
  const uint32_t lds_x = static_cast<uint32_t>(reinterpret_cast<size_t>((__attribute__((address_space(3))) uint8_t*)smem));
  const uint32_t lds_sum = lds_x + qmm_x_bytes(TT, FEW) + qmm_scale_bytes(NPROJ);

  // weight pointers of this workgroup's projections
  const uint8_t* Wp[NPROJ];
  const uint16_t* Sp[NPROJ];
  const uint16_t* Bp[NPROJ];
  uint32_t row_base[NPROJ];  // first weight row of each of this wave's 32-row blocks
#pragma unroll
  for (int p = 0; p < NPROJ; ++p) {
    const int t = a.pair_rows ? 0 : p;
    if (a.dense_mode) {
      Wp[p] = static_cast<const uint8_t*>(a.dense[t].weights);
      Sp[p] = a.dense[t].scales;
      Bp[p] = a.dense[t].biases;
    } else {
      const uint8_t* blob = a.expert_base + static_cast<size_t>(expert) * a.expert_stride;
      Wp[p] = blob + a.w_off[t];
      Sp[p] = reinterpret_cast<const uint16_t*>(blob + a.s_off[t]);
      Bp[p] = reinterpret_cast<const uint16_t*>(blob + a.b_off[t]);
    }
    // (a width that is no multiple of the workgroup's rows: the last slice's waves past the end compute the last
    // 32 rows again and store nothing)
    row_base[p] = (slice * kQmmWaves + wv) * wave_rows + (a.pair_rows ? 32u * p : 0u);
    if (!NG8) row_base[p] = min(row_base[p], a.rows - 32u);
  }
  const uint32_t ng_ld = a.ng_ld ? a.ng_ld : ng;
  const size_t row_bytes = static_cast<size_t>(ng_ld) * kGB;

  // ---- everything the tile needs that depends only on the tile: issued back to back.
  // Routes past `count` read the tile's last route instead (finite data, results discarded).
  // x is requested straight into LDS, 8 tokens x 8 runs of 8 values an instruction: lane l brings a run of token l / 8 of the eight
  const uint32_t st_n = 8 * wv + (lane >> 3);  // (and, of a tile of 64, token st_n + 32)
  uint32_t xrow[NT], st_row[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    xrow[nt] = pair_start + min(32 * nt + m, count - 1);
    st_row[nt] = pair_start + min(32 * nt + st_n, count - 1);
  }
  uint32_t slot = pair_start + min(threadIdx.x & 63u, count - 1);
  // the routes' records are requested here and looked at behind the code loads below, which do not depend on
  // them: the first codes are then on their way one memory round trip earlier
  mf_pair pr{};
  uint32_t tok_st[NT] = {}, tok[NT] = {};
  if (!a.dense_mode) {
    pr = a.sorted[slot];
    if (a.gather) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        tok_st[nt] = a.sorted[st_row[nt]].token;
        tok[nt] = a.sorted[xrow[nt]].token;
      }
    }
  }
  // (addresses of codes and tables: a uniform base, which the scalar unit moves along, and the lane's 32-bit offset)
  const uint8_t* wbase[NPROJ];
  using Codes = QmmCodes<BITS, SWAPPED>;
  const uint32_t gstride = a.tiled ? 32u * kGB : kGB;  // bytes from a group's codes to the next group's
  const uint32_t second = static_cast<uint32_t>(Codes::second(row_bytes, a.tiled));
  const uint32_t lane_off = static_cast<uint32_t>(Codes::lane_offset(lane, row_bytes, a.tiled));
  const uint32_t last_pair = (ng - 1) & ~1u;
  // (the last pair of an odd number of groups is half a pair: the lanes that would ask for its second group ask for the first)
  const uint32_t last_off = lane_off - (!NG8 && (ng & 1u) ? Codes::lane_group(lane) * gstride : 0u);
  // part i of the pair of groups from g on; past the end: the last pair again
  auto codes_at = [&](int p, uint32_t g, int i) __attribute__((always_inline)) {
    const uint32_t gc = min(g, last_pair);
    return wbase[p] + (gc * gstride + (i ? second : 0u)) + (!NG8 && gc == last_pair ? last_off : lane_off);
  };
  // pairs of groups in flight: one for 4-bit codes on tiles of 32, whose 168 registers do not hold a second (with it, 31 values went
  // through scratch memory: 2816 x 704, 300 tokens, gate / up 60 -> 100 us; 93 tokens of the Qwen shape 31 -> 37)
  constexpr int kRing = FEW ? 4 : NT == 1 && BITS == 4 ? 1 : 2;
  RegArray<Codes, kRing> cur[NPROJ];
#pragma unroll
  for (int p = 0; p < NPROJ; ++p) {
    wbase[p] = Wp[p] + row_base[p] * row_bytes + static_cast<size_t>(g_off) * gstride;
#pragma unroll
    for (int u = 0; u < kRing; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i) cur[p][u].load(i, codes_at(p, 2 * u, i));
  }
  // Scale (what = 0) or bias words (1) of the lane's row of projection p in a step of 16 K groups: groups g0 + 8h .. + 7
  auto tab_fetch = [&](int what, int p, uint32_t g0) __attribute__((always_inline)) -> uint4 {
    const uint16_t* table = (what ? Bp[p] : Sp[p]) + static_cast<size_t>(row_base[p]) * ng_ld + g_off;
    const uint32_t gl = g0 + 8 * h;
    const uint32_t gc = gl < ng ? gl : 0;  // a lane without groups reads group 0 and drops it
    // (whole 16-byte loads at any group and alignment; in the last step they end at the row's end and tab_step moves them down: done
    // here, it would wait for them and for every request in front of them)
    return load_16_bytes(table + (m * ng_ld + (NG8 ? gc : min(gc, ng - 8))));
  };
  uint4 tab[2][NPROJ];  // of the next step
#pragma unroll
  for (int p = 0; p < NPROJ; ++p)
#pragma unroll
    for (int what = 0; what < 2; ++what)
      tab[what][p] = NG8 || ng >= 8 ? tab_fetch(what, p, 0)
                                    : load_bf16x8_guarded((what ? Bp[p] : Sp[p]) + static_cast<size_t>(row_base[p] + m) * ng_ld + g_off, h ? 0u : ng);
  __builtin_amdgcn_sched_barrier(0);  // (keeps the look at the routes behind the loads that do not depend on them)
  if (!a.dense_mode) {
    if (a.gather) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        st_row[nt] = tok_st[nt];
        xrow[nt] = tok[nt];
      }
    }
    if (a.epi == 1 || a.epi == 3) slot = pr.token * a.top_k + pr.rank;
  }
  const float row_max = a.row_max[a.dense_mode ? pair_start + min(threadIdx.x & 63u, count - 1) : pr.token];
  // The place in the 128 bytes of a token's group where run c lies: c ^ (token / 2 % 8), so that the 16 lanes that read one run of
  // as many tokens together meet all the banks.
  const uint8_t* x_src[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    x_src[nt] = reinterpret_cast<const uint8_t*>(a.x + static_cast<size_t>(st_row[nt]) * a.x_stride + static_cast<size_t>(g_off) * kGroup) +
                ((lane & 7u) ^ ((st_n >> 1) & 7u)) * 16u;
  // K groups g and g + 1 of the tile's first `blocks` blocks of 32 tokens into a stage of the ring (an odd number of groups: the
  // last pair's second group is the last one again, and not multiplied)
  auto x_request = [&](uint32_t g, uint32_t stage, int blocks) __attribute__((always_inline)) {
#pragma unroll
    for (int gi = 0; gi < 2; ++gi)
#pragma unroll
      for (int nt = 0; nt < blocks; ++nt)
        load_to_lds(x_src[nt] + (NG8 ? g + gi : min(g + gi, ng - 1)) * 128u,
                    lds_x + ((stage * 2 + gi) * TT + nt * 32 + wv * 8) * 128);
  };
  // the group sums of a step, for the bias terms: three bf16 parts of 8 groups by half, token by lane
  auto sums_request = [&](uint32_t g0, int blocks) __attribute__((always_inline)) {
    const uint32_t gl = g0 + 8 * h, gc = gl < ng ? gl : 0;
#pragma unroll
    for (int i = 0; i < 3 * blocks; ++i)
      if (wv == i % kQmmWaves)
        load_to_lds(a.sumx + xrow[i / 3] * group_sum_words(ng_ld) + (g_off + gc) / 8 * 24 + 8 * (i % 3), lds_sum + i * 1024);
  };
  qmm_trace(a, work, 1);

  if (threadIdx.x < TT) s_slot[threadIdx.x] = threadIdx.x < count ? slot : 0xFFFFFFFFu;

  f32x16_t acc[NPROJ][NT];
#pragma unroll
  for (int p = 0; p < NPROJ; ++p)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[p][nt][r] = 0.0f;

  // A tile of at most 32 routes fills only the first token block: the second block's matrix
  // instructions and scale multiplies are left out (NTA = 1); its accumulators stay zero and its
  // output slots are empty.  Of a tile of at most 8 routes (most tiles of a short prompt) a lane's first four results are all
  // there is: only those are scaled (RES), 4 of 16 multiply-adds per group and row block.
  auto tile_body = [&](auto nta_c, auto res_c) {
  constexpr int NTA = decltype(nta_c)::value, RES = decltype(res_c)::value;
  // Behind a pair's x a wave requests kCodeLoads loads of codes, and before that pair's turn the x of every further stage and as many
  // codes again: kBehind, of which none may be left out.
  constexpr int kStages = qmm_stages(FEW), kCodeLoads = NPROJ * (BITS == 4 ? 2 : 1);
  constexpr int kBehind = (kStages - 2) * (kCodeLoads + 2 * NTA) + kCodeLoads;
  sums_request(0, NTA);
  x_request(0, 0, NTA);
  if constexpr (FEW) {
#pragma unroll
    for (int u = 1; u < kStages - 1; ++u) x_request(min(2u * u, last_pair), u, NTA);
  }
  if (threadIdx.x < TT) {
    s_rel[threadIdx.x] = rel_of_scale(a.act_rows ? act_scale(row_max) : row_scale(row_max));
    s_act[threadIdx.x] = act_scale(row_max);
  }
  uint32_t rd_col[4];
#pragma unroll
  for (int sidx = 0; sidx < 4; ++sidx) rd_col[sidx] = m * 8 + ((4 * h + sidx) ^ ((m >> 1) & 7u));
  // Per step of 16 groups: the scales of the wave's rows, times the powers of two that codes and rows carry, into the
  // [g][row] table, and the bias term: acc[token, row] += sumx[token, g] * B[row, g].
  auto tab_step = [&](uint32_t g0) __attribute__((always_inline)) {
    const bool have = g0 + 8 * h < ng;
    uint4 ab[NPROJ];
#pragma unroll
    for (int p = 0; p < NPROJ; ++p) {
      uint4 S = tab[0][p], B = tab[1][p];
      if (!NG8 && ng >= 8 && g0 + kTabStep > ng) {
        const uint32_t gc = have ? g0 + 8 * h : 0, skip = gc - min(gc, ng - 8);
        S = drop_bf16(S, skip);
        B = drop_bf16(B, skip);
      }
      float* to = s_scale + p * (kTabStep * 32) + 8 * h * 32 + m;
      const uint32_t w[4] = {S.x, S.y, S.z, S.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        to[2 * i * 32] = QmmCodes<BITS>::kScaleMul * bf16_lo(w[i]);
        to[(2 * i + 1) * 32] = QmmCodes<BITS>::kScaleMul * bf16_hi(w[i]);
      }
      // ternary rows store no biases: the bias is -scale (the table pointer is the scale table then)
      ab[p] = a.ternary ? make_uint4(B.x ^ 0x80008000u, B.y ^ 0x80008000u, B.z ^ 0x80008000u, B.w ^ 0x80008000u) : B;
      if (!have) ab[p] = make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int nt = 0; nt < NTA; ++nt)
#pragma unroll
      for (int part = 0; part < 3; ++part) {
        const uint4 sum = s_sum[(nt * 3 + part) * 64 + lane];
#pragma unroll
        for (int p = 0; p < NPROJ; ++p) acc[p][nt] = mfma_bf16(sum, ab[p], acc[p][nt]);
      }
  };
  wait_loads<0>();
  qmm_trace(a, work, 2);

  // Weight codes run kRing pairs of K groups ahead in a ring of registers (the expert's bytes come from HBM); x rows come from L2
  // kStages - 1 pairs ahead, into the stage that was read last.
  Codes now[NPROJ];
  for (uint32_t g0 = 0; g0 < ng; g0 += 2 * kStages) {
#pragma unroll
    for (int uu = 0; uu < kStages; ++uu) {  // pair of K groups g0 + 2uu, g0 + 2uu + 1 in stage uu
      const uint32_t gu = g0 + 2 * uu;
      if (!NG8 && gu >= ng) break;
      wait_loads<kBehind>();  // this wave's part of stage uu is there
      __syncthreads();        // stage uu is complete, the stage before it is no longer read
      // The pair's codes are taken up in front of the request for x: the compiler counts the loads it knows, so behind
      // that request its wait for them would be one for x, too.
#pragma unroll
      for (int p = 0; p < NPROJ; ++p) {
        if constexpr (BITS == 2) now[p] = cur[p][uu % kRing];  // (all four registers of the pair are one load, which leaves below)
        Codes& codes = BITS == 2 ? now[p] : cur[p][uu % kRing];
        codes.settle();
#pragma unroll
        for (auto& w : codes.w) asm volatile("" : "+v"(w));
      }
      if constexpr (FEW) x_request(min(gu + 2 * (kStages - 1), last_pair), (uu + kStages - 1) % kStages, NTA);
      else if (gu + 2 < ng) x_request(gu + 2, uu ^ 1, NTA);
      if constexpr (BITS == 2) {
#pragma unroll
        for (int p = 0; p < NPROJ; ++p) cur[p][uu % kRing].load(1, codes_at(p, gu + 2 * kRing, 1));
      }
      // tables: a step's sums are requested when everybody has read the step's before, its scales and biases a pair ahead
      if (uu == 0 && g0 % kTabStep == 0) tab_step(g0);
      if (uu == 1 && g0 % kTabStep == 0 && g0 + kTabStep < ng) sums_request(g0 + kTabStep, NTA);
      if (uu == kStages - 1 && g0 % kTabStep == kTabStep - 2 * kStages && g0 + 2 * kStages < ng) {
#pragma unroll
        for (int p = 0; p < NPROJ; ++p)
#pragma unroll
          for (int what = 0; what < 2; ++what) tab[what][p] = tab_fetch(what, p, g0 + 2 * kStages);
      }
#pragma unroll
      for (int gi = 0; gi < 2; ++gi) {
        const uint32_t g = gu + gi;
        if (!NG8 && g >= ng) {  // the half pair at the end of an odd number of groups; its loads leave on either way, which keeps the compiler's count of them
          if constexpr (BITS != 2) {
#pragma unroll
            for (int p = 0; p < NPROJ; ++p) cur[p][uu % kRing].load(gi, codes_at(p, gu + 2 * kRing, gi));
          }
          break;
        }
        // ---- matrix core: tmp[token, row] = sum over the group of x * q, times the powers of two kScaleMul takes back
        const uint4* buf = s_x + (2 * uu + gi) * kXGroup;
        uint4 bx[2][4];
#pragma unroll
        for (int nt = 0; nt < NTA; ++nt)
#pragma unroll
          for (int s = 0; s < 4; ++s) bx[nt][s] = buf[nt * 256 + rd_col[s]];
#pragma unroll
        for (int p = 0; p < NPROJ; ++p) {
          const float sc = s_scale[(p * kTabStep + g % kTabStep) * 32 + m];
          f32x16_t tmp[2];
#pragma unroll
          for (int nt = 0; nt < NTA; ++nt)
#pragma unroll
            for (int r = 0; r < 16; ++r) tmp[nt][r] = 0.0f;
          if constexpr (BITS == 2) group_products<BITS, NTA>(now[p], gi, bx, tmp, [](int) {});
          else group_products<BITS, NTA>(cur[p][uu % kRing], gi, bx, tmp, [](int) {});
          // the registers that held this group's codes take their part of the pair two ahead
          // (past the end the last pair is read again: no branch inside the unrolled body)
          if constexpr (BITS != 2) cur[p][uu % kRing].load(gi, codes_at(p, gu + 2 * kRing, gi));
#pragma unroll
          for (int nt = 0; nt < NTA; ++nt)
#pragma unroll
            for (int r = 0; r < RES; ++r) acc[p][nt][r] = __builtin_fmaf(sc, tmp[nt][r], acc[p][nt][r]);
          if constexpr (NT == 1 && !FEW) __builtin_amdgcn_sched_barrier(0);  // one unit at a time: the registers of three waves
        }
      }
      // (the sums are wanted here: without this a pair's products are kept beyond the branches behind it)
#pragma unroll
      for (int p = 0; p < NPROJ; ++p)
#pragma unroll
        for (int nt = 0; nt < NTA; ++nt) asm volatile("" : "+v"(acc[p][nt]));
    }
  }
  if constexpr (FEW) wait_loads<0>();  // (what was requested past the end: the ring is used again, and LDS is given back)
  // (results that do not exist: not kept through the loop)
#pragma unroll
  for (int p = 0; p < NPROJ; ++p)
#pragma unroll
    for (int r = RES; r < 16; ++r) acc[p][0][r] = 0.0f;
  };  // tile_body
  // (the one-projection form keeps to its budget of 168 registers, three waves per SIMD, with one body only)
  using two = std::integral_constant<int, 2>;
  using one = std::integral_constant<int, 1>;
  if constexpr (NT > 1) {
    if (NPROJ == 1 || count > 32) tile_body(two{}, std::integral_constant<int, 16>{});
    else if (count > 8) tile_body(one{}, std::integral_constant<int, 16>{});
    else tile_body(one{}, std::integral_constant<int, 4>{});
  } else {
    if (count > 16) tile_body(one{}, std::integral_constant<int, 16>{});
    else if (count > 8) tile_body(one{}, std::integral_constant<int, 8>{});
    else tile_body(one{}, std::integral_constant<int, 4>{});
  }

  qmm_trace(a, work, 3);
  // ---- epilogue: the lane holds weight row row_base[p] + m for tokens 8j + 4h + i of each 32-token block
  const uint32_t row_raw = (slice * kQmmWaves + wv) * wave_rows;  // past a.rows: this wave has no rows of its own
  const bool far = __any(s_rel[lane & (TT - 1)] != 1.0f || s_act[lane & (TT - 1)] != kRowScale);  // a row out of the ordinary window
  auto bring_back = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4 rel = *reinterpret_cast<const float4*>(s_rel + nt * 32 + 8 * j + 4 * h);
        const float r[4] = {rel.x, rel.y, rel.z, rel.w};
#pragma unroll
        for (int p = 0; p < NPROJ; ++p)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[p][nt][4 * j + i] *= r[i];
      }
  };
  if (a.epi == 0) {
    // SwiGLU, narrowed to bf16 (at the scale of the token's activations), transposed through the (now free) x ring so that a lane stores
    // 16 bytes of one token: [token][32 rows] per wave, the rows of a run of 8 in the
    // (0,4,1,5,2,6,3,7) order phase 2 reads, i.e. rows r and r + 4 share a 32-bit word.
    __syncthreads();  // every wave is past its last read of the ring
    uint32_t* so = reinterpret_cast<uint32_t*>(s_x) + wv * (TT * 16);
    const bool upper = (m >> 2) & 1u;
    const uint32_t dw = ((m & ~7u) >> 1) + (m & 3u);  // word of the row pair (r, r + 4)
    // The activation's variants are chosen outside the element loops (one uniform branch: Maple's or the
    // ordinary one) and, for the ordinary one, by selects -- narrowed or not, clamped or not -- so that the
    // 64 exponentials and reciprocals of a lane are one block of code the compiler can interleave (with
    // the three tests inside the loops every element was a block of its own).
    const bool clamp = a.limit > 0.0f, narrow = a.narrow != 0;
    auto swiglu_block = [&](auto maple_tag, auto far_tag) __attribute__((always_inline)) {
      constexpr bool kMaple = decltype(maple_tag)::value;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        if (nt == 1 && count <= 32) break;  // no route in the second block: its slots are empty
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (j == 1 && count <= 8) break;
          if (NT == 1 && j == 2 && count <= 16) break;
          uint32_t bits[4];
          float scale[4] = {kRowScale, kRowScale, kRowScale, kRowScale};
          if constexpr (decltype(far_tag)::value) {
            const float4 scales = *reinterpret_cast<const float4*>(s_act + nt * 32 + 8 * j + 4 * h);
            scale[0] = scales.x; scale[1] = scales.y; scale[2] = scales.z; scale[3] = scales.w;
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float gv = acc[0][nt][4 * j + i], uv = acc[NPROJ - 1][nt][4 * j + i];
            if constexpr (kMaple) {  // maple_moe.metal:153-164
              bits[i] = f_to_bf16(maple_swiglu(gv, uv) * scale[i]);
            } else {
              const float gr = round_bf16(gv), ur = round_bf16(uv);
              const float g0 = narrow ? gr : gv, u0 = narrow ? ur : uv;
              gv = clamp ? fminf(g0, a.limit) : g0;  // (selects, so that a NaN stays one without a clamp)
              uv = clamp ? fminf(fmaxf(u0, -a.limit), a.limit) : u0;
              bits[i] = f_to_bf16(fast_silu(gv) * uv * scale[i]);
            }
          }
          // lanes m and m ^ 4 trade halves: the lower lane ends with tokens i = 0, 1 of both rows,
          // the upper lane with tokens i = 2, 3
          const uint32_t t01 = bits[0] | (bits[1] << 16), t23 = bits[2] | (bits[3] << 16);
          const uint32_t keep = upper ? t23 : t01;
          const uint32_t got = static_cast<uint32_t>(
              __builtin_amdgcn_ds_swizzle(static_cast<int>(upper ? t01 : t23), 0x101F));  // lane ^ 4
          const uint32_t lo_row = upper ? got : keep, hi_row = upper ? keep : got;
          const uint32_t tok = nt * 32 + 8 * j + 4 * h + (upper ? 2u : 0u);
          so[tok * 16 + dw] = __builtin_amdgcn_perm(hi_row, lo_row, 0x05040100u);
          so[(tok + 1) * 16 + dw] = __builtin_amdgcn_perm(hi_row, lo_row, 0x07060302u);
        }
      }
    };
    if (__builtin_expect(far, 0)) {
      bring_back();
      if (a.maple) swiglu_block(std::true_type{}, std::true_type{});
      else swiglu_block(std::false_type{}, std::true_type{});
    } else if (a.maple) swiglu_block(std::true_type{}, std::false_type{});
    else swiglu_block(std::false_type{}, std::false_type{});
    __syncthreads();
    // the sums of the slice's two groups: two waves' rows each, four threads a (token, group), 16 values of every thread
    {
      const uint32_t ng_out = a.rows / kGroup, part = threadIdx.x & 3u;
#pragma unroll
      for (int it = 0; it < TT / 32; ++it) {
        if (it == 1 && count <= 32) break;
        const uint32_t task = it * 64 + (threadIdx.x >> 2), tok = task >> 1, gi = task & 1u, g = slice * 2 + gi;
        const uint32_t* half = reinterpret_cast<const uint32_t*>(s_x) + (2 * gi + (part >> 1)) * (TT * 16) + tok * 16 + (part & 1u) * 8;
        const uint4 v0 = *reinterpret_cast<const uint4*>(half), v1 = *reinterpret_cast<const uint4*>(half + 4);
        // (each times 2^-64 first: at their scale the sum of large ones would overflow)
        const uint32_t pairs[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        float pair[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) pair[i] = bf16_lo(pairs[i]) * kRowUnscale + bf16_hi(pairs[i]) * kRowUnscale;
        float sum = ((pair[0] + pair[1]) + (pair[2] + pair[3])) + ((pair[4] + pair[5]) + (pair[6] + pair[7]));
        sum = group_sum(sum, 4);
        const uint32_t sl = s_slot[tok];
        if (part == 0 && sl != 0xFFFFFFFFu && g < ng_out)
          store_group_sum(a.out_sums + sl * group_sum_words(ng_out), g, ng_out, sum);
      }
    }
    const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
    for (int it = 0; it < TT / 16; ++it) {
      if (it == 2 && count <= 32) break;
      const uint32_t c = it * 64 + lane, tok = c >> 2, part = c & 3u;
      const uint32_t sl = s_slot[tok];
      const uint4 v = reinterpret_cast<const uint4*>(so)[c];
      if (sl != 0xFFFFFFFFu && (NG8 || row_raw < a.rows))
        *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(out_base) + static_cast<size_t>(sl) * a.rows + row_base[0] +
                                  part * 8) = v;
    }
  } else {
    if (__builtin_expect(far, 0)) bring_back();
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if (nt == 1 && count <= 32) break;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j == 1 && count <= 8) break;
        if (NT == 1 && j == 2 && count <= 16) break;
        const uint4 sl = *reinterpret_cast<const uint4*>(s_slot + nt * 32 + 8 * j + 4 * h);
        const uint32_t slot[4] = {sl.x, sl.y, sl.z, sl.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (slot[i] == 0xFFFFFFFFu) continue;
          const size_t at = static_cast<size_t>(slot[i]) * a.rows;
#pragma unroll
          for (int p = 0; p < NPROJ; ++p) {
            if (p > 0 && !a.pair_rows && !out2_base) break;
            if (!NG8 && row_raw + (a.pair_rows ? 32u * p : 0u) >= a.rows) break;
            uint8_t* ob = (p > 0 && !a.pair_rows) ? out2_base : out_base;  // the second projection's own buffer
            if (a.epi == 1) reinterpret_cast<float*>(ob)[at + row_base[p] + m] = acc[p][nt][4 * j + i];
            else reinterpret_cast<uint16_t*>(ob)[at + row_base[p] + m] = f_to_bf16(acc[p][nt][4 * j + i]);
          }
        }
      }
    }
  }
  qmm_trace(a, work, 4);
}

// (Both parts of a launch read their codes in the form SWAPPED names; without it 2-bit codes have to be tiled.  The dense
// problem beside 2-bit experts is 4-bit and goes through qmm_mixed_kernel: the launchers refuse a 2-bit one beside a tiled pool.)
template <int TT, int BITS, int NPROJ, bool NG8, bool SWAPPED, bool FEW = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(qmm_waves(TT, NPROJ, FEW), qmm_waves(TT, NPROJ, FEW))))
void qmm_kernel(const QmmLaunch launch) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  bool second;
  const QmmPlace at = qmm_place(launch.per_xcd, second);
  const QmmArgs& a = launch.part[second ? 1 : 0];
  qmm_item<TT, BITS, NPROJ, NG8, SWAPPED, FEW>(a, at, smem);
}

// 2-bit (or ternary) routed experts and a 4-bit shared expert in one launch: a launch of its own leaves the shared
// expert's few, long work items on a handful of CUs (large 2-bit layer, 32 tokens: 39 + 25 us beside 127 + 69; 777
// tokens: 53 + 33 beside 388 + 207).
template <int TT, int NPROJ, bool NG8, bool SWAPPED, bool FEW = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(qmm_waves(TT, NPROJ, FEW), qmm_waves(TT, NPROJ, FEW))))
void qmm_mixed_kernel(const QmmLaunch launch) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  bool second;
  const QmmPlace at = qmm_place(launch.per_xcd, second);
  const QmmArgs& a = launch.part[second ? 1 : 0];
  if (a.dense_mode) qmm_item<TT, 4, NPROJ, NG8, true, FEW>(a, at, smem);
  else qmm_item<TT, 2, NPROJ, NG8, SWAPPED, FEW>(a, at, smem);
}

// ---- the same product for a short contraction (K <= 512: the down projections) ----
// With K this short the x tile of a workgroup (64 routes x K bf16 <= 64 KB) stays in LDS whole, so a
// workgroup stages it once and then walks over `slices` consecutive 256-row slices of the weight matrix
// without any further workgroup barrier: the waves run free, each wave's next-slice codes and scale / bias
// words are requested while it still multiplies the current slice, and the stores of a finished slice
// drain while the next one starts.  (qmm_kernel re-stages x through a two-stage ring for every 128 or 256
// rows, four barriers per 8 groups, and pays its set-up -- tile, routes, tables, 3 us -- per slice.)
// A wave owns two consecutive 32-row blocks (64 rows).  Routes past the tile's count repeat the tile's
// last route in every respect, its output slot included: they store the same values to the same place,
// and no store needs a branch.
struct KresLaunch {
  QmmArgs part[2];
  uint32_t per_xcd[2];   // work items of each part on one XCD (grid = 8 * their sum)
  uint32_t slices[2];    // 256-row slices one work item walks (divides rows / 256)
};

// the columns by which run c of 8 values is turned in the x tile
template <int TT> __device__ __forceinline__ uint32_t kres_turn(uint32_t c) { return TT == 32 ? 2 * c : 4 * ((c & 3) >> 1) + 8 * (c >> 2); }

template <int NG> __device__ __forceinline__ uint4 load_groups_bf16(const uint16_t* p) {  // NG bf16, zero-padded to 8
  if constexpr (NG >= 8) {
    return *reinterpret_cast<const uint4*>(p);
  } else if constexpr (NG == 4) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    return make_uint4(v.x, v.y, 0, 0);
  } else {
    return make_uint4(*reinterpret_cast<const uint32_t*>(p), 0, 0, 0);
  }
}

template <int TT, int BITS, int NG, bool SWAPPED>
__device__ __forceinline__ void qmm_kres_item(const QmmArgs& a, const QmmPlace& place, uint32_t n_walk, uint8_t* smem) {
  static_assert(NG == 2 || NG == 4 || NG == 8, "K is 128, 256 or 512");
  constexpr int NT = TT / 32;           // token blocks of a tile
  constexpr uint32_t kXGroup = TT * 8;  // 16-byte pieces of one K group of the x tile
  constexpr uint32_t kGB = QmmCodes<BITS>::kGroupBytes;  // bytes of one K group of one weight row
  using Codes = QmmCodes<BITS, SWAPPED>;
  constexpr int kRing = NG < 4 || TT == 32 ? 1 : 2;  // pairs of groups in flight per row block
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint32_t m = lane & 31, h = lane >> 5;
  const uint32_t items_per_tile = a.rows / (256u * n_walk);
  const uint32_t work = qmm_work(a, place, items_per_tile);
  uint32_t tile_id = work / items_per_tile, slice0 = (work % items_per_tile) * n_walk;
  if (a.dense_mode) {
    if (work >= a.dense_items) return;
    tile_id = a.tile_major ? work / items_per_tile : work % a.dense_tiles;
    slice0 = (a.tile_major ? work % items_per_tile : work / a.dense_tiles) * n_walk;
    if (tile_id >= a.dense_tiles) return;
  }
  qmm_trace(a, work, 0);

  uint32_t expert = 0, pair_start, count;
  if (a.dense_mode) {
    pair_start = tile_id * TT;
    count = min(static_cast<uint32_t>(TT), a.dense_rows - pair_start);
  } else {
    if (work == kNoWork) return;
    const uint4 tv = *reinterpret_cast<const uint4*>(a.tiles + tile_id);
    const Tile t{tv.x, tv.y, tv.z, tv.w};
    expert = t.expert;
    pair_start = t.pair_start;
    count = t.count;
  }
  uint4* s_x = reinterpret_cast<uint4*>(smem);                                  // [NG groups][kXGroup]
  uint32_t* s_slot = reinterpret_cast<uint32_t*>(smem + NG * kXGroup * 16);     // [TT]

  const uint8_t* W;
  const uint16_t* Sp;
  const uint16_t* Bp;
  if (a.dense_mode) {
    W = static_cast<const uint8_t*>(a.dense[0].weights);
    Sp = a.dense[0].scales;
    Bp = a.dense[0].biases;
  } else {
    const uint8_t* blob = a.expert_base + static_cast<size_t>(expert) * a.expert_stride;
    W = blob + a.w_off[0];
    Sp = reinterpret_cast<const uint16_t*>(blob + a.s_off[0]);
    Bp = reinterpret_cast<const uint16_t*>(blob + a.b_off[0]);
  }
  constexpr uint32_t kRowBytes = NG * kGB;
  // the lane's weight row of block p of slice w: row0 + 256 w + 32 p
  const uint32_t row0 = (slice0 * kQmmWaves + wv) * 64 + m;
  const uint32_t pair_stride = a.tiled ? 64u * kGB : 2u * kGB;
  const size_t second = Codes::second(kRowBytes, a.tiled);
  const uint8_t* wrow = W + static_cast<size_t>(row0 - m) * kRowBytes + Codes::lane_offset(lane, kRowBytes, a.tiled);
  const uint16_t* srow = Sp + static_cast<size_t>(row0) * NG;
  const uint16_t* brow = Bp + static_cast<size_t>(row0) * NG;

  // ---- everything issued back to back: codes of the first slice, its scale / bias words, the x tile
  RegArray<Codes, kRing> cur[2];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int u = 0; u < kRing; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i) cur[p][u].load(i, wrow + p * 32 * kRowBytes + u * pair_stride + (i ? second : 0));
  uint4 nS[2], nB[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    nS[p] = load_groups_bf16<NG>(srow + p * 32 * NG);
    nB[p] = load_groups_bf16<NG>(brow + p * 32 * NG);
  }
  // staging: 256 / TT threads a route, kPieces neighbouring runs of 8 values of every group each
  constexpr int kPieces = TT / 32, kPerRoute = 256 / TT;
  const uint32_t st_i = threadIdx.x / kPerRoute, st_q = threadIdx.x % kPerRoute;
  const uint16_t* st_src = a.x + static_cast<size_t>(pair_start + min(st_i, count - 1)) * a.x_stride + st_q * 8 * kPieces;
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
  u32x4_t xv[kPieces * NG];
#pragma unroll
  for (int g = 0; g < kPieces * NG; ++g)
    xv[g] = *reinterpret_cast<const u32x4_t*>(st_src + (g / kPieces) * kGroup + (g % kPieces) * 8);
  uint4 b_term[NT][2];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const uint16_t* sp = a.sumx + static_cast<size_t>(pair_start + min(32 * nt + m, count - 1)) * group_sum_words(NG);
    b_term[nt][0] = *reinterpret_cast<const uint4*>(sp + 8 * h);
    b_term[nt][1] = *reinterpret_cast<const uint4*>(sp + 16);
    if (h) b_term[nt][1] = make_uint4(0, 0, 0, 0);
  }
  // (every wave: lane i holds route i's slot and token)
  uint32_t slot = pair_start + min(lane & (TT - 1), count - 1), token = slot;
  if (!a.dense_mode) {
    const mf_pair pr = a.sorted[slot];
    token = pr.token;
    if (a.epi == 1 || a.epi == 3) slot = pr.token * a.top_k + pr.rank;
  }
  qmm_trace(a, work, 1);

  // ---- x tile into LDS: [group][block of 32 routes][s][h][32 routes, turned by kres_turn] x 16 B, run c = s + 4 h of a group
  {
    // (the 16 lanes that store together hold four runs of 8 of four routes each, or eight of two: the column is rotated so
    // that they hit different bank groups)
    const uint32_t st_nt = st_i >> 5, st_n = st_i & 31;
    uint32_t st_slot[kPieces];
#pragma unroll
    for (int u = 0; u < kPieces; ++u) {
      const uint32_t c = kPieces * st_q + u;
      st_slot[u] = ((st_nt * 4 + (c & 3)) * 2 + (c >> 2)) * 32 + ((st_n + kres_turn<TT>(c)) & 31);
    }
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int u = 0; u < kPieces; ++u) *reinterpret_cast<u32x4_t*>(s_x + g * kXGroup + st_slot[u]) = xv[kPieces * g + u];
    if (threadIdx.x < TT) s_slot[threadIdx.x] = slot;
  }
  uint32_t rd_col[4];
#pragma unroll
  for (int sidx = 0; sidx < 4; ++sidx) rd_col[sidx] = (m + kres_turn<TT>(sidx + 4 * h)) & 31;
  __syncthreads();  // the only workgroup barrier: from here on the waves run on their own
  qmm_trace(a, work, 2);
  const float row_max = a.row_max[token];  // (looked at in front of the first stores)
  // The sums of the lane's routes: K slots 8h..8h+7 of the bias product are groups 0..7 twice, the first parts for
  // h = 0 and the second ones for h = 1, then the third for h = 0 -- two products instead of three.
  // A tile of at most 32 routes fills only the first route block (NTA = 1): the second block, whose routes
  // would all repeat the last route, is left out of the products, the scale multiplies and the stores.
  // (RES = 4 for a tile of at most 8 routes: as in qmm_item)
  auto tile_body = [&](auto nta_c, auto res_c) {
  constexpr int NTA = decltype(nta_c)::value, RES = decltype(res_c)::value;
  for (uint32_t w = 0; w < n_walk; ++w) {
    const uint32_t step = w + 1 < n_walk ? 1u : 0u;  // the last slice requests itself again: no branch around loads
    const uint8_t* wnext = wrow + static_cast<size_t>(step) * 256 * kRowBytes;
    // scale words of this slice; bias operand: the biases, for both halves;
    // ternary rows store no biases: theirs is -scale (the bias pointer is the scale table then)
    uint4 Sv[2], bop[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      Sv[p] = nS[p];
      const uint32_t flip = a.ternary ? 0x80008000u : 0u;
      bop[p] = make_uint4(nB[p].x ^ flip, nB[p].y ^ flip, nB[p].z ^ flip, nB[p].w ^ flip);
    }
    f32x16_t acc[2][NT];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int nt = 0; nt < NTA; ++nt) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[p][nt][r] = 0.0f;
#pragma unroll
        for (int term = 0; term < 2; ++term) acc[p][nt] = mfma_bf16(b_term[nt][term], bop[p], acc[p][nt]);
      }
    // the next slice's scale / bias words (the registers are free again)
    srow += step * 256 * NG;
    brow += step * 256 * NG;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      nS[p] = load_groups_bf16<NG>(srow + p * 32 * NG);
      nB[p] = load_groups_bf16<NG>(brow + p * 32 * NG);
    }
    // x of a group comes out of LDS one group ahead, into the registers the matrix core has just read
    uint4 bx[2][4];
    if (w == 0) {
#pragma unroll
      for (int nt = 0; nt < NTA; ++nt)
#pragma unroll
        for (int s = 0; s < 4; ++s) bx[nt][s] = s_x[((nt * 4 + s) * 2 + h) * 32 + rd_col[s]];
    }
    Codes now[2];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const uint4* nbuf = s_x + ((g + 1) % NG) * kXGroup;  // after the last group: group 0 again, for the next slice
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const uint32_t sw[4] = {Sv[p].x, Sv[p].y, Sv[p].z, Sv[p].w};
        const float sc = QmmCodes<BITS>::kScaleMul * ((g & 1) ? bf16_hi(sw[g >> 1]) : bf16_lo(sw[g >> 1]));
        f32x16_t tmp[2];
#pragma unroll
        for (int nt = 0; nt < NTA; ++nt)
#pragma unroll
          for (int r = 0; r < 16; ++r) tmp[nt][r] = 0.0f;
        constexpr int kPairs = NG / 2;
        Codes& codes = cur[p][(g / 2) % kRing];
        const int ahead = g / 2 + kRing;
        const uint8_t* next_pair = ahead < kPairs ? wrow + p * 32 * kRowBytes + ahead * pair_stride
                                                  : wnext + p * 32 * kRowBytes + (ahead - kPairs) * pair_stride;
        if (g % 2 == 0) {
          if constexpr (BITS == 2) {
            now[p] = codes;
            codes.load(1, next_pair);
            now[p].settle();
          } else codes.settle();
        }
        group_products<BITS, NTA>(BITS == 2 ? now[p] : codes, g % 2, bx, tmp, [&](int s) {
          if (p == 1) {  // both row blocks have read x slot s of this group
            bx[0][s] = nbuf[((0 * 4 + s) * 2 + h) * 32 + rd_col[s]];
            if (NTA > 1) bx[1][s] = nbuf[((1 * 4 + s) * 2 + h) * 32 + rd_col[s]];
          }
        });
        // the registers take the codes kRing pairs on: of this slice, or of the next one
        if constexpr (BITS != 2) codes.load(g % 2, next_pair + (g % 2 ? second : 0));
#pragma unroll
        for (int nt = 0; nt < NTA; ++nt)
#pragma unroll
          for (int r = 0; r < RES; ++r) acc[p][nt][r] = __builtin_fmaf(sc, tmp[nt][r], acc[p][nt][r]);
        // the sums are wanted here, not after the last group: without this the compiler keeps every
        // group's products and adds them up at the end of the slice, out of scratch memory
        if constexpr (NTA > 1) asm volatile("" : "+v"(acc[p][0]), "+v"(acc[p][NT - 1]));
        else asm volatile("" : "+v"(acc[p][0]));
        __builtin_amdgcn_sched_barrier(0);  // one unit at a time: hoisted loads would cost more registers than exist
      }
    }
    if (w + 1 == n_walk) qmm_trace(a, work, 3);
    const float rel = rel_of_scale(a.act_rows ? act_scale(row_max) : row_scale(row_max));
    if (__builtin_expect(__any(rel != 1.0f), 0)) {  // a row out of the ordinary window among the tile's
#pragma unroll
      for (int nt = 0; nt < NTA; ++nt)
#pragma unroll
        for (int r = 0; r < RES; ++r) {
          const float v = __shfl(rel, static_cast<int>(nt * 32 + 8 * (r / 4) + 4 * h + r % 4));
          acc[0][nt][r] *= v;
          acc[1][nt][r] *= v;
        }
    }
    // ---- stores: the lane holds rows row + 32 p for routes 8j + 4h + i of each 32-route block
    const uint32_t row = row0 + w * 256;
    // byte offsets fit 32 bits (the launcher checks): one multiply-add per route, the base stays scalar
    if (a.epi == 1) {
      uint8_t* out = static_cast<uint8_t*>(a.out);
      const uint32_t pitch = a.rows * 4, col = row * 4;
#pragma unroll
      for (int nt = 0; nt < NTA; ++nt) {
#pragma unroll
        for (int j = 0; j < RES / 4; ++j) {
          const uint4 sl = *reinterpret_cast<const uint4*>(s_slot + nt * 32 + 8 * j + 4 * h);
          const uint32_t sl4[4] = {sl.x, sl.y, sl.z, sl.w};
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float* o = reinterpret_cast<float*>(out + (sl4[i] * pitch + col));
            o[0] = acc[0][nt][4 * j + i];
            o[32] = acc[1][nt][4 * j + i];
          }
        }
      }
    } else {
      uint8_t* out = static_cast<uint8_t*>(a.out);
      const uint32_t pitch = a.rows * 2, col = row * 2;
#pragma unroll
      for (int nt = 0; nt < NTA; ++nt) {
#pragma unroll
        for (int j = 0; j < RES / 4; ++j) {
          const uint4 sl = *reinterpret_cast<const uint4*>(s_slot + nt * 32 + 8 * j + 4 * h);
          const uint32_t sl4[4] = {sl.x, sl.y, sl.z, sl.w};
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            uint16_t* o = reinterpret_cast<uint16_t*>(out + (sl4[i] * pitch + col));
            o[0] = f_to_bf16(acc[0][nt][4 * j + i]);
            o[32] = f_to_bf16(acc[1][nt][4 * j + i]);
          }
        }
      }
    }
    wrow = wnext;
  }
  };  // tile_body
  using two = std::integral_constant<int, 2>;
  using one = std::integral_constant<int, 1>;
  if constexpr (NT > 1) {
    if (count > 32) tile_body(two{}, std::integral_constant<int, 16>{});
    else if (count > 8) tile_body(one{}, std::integral_constant<int, 16>{});
    else tile_body(one{}, std::integral_constant<int, 4>{});
  } else {
    if (count > 16) tile_body(one{}, std::integral_constant<int, 16>{});
    else if (count > 8) tile_body(one{}, std::integral_constant<int, 8>{});
    else tile_body(one{}, std::integral_constant<int, 4>{});
  }
  qmm_trace(a, work, 4);
}

template <int TT, int BITS, int NG, bool SWAPPED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(qmm_waves(TT, 2), qmm_waves(TT, 2))))
void qmm_kres_kernel(const KresLaunch launch) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  bool second;
  const QmmPlace at = qmm_place(launch.per_xcd, second);
  const QmmArgs& a = launch.part[second ? 1 : 0];
  const uint32_t walk = launch.slices[second ? 1 : 0];
  qmm_kres_item<TT, BITS, NG, SWAPPED>(a, at, walk, smem);
}

template <int TT, int NG, bool SWAPPED>  // as qmm_mixed_kernel
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(qmm_waves(TT, 2), qmm_waves(TT, 2))))
void qmm_kres_mixed_kernel(const KresLaunch launch) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  bool second;
  const QmmPlace at = qmm_place(launch.per_xcd, second);
  const uint32_t walk = launch.slices[second ? 1 : 0];
  const QmmArgs& a = launch.part[second ? 1 : 0];
  if (a.dense_mode) qmm_kres_item<TT, 4, NG, true>(a, at, walk, smem);
  else qmm_kres_item<TT, 2, NG, SWAPPED>(a, at, walk, smem);
}

// ------------------------------------------------------------------ launches

// Work items of a dense problem that one XCD gets: an eighth, but at least 4 while there are any -- a handful
// of items (the shared expert beside the routed experts of a short batch) runs faster on few XCDs, whose L2
// serves the x rows and weight rows they share, than spread one to an XCD (Qwen shape, 128 tokens: layer 81 us
// against 89 us).
inline uint32_t dense_per_xcd(uint32_t items) { return std::max((items + 7) / 8, std::min(items, 4u)); }
// Whether an XCD should own tiles (and stream all weight rows) or row slices (and stream all of x): whichever
// streams fewer bytes.  code_bits: 4 or 2.
inline int dense_tile_major(uint32_t rows, uint32_t x_rows, int code_bits) {
  return static_cast<uint64_t>(rows) * code_bits <= static_cast<uint64_t>(x_rows) * 16;
}

template <int TT>
hipError_t launch_kres_tiles(hipStream_t s, int bits, const QmmArgs& a, uint32_t tile_slots, const QmmArgs* b,
                             uint32_t b_tile_slots) {
  KresLaunch launch{};
  const bool tiled = a.tiled || (b && b->tiled);  // which form of the code loads: QmmCodes
  if (bits == 2 && tiled && !(a.tiled && (!b || b->tiled))) return hipErrorInvalidValue;
  for (int part = 0; part < (b ? 2 : 1); ++part) {
    QmmArgs& q = launch.part[part];
    q = part ? *b : a;
    const uint32_t slots = part ? b_tile_slots : tile_slots;
    const uint32_t n_slices = q.rows / 256;
    // two slices per work item halve the set-up per slice and still leave several rounds of work items
    // (Qwen shape, 2048 tokens, whole layer: 331 us with one slice, 325 with two, 330 with four, 334 with eight)
    const uint32_t walk = n_slices % 2 == 0 ? 2 : 1;
    launch.slices[part] = walk;
    if (q.dense_mode) {
      q.dense_tiles = slots;
      q.tile_major = dense_tile_major(q.rows, q.dense_rows, part_bits(bits, q));
      q.dense_items = slots * (n_slices / walk);
      launch.per_xcd[part] = dense_per_xcd(q.dense_items);
    } else {
      launch.per_xcd[part] = slots / 8 * (n_slices / walk);
    }
  }
  const dim3 grid(8 * (launch.per_xcd[0] + launch.per_xcd[1])), block(256);
  if (grid.x == 0) return hipSuccess;
  const uint32_t ng = a.kdim / kGroup;
  const size_t lds = static_cast<size_t>(ng) * TT * 128 + TT * 4;
#define MF_KRES_L(...)                                                                                 \
  do {                                                                                                 \
    const hipError_t e = allow_lds<__VA_ARGS__>(lds, kMaxLds);                                         \
    if (e != hipSuccess) return e;                                                                     \
    __VA_ARGS__<<<grid, block, lds, s>>>(launch);                                                      \
  } while (0)
#define MF_KRES(N)                                                                                     \
  do {                                                                                                 \
    if (bits == kMixedBits && tiled) MF_KRES_L(qmm_kres_mixed_kernel<TT, N, false>);                       \
    else if (bits == kMixedBits) MF_KRES_L(qmm_kres_mixed_kernel<TT, N, true>);                            \
    else if (bits == 4 && tiled) MF_KRES_L(qmm_kres_kernel<TT, 4, N, false>);                              \
    else if (bits == 4) MF_KRES_L(qmm_kres_kernel<TT, 4, N, true>);                                        \
    else if (tiled) MF_KRES_L(qmm_kres_kernel<TT, 2, N, false>);                                           \
    else MF_KRES_L(qmm_kres_kernel<TT, 2, N, true>);                                                       \
  } while (0)
  if (ng == 8) MF_KRES(8); else if (ng == 4) MF_KRES(4); else MF_KRES(2);
#undef MF_KRES_L
#undef MF_KRES
  return hipGetLastError();
}

template <int TT>
hipError_t launch_qmm_tiles(hipStream_t s, int bits, const QmmArgs& a, int nproj, uint32_t tile_slots, const QmmArgs* b,
                            uint32_t b_tile_slots, bool few) {
  QmmLaunch launch{};
  const bool tiled = a.tiled || (b && b->tiled);  // which form of the code loads: QmmCodes
  if (bits == 2 && tiled && !(a.tiled && (!b || b->tiled))) return hipErrorInvalidValue;
  bool ng8 = true;
  for (int part = 0; part < (b ? 2 : 1); ++part) {
    QmmArgs& q = launch.part[part];
    q = part ? *b : a;
    const uint32_t slots = part ? b_tile_slots : tile_slots;
    const uint32_t slice_rows = kQmmRows * (q.pair_rows ? nproj : 1), n_slices = (q.rows + slice_rows - 1) / slice_rows;
    if (q.dense_mode) {
      q.dense_tiles = slots;
      q.tile_major = dense_tile_major(q.rows * (q.pair_rows ? 1 : nproj), q.dense_rows, part_bits(bits, q));
      q.dense_items = slots * n_slices * std::max(1u, q.n_win);
      launch.per_xcd[part] = dense_per_xcd(q.dense_items);
    } else {
      launch.per_xcd[part] = slots / 8 * n_slices;
    }
    ng8 = ng8 && (q.n_win > 1 ? q.ng_ld : q.kdim / kGroup) % 8 == 0 && q.rows % slice_rows == 0;
  }
  const dim3 grid(8 * (launch.per_xcd[0] + launch.per_xcd[1])), block(256);
  const size_t lds = qmm_lds_bytes(TT, nproj, TT == kSmallTile && few);
  if (grid.x == 0) return hipSuccess;
#define MF_QMM_L(...)                                                                                  \
  do {                                                                                                 \
    const hipError_t e = allow_lds<__VA_ARGS__>(lds, kMaxLds);                                         \
    if (e != hipSuccess) return e;                                                                     \
    __VA_ARGS__<<<grid, block, lds, s>>>(launch);                                                      \
  } while (0)
#define MF_QMM_FORM(KERNEL, ...)                                                                       \
  do {                                                                                                 \
    if constexpr (TT == kSmallTile) {                                                                  \
      if (few) { MF_QMM_L(KERNEL<__VA_ARGS__, true>); break; }                                         \
    }                                                                                                  \
    MF_QMM_L(KERNEL<__VA_ARGS__, false>);                                                              \
  } while (0)
#define MF_QMM(P, G)                                                                                   \
  do {                                                                                                 \
    if (bits == kMixedBits && tiled) MF_QMM_FORM(qmm_mixed_kernel, TT, P, G, false);                       \
    else if (bits == kMixedBits) MF_QMM_FORM(qmm_mixed_kernel, TT, P, G, true);                            \
    else if (bits == 4 && tiled) MF_QMM_FORM(qmm_kernel, TT, 4, P, G, false);                              \
    else if (bits == 4) MF_QMM_FORM(qmm_kernel, TT, 4, P, G, true);                                        \
    else if (tiled) MF_QMM_FORM(qmm_kernel, TT, 2, P, G, false);                                           \
    else MF_QMM_FORM(qmm_kernel, TT, 2, P, G, true);                                                       \
  } while (0)
  if (nproj == 2) { if (ng8) MF_QMM(2, true); else MF_QMM(2, false); }
  else { if (ng8) MF_QMM(1, true); else MF_QMM(1, false); }
#undef MF_QMM
#undef MF_QMM_FORM
#undef MF_QMM_L
  return hipGetLastError();
}



}  // namespace mf
