// The fused decode layer: one launch per MoE layer.
//
// A grid of one 1024-thread workgroup per CU stays resident for the whole layer:
//
//   A  router logits (one wave per expert row), the scalar shared gate w_sg.x,
//      shared-expert gate/up/activation rows
//      -> every workgroup gathers the logits and selects the top-k itself (cheap and
//         deterministic: rank counting over the logits in LDS, all waves)
//   B  routed gate/up/activation rows of the K selected experts of every token
//   C  the workgroups are split among the tokens, each owns output rows of one: the
//      shared expert's down rows of those rows (-> gated h1, kept in LDS), then the
//      routed down rows.  A wave takes one slot of a unit of rows and weights its values; one
//      thread per row adds a row's K values to h1 in rank order.  With one or two units per
//      workgroup they go round by round, with three and more a wave takes its share of all
//      (unit, slot) pairs, four requested ahead.
//
// Workgroups exchange three small vectors through HBM: logits, shared
// activations, routed activations.  There is no grid barrier.  Every exchanged
// word carries the launch's epoch as a tag (fp32 logits: a 32-bit tag beside the
// value; bf16 activations: a 16-bit tag above the value), producers write them
// with device-coherent stores and go on, consumers poll the data itself with
// device-coherent loads into LDS until every tag they need is current.  This
// costs one store propagation plus about one load round trip per exchange
// (0.55 - 0.65 us between two workgroups, on the same XCD or not);
// a barrier built on a flag or counter costs a store acknowledgement, the flag's
// own propagation, a poll and then the data load.  The epoch is a per-workgroup counter
// in the workspace that every workgroup raises by one per launch, so all
// workgroups agree on it without talking, nothing is reset between launches
// and a captured HIP graph can replay the launch.  One token slot of the
// activation buffers (epoch mod 8, if unused by this launch) is re-tagged per
// launch so that no stale word is ever older than 8 launches: a 16-bit tag can
// never alias.
//
// Producers write whole 64-byte pieces.  Work is dealt in chunks of consecutive rows, one chunk
// per workgroup, the waves' results meet in LDS and one store instruction writes the chunk:
// when neighbouring words of a line are written through by different workgroups (different
// XCDs), the partial-line writes serialise in the memory system and the gather of a 16 KiB
// vector by all workgroups takes 3.3 us instead of 1.4 us (2 KiB: 2.4 against 1.2 us).
//
// Nothing but the router decides which weights are read, so stage C's packed
// codes are requested before the routed activations are polled: their HBM
// latency hides behind the wait.
//
// Consumers spin on data other workgroups produce, so every workgroup of the
// grid has to be resident at once: the launcher never asks for more workgroups
// than CUs and the kernel needs a whole CU (1024 threads, <= 128 VGPRs).  Waits
// are bounded: a poll that does not complete within kSpinLimit tries sets the
// status word, the workgroup writes NaN to the output rows it owns and the grid drains.
#include <algorithm>
#include <type_traits>

#include "mf_device.h"
#include "mf_internal.h"
#include "mf_router.h"

#pragma clang fp contract(off)

namespace mf {

constexpr uint32_t kFusedThreads = 1024;
constexpr uint32_t kFusedWaves = kFusedThreads / kWave;
constexpr uint32_t kSpinLimit = 1u << 17;  // x ~0.6 us per poll
constexpr uint32_t kRouterChunk = 8;       // router rows per workgroup chunk: 8 tagged logits = 64 bytes
constexpr uint32_t kRankCountLimit = 1u << 18;  // T * E * E up to which the top-k counts ranks
constexpr uint32_t kRankWords = 2048;      // ... and T * E it may have then
constexpr uint32_t kWaveSelect = 128;      // experts up to which a wave per token selects instead
constexpr uint32_t kMaxH1 = 2048;          // output rows of one token a workgroup may own

// A lane's step of a row: codes and the table entries of its group as they come from memory.  The entries become
// numbers where they are used (scale(), bias()), behind an empty asm statement: converted next to their load they
// would be waited for there, in front of everything that was to run while they are on their way.  They stay 16 bits
// wide until then for the same reason: widened in front of a loop's branch back, they are waited for at that branch.
template <int BITS> struct Chunk {
  uint4 codes;
  uint16_t sraw, braw;
  __device__ __forceinline__ float scale() const {
    uint16_t r = sraw;
    asm volatile("" : "+v"(r));
    return bf16_to_f(r);
  }
  __device__ __forceinline__ float bias() const {
    if constexpr (BITS == kBitsTernary) return -scale();
    uint16_t r = braw;
    asm volatile("" : "+v"(r));
    return bf16_to_f(r);
  }
};

template <class T>
__device__ __forceinline__ const __attribute__((address_space(1))) T* global_ptr(const void* p) {
  return reinterpret_cast<const __attribute__((address_space(1))) T*>(reinterpret_cast<uint64_t>(p));
}

template <int BITS>
__device__ __forceinline__ Chunk<BITS> load_chunk(const uint8_t* wrow, const uint16_t* srow,
                                                  const uint16_t* brow, uint32_t e0) {
  Chunk<BITS> c;
  // (global loads by name: a base made of two readlanes is a flat address to the compiler, and a flat load in flight is
  // waited for with every LDS read)
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 q = *global_ptr<u32x4>(wrow + static_cast<size_t>(e0) * Store<BITS>::kBits / 8);
  c.codes = make_uint4(q.x, q.y, q.z, q.w);
  c.sraw = *global_ptr<uint16_t>(srow + e0 / kGroup);
  if constexpr (BITS == kBitsTernary) c.braw = 0;
  else c.braw = *global_ptr<uint16_t>(brow + e0 / kGroup);
  return c;
}

// lane partial of one row of N elements against x (16-byte aligned bf16, global
// or LDS); `first` may carry the already loaded chunk of the first step.
template <int BITS>
__device__ __forceinline__ float row_partial(const uint8_t* wrow, const uint16_t* srow,
                                             const uint16_t* brow, const uint16_t* x, uint32_t N,
                                             uint32_t sub, uint32_t lpr, bool have_first,
                                             const Chunk<BITS> first) {
  constexpr uint32_t EPL = Fmt<BITS>::kElemsPer16B;
  float acc = 0.0f;
  for (uint32_t e0 = sub * EPL; e0 < N; e0 += lpr * EPL) {
    // plain scalars, not a struct select: the prefetched chunk must stay in registers
    uint4 codes = first.codes;
    float s = first.scale(), b = first.bias();
    if (!(have_first && e0 == sub * EPL)) {
      codes = load_codes16<true>(wrow + static_cast<size_t>(e0) * Store<BITS>::kBits / 8);
      load_scale_bias<BITS>(srow, brow, e0, s, b);
    }
    const XSlice<BITS> xs = load_xslice<BITS, kXAligned>(x + e0);
    acc = __builtin_fmaf(s, codes_dot<BITS>(codes, xs), acc);
    acc = __builtin_fmaf(b, xs.sum, acc);
  }
  return acc;
}

// gate and up rows of one projection pair sharing the x loads
template <int BITS>
__device__ __forceinline__ void gate_up_partial(const uint8_t* gw, const uint16_t* gs,
                                                const uint16_t* gb, const uint8_t* uw,
                                                const uint16_t* us, const uint16_t* ub,
                                                const uint16_t* x, uint32_t N, uint32_t sub,
                                                uint32_t lpr, float& ga, float& ua) {
  constexpr uint32_t EPL = Fmt<BITS>::kElemsPer16B;
  ga = ua = 0.0f;
  for (uint32_t e0 = sub * EPL; e0 < N; e0 += lpr * EPL) {
    const Chunk<BITS> g = load_chunk<BITS>(gw, gs, gb, e0);
    const Chunk<BITS> u = load_chunk<BITS>(uw, us, ub, e0);
    const XRaw<BITS> xr = load_xraw<BITS>(x + e0);
    issue_fence();
    const XSlice<BITS> xs = make_xslice<BITS>(xr);
    const float gd = codes_dot<BITS>(g.codes, xs), ud = codes_dot<BITS>(u.codes, xs);
    ga = __builtin_fmaf(g.scale(), gd, ga);
    ga = __builtin_fmaf(g.bias(), xs.sum, ga);
    ua = __builtin_fmaf(u.scale(), ud, ua);
    ua = __builtin_fmaf(u.bias(), xs.sum, ua);
  }
}

// n / d for n < 2^31 as a multiplication: the dimensions of most instances are launch arguments, a division by one
// expands to some thirty instructions, and with sixteen waves on a CU an instruction that every wave executes costs 5 ns.
struct FastDiv {
  uint32_t m, add, sh;
};
__device__ __forceinline__ uint32_t fdiv(uint32_t n, const FastDiv& f) { return (__umulhi(n, f.m) + (n & f.add)) >> f.sh; }
static FastDiv make_fastdiv(uint32_t d) {
  if (d <= 1) return FastDiv{0u, ~0u, 0u};
  uint32_t s = 1;
  while (s < 31 && (1u << s) < d) ++s;
  return FastDiv{static_cast<uint32_t>((1ull << (31 + s)) / d + 1), 0u, s - 1};
}

// Launch geometry: what follows from the shape and the number of workgroups (uniform, made on the host once per launch)
struct FusedGeo {
  uint32_t b_per_wg;   // units (rpw rows of one routed slot) a workgroup takes in stage B
  uint32_t c_wgs;      // workgroups that share one token's output rows in stage C
  uint32_t c_units;    // output units of one workgroup: per round (rows form) or in all (units form)
  uint32_t c_rounds;   // rounds (rows form)
  uint8_t lpr_d, lpr_f, lpr_sd, lpr_sf;  // log2 of the lanes per row: rows of D and F (routed), of D and Fs (shared)
  FastDiv E, n_sl, rgf, K, srg, c_wgs_div, rpr, x_runs;
};

struct FusedArgs {
  const uint16_t* router_w;
  const uint8_t* expert_base;
  size_t expert_stride;
  mf_expert_offsets off;
  mf_qtensor sg, su, sd;
  const uint16_t* w_sg;
  // the scalar gate as 8-bit affine codes [1, D] with its scale / bias tables (null: w_sg, or no gate)
  const uint8_t* gq_w;
  const uint16_t* gq_s;
  const uint16_t* gq_b;
  const uint16_t* x;
  uint16_t* y;
  uint16_t* hidden;
  // NORM instances: x is made inside the launch from hidden (+ delta) -- see the kernel's prologue
  const uint16_t* delta;   // [T, D] added to hidden first, or null
  const uint16_t* norm_w;  // [D] RMSNorm weight
  float norm_eps;
  uint32_t xn_off;         // byte offset of the normalised rows [T, D] in LDS
  uint32_t* out_idx;
  float* out_w;
  // exchange buffers (workspace of the handle)
  unsigned long long* t_logits;  // [T, E] (value bits | epoch << 32)
  uint32_t* t_sact;              // [MF_MAX_TOKENS, Fs + 4] (bf16 | tag << 16); word Fs = gate
  uint32_t* t_acts;              // [MF_MAX_TOKENS, K, F]
  uint32_t* epoch;               // one counter per workgroup
  uint32_t* status;
  unsigned long long* trace;     // phase timestamps, 8 per workgroup, or nullptr
  uint32_t D, F, E, K, T, Fs;
  int router_mode;
  float limit;
  int maple;  // MapleMoE's rounding points (mf_moe_config::maple_rounding)
  uint32_t stage_words;  // words of the LDS staging area
  int xprep;             // the routed rows read x from LDS, permuted and summed once per workgroup
  FusedGeo g;
};

__device__ __forceinline__ void store_u64_agent(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// a bounded wait ran out: the status word tells the host, the LDS flag makes this workgroup
// write NaN instead of a result
__device__ __forceinline__ void give_up(uint32_t* status, uint32_t* s_fail, uint32_t lane) {
  if (lane == 0) {
    store_u32_agent(status, 1u);
    *s_fail = 1u;
  }
}

// phase trace: the 100 MHz wall clock at every stage boundary, thread 0 of each workgroup
__device__ __forceinline__ void trace_mark(const FusedArgs& a, uint32_t slot) {
  if (a.trace && threadIdx.x == 0) a.trace[blockIdx.x * 8 + slot] = wall_clock64();
}

// Shape specialisation (the reference's FC_MOE_D / FC_MOE_F / FC_MOE_TOP_K function
// constants, moe.metal:13-16): a StaticShape turns the dimensions it names into
// compile-time constants (kDyn leaves one to the arguments), which unrolls the row
// loops and removes most of the control flow -- the launch executes each
// instruction once per wave, so code size is instruction-fetch latency.
// RuntimeShape reads every dimension from the arguments and handles everything else.
// kGiven: the routing is the caller's (written by an earlier launch, e.g. a family router): the kernel
// has no router rows, no logits exchange and no top-k, and reads indices and weights instead of
// writing them.  A compile-time property, so the kernels that route keep their code as it is.
constexpr uint32_t kDyn = 0xFFFFFFFFu;  // a dimension read from the arguments
// kAnyE: the number of experts need not be a multiple of four (an instance of its own: the few instructions more cost the
// others 4 % of a small layer)
template <bool GIVEN = false, bool ANYE = false>
struct RuntimeShapeT {
  static constexpr bool kStatic = false, kGiven = GIVEN, kAnyE = ANYE;
  static constexpr uint32_t D = kDyn, F = kDyn, E = kDyn, K = kDyn, T = kDyn, Fs = kDyn;
  static constexpr uint32_t Mode = kDyn, Maple = kDyn, NoLimit = 0, XPrep = kDyn;
};
using RuntimeShape = RuntimeShapeT<false>;
// MODE_ / MAPLE_: the router mode and the Maple rounding flag as literals (kDyn: from the arguments);
// NOLIMIT_ = 1: the layer has no SwiGLU clamp; XPREP_ = 1: the x slices are kept in LDS.
template <uint32_t D_, uint32_t F_, uint32_t E_, uint32_t K_, uint32_t T_, uint32_t Fs_, bool GIVEN = false,
          uint32_t MODE_ = kDyn, uint32_t MAPLE_ = kDyn, uint32_t NOLIMIT_ = 0, uint32_t XPREP_ = kDyn>
struct StaticShape {
  static constexpr bool kStatic = D_ != kDyn && F_ != kDyn && E_ != kDyn && K_ != kDyn && T_ != kDyn && Fs_ != kDyn;
  static constexpr bool kGiven = GIVEN, kAnyE = E_ != kDyn && E_ % 4 != 0;
  static constexpr uint32_t D = D_, F = F_, E = E_, K = K_, T = T_, Fs = Fs_;
  static constexpr uint32_t Mode = MODE_, Maple = MAPLE_, NoLimit = NOLIMIT_, XPrep = XPREP_;
};

// rows one wave takes per step when a row has n elements (compile-time twin of
// 64 >> lanes_per_row_log2_dev)
constexpr uint32_t static_rows_per_wave(uint32_t n, uint32_t elems_per_lane) {
  uint32_t need = (n + elems_per_lane - 1) / elems_per_lane, lanes = 1;
  while (lanes < need && lanes < 64) lanes *= 2;
  return 64u / lanes;
}

// The launch geometry as one function of the shape, for the host (every instance) and at compile time (the one-token
// instances with literal dimensions, which the launcher picks for kStaticWgs workgroups only).
constexpr uint32_t kStaticWgs = 256;

// Units of stage B one workgroup takes: an equal share, in whole 64-byte pieces of the exchanged activations (one
// writer per memory line) while a wave then has one unit at most (1024 x 384, 48 experts, one token: 11.8 us, in 32-byte
// pieces 11.9), else in 16-byte pieces: the 2816 x 704 layer would have 176 of 256 workgroups at work with 32 units each
// (its router, layer and MLP 33.2 us, with 24 units on 235 workgroups 31.5; 1600 x 960, 100 experts, top 5: 19.6 / 18.1).
constexpr uint32_t fused_b_per_wg(uint32_t epl, uint32_t d, uint32_t f, uint32_t k, uint32_t t, uint32_t n_wg) {
  const uint32_t rpw = static_rows_per_wave(d, epl);
  const uint32_t n = t * k * ((f + rpw - 1) / rpw), piece = rpw < 16 ? 16 / rpw : 1;
  const uint32_t share = (n + n_wg - 1) / n_wg, whole = (share + piece - 1) / piece * piece;
  if (whole <= kFusedWaves) return whole;
  const uint32_t part = rpw < 4 ? 4 / rpw : 1;
  return (share + part - 1) / part * part;
}

// How stage C deals a token's output rows.  Rows form: a unit's K slots on K waves, their values meet in LDS -- all
// waves work although a workgroup has only a unit or two.  Units form: the (unit, slot) pairs of all units go to the
// waves in turn with four requested ahead, and all values meet once -- from three units per workgroup on (large 2-bit
// layer, one token: 8 units; most shapes at several tokens), while a row is one step of 64 lanes.  (With a unit's slots on one wave, one after the other, eleven waves of sixteen
// worked at five tokens of the Qwen shape, and six of sixteen at one token of the 2816 x 704 layer.)  Launch, us, before
// and now: Qwen shape 16.0 / 15.2 (two tokens), 26.7 / 26.2 (five), 32.2 / 31.1 (six); large 2-bit layer 52.3 / 50.2
// (two), 145 / 138 (eight); ternary layer of 256 experts 18.4 / 17.3 (four).
struct FusedSplit {
  bool by_units;
  uint32_t wgs, units, rounds;  // workgroups per token; units per workgroup (rows form: and round); rounds
};
constexpr FusedSplit fused_split(uint32_t epl, uint32_t d, uint32_t f, uint32_t k, uint32_t t, uint32_t n_wg, bool units_fit = true) {
  const uint32_t rpw = static_rows_per_wave(f, epl), rg = (d + rpw - 1) / rpw, wgs = n_wg / t;
  const uint32_t share = (rg + wgs - 1) / wgs;
  const bool by_units = units_fit && share >= 3 && f <= 64 * epl;
  const uint32_t per_round = kFusedWaves / k < share ? kFusedWaves / k : share;
  const uint32_t units = by_units ? share : per_round;
  return FusedSplit{by_units, wgs, units, by_units ? 1 : (rg + wgs * units - 1) / (wgs * units)};
}

// stage A: waves that poll for n2 16-byte pieces of tagged logits, and waves that build n slices of x
__host__ __device__ __forceinline__ uint32_t fused_poll_waves(uint32_t n2) {
  const uint32_t w = (n2 + kWave - 1) / kWave;
  return w < 8 ? w : 8;
}
// (a run: up to 64 slices of one token, on the lanes of a wave, or all of them on half a wave's where that holds them)
__host__ __device__ __forceinline__ uint32_t fused_x_runs(uint32_t n_sl) { return (n_sl + kWave - 1) / kWave; }
__host__ __device__ __forceinline__ uint32_t fused_slice_waves(uint32_t t, uint32_t n_sl, uint32_t n_poll) {
  const uint32_t w = n_sl <= kWave / 2 ? (t + 1) / 2 : t * fused_x_runs(n_sl);
  return w < kFusedWaves - n_poll - 4 ? w : kFusedWaves - n_poll - 4;
}

template <int BITS, int SBITS, class S, bool NORM, bool UNITS>
__global__ __launch_bounds__(kFusedThreads) void fused_decode_kernel(const FusedArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const uint32_t D = S::D != kDyn ? S::D : a.D, F = S::F != kDyn ? S::F : a.F;
  const uint32_t E = S::E != kDyn ? S::E : a.E, K = S::K != kDyn ? S::K : a.K;
  const uint32_t T = S::T != kDyn ? S::T : a.T, Fs = S::Fs != kDyn ? S::Fs : a.Fs;
  const int router_mode = S::Mode != kDyn ? static_cast<int>(S::Mode) : a.router_mode;
  const bool maple = S::Maple != kDyn ? S::Maple != 0u : a.maple != 0;
  const float limit = S::NoLimit ? 0.0f : a.limit;
  const bool xprep = S::XPrep != kDyn ? S::XPrep != 0u : a.xprep != 0;
  // LDS carve-up (the launcher sizes it with fused_lds_bytes)
  uint32_t* s_idx = reinterpret_cast<uint32_t*>(smem);                 // [8*8]
  float* s_w = reinterpret_cast<float*>(smem + 256);                    // [8*8]
  float* s_sc = reinterpret_cast<float*>(smem + 512);                   // [8*8] selected scores
  uint32_t* s_flag = reinterpret_cast<uint32_t*>(smem + 768);           // [8] token has a non-finite logit
  uint32_t* s_fail = reinterpret_cast<uint32_t*>(smem + 800);           // a bounded wait gave up; [1]: selection fallback
  float* s_v = reinterpret_cast<float*>(smem + 1024);                   // [16][64]
  float* s_h1 = reinterpret_cast<float*>(smem + 1024 + 4096);           // [kMaxH1]
  uint32_t* s_rank = reinterpret_cast<uint32_t*>(smem + 1024 + 4096 + kMaxH1 * 4);  // [kRankWords]
  uint8_t* dyn = smem + 1024 + 4096 + kMaxH1 * 4 + kRankWords * 4;
  const uint32_t Ep = S::kAnyE ? (E + 3) & ~3u : E;  // logits per token in LDS: the selection reads them four at a time, -inf behind the last
  float* s_lg = reinterpret_cast<float*>(dyn);                          // [MF_MAX_TOKENS][Ep]
  uint32_t* s_sact = reinterpret_cast<uint32_t*>(dyn + MF_MAX_TOKENS * Ep * 4);  // [(Fs+4)/2]
  uint32_t* s_acts = s_sact + (((Fs + 4) / 2 + 3) & ~3u);               // [K*F/2], 16-byte aligned
  // the routed activations as 16-byte blocks in the order of the x slices: block q of slice sl at q * act_ld + sl (an
  // odd stride: the lanes that write a slice's blocks and those that read one block of many slices both spread over
  // the banks; row by row the readers' slices lay 64 or 128 bytes apart, four or eight of 16 lanes on one bank)
  const uint32_t act_ld = (K * F / Fmt<BITS>::kElemsPer16B) | 1u;
  uint32_t* s_stage = s_acts + Fmt<BITS>::kElemsPer16B / 8 * 4 * act_ld;  // chunk staging, a.stage_words
  const uint32_t sact_stride = Fs + 4;  // words per token in t_sact

  const uint32_t lane = threadIdx.x & 63;
  // the wave index as a scalar: what derives from it (rows, experts, base addresses) is then
  // computed once per wave by the scalar unit instead of per lane
  const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t G = S::kStatic ? kStaticWgs : gridDim.x, wg = blockIdx.x;
  constexpr FusedSplit kSplit =
      S::kStatic ? fused_split(Fmt<BITS>::kElemsPer16B, S::D, S::F, S::K, 1, kStaticWgs) : FusedSplit{UNITS, 0, 0, 0};
  static_assert(!S::kStatic || (S::T == 1 && kSplit.by_units == UNITS), "an instance with every dimension literal has the form of its shape");
  // x slices of the routed rows, built once per workgroup (when a.xprep)
  constexpr uint32_t kEPL = Fmt<BITS>::kElemsPer16B;
  const uint32_t n_sl = D / kEPL;  // slices per token (the last partial slice, if any, is not kept)
  uint4* s_xq = reinterpret_cast<uint4*>(s_stage + a.stage_words);
  float* s_xsum = reinterpret_cast<float*>(s_xq + T * (XSlice<BITS>::kPairs / 4) * n_sl);

  // The launch epoch comes out of device memory (a captured graph replays the launch with the same
  // arguments) and is first needed when a result is tagged.  The load is requested here; every
  // user takes the value through epoch_now(), whose empty asm statement keeps the compiler from
  // waiting for it any earlier -- in particular not before the first rows' loads are out.
  uint32_t epoch_lane_off = 0;
  asm volatile("" : "+v"(epoch_lane_off));
  const uint32_t epoch_raw =
      __hip_atomic_load(&a.epoch[wg] + epoch_lane_off, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  auto epoch_now = [&]() __attribute__((always_inline)) {
    uint32_t e = epoch_raw;
    asm volatile("" : "+v"(e));
    return e + 1u;
  };
  trace_mark(a, 0);
  // NORM: the step in front of the layer inside the launch (RealForwardRunner.swift:2799-2808: hidden += delta,
  // x = RMSNorm(hidden) * weight).  Every workgroup makes the normalised rows for itself, in LDS, with the
  // instruction order of residual_rmsnorm_kernel (256 threads per row, element i + 256 j on thread i, fmaf
  // chain, neighbour-first butterfly, (s0 + s1) + (s2 + s3)), so x has the bits of that launch; everything
  // below reads x from LDS.  hidden itself is written once, at the end, by the workgroup that owns the
  // element: bf16(bf16(hidden + delta) + y).  A workgroup that other workgroups do not wait for (no row of
  // stages A and B) may read hidden while it is being written: its x then is of no consequence.
  const uint16_t* xin = a.x;
  // (NORM) the first router row of a wave: its weights are requested ahead of the norm, which has a memory
  // round trip of its own to wait for -- rows of up to 2048 elements, four chunks per lane
  uint4 pre_w[4];
  bool pre_router = false;
  if constexpr (NORM && !S::kGiven) {
    const uint32_t row = wg * kRouterChunk + wv;
    pre_router = D <= 2048 && D % 8 == 0 && wv < kRouterChunk && row < E * T;
    if (pre_router) {
      const uint16_t* wr = a.router_w + static_cast<size_t>(row % E) * D;
#pragma unroll
      for (int sidx = 0; sidx < 4; ++sidx) {
        const uint32_t c = lane + sidx * kWave;
        pre_w[sidx] = c < D / 8 ? load_x8<true>(wr + c * 8) : make_uint4(0, 0, 0, 0);
      }
    }
  }
  if constexpr (NORM) {
    uint16_t* s_xn = reinterpret_cast<uint16_t*>(smem + a.xn_off);
    float* s_part = s_v;  // [token][4 waves of its row]; s_v is free until stage C
    // The rows come in as 16-byte pieces, every piece once per workgroup (piece c on thread c % 1024), with
    // the matching piece of delta and of the weights in the same round trip; bf16(hidden + delta) goes to
    // LDS, the sums read it from there in the norm kernel's order, and each piece's owner scales it in
    // place.  (Element by element from global memory, the delta loads sat behind a branch each: eight
    // round trips in a row, 3.9 us before the first row could start.)
    constexpr uint32_t kPc = MF_MAX_TOKENS * 4096 / 8 / kFusedThreads;  // pieces per thread at most
    const uint32_t ppr = D / 8, n_pc = T * ppr;
    const uint16_t* dsrc = a.delta ? a.delta : a.hidden;  // (always a valid address: no branch around the load)
    const bool has_delta = a.delta != nullptr;
    uint4 hv[kPc], nv[kPc];
#pragma unroll
    for (uint32_t p = 0; p < kPc; ++p) {
      const uint32_t c = threadIdx.x + kFusedThreads * p;
      if (c < n_pc) {
        const uint4 h4 = load_x8<true>(a.hidden + static_cast<size_t>(c) * 8);
        const uint4 d4 = load_x8<true>(dsrc + static_cast<size_t>(c) * 8);
        nv[p] = load_x8<true>(a.norm_w + static_cast<size_t>(c % ppr) * 8);
        const uint32_t hw[4] = {h4.x, h4.y, h4.z, h4.w}, dw[4] = {d4.x, d4.y, d4.z, d4.w};
        uint32_t o[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint16_t lo = f_to_bf16(bf16_to_f(static_cast<uint16_t>(hw[q] & 0xffffu)) +
                                        bf16_to_f(static_cast<uint16_t>(dw[q] & 0xffffu)));
          const uint16_t hi = f_to_bf16(bf16_to_f(static_cast<uint16_t>(hw[q] >> 16)) +
                                        bf16_to_f(static_cast<uint16_t>(dw[q] >> 16)));
          o[q] = has_delta ? (static_cast<uint32_t>(lo) | (static_cast<uint32_t>(hi) << 16)) : hw[q];
        }
        hv[p] = make_uint4(o[0], o[1], o[2], o[3]);
        *reinterpret_cast<uint4*>(s_xn + static_cast<size_t>(c) * 8) = hv[p];
      }
    }
    __syncthreads();
    const uint32_t grp = threadIdx.x >> 8, ti = threadIdx.x & 255u;
    for (uint32_t tok0 = 0; tok0 < T; tok0 += 4) {
      const uint32_t tok = tok0 + grp;
      float acc = 0.0f;
      if (tok < T) {
#pragma unroll
        for (uint32_t j = 0; j < 16; ++j) {  // D <= 4096
          const uint32_t i = ti + 256u * j;
          if (i < D) {
            const float v = bf16_to_f(s_xn[static_cast<size_t>(tok) * D + i]);
            acc = __builtin_fmaf(v, v, acc);
          }
        }
      }
      acc = wave_sum(acc);
      if (lane == 0 && tok < T) s_part[4 * tok + (wv & 3u)] = acc;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t p = 0; p < kPc; ++p) {
      const uint32_t c = threadIdx.x + kFusedThreads * p;
      if (c < n_pc) {
        const uint32_t tok = c / ppr;
        const float total = (s_part[4 * tok] + s_part[4 * tok + 1]) + (s_part[4 * tok + 2] + s_part[4 * tok + 3]);
        const float inv = 1.0f / __builtin_sqrtf(total / static_cast<float>(D) + a.norm_eps);
        const uint32_t hw[4] = {hv[p].x, hv[p].y, hv[p].z, hv[p].w}, nw4[4] = {nv[p].x, nv[p].y, nv[p].z, nv[p].w};
        uint32_t o[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint16_t lo = f_to_bf16(bf16_to_f(static_cast<uint16_t>(hw[q] & 0xffffu)) * inv *
                                        bf16_to_f(static_cast<uint16_t>(nw4[q] & 0xffffu)));
          const uint16_t hi = f_to_bf16(bf16_to_f(static_cast<uint16_t>(hw[q] >> 16)) * inv *
                                        bf16_to_f(static_cast<uint16_t>(nw4[q] >> 16)));
          o[q] = static_cast<uint32_t>(lo) | (static_cast<uint32_t>(hi) << 16);
        }
        *reinterpret_cast<uint4*>(s_xn + static_cast<size_t>(c) * 8) = make_uint4(o[0], o[1], o[2], o[3]);
      }
    }
    __syncthreads();
    xin = s_xn;
    trace_mark(a, 7);
  }
  // ranks are counted over all experts when that is cheap enough, else one wave per token sorts
  const bool rank_count = !S::kGiven && T * E * E <= kRankCountLimit && T * Ep <= kRankWords;
  // Who does what while the logits are on their way: the top waves poll for them (n_poll waves),
  // the waves below those build the x slices, the bottom waves have the rows of stage A.
  const uint32_t n2 = S::kGiven ? 0 : (S::kAnyE ? T * E + 1 : T * E) / 2;  // 16-byte pieces of tagged logits
  const uint32_t n_poll = fused_poll_waves(n2), n_xw = fused_slice_waves(T, n_sl, n_poll);
  const uint32_t x_runs = fused_x_runs(n_sl);

  // The scales of every token's activations and x.  Tokens of several runs: the runs' largest magnitudes, times kRowScale, first, and the
  // scales behind the requests of stage B.  (s_v is free until stage C.)
  float* s_scale = s_v;
  float* s_xscale = s_v + MF_MAX_TOKENS;
  float* s_most = s_v + 2 * MF_MAX_TOKENS;

  // ------------------------------------------------------------- stage A
  // Router rows are on the critical path and their logits are gathered by everybody: they go in
  // chunks of kRouterChunk consecutive rows to the first workgroups (a wave each; the chunk
  // leaves as one 64-byte store).  The shared expert's rows and the scalar-gate rows are needed
  // much later; they are dealt one at a time over the waves of the other workgroups (their
  // dot products are vector-ALU work: spread thin, they cost no workgroup more than a row or two).
  {
    const uint32_t lpr_log2 = S::D != kDyn ? lanes_per_row_log2_dev(D, Fmt<SBITS>::kElemsPer16B) : a.g.lpr_sd;
    const uint32_t lpr = 1u << lpr_log2, rpw = 64u >> lpr_log2;
    const uint32_t n_rows_r = S::kGiven ? 0 : E * T;
    const uint32_t n_rc = (n_rows_r + kRouterChunk - 1) / kRouterChunk;
    unsigned long long* s_stage64 = reinterpret_cast<unsigned long long*>(s_stage);
    for (uint32_t ci = wg; ci < n_rc; ci += G) {
      const uint32_t row = ci * kRouterChunk + wv;
      if (wv < kRouterChunk && row < n_rows_r) {
        const uint32_t tok = S::E != kDyn ? row / E : fdiv(row, a.g.E), e = row - tok * E;
        float v;
        if (NORM && pre_router && ci == wg) {  // the weights are here already: dot_bf16_row's products in its order
          const uint16_t* xr = xin + static_cast<size_t>(tok) * D;
          float acc = 0.0f;
#pragma unroll
          for (int sidx = 0; sidx < 4; ++sidx) {
            const uint32_t c = lane + sidx * kWave;
            if (c < D / 8) acc = fma_chunk_bf16(pre_w[sidx], load_x8<true>(xr + c * 8), acc);
          }
          v = wave_sum(acc);
        } else {
          v = dot_bf16_row(a.router_w + static_cast<size_t>(e) * D, xin + static_cast<size_t>(tok) * D, D, lane);
        }
        if (lane == 0) s_stage64[wv] = (static_cast<unsigned long long>(epoch_now()) << 32) | __float_as_uint(v);
      }
      __syncthreads();
      if (wv == 0 && lane < kRouterChunk && ci * kRouterChunk + lane < n_rows_r)
        store_u64_agent(&a.t_logits[ci * kRouterChunk + lane], s_stage64[lane]);
      if (ci + G < n_rc) __syncthreads();  // the staging words are reused
    }
    const uint32_t skip = n_rc < G ? n_rc : 0;  // workgroups [0, skip) had router rows
    const uint32_t n_gate = (Fs && (a.w_sg || a.gq_w)) ? T : 0;
    const uint32_t srg = (Fs + rpw - 1) >> (6 - lpr_log2);
    const uint32_t n_items = n_gate + T * srg;
    const uint32_t Gs = G - skip;
    for (uint32_t item = wg >= skip ? wv * Gs + (wg - skip) : n_items; item < n_items; item += kFusedWaves * Gs) {
      if (item < n_gate) {
        const uint32_t tok = item;
        const float v = a.gq_w ? dot_q8_row(a.gq_w, a.gq_s, a.gq_b, xin + static_cast<size_t>(tok) * D, D, lane, true)
                               : dot_bf16_row(a.w_sg, xin + static_cast<size_t>(tok) * D, D, lane);
        if (lane < 4)  // the gate rides behind the token's shared activations
          store_u32_agent(&a.t_sact[static_cast<size_t>(tok) * sact_stride + Fs + lane],
                          (lane == 0 ? static_cast<uint32_t>(f_to_bf16(v)) : 0u) | (epoch_now() << 16));
      } else {
        const uint32_t it = item - n_gate;
        // (no shared expert: this branch is never taken)
        const uint32_t tok = S::Fs != kDyn && S::D != kDyn ? (srg ? it / srg : 0u) : fdiv(it, a.g.srg);
        const uint32_t row = (it - tok * srg) * rpw + (lane >> lpr_log2);
        const uint32_t sub = lane & (lpr - 1);
        const bool ok = row < Fs;
        const size_t r = ok ? row : 0;
        const uint32_t ng = D / kGroup;
        const size_t rb = static_cast<size_t>(D) * Store<SBITS>::kBits / 8;
        float ga = 0.0f, ua = 0.0f;
        if (ok)
          gate_up_partial<SBITS>(static_cast<const uint8_t*>(a.sg.weights) + r * rb,
                                 a.sg.scales + r * ng, a.sg.biases + r * ng,
                                 static_cast<const uint8_t*>(a.su.weights) + r * rb,
                                 a.su.scales + r * ng, a.su.biases + r * ng,
                                 xin + static_cast<size_t>(tok) * D, D, sub, lpr, ga, ua);
        const float g = group_sum(ga, static_cast<int>(lpr));
        const float u = group_sum(ua, static_cast<int>(lpr));
        if (ok && sub == 0) {
          // dequant_int4.metal:240-245: gate and up narrowed before the activation
          const float rg = round_bf16(g), ru = round_bf16(u);
          store_u32_agent(&a.t_sact[static_cast<size_t>(tok) * sact_stride + row],
                          static_cast<uint32_t>(f_to_bf16(mf_silu(rg) * ru)) | (epoch_now() << 16));
        }
      }
    }
    // the x slices of the routed rows, and the scales: a wave takes whole runs, two tokens' where half of its lanes hold one
    // (us a layer, a wave a token before: 1024 x 384, two tokens 13.8 -> 13.1; 256 ternary experts of 512, eight 24.0 -> 22.9; large 2-bit layer, eight
    // 122 -> 120.7; 2816 x 704, two 40.6 -> 40.1)
    if (wv + n_poll + n_xw >= kFusedWaves && wv + n_poll < kFusedWaves) {
      const uint32_t half = n_sl <= kWave / 2 ? 1u : 0u, run_lane = lane & ((kWave >> half) - 1), runs = T * x_runs;
      for (uint32_t r0 = (wv + n_poll + n_xw - kFusedWaves) << half; r0 < runs; r0 += n_xw << half) {
        const uint32_t run = r0 + (lane >> (6 - half));
        const uint32_t tok = S::T == 1 ? 0u : S::D != kDyn ? run / x_runs : fdiv(run, a.g.x_runs);
        const uint32_t sl = (run - tok * x_runs) * kWave + run_lane;
        float largest = 0.0f;
        if (run < runs && sl < n_sl) {
          const XSlice<BITS> xs = load_expert_x<BITS, true>(xin + static_cast<size_t>(tok) * D + sl * kEPL, kRowScale, &largest);
          if (xprep) store_xslice_lds<BITS>(s_xq, s_xsum, tok, n_sl, sl, xs);
        }
        const float2 most = half_wave_max(largest);
        largest = half ? (lane < kWave / 2 ? most.x : most.y) : fmaxf(most.x, most.y);
        if (run < runs && run_lane == 0) {
          if (x_runs == 1) {
            s_scale[tok] = act_scale(largest);
            s_xscale[tok] = row_scale(largest);
          } else {
            s_most[run] = largest;
          }
        }
      }
    }
  }
  const uint32_t epoch = epoch_now();
  const uint32_t tag16 = epoch & 0xFFFFu;
  for (uint32_t i = threadIdx.x; i < kRankWords; i += kFusedThreads) s_rank[i] = 0u;
  if (threadIdx.x < MF_MAX_TOKENS * MF_MAX_TOPK) {
    s_idx[threadIdx.x] = 0u;
    s_sc[threadIdx.x] = -__builtin_inff();
  }
  if (threadIdx.x < MF_MAX_TOKENS + 2) s_flag[threadIdx.x] = 0u;  // + s_fail and the selection's fallback flag behind it
  if (S::kAnyE && threadIdx.x < T * 4) {
    const uint32_t i = E + (threadIdx.x & 3u);
    if (i < Ep) s_lg[(threadIdx.x >> 2) * Ep + i] = -__builtin_inff();
  }
  {
    // keep every word of the activation buffers recently tagged (see the top)
    const uint32_t ts = epoch % MF_MAX_TOKENS;
    if (ts >= T) {
      const uint32_t gtid = wg * kFusedThreads + threadIdx.x, gthreads = G * kFusedThreads;
      for (uint32_t i = gtid * 4; i < K * F; i += gthreads * 4)  // K * F is a multiple of 64
        store_u32x4_agent(&a.t_acts[static_cast<size_t>(ts) * K * F + i], tag16 << 16);
      for (uint32_t i = gtid; i < (Fs ? sact_stride : 0); i += gthreads)
        store_u32_agent(&a.t_sact[static_cast<size_t>(ts) * sact_stride + i], tag16 << 16);
    }
  }
  trace_mark(a, 1);

  // ------------------------------------------------------- logits, top-k
  if constexpr (!S::kGiven) {
    // every lane takes two tagged logits
    if (wv + n_poll >= kFusedWaves) {
      for (uint32_t p0 = (kFusedWaves - 1 - wv) * kWave; p0 < n2; p0 += n_poll * kWave) {
        const uint32_t p = p0 + lane;
        const bool in = p < n2;
        uint4 v = make_uint4(0, epoch, 0, epoch);
        for (uint32_t spins = 0;; ++spins) {
          if (in) v = load_u32x4_agent(a.t_logits + 2 * p);
          if (__all(!in || (v.y == epoch && (v.w == epoch || (S::kAnyE && 2 * p + 1 == T * E))))) break;  // (an odd number: half a piece)
          if (spins > kSpinLimit) {
            give_up(a.status, s_fail, lane);
            break;
          }
          __builtin_amdgcn_s_sleep(1);
        }
        if (in) {  // rank counting wants no NaN among the scores it compares
          const bool clean = rank_count && router_mode == 0;
          uint32_t at[2] = {2 * p, 2 * p + 1};
          if constexpr (S::kAnyE) {
            at[0] += fdiv(at[0], a.g.E) * (Ep - E);
            at[1] += fdiv(at[1], a.g.E) * (Ep - E);
          }
          s_lg[at[0]] = clean ? score_or_ninf(__uint_as_float(v.x)) : __uint_as_float(v.x);
          if (!S::kAnyE || 2 * p + 1 < T * E) s_lg[at[1]] = clean ? score_or_ninf(__uint_as_float(v.z)) : __uint_as_float(v.z);
        }
      }
    }
    __syncthreads();
    trace_mark(a, 2);
    if (rank_count && router_mode == 0 && E <= kWaveSelect && 4 * K <= E) {
      // Few experts: a wave per token takes the best K times in registers, without a barrier before its result.  Layer of 1024 x 384, us,
      // counted / by waves, one and eight tokens: 48 experts, top 4 12.1 / 11.5, 17.5 / 15.5, top 8 12.7 / 12.6, 21.6 / 20.3; 96, top 4
      // 12.7 / 11.6, 20.4 / 15.6; 128, top 4 12.5 / 11.6, 17.4 / 15.7, top 8 13.5 / 12.8, 21.9 / 20.4.  Counting stays where there is
      // little to count (30 experts, top 8, eight tokens: 38.5, by waves 40.2) and behind a full softmax, whose wave would do
      // both (64 experts: 12.0, 12.6).  The line is where two logits a lane end; four a lane (no instance has them) measured 160 experts, top 4
      // 13.3 / 11.9, 26.4 / 16.4; 256, top 8, one, four and eight tokens 13.4 / 13.3, 17.1 / 16.4, 21.6 / 21.7.
      if (wv < T) {
        if (E <= kWave) topk_select_sorted<1, 3>(s_lg + wv * Ep, E, K, s_idx + wv * K, s_sc + wv * K, lane);
        else topk_select_sorted<2, 3>(s_lg + wv * Ep, E, K, s_idx + wv * K, s_sc + wv * K, lane);
      }
    } else if (rank_count) {
      if (router_mode != 0) {  // full softmax first: the probabilities replace the logits
        if (wv < T && !full_softmax_probs(s_lg + wv * Ep, s_lg + wv * Ep, E, lane)) {
          if (lane == 0) s_flag[wv] = 1u;  // the token routes nowhere; its scores only have to be comparable
          for (uint32_t i = lane; i < E; i += kWave) s_lg[wv * Ep + i] = 0.0f;
        }
        __syncthreads();
      }
      bool counted = false;
      if (topk_prefilter_fits(T, Ep, K, kFusedWaves)) {
        topk_prefilter(s_lg, s_rank, s_fail + 1, T, Ep, K, s_idx, s_sc, wv, lane);
        counted = s_fail[1] == 0u;  // else too many experts passed the prefilter: rank everything
        if (!counted) {
          __syncthreads();
          for (uint32_t i = threadIdx.x; i < kRankWords; i += kFusedThreads) s_rank[i] = 0u;
          __syncthreads();
        }
      }
      if (!counted) {
        topk_rank_count(s_lg, s_rank, T, Ep, wv, lane, kFusedWaves);
        __syncthreads();
        topk_rank_emit(s_lg, s_rank, T, Ep, K, s_idx, s_sc, threadIdx.x, kFusedThreads);
      }
      if (router_mode != 0) {  // a token with a non-finite logit routes nowhere (maple_moe.metal:62-119)
        __syncthreads();
        if (threadIdx.x < T * K && s_flag[threadIdx.x / K]) s_idx[threadIdx.x] = E;
      }
      // the routing weights follow after stage B: nothing needs them before stage C
    } else if (wv < T) {
      if (router_mode == 0) topk_select_fast(s_lg + wv * Ep, E, K, s_idx + wv * K, s_w + wv * K, lane);
      else topk_full_softmax_fast(s_lg + wv * Ep, s_lg + wv * Ep, E, K, s_idx + wv * K, s_w + wv * K, lane);
    }
    __syncthreads();
  } else {  // routing written by an earlier launch on the stream (a family router): read, never written
    trace_mark(a, 2);
    if (threadIdx.x < T * K) {
      s_idx[threadIdx.x] = a.out_idx[threadIdx.x];
      s_w[threadIdx.x] = a.out_w[threadIdx.x];
    }
    __syncthreads();
  }
  trace_mark(a, 3);

  // ------------------------------------------------------------- what stage C will read
  // The workgroups are split among the tokens: c_wgs of them own the output rows of one token, so a workgroup gathers
  // one token's activations (T tokens' by every workgroup one after the other: T waits, and T times the bytes past
  // every cache).  A unit is rpw output rows of the token.
  const uint32_t lpr_log2 = S::F != kDyn ? lanes_per_row_log2_dev(F, Fmt<BITS>::kElemsPer16B) : a.g.lpr_f;
  const uint32_t lpr = 1u << lpr_log2, rpw_log2 = 6 - lpr_log2, rpw = 1u << rpw_log2;
  const uint32_t rg_per_tok = (D + rpw - 1) >> rpw_log2;  // units of a token
  const uint32_t c_wgs = S::kStatic ? kSplit.wgs : a.g.c_wgs;
  const uint32_t tok = S::T == 1 ? 0u : fdiv(wg, a.g.c_wgs_div), wl = wg - tok * c_wgs;
  const uint32_t sub = lane & (lpr - 1), rloc = lane >> lpr_log2;
  const uint32_t ng = F / kGroup;
  const size_t rb = static_cast<size_t>(F) * Store<BITS>::kBits / 8;
  const uint32_t ub = S::kStatic ? kSplit.units : a.g.c_units;
  // The output row behind index i of the workgroup's rows (LDS order): rows form -- round by round, ub units each;
  // units form -- one run of units.
  const uint32_t rounds = UNITS ? 1u : S::kStatic ? kSplit.rounds : a.g.c_rounds, rows_per_round = ub << rpw_log2;
  auto row_at = [&](uint32_t i) __attribute__((always_inline)) {
    if constexpr (UNITS) return (wl * ub << rpw_log2) + i;
    const uint32_t round = rounds == 1 ? 0u : fdiv(i, a.g.rpr), in_round = i - round * rows_per_round;
    return ((round * c_wgs + wl) * ub << rpw_log2) + in_round;
  };
  // shared-expert down rows: srpw rows per wave step
  const uint32_t slpr_log2 = !Fs ? 0u : S::Fs != kDyn ? lanes_per_row_log2_dev(Fs, Fmt<SBITS>::kElemsPer16B) : a.g.lpr_sf;
  const uint32_t slpr = 1u << slpr_log2, srpw = 64u >> slpr_log2;

  // What the router decided is all a down row needs to be requested: the first codes leave before anything is
  // waited for.  Rows form: slot wv % K of unit wv / K of the first round.  Units form: pair wv, wv + 16, ... of the
  // (unit, slot) pairs, slots fastest; four of them are in flight.
  constexpr uint32_t kEPLF = Fmt<BITS>::kElemsPer16B;
  constexpr int kRing = UNITS ? 4 : 1;
  Chunk<BITS> ring[kRing];
  const uint32_t e0 = sub * kEPLF;
  const bool lane_in = e0 < F;
  const uint32_t e0c = lane_in ? e0 : 0u;
  // (unit, slot) of the wave's first pair: of the round in the rows form, of all in the units form
  const uint32_t unit_local = S::K != kDyn ? wv / K : fdiv(wv, a.g.K), slot = wv - unit_local * K;
  // units form: the slots' blobs and weights, a slot per lane
  uint32_t base_lo = 0, base_hi = 0;
  float w_lane = 0.0f;
  const uint32_t u_first = wl * ub, u_n = u_first < rg_per_tok ? (rg_per_tok - u_first < ub ? rg_per_tok - u_first : ub) : 0;
  const uint32_t n_pairs = u_n * K, n_mine = UNITS && wv < n_pairs ? (n_pairs - wv + kFusedWaves - 1) / kFusedWaves : 0u;
  const uint32_t step_units = S::K != kDyn ? kFusedWaves / K : fdiv(kFusedWaves, a.g.K), step_slots = kFusedWaves - step_units * K;
  uint32_t f_unit = unit_local, f_slot = slot;    // the next (unit, slot) to request
  auto request = [&](const uint8_t* blob, uint32_t row) __attribute__((always_inline)) {
    const uint32_t rc = row < D ? row : 0u;
    return load_chunk<BITS>(blob + a.off.down_w + rc * rb,
                            reinterpret_cast<const uint16_t*>(blob + a.off.down_s) + static_cast<size_t>(rc) * ng,
                            reinterpret_cast<const uint16_t*>(blob + a.off.down_b) + static_cast<size_t>(rc) * ng, e0c);
  };
  auto next_pair = [&](uint32_t& unit, uint32_t& sl) __attribute__((always_inline)) {
    unit += step_units;
    sl += step_slots;
    if (sl >= K) {
      sl -= K;
      ++unit;
    }
  };
  auto fetch_unit = [&](Chunk<BITS>& c) __attribute__((always_inline)) {
    const uint64_t base = (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(base_hi), f_slot))) << 32) |
                          static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(base_lo), f_slot));
    c = request(reinterpret_cast<const uint8_t*>(base), ((u_first + (f_unit < u_n ? f_unit : 0u)) << rpw_log2) + rloc);
    next_pair(f_unit, f_slot);
  };
  auto fetch_first = [&](Chunk<BITS>& c) __attribute__((always_inline)) {
    const uint32_t unit = wl * ub + unit_local;
    const uint32_t expert = __builtin_amdgcn_readfirstlane(s_idx[tok * K + slot]);
    c = request(a.expert_base + static_cast<size_t>(expert < E ? expert : 0u) * a.expert_stride, (unit << rpw_log2) + rloc);
  };
  // first shared-expert down chunk of a wave
  const uint32_t sng = Fs ? Fs / kGroup : 0;
  const size_t srb = static_cast<size_t>(Fs) * Store<SBITS>::kBits / 8;
  const uint32_t n_slots = !Fs ? 0u : UNITS ? u_n << rpw_log2 : rounds * rows_per_round;
  const uint32_t ssub = lane & (slpr - 1);
  Chunk<SBITS> spre{};
  bool have_spre = false;
  // When the requests go out.  Rows form: behind stage B's first (and mostly only) ones, so that the codes are here when
  // the activations are and no poll for activations has to wait for them -- a wave's loads return in order (small 4-bit
  // layer 12.4 -> 11.5 us, ternary layer 12.6 -> 12.3).  Units form: behind stage B, whose own stream of rows they
  // would sit in (Qwen shape, five tokens, as it was then: 26.4 us, with the early requests 28.9).
  auto request_down_rows = [&]() __attribute__((always_inline)) {
    if constexpr (UNITS) {
      const uint32_t expert = lane < K ? s_idx[tok * K + lane] : E;
      const uint64_t base = reinterpret_cast<uint64_t>(a.expert_base + static_cast<size_t>(expert < E ? expert : 0u) * a.expert_stride);
      base_lo = static_cast<uint32_t>(base);
      base_hi = static_cast<uint32_t>(base >> 32);
      if (n_mine) {
  #pragma unroll
        for (int i = 0; i < kRing; ++i) fetch_unit(ring[i]);
      }
    } else if (S::kStatic || unit_local < ub) {  // (literal shapes: no branch around the loads)
      fetch_first(ring[0]);
    }
    if (Fs) {
      const uint32_t i = wv * srpw + (lane >> slpr_log2), row = row_at(i);
      if (i < n_slots && row < D && ssub * Fmt<SBITS>::kElemsPer16B < Fs) {
        spre = load_chunk<SBITS>(static_cast<const uint8_t*>(a.sd.weights) + row * srb,
                                 a.sd.scales + static_cast<size_t>(row) * sng,
                                 a.sd.biases + static_cast<size_t>(row) * sng,
                                 ssub * Fmt<SBITS>::kElemsPer16B);
        have_spre = true;
      }
    }
  };

  // lane t: the scale of token t's x (one token: the same in every lane); read behind the first requests of stage B
  float x_scale = kRowScale;
  auto of_token = [&](float v, uint32_t token) __attribute__((always_inline)) { return S::T == 1 ? v : readlane_f(v, static_cast<int>(token)); };

  // ------------------------------------------------------------- stage B
  // Every workgroup takes a run of consecutive units (rpw rows of one routed slot), its waves
  // take them in turn; gate and up sums meet in LDS, the first threads turn them into
  // activations (one exp and one division per thread instead of per wave) and the run leaves as
  // one contiguous piece.  A wave with several units (or rows of several steps) requests the next
  // step's codes before it multiplies the present ones.
  {
    const uint32_t lpr_log2 = S::D != kDyn ? lanes_per_row_log2_dev(D, kEPL) : a.g.lpr_d;
    const uint32_t lpr = 1u << lpr_log2, rpw_log2 = 6 - lpr_log2, rpw = 1u << rpw_log2;
    const uint32_t rgf = (F + rpw - 1) >> rpw_log2;   // units per (token, slot)
    const uint32_t n_items = T * K * rgf;
    const uint32_t per_wg = S::kStatic ? fused_b_per_wg(kEPL, S::D, S::F, S::K, 1, kStaticWgs) : a.g.b_per_wg;
    const uint32_t first = wg * per_wg;
    const uint32_t last = first + per_wg < n_items ? first + per_wg : n_items;
    float* s_gu = reinterpret_cast<float*>(s_stage);  // (gate sum, up sum) per staged row
    const uint32_t sub = lane & (lpr - 1), rloc = lane >> lpr_log2;
    const uint32_t ng = D / kGroup;
    const size_t rb = static_cast<size_t>(D) * Store<BITS>::kBits / 8;
    const uint32_t steps = (D + lpr * kEPL - 1) / kEPL >> lpr_log2;  // 16-byte steps of a lane along a row
    auto pair_of = [&](uint32_t item) __attribute__((always_inline)) {
      return S::F != kDyn && S::D != kDyn ? item / rgf : fdiv(item, a.g.rgf);
    };
    struct Step {
      Chunk<BITS> g, u;
      uint32_t tok, e0;  // where its x slice lies; ok: the lane has a row and the slot an expert
      bool ok;
    };
    // one step's codes and table entries, without a branch around the loads: a lane without a row (or past the row's
    // end), or a router sentinel, reads something that exists and its sums stay 0
    auto fetch = [&](uint32_t item, uint32_t step, Step& c) __attribute__((always_inline)) {
      const uint32_t pair = pair_of(item);
      const uint32_t row = ((item - pair * rgf) << rpw_log2) + rloc;
      const uint32_t expert = __builtin_amdgcn_readfirstlane(s_idx[pair]);
      c.e0 = (step * lpr + sub) * kEPL;
      c.ok = row < F && expert < E && c.e0 < D;
      if (!(c.e0 < D)) c.e0 = 0;
      c.tok = S::K != kDyn ? pair / K : fdiv(pair, a.g.K);
      const uint8_t* blob = a.expert_base + static_cast<size_t>(expert < E ? expert : 0u) * a.expert_stride;
      const uint32_t rc = row < F ? row : 0u;
      const size_t tb = static_cast<size_t>(rc) * ng;
      c.g = load_chunk<BITS>(blob + a.off.gate_w + rc * rb, reinterpret_cast<const uint16_t*>(blob + a.off.gate_s) + tb,
                             reinterpret_cast<const uint16_t*>(blob + a.off.gate_b) + tb, c.e0);
      c.u = load_chunk<BITS>(blob + a.off.up_w + rc * rb, reinterpret_cast<const uint16_t*>(blob + a.off.up_s) + tb,
                             reinterpret_cast<const uint16_t*>(blob + a.off.up_b) + tb, c.e0);
    };
    float ga = 0.0f, ua = 0.0f;
    auto multiply = [&](uint32_t item, uint32_t step, const Step& c) __attribute__((always_inline)) {
      float largest = 0.0f;
      const XSlice<BITS> xs = xprep ? load_xslice_lds<BITS>(s_xq, c.tok, n_sl, c.e0 / kEPL, s_xsum[c.tok * n_sl + c.e0 / kEPL], code_unscale<BITS>(of_token(x_scale, c.tok)))
                                    : load_expert_x<BITS, true>(xin + static_cast<size_t>(c.tok) * D + c.e0, of_token(x_scale, c.tok), &largest);
      const float gd = expert_dot<BITS>(c.g.codes, xs), ud = expert_dot<BITS>(c.u.codes, xs);
      if (c.ok) {
        ga = __builtin_fmaf(c.g.scale(), gd, ga);
        ga = __builtin_fmaf(c.g.bias(), xs.sum, ga);
        ua = __builtin_fmaf(c.u.scale(), ud, ua);
        ua = __builtin_fmaf(c.u.bias(), xs.sum, ua);
      }
      if (step + 1 == steps) {  // the row is complete
        const float g = group_sum(ga, static_cast<int>(lpr));
        const float u = group_sum(ua, static_cast<int>(lpr));
        if (sub == 0) {
          float* dst = s_gu + 2 * (((item - first) << rpw_log2) + rloc);
          dst[0] = g;
          dst[1] = u;
        }
        ga = ua = 0.0f;
      }
    };
    uint32_t item = first + wv, step = 0;
    Step cur{};
    if (S::kStatic || item < last) fetch(item < n_items ? item : 0u, 0, cur);  // (literal shapes: no branch around the loads)
    if constexpr (!UNITS) request_down_rows();
    issue_fence();
    x_scale = s_xscale[S::T == 1 ? 0u : lane & (MF_MAX_TOKENS - 1)];
    if (x_runs != 1) {
      const float* of_lane = s_most + (lane < T ? lane * x_runs : 0u);
      float most = of_lane[0];
      for (uint32_t r = 1; r < x_runs; ++r) most = fmaxf(most, of_lane[r]);
      if (S::T == 1) most = readlane_f(most, 0);
      x_scale = row_scale(most);
      if (threadIdx.x < T) s_scale[threadIdx.x] = act_scale(most);  // (read behind the barriers of stage B)
    }
    // A token out of the ordinary window of magnitudes has its slices made again (the same for all waves)
    const bool again = S::T == 1 ? __any(x_scale != kRowScale) : __any(lane < T && x_scale != kRowScale);
    if (__builtin_expect(xprep && again, 0)) {
      for (uint32_t t = 0; t < T; ++t) {
        const float scale = of_token(x_scale, t);
        if (scale == kRowScale) continue;
        stage_expert_x<BITS>(s_xq + t * (XSlice<BITS>::kPairs / 4) * n_sl, s_xsum + t * n_sl, n_sl, n_sl, scale, xin + static_cast<size_t>(t) * D);
      }
      __syncthreads();
    }
    if (item < last) {
      for (;;) {
        uint32_t nitem = item, nstep = step + 1;
        if (nstep == steps) {
          nstep = 0;
          nitem += kFusedWaves;
        }
        if (nitem >= last) break;
        Step nxt;
        fetch(nitem, nstep, nxt);
        issue_fence();
        multiply(item, step, cur);
        cur = nxt;
        item = nitem;
        step = nstep;
      }
      multiply(item, step, cur);
    }
    __syncthreads();
    // staged row (item - first) * rpw + r is activation (item % rgf) * rpw + r of pair item / rgf
    const uint32_t n_words = first < last ? (last - first) << rpw_log2 : 0;
    for (uint32_t i = threadIdx.x; i < n_words; i += kFusedThreads) {
      const uint32_t it = first + (i >> rpw_log2), pair = pair_of(it);
      const uint32_t row = ((it - pair * rgf) << rpw_log2) + (i & (rpw - 1));
      // moe.metal:27-34, 528; maple_moe.metal:153-164; exchanged at the scale that the slices of the token's activations have
      const float scale = s_scale[S::T == 1 ? 0u : S::K != kDyn ? pair / K : fdiv(pair, a.g.K)];
      const float act = bf16_to_f(routed_activation(s_gu[2 * i], s_gu[2 * i + 1], limit, maple)) * scale;
      const uint32_t word = (__float_as_uint(act) >> 16) | (tag16 << 16);
      if (row < F) store_u32_agent(&a.t_acts[static_cast<size_t>(pair) * F + row], word);
    }
  }
  trace_mark(a, 4);
  // routing weights of token t by the wave 15 - t (rank counting left scores, not weights)
  if (rank_count && wv + T >= kFusedWaves) {
    const uint32_t tok = kFusedWaves - 1 - wv;
    const float my_score = lane < K ? s_sc[tok * K + lane] : -__builtin_inff();
    float wgt = router_mode == 0 ? topk_weight_of_rank<0>(my_score, K) : topk_weight_of_rank<1>(my_score, K);
    if (s_flag[tok]) wgt = 0.0f;  // maple_moe.metal:62-119: a non-finite logit routes nowhere
    if (lane < K) s_w[tok * K + lane] = wgt;
  }

  // ------------------------------------------------------------- stage C
  if (tok < T) {
    if constexpr (UNITS) request_down_rows();
    // the scale of the token's activations, in a vector register: the scalar ones are all taken
    float act_sc = s_scale[S::T == 1 ? 0u : tok];
    asm volatile("" : "+v"(act_sc));
    // Gather what other workgroups produced: the routed activations [K*F] and the shared
    // activations (+ gate) [Fs (+4)], 256 words per wave step, two steps in flight.
    // The shared activations were written in stage A, long ago: when the routed words fit the
    // other waves' first poll step, the workgroup fetches the shared words first (they are there:
    // one round trip, during which the routed words are still on their way anyway) and the few
    // waves that own the shared-expert down rows compute the gated shared output h1 while the
    // rest of the workgroup polls for the routed words -- h1 leaves the critical path.
    const bool gated = a.w_sg || a.gq_w;
    const uint32_t n_a = K * F, n_s = Fs ? (gated ? Fs + 4 : Fs) : 0;
    const AgentBuf ba = make_agent_buf(a.t_acts + static_cast<size_t>(tok) * n_a);
    const AgentBuf bs = make_agent_buf(a.t_sact + static_cast<size_t>(tok) * sact_stride);
    const uint32_t want = tag16 << 16;
    // waves [w0, w0 + nw) gather words [first, first + count) of the virtual array [acts | sact]
    auto gather = [&](uint32_t first, uint32_t count, uint32_t w0, uint32_t nw) __attribute__((always_inline)) {
      const uint32_t step = nw * 4 * kWave, end = first + count;
      for (uint32_t c0 = first + (wv - w0) * 4 * kWave; c0 < end; c0 += 2 * step) {
        const uint32_t i0 = c0 + 4 * lane, i1 = i0 + step;
        const bool in0 = i0 < end, in1 = i1 < end;
        uint4 v0 = make_uint4(want, want, want, want), v1 = v0;
        for (uint32_t spins = 0;; ++spins) {
          if (in0) v0 = i0 < n_a ? load_u32x4_agentbuf(ba, i0 * 4) : load_u32x4_agentbuf(bs, (i0 - n_a) * 4);
          if (in1) v1 = i1 < n_a ? load_u32x4_agentbuf(ba, i1 * 4) : load_u32x4_agentbuf(bs, (i1 - n_a) * 4);
          const uint32_t diff = (v0.x ^ want) | (v0.y ^ want) | (v0.z ^ want) | (v0.w ^ want) |
                                (v1.x ^ want) | (v1.y ^ want) | (v1.z ^ want) | (v1.w ^ want);
          if (__all((diff >> 16) == 0)) break;
          if (spins > kSpinLimit) {
            give_up(a.status, s_fail, lane);
            break;
          }
          __builtin_amdgcn_s_sleep(1);
        }
        auto put = [&](uint32_t i, const uint4& v) __attribute__((always_inline)) {  // four activations from element i on
          uint32_t* dst = i < n_a ? s_acts + ((i % kEPLF / 8) * act_ld + i / kEPLF) * 4 + i % 8 / 2 : s_sact + (i - n_a) / 2;
          *reinterpret_cast<uint2*>(dst) =
              make_uint2(__builtin_amdgcn_perm(v.y, v.x, 0x05040100u), __builtin_amdgcn_perm(v.w, v.z, 0x05040100u));
        };
        if (in0) put(i0, v0);
        if (in1) put(i1, v1);
      }
    };
    // gated shared output h1 of the output rows this workgroup owns; waves [0, nw) share the rows
    auto shared_rows = [&](uint32_t nw) __attribute__((always_inline)) {
      const float gate = gated ? bf16_lo(s_sact[Fs / 2]) : 0.0f;
      for (uint32_t s0 = wv * srpw; s0 < n_slots; s0 += nw * srpw) {
        const uint32_t i = s0 + (lane >> slpr_log2), row = row_at(i);
        const bool ok = i < n_slots && row < D;
        float part = 0.0f;
        if (ok)
          part = row_partial<SBITS>(static_cast<const uint8_t*>(a.sd.weights) + row * srb,
                                    a.sd.scales + static_cast<size_t>(row) * sng,
                                    a.sd.biases + static_cast<size_t>(row) * sng,
                                    reinterpret_cast<const uint16_t*>(s_sact), Fs, ssub, slpr,
                                    have_spre && s0 == wv * srpw, spre);
        const float v = group_sum(part, static_cast<int>(slpr));
        if (ok && ssub == 0) {
          float h = round_bf16(v);  // dequant_int4.metal:177-180
          if (gated) h = round_bf16(h / (1.0f + mf_exp(-gate)));  // utility.metal:49-59
          s_h1[i] = h;
        }
      }
    };
    // waves that own shared rows when the rows are dealt one wave step each
    const uint32_t sh_waves = Fs ? (n_slots + srpw - 1) >> (6 - slpr_log2) : 0;
    const bool split = Fs && sh_waves <= 4 && n_a <= (kFusedWaves - sh_waves) * 8 * kWave;
    if (split) {
      gather(n_a, n_s, 0, kFusedWaves);  // first try succeeds: one round trip
      __syncthreads();
      if (wv < sh_waves) shared_rows(sh_waves);
      else gather(0, n_a, sh_waves, kFusedWaves - sh_waves);
      __syncthreads();
      trace_mark(a, 5);
    } else {
      gather(0, n_a + n_s, 0, kFusedWaves);
      __syncthreads();
      trace_mark(a, 5);
      if (Fs) shared_rows(kFusedWaves);
    }

    auto store_row = [&](uint32_t row, float acc, bool failed) __attribute__((always_inline)) {
      const size_t o = static_cast<size_t>(tok) * D + row;
      const uint16_t yb = failed ? static_cast<uint16_t>(0x7FC0u) : f_to_bf16(acc);
      a.y[o] = yb;
      if (a.hidden && !failed) {  // residual_add_fp16, utility.metal:83-92
        uint16_t hv = a.hidden[o];
        if constexpr (NORM) {  // the residual add in front of the norm, made here for good
          if (a.delta) hv = f_to_bf16(bf16_to_f(hv) + bf16_to_f(a.delta[o]));
        }
        a.hidden[o] = f_to_bf16(bf16_to_f(hv) + bf16_to_f(yb));
      }
    };

    // The lane slices of the activations (permuted pairs and their sum) are the same for every output row: made once, in
    // place, in the layout of the x slices.  A thread reads and writes the blocks of its own part of a slice only.
    const uint32_t spl = F / kEPLF;
    uint4* acts4 = reinterpret_cast<uint4*>(s_acts);
    float* s_asum = reinterpret_cast<float*>(s_stage);
    // (Rows form: a wave meets one slice or two and makes them itself for less than the barrier costs -- 2816 x 448, 2-bit,
    // norm in front: 17.9 us staged, 17.4 -- except the 64-element slices of a literal shape: ternary layer 12.2 / 12.0.)
    constexpr bool kStageActs = UNITS || (BITS != kBits4 && S::kStatic);
    for (uint32_t i = threadIdx.x; kStageActs && i < 4 * K * spl; i += kFusedThreads) {
      constexpr int kW = kPartWords<BITS>;
      const uint32_t sl = i >> 2, part = i & 3u;
      uint32_t raw[kW], p[kW];
#pragma unroll
      for (int q = 0; q < kW / 4; ++q) {
        const uint4 v = acts4[(part * (kW / 4) + q) * act_ld + sl];
        raw[4 * q] = v.x; raw[4 * q + 1] = v.y; raw[4 * q + 2] = v.z; raw[4 * q + 3] = v.w;
      }
      float sum = expert_x_part<BITS, true>(raw, p, act_sc, nullptr);
      sum += dpp_f<0xB1>(sum);
      sum += dpp_f<0x4E>(sum);
#pragma unroll
      for (int q = 0; q < kW / 4; ++q) acts4[(part * (kW / 4) + q) * act_ld + sl] = make_uint4(p[4 * q], p[4 * q + 1], p[4 * q + 2], p[4 * q + 3]);
      if (part == 0) s_asum[sl] = sum;
    }
    if (kStageActs) __syncthreads();
    auto act_slice = [&](uint32_t sl) __attribute__((always_inline)) {
      const XSlice<BITS> xs = load_xslice_lds<BITS>(acts4, 0, act_ld, sl, kStageActs ? s_asum[sl] : 0.0f, code_unscale<BITS>(act_sc));
      if constexpr (kStageActs) return xs;
      else return permuted_expert_x<BITS>(xs, act_sc);
    };

    if constexpr (UNITS) {
      const bool failed = *s_fail != 0u;  // a wait gave up: no result, and hidden stays as it is
      const uint64_t live = __ballot((lane < K ? s_idx[tok * K + lane] : E) < E);
      w_lane = lane < K ? s_w[tok * K + lane] : 0.0f;
      float* s_pv = reinterpret_cast<float*>(s_xq);  // [unit][slot][row of the unit]; the x slices have had their use
      uint32_t c_unit = unit_local, c_slot = slot;   // the (unit, slot) at hand
      auto take = [&](const Chunk<BITS>& c) __attribute__((always_inline)) {
        const XSlice<BITS> xs = act_slice(c_slot * spl + (lane_in ? sub : 0u));
        float part = __builtin_fmaf(c.scale(), expert_dot<BITS>(c.codes, xs), 0.0f);  // the one step of a row
        part = __builtin_fmaf(c.bias(), xs.sum, part);
        const float v = group_sum(lane_in ? part : 0.0f, static_cast<int>(lpr));
        // moe.metal:1262; maple_moe.metal:258 (the down output is a bf16 number first)
        if (sub == 0) s_pv[((c_unit * K + c_slot) << rpw_log2) + rloc] = readlane_f(w_lane, static_cast<int>(c_slot)) * (maple ? round_bf16(v) : v);
        next_pair(c_unit, c_slot);
      };
      uint32_t n = 0;
      for (; n + 2 * kRing <= n_mine; n += kRing) {
#pragma unroll
        for (int i = 0; i < kRing; ++i) {
          take(ring[i]);
          fetch_unit(ring[i]);
        }
      }
      // what is left: up to four that are on their way and up to three that are not (no register with a request on its
      // way is moved: that would wait for it)
#pragma unroll
      for (int i = 0; i < kRing; ++i) {
        if (n + i < n_mine) take(ring[i]);
        if (n + kRing + i < n_mine) fetch_unit(ring[i]);
      }
      n += kRing;
#pragma unroll
      for (int i = 0; i + 1 < kRing; ++i)
        if (n + i < n_mine) take(ring[i]);
      __syncthreads();
      for (uint32_t i = threadIdx.x; i < u_n << rpw_log2; i += kFusedThreads) {  // sums in rank order, residual first
        const uint32_t row = (u_first << rpw_log2) + i;
        if (row < D) {
          const float* pv = s_pv + (((i >> rpw_log2) * K) << rpw_log2) + (i & (rpw - 1));
          float vk[MF_MAX_TOPK];
#pragma unroll
          for (uint32_t k = 0; k < MF_MAX_TOPK; ++k) vk[k] = pv[(k < K ? k : 0u) << rpw_log2];
          float acc = Fs ? s_h1[i] : 0.0f;
#pragma unroll
          for (uint32_t k = 0; k < MF_MAX_TOPK; ++k)
            if ((live >> k) & 1ull) acc = acc + vk[k];
          store_row(row, acc, failed);
        }
      }
    } else {
      for (uint32_t round = 0; round < rounds; ++round) {
        const uint32_t unit = (round * c_wgs + wl) * ub + unit_local;
        if (unit_local < ub && unit < rg_per_tok) {
          const uint32_t row = (unit << rpw_log2) + rloc;
          const uint32_t pair = tok * K + slot;
          const uint32_t expert = __builtin_amdgcn_readfirstlane(s_idx[pair]);
          float part = 0.0f;
          if (expert < E) {  // (the same for all lanes)
            const uint8_t* blob = a.expert_base + static_cast<size_t>(expert) * a.expert_stride;
            const uint32_t rc = row < D ? row : 0u;
            const uint8_t* wrow = blob + a.off.down_w + rc * rb;
            const uint16_t* srow = reinterpret_cast<const uint16_t*>(blob + a.off.down_s) + rc * ng;
            const uint16_t* brow = reinterpret_cast<const uint16_t*>(blob + a.off.down_b) + rc * ng;
            for (uint32_t first = 0; first < F; first += lpr * kEPLF) {  // the steps of a row
              const uint32_t e = first + e0, ec = e < F ? e : 0u;
              Chunk<BITS> c = ring[0];
              if (!(round == 0 && first == 0)) c = load_chunk<BITS>(wrow, srow, brow, ec);
              const XSlice<BITS> xs = act_slice(slot * spl + ec / kEPLF);
              const float dot = expert_dot<BITS>(c.codes, xs);
              if (e < F) {
                part = __builtin_fmaf(c.scale(), dot, part);
                part = __builtin_fmaf(c.bias(), xs.sum, part);
              }
            }
          }
          const float v = group_sum(part, static_cast<int>(lpr));
          // moe.metal:1262; maple_moe.metal:258 (the down output is a bf16 number first)
          if (sub == 0) s_v[wv * kWave + rloc] = s_w[pair] * (maple ? round_bf16(v) : v);
        }
        __syncthreads();
        if (threadIdx.x < rows_per_round) {
          const uint32_t ul = threadIdx.x >> rpw_log2, rr = threadIdx.x & (rpw - 1);
          const uint32_t row = (((round * c_wgs + wl) * ub + ul) << rpw_log2) + rr;
          if (row < D) {
            // the K weighted values first (independent LDS reads: one round of latency, not K),
            // then the sum in rank order, residual first
            float vk[MF_MAX_TOPK];
            bool live[MF_MAX_TOPK];
#pragma unroll
            for (uint32_t k = 0; k < MF_MAX_TOPK; ++k) {
              live[k] = k < K && s_idx[tok * K + (k < K ? k : 0)] < E;
              vk[k] = s_v[(ul * K + (k < K ? k : 0)) * kWave + rr];
            }
            float acc = Fs ? s_h1[round * rows_per_round + threadIdx.x] : 0.0f;
#pragma unroll
            for (uint32_t k = 0; k < MF_MAX_TOPK; ++k)
              if (live[k]) acc = acc + vk[k];
            store_row(row, acc, *s_fail != 0u);  // a wait gave up: no result, and hidden stays as it is
          }
        }
        // The next round overwrites s_v.  Behind the last round nothing is left to protect, and a barrier there only
        // makes every wave wait for the acknowledgement of the stores of y.
        if (round + 1 < rounds) __syncthreads();
      }
    }
  }
  if constexpr (!S::kGiven) {
    if (wg == 0 && threadIdx.x < T * K) {  // s_w was complete before stage C's first barrier
      if (a.out_idx) a.out_idx[threadIdx.x] = s_idx[threadIdx.x];
      if (a.out_w) a.out_w[threadIdx.x] = s_w[threadIdx.x];
    }
  }
  if (threadIdx.x == 0) a.epoch[wg] = epoch;
  trace_mark(a, 6);
}

// Host side: how a launch divides its work.
static uint32_t fused_epl(const mf_moe_config& c) { return c.bits == MF_BITS_4 ? 32 : 64; }

static uint32_t fused_b_per_wg(const mf_moe_config& c, uint32_t num_cu, uint32_t t) {
  return fused_b_per_wg(fused_epl(c), c.d, c.f, c.top_k, t, num_cu);
}
static FusedGeo fused_geo(const mf_moe_config& c, uint32_t num_cu, uint32_t t, const FusedSplit& sp) {
  const uint32_t epl = fused_epl(c), sepl = c.shared_bits == MF_BITS_4 ? 32 : 64;
  FusedGeo g{};
  g.b_per_wg = fused_b_per_wg(c, num_cu, t);
  g.c_wgs = sp.wgs;
  g.c_units = sp.units;
  g.c_rounds = sp.rounds;
  g.lpr_d = static_cast<uint8_t>(lanes_per_row_log2_dev(c.d, epl));
  g.lpr_f = static_cast<uint8_t>(lanes_per_row_log2_dev(c.f, epl));
  g.lpr_sd = static_cast<uint8_t>(c.shared_f ? lanes_per_row_log2_dev(c.d, sepl) : 0);
  g.lpr_sf = static_cast<uint8_t>(c.shared_f ? lanes_per_row_log2_dev(c.shared_f, sepl) : 0);
  const uint32_t rpw_d = 64u >> g.lpr_d, rpw_f = 64u >> g.lpr_f, rpw_sd = 64u >> g.lpr_sd;
  g.E = make_fastdiv(c.num_experts);
  g.n_sl = make_fastdiv(c.d / epl);
  g.rgf = make_fastdiv((c.f + rpw_d - 1) / rpw_d);
  g.K = make_fastdiv(c.top_k);
  g.x_runs = make_fastdiv(fused_x_runs(c.d / epl));
  g.srg = make_fastdiv((c.shared_f + rpw_sd - 1) / rpw_sd);
  g.c_wgs_div = make_fastdiv(sp.wgs);
  g.rpr = make_fastdiv(sp.units * rpw_f);
  return g;
}

// words of the LDS staging area: a chunk of router logits in stage A, the (gate, up) sums of a
// workgroup's run of routed rows in stage B
// (and, in stage C, the sums of the activation slices)
static uint32_t fused_stage_words(const mf_moe_config& c, uint32_t num_cu, uint32_t t) {
  const uint32_t epl = fused_epl(c), rpw = 64u >> lanes_per_row_log2_dev(c.d, epl);
  const uint32_t words = std::max(2 * fused_b_per_wg(c, num_cu, t) * rpw, c.top_k * (c.f / epl));
  return words < 64 ? 64 : (words + 3) & ~3u;
}
// words of the x slices of the routed rows (permuted pairs + sum per slice)
static uint32_t fused_xprep_words(const mf_moe_config& c, uint32_t t) {
  const uint32_t epl = c.bits == MF_BITS_4 ? 32 : 64;
  return t * (c.d / epl) * (epl / 2 + 1);
}
static size_t fused_lds_base(const mf_moe_config& c, uint32_t num_cu, uint32_t t) {
  const size_t sact_words = ((c.shared_f + 4) / 2 + 3) & ~size_t(3);
  const uint32_t epl = fused_epl(c);
  const size_t acts_words = static_cast<size_t>(epl / 8 * 4) * ((c.top_k * c.f / epl) | 1u);
  return 1024 + 4096 + kMaxH1 * 4 + kRankWords * 4 + static_cast<size_t>(MF_MAX_TOKENS) * ((c.num_experts + 3) & ~3u) * 4 +
         4 * (sact_words + acts_words + fused_stage_words(c, num_cu, t));
}
constexpr size_t kFusedLdsLimit = 150 * 1024;
// units form of stage C: a value per slot and output row of a workgroup, where the x slices were
static uint32_t fused_pv_words(const mf_moe_config& c, const FusedSplit& sp) {
  return sp.by_units ? sp.units * (64u >> lanes_per_row_log2_dev(c.f, fused_epl(c))) * c.top_k : 0;
}
// what the normalised rows of a launch that makes x itself take beside the rest
static size_t fused_norm_bytes(const mf_moe_config& c, uint32_t t, bool norm) { return norm ? 16 + static_cast<size_t>(t) * c.d * 2 : 0; }
static FusedSplit fused_split(const mf_moe_config& c, uint32_t num_cu, uint32_t t, bool norm) {
  FusedSplit sp = fused_split(fused_epl(c), c.d, c.f, c.top_k, t, num_cu);
  if (fused_lds_base(c, num_cu, t) + 4 * static_cast<size_t>(fused_pv_words(c, sp)) + fused_norm_bytes(c, t, norm) > kFusedLdsLimit)
    sp = fused_split(fused_epl(c), c.d, c.f, c.top_k, t, num_cu, false);
  return sp;
}
// the x slices are kept in LDS when they fit beside everything else
static bool fused_xprep(const mf_moe_config& c, uint32_t num_cu, uint32_t t) {
  return fused_lds_base(c, num_cu, t) + 4 * static_cast<size_t>(fused_xprep_words(c, t)) <= kFusedLdsLimit;
}
static size_t fused_lds_bytes(const mf_moe_config& c, uint32_t num_cu, uint32_t t, bool norm) {
  const size_t pv = fused_pv_words(c, fused_split(c, num_cu, t, norm)), xs = fused_xprep(c, num_cu, t) ? fused_xprep_words(c, t) : 0;
  return fused_lds_base(c, num_cu, t) + 4 * std::max(pv, xs);
}

// whether the rows of one token that a workgroup owns fit the h1 array (every token needs a workgroup)
static bool fused_rows_fit(const mf_moe_config& c, uint32_t num_cu, uint32_t t, bool norm) {
  const FusedSplit sp = fused_split(c, num_cu, t, norm);
  return sp.rounds * sp.units * (64u >> lanes_per_row_log2_dev(c.f, fused_epl(c))) <= kMaxH1;
}

bool fused_supported(const mf_moe& h, const mf_moe_layer_weights& w, const void* x, const void* y,
                     const void* hidden, uint32_t t) {
  const mf_moe_config& c = h.cfg;
  if (c.gate_group_size == 32) return false;  // a gate projection at group 32 runs on the chain of launches
  const bool combo = (c.bits == MF_BITS_4 && (!c.shared_f || c.shared_bits == MF_BITS_4)) ||
                     (c.bits == MF_BITS_2 && (!c.shared_f || c.shared_bits == MF_BITS_4 ||
                                              c.shared_bits == MF_BITS_2)) ||
                     (c.bits == MF_BITS_TERNARY && (!c.shared_f || c.shared_bits == MF_BITS_4));
  if (!combo || c.d % 8 != 0) return false;
  if (t * fused_x_runs(c.d / fused_epl(c)) > kFusedWaves * kWave - 2 * MF_MAX_TOKENS) return false;  // (hidden sizes from 260 000 on)
  if (fused_lds_base(c, static_cast<uint32_t>(h.ctx->num_cu), t) > kFusedLdsLimit) return false;
  if (static_cast<uint32_t>(h.ctx->num_cu) < t || !fused_rows_fit(c, static_cast<uint32_t>(h.ctx->num_cu), t, false)) return false;
  const uint32_t offs = w.offsets.gate_w | w.offsets.up_w | w.offsets.down_w;
  if (!aligned16(w.expert_base) || w.expert_stride % 16 || offs % 16) return false;
  if (!aligned16(w.router_w) || !aligned16(x) || !aligned16(y)) return false;
  if (hidden && !aligned16(hidden)) return false;
  if (c.shared_f) {
    if (!aligned16(w.shared_gate.weights) || !aligned16(w.shared_up.weights) ||
        !aligned16(w.shared_down.weights))
      return false;
    if (w.w_sg && !w.w_sg_q8.weights && !aligned16(w.w_sg)) return false;
    if (w.w_sg_q8.weights && (reinterpret_cast<uintptr_t>(w.w_sg_q8.weights) & 7u)) return false;
  }
  return true;
}

// Whether the launch can make x itself (NORM instances): own routing, rows of at most 4096 elements, room in
// LDS for the normalised rows, everything the plain launch needs
bool fused_norm_supported(const mf_moe& h, const mf_moe_layer_weights& w, const void* y, const void* hidden,
                          const void* delta, const void* norm_w, uint32_t t) {
  const mf_moe_config& c = h.cfg;
  if (!w.router_w || !hidden || !norm_w || c.d > 4096) return false;
  if (!aligned16(hidden) || !aligned16(norm_w) || (delta && !aligned16(delta))) return false;
  if (!fused_supported(h, w, hidden, y, hidden, t)) return false;  // (x stands in as an aligned pointer)
  const uint32_t num_cu = static_cast<uint32_t>(h.ctx->num_cu);
  return fused_rows_fit(c, num_cu, t, true) && fused_lds_bytes(c, num_cu, t, true) + fused_norm_bytes(c, t, true) <= kFusedLdsLimit;
}

// One instance in the form (rows or units of stage C) its shape takes; an instance with every dimension literal exists
// in one form only.
template <int BITS, int SBITS, class S, bool NORM>
static hipError_t launch_instance(bool by_units, dim3 grid, dim3 block, size_t lds, hipStream_t s, const FusedArgs& a) {
  auto go = [&](auto units) {
    constexpr auto kKernel = fused_decode_kernel<BITS, SBITS, S, NORM, decltype(units)::value>;
    const hipError_t e = allow_lds<kKernel>(lds, kFusedLdsLimit);
    if (e != hipSuccess) return e;
    kKernel<<<grid, block, lds, s>>>(a);
    return hipGetLastError();
  };
  if constexpr (S::kStatic) {
    return go(std::bool_constant<fused_split(Fmt<BITS>::kElemsPer16B, S::D, S::F, S::K, 1, kStaticWgs).by_units>{});
  } else {
    if (by_units) return go(std::true_type{});
    return go(std::false_type{});
  }
}

hipError_t launch_fused_decode(hipStream_t s, const mf_moe& h, const mf_moe_layer_weights& w,
                               const uint16_t* x, uint32_t t, uint16_t* y, uint16_t* hidden,
                               uint32_t* out_idx, float* out_w, const FusedNorm* norm) {
  const mf_moe_config& c = h.cfg;
  FusedArgs a{};
  a.router_w = w.router_w;
  a.expert_base = static_cast<const uint8_t*>(w.expert_base);
  a.expert_stride = w.expert_stride;
  a.off = w.offsets;
  a.sg = w.shared_gate;
  a.su = w.shared_up;
  a.sd = w.shared_down;
  const bool gate_q8 = c.shared_f && w.w_sg_q8.weights;
  a.w_sg = c.shared_f && !gate_q8 ? w.w_sg : nullptr;
  a.gq_w = gate_q8 ? static_cast<const uint8_t*>(w.w_sg_q8.weights) : nullptr;
  a.gq_s = gate_q8 ? w.w_sg_q8.scales : nullptr;
  a.gq_b = gate_q8 ? w.w_sg_q8.biases : nullptr;
  a.x = x;
  a.y = y;
  a.hidden = hidden;
  a.out_idx = out_idx;
  a.out_w = out_w;
  a.t_logits = h.ws.t_logits;
  a.t_sact = h.ws.t_sact;
  a.t_acts = h.ws.t_acts;
  a.epoch = h.ws.epoch;
  a.status = h.ws.status;
  a.trace = h.trace;
  a.D = c.d;
  a.F = c.f;
  a.E = c.num_experts;
  a.K = c.top_k;
  a.T = t;
  a.Fs = c.shared_f;
  a.router_mode = c.router_mode;
  a.limit = c.swiglu_limit;
  a.maple = static_cast<int>(c.maple_rounding);
  const dim3 grid(static_cast<uint32_t>(h.ctx->num_cu)), block(kFusedThreads);
  const uint32_t num_cu = static_cast<uint32_t>(h.ctx->num_cu);
  size_t lds = fused_lds_bytes(c, num_cu, t, norm != nullptr);
  a.stage_words = fused_stage_words(c, num_cu, t);
  a.xprep = fused_xprep(c, num_cu, t) ? 1 : 0;
  if (norm) {  // the normalised rows behind everything else in LDS
    a.delta = norm->delta;
    a.norm_w = norm->weight;
    a.norm_eps = norm->eps;
    a.xn_off = static_cast<uint32_t>((lds + 15) & ~size_t(15));
    lds = a.xn_off + static_cast<size_t>(t) * c.d * 2;
  }
  const FusedSplit sp = fused_split(c, num_cu, t, norm != nullptr);
  a.g = fused_geo(c, num_cu, t, sp);
#define MF_FUSED(B, SB, SHAPE) return launch_instance<B, SB, SHAPE, false>(sp.by_units, grid, block, lds, s, a)
#define MF_FUSED_N(B, SB, SHAPE) return launch_instance<B, SB, SHAPE, true>(sp.by_units, grid, block, lds, s, a)
  const bool one = t == 1 && num_cu == kStaticWgs;  // the instances with every dimension literal
  // Shape-specialised instances: a layer shape's dimensions as literals with the token rows read from the
  // arguments (Tn), and the one-token launch with T = 1 as a literal as well (T1: it drops the code of the
  // token loop; Qwen shape 12.3 us against 13.5 us through Tn).  Which literal buys what, Qwen shape, 4
  // token rows: none 40.2 us, T alone 39.8, top_k 37.5, top_k + experts 36.5, d + f 35.1, d + f + top_k 33.9,
  // those + shared_f 29.1, all but T 27.2, all 27.1.
  using QwenT1 = StaticShape<2048, 512, 256, 8, 1, 512, false, 0, 0, 1, 1>;
  using QwenTn = StaticShape<2048, 512, 256, 8, kDyn, 512, false, 0>;
  const bool qwen = c.bits == MF_BITS_4 && c.shared_bits == MF_BITS_4 && c.d == 2048 &&
                    c.f == 512 && c.num_experts == 256 && c.top_k == 8 && c.shared_f == 512 &&
                    c.router_mode == MF_ROUTER_TOPK_SOFTMAX;
  // the large 2-bit layer (hidden 4096, 256 experts of 2048, top-6, 4-bit shared expert of 2048)
  using Big2T1 = StaticShape<4096, 2048, 256, 6, 1, 2048, false, 0, 0, 0, 1>;
  using Big2Tn = StaticShape<4096, 2048, 256, 6, kDyn, 2048, false, 0>;
  const bool big2 = c.bits == MF_BITS_2 && c.shared_bits == MF_BITS_4 && c.d == 4096 && c.f == 2048 &&
                    c.num_experts == 256 && c.top_k == 6 && c.shared_f == 2048 &&
                    c.router_mode == MF_ROUTER_TOPK_SOFTMAX;
  // the ternary layer (hidden 2048, 64 experts of 1024, top-8, no shared expert)
  using TernT1 = StaticShape<2048, 1024, 64, 8, 1, 0, false, 1, 1, 1, 1>;
  using TernTn = StaticShape<2048, 1024, 64, 8, kDyn, 0>;
  const bool tern = c.bits == MF_BITS_TERNARY && c.d == 2048 && c.f == 1024 && c.num_experts == 64 &&
                    c.top_k == 8 && c.shared_f == 0;
  // MaplePreview's ternary layer (ModelTypes.swift:515-560: hidden 2048, 256 experts of 512, top-8, no shared expert)
  using MapleT1 = StaticShape<2048, 512, 256, 8, 1, 0, false, 1, 1, 1, 1>;
  using MapleTn = StaticShape<2048, 512, 256, 8, kDyn, 0>;
  const bool maple = c.bits == MF_BITS_TERNARY && c.d == 2048 && c.f == 512 && c.num_experts == 256 &&
                     c.top_k == 8 && c.shared_f == 0;
  const bool no_limit = c.swiglu_limit == 0.0f;  // the one-token instances of the benchmark shapes have these flags as literals
  // the instances of the shapes listed for the build (fused_shapes.json): declarations here, the branches
  // that pick them below, ahead of the instances that read every dimension from the arguments
#define MF_SHAPES_DECLARE
#include "fused_shapes.inc"
#undef MF_SHAPES_DECLARE
  using Given = RuntimeShapeT<true>;
  using Big2T1Given = StaticShape<4096, 2048, 256, 6, 1, 2048, true>;
  using QwenT1Given = StaticShape<2048, 512, 256, 8, 1, 512, true, kDyn, 0, 1, 1>;
  using QwenTnGiven = StaticShape<2048, 512, 256, 8, kDyn, 512, true>;
  // (with the routing given the router mode plays no part: the shapes are recognised without it)
  const bool qwen_dims = c.bits == MF_BITS_4 && c.shared_bits == MF_BITS_4 && c.d == 2048 && c.f == 512 &&
                         c.num_experts == 256 && c.top_k == 8 && c.shared_f == 512;
  const bool lit = !h.generic_shape;  // shape instances allowed
  using AnyE = RuntimeShapeT<false, true>;
  const bool any_e = c.num_experts % 4 != 0;
  if (norm) {  // x made inside the launch: the Qwen shape's instances and the ones that read every dimension
    if (lit && qwen && one && !c.maple_rounding && no_limit && a.xprep) MF_FUSED_N(kBits4, kBits4, QwenT1);
    else if (lit && qwen) MF_FUSED_N(kBits4, kBits4, QwenTn);
    else if (any_e && c.bits == MF_BITS_4) MF_FUSED_N(kBits4, kBits4, AnyE);
    else if (any_e && c.bits == MF_BITS_2 && c.shared_f && c.shared_bits == MF_BITS_2) MF_FUSED_N(kBits2, kBits2, AnyE);
    else if (any_e && c.bits == MF_BITS_2) MF_FUSED_N(kBits2, kBits4, AnyE);
    else if (any_e) MF_FUSED_N(kBitsTernary, kBits4, AnyE);
    else if (c.bits == MF_BITS_4) MF_FUSED_N(kBits4, kBits4, RuntimeShape);
    else if (c.bits == MF_BITS_2 && c.shared_f && c.shared_bits == MF_BITS_2) MF_FUSED_N(kBits2, kBits2, RuntimeShape);
    else if (c.bits == MF_BITS_2) MF_FUSED_N(kBits2, kBits4, RuntimeShape);
    else MF_FUSED_N(kBitsTernary, kBits4, RuntimeShape);
  }
  if (!w.router_w) {  // caller-given routing
    if (!lit) {
      if (c.bits == MF_BITS_4) MF_FUSED(kBits4, kBits4, Given);
      else if (c.bits == MF_BITS_2 && c.shared_f && c.shared_bits == MF_BITS_2) MF_FUSED(kBits2, kBits2, Given);
      else if (c.bits == MF_BITS_2) MF_FUSED(kBits2, kBits4, Given);
      else MF_FUSED(kBitsTernary, kBits4, Given);
    }
    else if (big2 && one) MF_FUSED(kBits2, kBits4, Big2T1Given);
    else if (qwen_dims && one && !c.maple_rounding && no_limit && a.xprep) MF_FUSED(kBits4, kBits4, QwenT1Given);
    else if (qwen_dims) MF_FUSED(kBits4, kBits4, QwenTnGiven);
#define MF_SHAPES_PICK_GIVEN
#include "fused_shapes.inc"
#undef MF_SHAPES_PICK_GIVEN
    else if (c.bits == MF_BITS_4) MF_FUSED(kBits4, kBits4, Given);
    else if (c.bits == MF_BITS_2 && c.shared_f && c.shared_bits == MF_BITS_2) MF_FUSED(kBits2, kBits2, Given);
    else if (c.bits == MF_BITS_2) MF_FUSED(kBits2, kBits4, Given);
    else MF_FUSED(kBitsTernary, kBits4, Given);
  } else if (any_e) {
    if (c.bits == MF_BITS_4) MF_FUSED(kBits4, kBits4, AnyE);
    else if (c.bits == MF_BITS_2 && c.shared_f && c.shared_bits == MF_BITS_2) MF_FUSED(kBits2, kBits2, AnyE);
    else if (c.bits == MF_BITS_2) MF_FUSED(kBits2, kBits4, AnyE);
    else MF_FUSED(kBitsTernary, kBits4, AnyE);
  } else if (!lit) {
    if (c.bits == MF_BITS_4) MF_FUSED(kBits4, kBits4, RuntimeShape);
    else if (c.bits == MF_BITS_2 && c.shared_f && c.shared_bits == MF_BITS_2) MF_FUSED(kBits2, kBits2, RuntimeShape);
    else if (c.bits == MF_BITS_2) MF_FUSED(kBits2, kBits4, RuntimeShape);
    else MF_FUSED(kBitsTernary, kBits4, RuntimeShape);
  } else if (qwen && one && !c.maple_rounding && no_limit && a.xprep) MF_FUSED(kBits4, kBits4, QwenT1);
  else if (qwen) MF_FUSED(kBits4, kBits4, QwenTn);
  else if (big2 && one && !c.maple_rounding && a.xprep) MF_FUSED(kBits2, kBits4, Big2T1);
  else if (big2) MF_FUSED(kBits2, kBits4, Big2Tn);
  else if (tern && one && c.router_mode == MF_ROUTER_FULL_SOFTMAX && c.maple_rounding && no_limit && a.xprep)
    MF_FUSED(kBitsTernary, kBits4, TernT1);
  else if (tern) MF_FUSED(kBitsTernary, kBits4, TernTn);
  else if (maple && one && c.router_mode == MF_ROUTER_FULL_SOFTMAX && c.maple_rounding && no_limit && a.xprep)
    MF_FUSED(kBitsTernary, kBits4, MapleT1);
  else if (maple) MF_FUSED(kBitsTernary, kBits4, MapleTn);
#define MF_SHAPES_PICK_OWN
#include "fused_shapes.inc"
#undef MF_SHAPES_PICK_OWN
  else if (c.bits == MF_BITS_4) MF_FUSED(kBits4, kBits4, RuntimeShape);
  else if (c.bits == MF_BITS_2 && c.shared_f && c.shared_bits == MF_BITS_2)
    MF_FUSED(kBits2, kBits2, RuntimeShape);
  else if (c.bits == MF_BITS_2) MF_FUSED(kBits2, kBits4, RuntimeShape);
  else MF_FUSED(kBitsTernary, kBits4, RuntimeShape);
#undef MF_FUSED
#undef MF_FUSED_N
}

}  // namespace mf
