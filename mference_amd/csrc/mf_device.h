// Device-side building blocks shared by every kernel: bf16 helpers, the
// deterministic exp, wave64 reductions and the per-lane packed-code dot products.
//
// Compile with -ffp-contract=off: every fused multiply-add below is spelled
// fmaf(); any other a*b+c is two roundings on purpose (the bit-exact paths
// rely on it).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mf {

constexpr int kWave = 64;    // gfx950 wavefront
constexpr int kGroup = 64;   // quantization group (Quantization.swift:5)

enum : int { kBitsTernary = 1, kBits2 = 2, kBits4 = 4, kBits8 = 8 };  // 8: GEMV, quantizer and scalar gate only

// elements covered by one 16-byte load of packed codes
template <int BITS> struct Fmt { static constexpr int kElemsPer16B = (BITS == kBits4) ? 32 : 64; };
// storage width of a format in bits per element (ternary is stored as 2-bit codes)
template <int BITS> struct Store { static constexpr int kBits = (BITS == kBits4) ? 4 : 2; };

// lanes of a wave that share one row of n elements (power of two, <= 64)
__host__ __device__ __forceinline__ uint32_t lanes_per_row_log2_dev(uint32_t n,
                                                                    uint32_t elems_per_lane) {
  const uint32_t need = (n + elems_per_lane - 1) / elems_per_lane;
  uint32_t l = 0;
  while ((1u << l) < need && l < 6) ++l;
  return l;
}

// ------------------------------------------------------------------ bf16

__device__ __forceinline__ float bf16_to_f(uint16_t b) {
  return __uint_as_float(static_cast<uint32_t>(b) << 16);
}
__device__ __forceinline__ float bf16_lo(uint32_t pair) { return __uint_as_float(pair << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t pair) { return __uint_as_float(pair & 0xFFFF0000u); }

// Quantization.swift:17-23: (bits + 0x7FFF + lsb) >> 16, no NaN special case.
__device__ __forceinline__ uint16_t f_to_bf16(float x) {
  uint32_t b = __float_as_uint(x);
  return static_cast<uint16_t>((b + 0x7FFFu + ((b >> 16) & 1u)) >> 16);
}
__device__ __forceinline__ float round_bf16(float x) { return bf16_to_f(f_to_bf16(x)); }

// ------------------------------------------------------------------- exp

// Deterministic exp: the same sequence of IEEE operations as the CPU oracle,
// so routing weights agree bit for bit.  Results below e^-86 are 0.
__device__ __forceinline__ float mf_exp(float x) {
  if (x != x) return x;
  if (x < -86.0f) return 0.0f;
  if (x > 88.0f) return __builtin_inff();
  float n = __builtin_rintf(x * 1.44269504088896341f);
  float r = __builtin_fmaf(-n, 0.693145751953125f, x);
  r = __builtin_fmaf(-n, 1.42860682030941723212e-6f, r);
  float p = 1.9875691500e-4f;
  p = __builtin_fmaf(p, r, 1.3981999507e-3f);
  p = __builtin_fmaf(p, r, 8.3334519073e-3f);
  p = __builtin_fmaf(p, r, 4.1665795894e-2f);
  p = __builtin_fmaf(p, r, 1.6666665459e-1f);
  p = __builtin_fmaf(p, r, 5.0000001201e-1f);
  float r2 = r * r;
  p = __builtin_fmaf(p, r2, r);
  p = p + 1.0f;
  int e = static_cast<int>(n) + 127;
  return p * __uint_as_float(static_cast<uint32_t>(e) << 23);
}

// log(t) for 1 <= t <= 2 (t = 1 + exp(-|x|) in the routers): 2*atanh((t-1)/(t+1)), odd series
// through s^15; the same IEEE sequence as the CPU oracle.
__device__ __forceinline__ float mf_log_1to2(float t) {
  const float s = (t - 1.0f) / (t + 1.0f);
  const float z = s * s;
  float p = 6.6666666667e-2f;
  p = __builtin_fmaf(p, z, 7.6923076923e-2f);
  p = __builtin_fmaf(p, z, 9.0909090909e-2f);
  p = __builtin_fmaf(p, z, 1.1111111111e-1f);
  p = __builtin_fmaf(p, z, 1.4285714286e-1f);
  p = __builtin_fmaf(p, z, 2.0e-1f);
  p = __builtin_fmaf(p, z, 3.3333333333e-1f);
  float r = s * z;
  r = __builtin_fmaf(r, p, s);
  return r + r;
}

// moe.metal:736-740
__device__ __forceinline__ float mf_sqrtsoftplus(float x) {
  const float sp = (x > 0.0f ? x : 0.0f) + mf_log_1to2(1.0f + mf_exp(-__builtin_fabsf(x)));
  return __builtin_sqrtf(sp);
}

// moe.metal:79-84
__device__ __forceinline__ float mf_silu(float x) { return x / (1.0f + mf_exp(-x)); }

// silu with the hardware exp2 / reciprocal (1 ulp each): the result is narrowed to bf16 right after
__device__ __forceinline__ float fast_silu(float x) {
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * -1.4426950408889634f));
}

// int8_gelu_pytorch_tanh (Metal/Quant/dequant_int8.metal:44-49): 0.5 x (1 + tanh(c (x + 0.044715 x^3))), the
// argument clamped to +-20; tanh(z) = 1 - 2 / (exp(2 z) + 1) on this build's exp, the same IEEE sequence as the
// CPU oracle.
__device__ __forceinline__ float mf_gelu_tanh(float x) {
  const float x3 = x * x * x;
  float inner = 0.7978845608028654f * (x + 0.044715f * x3);
  inner = fminf(fmaxf(inner, -20.0f), 20.0f);
  const float th = 1.0f - 2.0f / (mf_exp(2.0f * inner) + 1.0f);
  return 0.5f * x * (1.0f + th);
}

// MapleMoE's activation (maple_swiglu, maple_moe.metal:153-164): every intermediate is a bf16 number.
// min / clamp of bf16 numbers against +-7 and |x| stay bf16 numbers, so only the five arithmetic
// results are narrowed here.
__device__ __forceinline__ float maple_swiglu(float gate_projection, float up_projection) {
  const float gate = fminf(round_bf16(gate_projection), 7.0f);
  const float up = fminf(fmaxf(round_bf16(up_projection), -7.0f), 7.0f);
  const float exponent = round_bf16(mf_exp(fabsf(gate)));
  const float reciprocal = round_bf16(1.0f / round_bf16(1.0f + exponent));
  const float sigmoid = gate < 0.0f ? reciprocal : round_bf16(1.0f - reciprocal);
  return round_bf16(round_bf16(gate * sigmoid) * up);
}

// the routed experts' activation, narrowed once (moe.metal:27-34, 528) or in Maple's steps
__device__ __forceinline__ uint16_t routed_activation(float g, float u, float limit, bool maple) {
  if (maple) return f_to_bf16(maple_swiglu(g, u));
  if (limit > 0.0f) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
  }
  return f_to_bf16(mf_silu(g) * u);
}

// --------------------------------------------------------- wave reductions

// cross-lane move inside a row of 16 lanes (DPP); CTRL: 0xB1 = swap lanes
// (l, l^1), 0x4E = (l, l^2), 0x141 = mirror inside 8, 0x140 = mirror inside 16
template <int CTRL> __device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float readlane_f(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Sum over aligned groups of `lanes` lanes (power of two <= 64); every lane of
// a group ends with the group's sum.  The tree pairs neighbours first:
// (l, l^1), then (l, l^2), 4, 8, 16, 32 -- identical to an xor butterfly with
// ascending strides, which is the order the router's bit-exact contract names.
__device__ __forceinline__ float group_sum(float v, int lanes) {
  if (lanes >= 2) v = v + dpp_f<0xB1>(v);
  if (lanes >= 4) v = v + dpp_f<0x4E>(v);
  if (lanes >= 8) v = v + dpp_f<0x141>(v);
  if (lanes >= 16) v = v + dpp_f<0x140>(v);
  if (lanes >= 32) {
    const float r0 = readlane_f(v, 0), r1 = readlane_f(v, 16);
    const float r2 = readlane_f(v, 32), r3 = readlane_f(v, 48);
    const float lo = r0 + r1, hi = r2 + r3;
    if (lanes >= 64) v = lo + hi;
    else v = (threadIdx.x & 32) ? hi : lo;
  }
  return v;
}
__device__ __forceinline__ float wave_sum(float v) { return group_sum(v, kWave); }

// maximum over the wave, returned in every lane (no NaN inputs)
// the largest of the lower and of the upper half of a wave
__device__ __forceinline__ float2 half_wave_max(float v) {
  v = fmaxf(v, dpp_f<0xB1>(v));
  v = fmaxf(v, dpp_f<0x4E>(v));
  v = fmaxf(v, dpp_f<0x141>(v));
  v = fmaxf(v, dpp_f<0x140>(v));
  const float r0 = readlane_f(v, 0), r1 = readlane_f(v, 16);
  const float r2 = readlane_f(v, 32), r3 = readlane_f(v, 48);
  return make_float2(fmaxf(r0, r1), fmaxf(r2, r3));
}
__device__ __forceinline__ float wave_max(float v) {
  const float2 h = half_wave_max(v);
  return fmaxf(h.x, h.y);
}

// ------------------------------------------- device-coherent accesses
//
// Data that workgroups on different XCDs exchange inside one launch goes
// through these: `sc1` makes a store write through, and a load miss, every
// cache that is private to a CU or an XCD, so no bulk cache write-back or
// invalidate is needed around the grid barriers.

__device__ __forceinline__ void store_u16_agent(uint16_t* p, uint16_t v) {
  const uint32_t vv = v;
  asm volatile("global_store_short %0, %1, off sc1" : : "v"(p), "v"(vv) : "memory");
}
__device__ __forceinline__ uint16_t load_u16_agent(const uint16_t* p) {
  uint32_t r;
  asm volatile("global_load_ushort %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : "=v"(r) : "v"(p) : "memory");
  return static_cast<uint16_t>(r);
}
__device__ __forceinline__ void store_u32_agent(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// 16 bytes (16-byte aligned) written through as one request; readers rely on nothing wider than
// the 4-byte words being whole
__device__ __forceinline__ void store_u32x4_agent(uint32_t* p, uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
  const u32x4 v = {a, b, c, d};
  asm volatile("global_store_dwordx4 %0, %1, off sc1" : : "v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void store_u32x4_agent(uint32_t* p, uint32_t a) { store_u32x4_agent(p, a, a, a, a); }
__device__ __forceinline__ void store_f32_agent(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_f32_agent(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint4 load_u32x4_agent(const void* p) {
  uint4 r;
  asm volatile("global_load_dwordx4 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : "=v"(r) : "v"(p) : "memory");
  return r;
}
// Device-coherent 16-byte loads the compiler can schedule and wait for itself
// (several may be in flight): a raw buffer over [p, p + 2 GiB) read with sc1.
typedef __attribute__((ext_vector_type(4))) unsigned int mf_u32x4;
struct AgentBuf {
  __amdgpu_buffer_rsrc_t rsrc;
};
__device__ __forceinline__ AgentBuf make_agent_buf(const void* p) {
  AgentBuf b;
  b.rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, 0x7FFFFFFF, 0x00020000);
  return b;
}
__device__ __forceinline__ uint4 load_u32x4_agentbuf(const AgentBuf& b, uint32_t byte_offset) {
  const mf_u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(b.rsrc, static_cast<int>(byte_offset), 0,
                                                           16 /* sc1 */);
  return make_uint4(v.x, v.y, v.z, v.w);
}

// Nothing is moved across this point by the compiler: placed behind a group of loads it keeps
// them one batch of requests (the compiler otherwise sinks some of them below the arithmetic on
// the others, which turns one memory round trip into several).
__device__ __forceinline__ void issue_fence() { asm volatile("" ::: "memory"); }

// every store this wave has issued is acknowledged at its scope
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// An array kept in registers: every index is a literal once the loops are unrolled.  A call of index_past_the_end that is left then is an
// error of the build, so a loop that runs past the array does not compile (clang has no warning for it).
__device__ void index_past_the_end() __attribute__((error("index past the end of a register array")));
template <typename T, int N> struct RegArray {
  T v[N];
  __device__ __forceinline__ T& operator[](int i) {
    if (i >= N) index_past_the_end();
    return v[i];
  }
};

// LDS[lds + 16 * lane ...] = the 16 bytes at p of every lane (lds: a byte address, uniform), without a register in between.  The
// compiler does not know of the request: wait_loads stands in front of the first read, and a barrier behind it where another wave reads.
// (The address is an input in m0, so that the compiler writes that register and knows that it does; the wait state between is this asm's.)
__device__ __forceinline__ void load_to_lds(const void* p, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"{m0}"(lds), "v"(p) : "memory");
}
// every load of this wave but its newest N has arrived
template <int N> __device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// ------------------------------------------------------------- raw loads

__device__ __forceinline__ uint32_t load_u32_bytes(const uint8_t* p) {
  return static_cast<uint32_t>(p[0]) | (static_cast<uint32_t>(p[1]) << 8) |
         (static_cast<uint32_t>(p[2]) << 16) | (static_cast<uint32_t>(p[3]) << 24);
}

// 16 bytes of packed codes; ALIGNED = pointer is 16-byte aligned.
template <bool ALIGNED>
__device__ __forceinline__ uint4 load_codes16(const uint8_t* p) {
  if constexpr (ALIGNED) {
    return *reinterpret_cast<const uint4*>(p);
  } else {
    uint4 r;
    r.x = load_u32_bytes(p);
    r.y = load_u32_bytes(p + 4);
    r.z = load_u32_bytes(p + 8);
    r.w = load_u32_bytes(p + 12);
    return r;
  }
}

// 8 bf16 values as 4 packed pairs; ALIGNED = pointer is 16-byte aligned
// (otherwise 2-byte aligned).
template <bool ALIGNED>
__device__ __forceinline__ uint4 load_x8(const uint16_t* p) {
  if constexpr (ALIGNED) {
    return *reinterpret_cast<const uint4*>(p);
  } else {
    uint4 r;
    r.x = static_cast<uint32_t>(p[0]) | (static_cast<uint32_t>(p[1]) << 16);
    r.y = static_cast<uint32_t>(p[2]) | (static_cast<uint32_t>(p[3]) << 16);
    r.z = static_cast<uint32_t>(p[4]) | (static_cast<uint32_t>(p[5]) << 16);
    r.w = static_cast<uint32_t>(p[6]) | (static_cast<uint32_t>(p[7]) << 16);
    return r;
  }
}

// ------------------------------------------------- per-lane code x x dots
//
// One lane's share of a row is 16 bytes of codes: 32 four-bit elements (half a
// quantization group) or 64 two-bit elements (one group).  The dot product
// sum(q*x) runs on v_dot2c_f32_bf16: two codes are masked out of the packed
// word straight into the mantissas of a bf16 pair (0x4100 | q << 3 = 8 + q/2
// for 4-bit codes, 0x4080 | q << 5 = 4 + q for 2-bit codes, both exact),
// multiplied with a matching bf16 pair of x and accumulated in fp32; the
// offset * sum(x) this adds is taken off once per lane share.  Codes are
// paired (j, j + 4) for 4-bit and (j, j + 8) for 2-bit because those pairs sit
// 16 bits apart in the packed word; the x slice is permuted once to match and
// reused for every row that meets it (gate and up, several tokens' rows).

typedef __attribute__((ext_vector_type(2))) short mf_bf16x2;

__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float acc) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(mf_bf16x2, a),
                                         __builtin_bit_cast(mf_bf16x2, b), acc, false);
}

constexpr uint32_t kMagic128 = 0x43004300u;  // bf16 pair (128.0, 128.0)
// A masked code lands in the mantissa of a bf16 whose exponent is the smallest that leaves
// room for it: 4-bit codes in mantissa bits 3..6 under 2^3 (the number 8 + q/2), 2-bit codes
// in bits 5..6 under 2^2 (4 + q).  The dot product then carries offset * sum(x), removed in
// fp32 afterwards; the smaller the offset, the less of the fp32 mantissa that cancellation eats.
constexpr uint32_t kMagic8 = 0x41004100u;    // bf16 pair (8.0, 8.0)
constexpr uint32_t kMagic4 = 0x40804080u;    // bf16 pair (4.0, 4.0)
constexpr uint32_t kOnes = 0x3F803F80u;      // bf16 pair (1.0, 1.0)

// (v & mask) | magic in one instruction (v_and_or_b32).  A VOP3 instruction of this ISA takes
// one scalar source and no literal, so the mask has to sit in a scalar register and the magic in
// a vector register; the two empty asm statements only pin the constants there (they are pure,
// so the compiler hoists them out of loops) and the and-or itself stays an ordinary instruction
// the compiler schedules and guards: written as inline asm it would escape the hazard checks
// between a matrix instruction that still reads an operand and the next write of that register.
__device__ __forceinline__ uint32_t pin_sgpr(uint32_t x) {
  uint32_t r;
  asm("" : "=s"(r) : "0"(x));
  return r;
}
__device__ __forceinline__ uint32_t pin_vgpr(uint32_t x) {
  uint32_t r;
  asm("" : "=v"(r) : "0"(x));
  return r;
}
__device__ __forceinline__ uint32_t and_or(uint32_t v, uint32_t mask, uint32_t magic) {
  return (v & pin_sgpr(mask)) | pin_vgpr(magic);
}

// ---- matrix-core forms of the same embedding
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;

__device__ __forceinline__ f32x16_t mfma_bf16(const uint4& a, const uint4& b, const f32x16_t& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// one packed word of 4-bit codes -> MFMA operand: pairs (q0,q4),(q1,q5),(q2,q6),(q3,q7) as the
// bf16 numbers 8 + q/2 (exponent 2^3, the code in mantissa bits 3..6).  16 is the smallest offset
// a mask-and-or can give a 4-bit code, and the offset matters: the matrix core accumulates
// offset * sum(x) alongside the signal and the correction term takes it out again in fp32.
__device__ __forceinline__ uint4 expand_q4(uint32_t w) {
  return make_uint4(and_or(w << 3, 0x00780078u, kMagic8), and_or(w >> 1, 0x00780078u, kMagic8),
                    and_or(w >> 5, 0x00780078u, kMagic8), and_or(w >> 9, 0x00780078u, kMagic8));
}

// ---- codes as bf16 subnormals: the operands of the quantized matmuls
//
// A bf16 number with a zero exponent field is its mantissa times 2^-133, one with exponent 1 is (128 + mantissa) times
// 2^-133: the low byte u of a 16-bit word whose upper byte is zero IS the number u * 2^-133, and the matrix cores (and
// v_dot2_f32_bf16) read it as that.  A code needs no magic or-ed in: its field is masked in place, at the top of the byte -- a 4-bit code
// in bits 4..7 is q * 2^-129, a 2-bit code in bits 6..7 is q * 2^-127 -- and nothing has to be taken off the sums afterwards.
// Measured against the numbers 8 + q/2 (4 + q) that a mask-and-or gives: an and takes 1.5 ns of a SIMD, an and-or 3.0; one K
// group of 64 with its operands in registers, two row blocks, two waves a SIMD: 357 -> 323 ns for two token
// blocks, 243 -> 198 for one, 222 -> 180 for one of at most 8 tokens; and a group's sum is 4 to 5 times nearer to its 64-bit value
// (relative rms 3.3e-8 -> 0.7e-8 on Gaussian rows, 7.9e-8 -> 1.8e-8 on SwiGLU outputs, 2.1e-7 -> 0.6e-7 beside an outlier of 1000).
// (Fields left where they are, at the bottom of the byte, would save half of the shifts: 292 / 167 / 147 ns.  The matrix core
// aligns products by the operands' exponents, though, and the small ones then lose bits: 1.1e-7 on SwiGLU outputs.)
// The rows that meet such codes are kept times 2^64 (kRowScale), so that products stay in the range of ordinary fp32
// numbers; the group's scale takes the powers of two back.  A sum then keeps all 24 bits down to 2^-61, and values may reach
// 2^57 (64 of them against codes of 15 stay finite).  What leaves that window takes another power of two, chosen by the largest
// magnitude: 2^2 for large values, 2^126 for small ones.  So a bf16 number of any size has its product, as with numbers under an offset.
constexpr float kRowScale = 0x1p64f, kRowUnscale = 0x1p-64f;
// m: the largest magnitude, times kRowScale (infinite where that overflows)
// (magnitudes compare as their bits do: where they are the same for a wave, on the scalar unit)
__device__ __forceinline__ float scale_of_window(float m, float low, float high) {
  const uint32_t b = __float_as_uint(m);
  return b >= __float_as_uint(high) ? 0x1p2f : b - 1u < __float_as_uint(low) - 1u ? 0x1p126f : kRowScale;
}
__device__ __forceinline__ float row_scale(float m) { return scale_of_window(m, 0x1p5f, 0x1p121f); }
// ... by the sum of the squares of up to 192 numbers (infinite, or zero, where that is what they come to)
__device__ __forceinline__ float scale_of_squares(float s) { return s < 0x1p-110f ? 0x1p126f : s < 0x1p113f ? kRowScale : 0x1p2f; }
// The activations between an MLP's products are scaled before the largest is known, by that of the token's x (m, as above): from
// 2^-20 to 2^20 in x they are products of two sums of such numbers and stay within 2^-61 .. 2^62 unless the weights do not.
__device__ __forceinline__ float act_scale(float m) { return scale_of_window(m, 0x1p44f, 0x1p84f); }

// the upper halves of two fp32 numbers, (lo, hi) in the lower and the upper half
__device__ __forceinline__ uint32_t upper_halves(float lo, float hi) {
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
// what a result of rows at `scale` lacks: a factor that is 1 for ordinary rows (the matmuls' tables hold the powers of two of those)
__device__ __forceinline__ float rel_of_scale(float scale) { return __uint_as_float(((2u * 127u + 64u) << 23) - __float_as_uint(scale)); }
// eight bf16 numbers of a row in the matmul's order (0,4,1,5,2,6,3,7) and times `scale`; their sum in *sum (unscaled); *largest (where
// given) is raised to the largest magnitude (at that scale)
__device__ __forceinline__ uint4 matmul_row8(const uint4& v, float scale, float* sum, float* largest = nullptr) {
  const float x0 = bf16_lo(v.x), x1 = bf16_hi(v.x), x2 = bf16_lo(v.y), x3 = bf16_hi(v.y);
  const float x4 = bf16_lo(v.z), x5 = bf16_hi(v.z), x6 = bf16_lo(v.w), x7 = bf16_hi(v.w);
  *sum = ((x0 + x1) + (x2 + x3)) + ((x4 + x5) + (x6 + x7));
  const float y0 = x0 * scale, y1 = x1 * scale, y2 = x2 * scale, y3 = x3 * scale, y4 = x4 * scale, y5 = x5 * scale, y6 = x6 * scale, y7 = x7 * scale;
  if (largest) *largest = fmaxf(*largest, fmaxf(fmaxf(fmaxf(fabsf(y0), fabsf(y1)), fmaxf(fabsf(y2), fabsf(y3))),
                                                fmaxf(fmaxf(fabsf(y4), fabsf(y5)), fmaxf(fabsf(y6), fabsf(y7)))));
  return make_uint4(upper_halves(y0, y4), upper_halves(y1, y5), upper_halves(y2, y6), upper_halves(y3, y7));
}

// The fp32 sums of a row's groups of 64 values (times 2^-64 and the row's scale: as they are for ordinary rows), as the matmuls read them for the bias term: three bf16 numbers each, which
// hold all 24 bits.  Per eight groups the eight first parts, then the second, then the third ones (48 bytes); groups past the
// row's last one are zeros.
__host__ __device__ __forceinline__ size_t group_sum_words(uint32_t ng) { return static_cast<size_t>((ng + 7) / 8) * 24; }
// sum of group g of ng; `row` = where the row's sums start
__device__ __forceinline__ void store_group_sum(uint16_t* row, uint32_t g, uint32_t ng, float sum) {
  const uint32_t hi = __float_as_uint(sum) & 0xFFFF0000u;
  const float r1 = sum - __uint_as_float(hi);
  const uint32_t mid = __float_as_uint(r1) & 0xFFFF0000u, lo = __float_as_uint(r1 - __uint_as_float(mid));
  uint16_t* at = row + g / 8 * 24 + g % 8;
  at[0] = static_cast<uint16_t>(hi >> 16);
  at[8] = static_cast<uint16_t>(mid >> 16);
  at[16] = static_cast<uint16_t>(lo >> 16);
  if (g + 1 == ng)
    for (uint32_t j = 1; (g + j) % 8; ++j) at[j] = at[8 + j] = at[16 + j] = 0;
}

// one packed word of 4-bit codes -> MFMA operand: pairs (q0,q4),(q1,q5),(q2,q6),(q3,q7)
__device__ __forceinline__ uint4 subnormal_q4(uint32_t w) {
  return make_uint4((w << 4) & 0x00F000F0u, w & 0x00F000F0u, (w >> 4) & 0x00F000F0u, (w >> 8) & 0x00F000F0u);
}
// one packed word of sixteen 2-bit codes -> two MFMA operands in the same pairing: the byte swap (B0, B2, B1, B3) puts
// code r and code r + 4 sixteen bits apart, and likewise 8 + r and 12 + r
__device__ __forceinline__ void subnormal_q2(uint32_t w, uint4& a, uint4& b) {
  const uint32_t v = __builtin_amdgcn_perm(w, w, 0x03010200u);
  a = make_uint4((v << 6) & 0x00C000C0u, (v << 4) & 0x00C000C0u, (v << 2) & 0x00C000C0u, v & 0x00C000C0u);
  b = make_uint4((v >> 2) & 0x00C000C0u, (v >> 4) & 0x00C000C0u, (v >> 6) & 0x00C000C0u, (v >> 8) & 0x00C000C0u);
}

// What the quantized matmuls need to know about a code width: a lane's share of one 64-wide group
// of its weight row is half the group -- 16 bytes of 4-bit codes or 8 bytes of 2-bit codes (ternary
// weights are 2-bit codes) -- and it becomes four MFMA operands of 8 bf16 numbers.
//
// Codes travel in pairs of groups.  Lane l = m + 32 h multiplies half h of row m of a 32-row block.  Asked for that
// way, from rows as they are, a load instruction touches 32 rows, 32 memory lines, for 1 KB (4-bit) or 512 B (2-bit),
// and the L1's line rate is a large part of what short batches cost.  So a lane asks for other bytes and
// the pair is put in order in registers (settle): 4-bit, two loads of 16 rows x 64 bytes (rows 0..15, then 16..31; the
// 16 lanes q of a quarter-wave take half q / 2 of group q % 2) and one row swap per register pair; 2-bit, one
// load of 32 rows x 32 bytes (the lanes of half h take group h) and one half-wave swap per register pair.
// SWAPPED = false: the lane asks for what it multiplies.  That is the better form for a tiled pool
// (tile_codes_kernel), where those bytes lie side by side and the swaps (2 of 66 vector instructions per group and
// row block; 4 of 55 of 2-bit codes and a tile of at most 32 routes) would buy nothing.  (Layers from the pool as loaded, in us, one piece per row -> this: Qwen shape, 93 tokens
// 89.9 -> 83.4; dense MLP 5120 x 17408, 150 rows, two of them 345 -> 337.  Qwen shape, 2048 tokens, tiled: 251 without
// the swaps, 254 with them.)
template <int BITS, bool SWAPPED = true> struct QmmCodes;
template <bool SWAPPED> struct QmmCodes<4, SWAPPED> {
  static constexpr uint32_t kGroupBytes = 32;     // one group of one row
  static constexpr float kScaleMul = 0x1p65f;     // q * 2^-129 meets x * 2^64
  uint32_t w[8];  // group 0: w[0..3], group 1: w[4..7]
  // which group of the pair the lane asks for first; its place in 32 rows as they are and in a tiled block; how far
  // behind the second load is
  static __device__ __forceinline__ uint32_t lane_group(uint32_t lane) { return SWAPPED ? (lane >> 4) & 1u : 0u; }
  static __device__ __forceinline__ size_t lane_offset(uint32_t lane, size_t row_bytes, bool tiled) {
    if (SWAPPED) return (lane & 15u) * row_bytes + lane_group(lane) * 32u + (lane >> 5) * 16u;
    return tiled ? lane * 16u : (lane & 31u) * row_bytes + (lane >> 5) * 16u;
  }
  static __device__ __forceinline__ size_t second(size_t row_bytes, bool tiled) {
    if (SWAPPED) return 16u * row_bytes;
    return tiled ? 1024u : 32u;
  }
  // the part of the pair whose registers are free once group i of the pair before has been multiplied (the second part lies
  // second() behind the first)
  __device__ __forceinline__ void load(int i, const uint8_t* p) {
    const uint4 v = *reinterpret_cast<const uint4*>(p);
    w[4 * i] = v.x; w[4 * i + 1] = v.y; w[4 * i + 2] = v.z; w[4 * i + 3] = v.w;
  }
  __device__ __forceinline__ void settle() {
    if (!SWAPPED) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const auto r = __builtin_amdgcn_permlane16_swap(w[i], w[4 + i], false, false);
      w[i] = r[0]; w[4 + i] = r[1];
    }
  }
};
template <bool SWAPPED> struct QmmCodes<2, SWAPPED> {  // (SWAPPED = false: only tiled)
  static constexpr uint32_t kGroupBytes = 16;
  static constexpr float kScaleMul = 0x1p63f;     // q * 2^-127 meets x * 2^64
  uint32_t w[4];  // group 0: w[0..1], group 1: w[2..3]
  static __device__ __forceinline__ uint32_t lane_group(uint32_t lane) { return SWAPPED ? lane >> 5 : 0u; }
  static __device__ __forceinline__ size_t lane_offset(uint32_t lane, size_t row_bytes, bool) {
    return SWAPPED ? (lane & 31u) * row_bytes + lane_group(lane) * 16u : lane * 16u;
  }
  static __device__ __forceinline__ size_t second(size_t, bool) { return 0; }
  __device__ __forceinline__ void load(int i, const uint8_t* p) {  // (all of the pair with its second part)
    if (i == 0) return;
    const uint4 v = *reinterpret_cast<const uint4*>(p);
    w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
  }
  __device__ __forceinline__ void settle() {
    if (!SWAPPED) return;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const auto r = __builtin_amdgcn_permlane32_swap(w[i], w[2 + i], false, false);
      w[i] = r[0]; w[2 + i] = r[1];
    }
  }
};

// tmp[token block] += x * codes over one group: 8 MFMAs; `after(s)` runs once both token blocks have
// issued theirs on operand s (the caller may then overwrite bx[.][s])
// (NTA = 1: only the first token block holds routes, the second is left alone)
// (g: which group of the settled pair)
template <int BITS, int NTA = 2, bool SWAPPED, typename After>
__device__ __forceinline__ void group_products(const QmmCodes<BITS, SWAPPED>& c, int g, const uint4 (&bx)[2][4], f32x16_t (&tmp)[2],
                                               After after) {
  if constexpr (BITS == 4) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const uint4 av = subnormal_q4(c.w[4 * g + s]);
      tmp[0] = mfma_bf16(bx[0][s], av, tmp[0]);
      if constexpr (NTA > 1) tmp[1] = mfma_bf16(bx[1][s], av, tmp[1]);
      after(s);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      uint4 a, b;
      subnormal_q2(c.w[2 * g + j], a, b);
      tmp[0] = mfma_bf16(bx[0][2 * j], a, tmp[0]);
      if constexpr (NTA > 1) tmp[1] = mfma_bf16(bx[1][2 * j], a, tmp[1]);
      after(2 * j);
      tmp[0] = mfma_bf16(bx[0][2 * j + 1], b, tmp[0]);
      if constexpr (NTA > 1) tmp[1] = mfma_bf16(bx[1][2 * j + 1], b, tmp[1]);
      after(2 * j + 1);
    }
  }
}

// 16 bytes from any address the element type allows (global memory takes unaligned vector loads)
__device__ __forceinline__ uint4 load_16_bytes(const void* p) {
  uint4 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}
// eight bf16 numbers without the first n (0..7); zeros follow
__device__ __forceinline__ uint4 drop_bf16(uint4 v, uint32_t n) {
  if (n & 4u) v = make_uint4(v.z, v.w, 0, 0);
  if (n & 2u) v = make_uint4(v.y, v.z, v.w, 0);
  if (n & 1u)
    v = make_uint4(__builtin_amdgcn_alignbit(v.y, v.x, 16), __builtin_amdgcn_alignbit(v.z, v.y, 16),
                   __builtin_amdgcn_alignbit(v.w, v.z, 16), v.w >> 16);
  return v;
}

// 8 bf16 from p, of which only the first `avail` exist (the rest read as 0)
__device__ __forceinline__ uint4 load_bf16x8_guarded(const uint16_t* p, uint32_t avail) {
  if (avail >= 8) return load_x8<false>(p);
  uint32_t v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = static_cast<uint32_t>(i) < avail ? p[i] : 0u;
  return make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16));
}

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

// The activations one lane meets, permuted for the pairing above, plus their sum.
template <int BITS> struct XSlice {
  static constexpr int kPairs = Fmt<BITS>::kElemsPer16B / 2;
  uint32_t p[kPairs];
  float sum;
  float unscale;  // (expert_dot's slices)
};

// raw: consecutive bf16 pairs (x0,x1),(x2,x3),... of the lane's slice
template <int BITS>
__device__ __forceinline__ void permute_x(const uint32_t* raw, XSlice<BITS>& xs) {
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < XSlice<BITS>::kPairs; ++i) sum = dot2_bf16(raw[i], kOnes, sum);
  xs.sum = sum;
  if constexpr (BITS == kBits4) {
    // per packed word: 8 elements = raw pairs r0..r3 -> (x0,x4),(x1,x5),(x2,x6),(x3,x7)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t r0 = raw[4 * j], r1 = raw[4 * j + 1], r2 = raw[4 * j + 2], r3 = raw[4 * j + 3];
      xs.p[4 * j + 0] = __builtin_amdgcn_perm(r2, r0, 0x05040100u);
      xs.p[4 * j + 1] = __builtin_amdgcn_perm(r2, r0, 0x07060302u);
      xs.p[4 * j + 2] = __builtin_amdgcn_perm(r3, r1, 0x05040100u);
      xs.p[4 * j + 3] = __builtin_amdgcn_perm(r3, r1, 0x07060302u);
    }
  } else {
    // per packed word: 16 elements = raw pairs r0..r7 -> (x_i, x_{i+8}), i = 0..7
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t lo = raw[8 * j + i], hi = raw[8 * j + 4 + i];
        xs.p[8 * j + 2 * i] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
        xs.p[8 * j + 2 * i + 1] = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
      }
    }
  }
}

enum XLoad : int { kXAligned = 0, kXUnaligned = 1 };

// loads and permutes the lane's slice of x starting at element pointer x
template <int BITS, int MODE>
__device__ __forceinline__ XSlice<BITS> load_xslice(const uint16_t* x) {
  constexpr int kQuads = Fmt<BITS>::kElemsPer16B / 8;
  uint32_t raw[kQuads * 4];
#pragma unroll
  for (int q = 0; q < kQuads; ++q) {
    const uint4 a = load_x8<MODE == kXAligned>(x + 8 * q);
    raw[4 * q] = a.x; raw[4 * q + 1] = a.y; raw[4 * q + 2] = a.z; raw[4 * q + 3] = a.w;
  }
  XSlice<BITS> xs;
  permute_x<BITS>(raw, xs);
  return xs;
}

// the same in two steps: request the lane's slice (16-byte aligned), permute it later
template <int BITS> struct XRaw { uint4 q[Fmt<BITS>::kElemsPer16B / 8]; };
template <int BITS>
__device__ __forceinline__ XRaw<BITS> load_xraw(const uint16_t* x) {
  XRaw<BITS> r;
#pragma unroll
  for (int q = 0; q < Fmt<BITS>::kElemsPer16B / 8; ++q) r.q[q] = load_x8<true>(x + 8 * q);
  return r;
}
template <int BITS>
__device__ __forceinline__ XSlice<BITS> make_xslice(const XRaw<BITS>& r) {
  constexpr int kQuads = Fmt<BITS>::kElemsPer16B / 8;
  uint32_t raw[kQuads * 4];
#pragma unroll
  for (int q = 0; q < kQuads; ++q) {
    raw[4 * q] = r.q[q].x; raw[4 * q + 1] = r.q[q].y; raw[4 * q + 2] = r.q[q].z; raw[4 * q + 3] = r.q[q].w;
  }
  XSlice<BITS> xs;
  permute_x<BITS>(raw, xs);
  return xs;
}

// sum over the lane's share of q * x
template <int BITS>
__device__ __forceinline__ float codes_dot(const uint4& codes, const XSlice<BITS>& xs) {
  const uint32_t ws[4] = {codes.x, codes.y, codes.z, codes.w};
  float dot = 0.0f;
  if constexpr (BITS == kBits4) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t w = ws[j];
      dot = dot2_bf16(and_or(w << 3, 0x00780078u, kMagic8), xs.p[4 * j + 0], dot);
      dot = dot2_bf16(and_or(w >> 1, 0x00780078u, kMagic8), xs.p[4 * j + 1], dot);
      dot = dot2_bf16(and_or(w >> 5, 0x00780078u, kMagic8), xs.p[4 * j + 2], dot);
      dot = dot2_bf16(and_or(w >> 9, 0x00780078u, kMagic8), xs.p[4 * j + 3], dot);
    }
    return 2.0f * __builtin_fmaf(-8.0f, xs.sum, dot);  // sum((8 + q/2) x) -> sum(q x)
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t w = ws[j];
      dot = dot2_bf16(and_or(w << 5, 0x00600060u, kMagic4), xs.p[8 * j + 0], dot);
      dot = dot2_bf16(and_or(w << 3, 0x00600060u, kMagic4), xs.p[8 * j + 1], dot);
      dot = dot2_bf16(and_or(w << 1, 0x00600060u, kMagic4), xs.p[8 * j + 2], dot);
#pragma unroll
      for (int i = 3; i < 8; ++i)
        dot = dot2_bf16(and_or(w >> (2 * i - 5), 0x00600060u, kMagic4), xs.p[8 * j + i], dot);
    }
    return __builtin_fmaf(-4.0f, xs.sum, dot);  // sum((4 + q) x) -> sum(q x)
  }
}

// The rows of the routed experts meet a token's slice on the matrix core: codes are bf16 subnormals at the top of a byte
// (above; the two-bit ones at two places with a sum each), four of them per v_mfma_f32_4x4x4_16b_bf16, whose blocks
// multiply the codes of every lane of a quad with the values of every lane of it -- the lane's own share is on the diagonal.
// Vector instructions are what the decode launch's routed stages wait for.  Per lane, 16 bytes and SIMD (four waves):
// codes under an offset for the two-element dot product 96 / 173 ns (4 / 2 bits), subnormals for it 80 / 139, here 67 / 122;
// error against 64 bits on normal values 2.1e-8 with the offset, 3.9e-9 / 3.4e-9 either way here (on SwiGLU outputs 5.4e-8, 1.1e-8).
// An expert's slice holds its values times a power of two (row_scale, of the slice or of its token; act_scale), in the order of the
// codes, their sum as it is, and what takes a dot product back to its own scale.  It is made in
// four parts of a code word each (the words of raw numbers, the same number of words out), whose
// sums are added (0 + 1) + (2 + 3).
template <int BITS> constexpr int kPartWords = Fmt<BITS>::kElemsPer16B / 8;
// 2^-k for scale 2^k, as a pair of bf16 numbers: against it a dot product gives the unscaled sum
__device__ __forceinline__ uint32_t unscale_pair(float scale) {
  const uint32_t b = (254u << 23) - __float_as_uint(scale);
  return __builtin_amdgcn_perm(b, b, 0x03020302u);
}
// q * 2^-129 (2 bits: q * 2^-127) met x * scale
template <int BITS>
__device__ __forceinline__ float code_unscale(float scale) {
  return __uint_as_float(((BITS == kBits4 ? 383u : 381u) << 23) - __float_as_uint(scale));
}
// SCALED: the raw words are at that scale already; else *largest is raised to the part's largest magnitude (at that scale)
template <int BITS, bool SCALED>
__device__ __forceinline__ float expert_x_part(const uint32_t* raw, uint32_t* p, float scale, float* largest) {
  constexpr int kSpan = kPartWords<BITS> / 2;  // words between an element and the one in the other half of a code word
#pragma unroll
  for (int i = 0; i < kSpan; ++i) {
    const uint32_t lo = raw[i], hi = raw[kSpan + i];
    uint32_t even, odd;
    if constexpr (SCALED) {
      even = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
      odd = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
    } else {
      const float e0 = bf16_lo(lo) * scale, e1 = bf16_lo(hi) * scale, o0 = bf16_hi(lo) * scale, o1 = bf16_hi(hi) * scale;
      even = upper_halves(e0, e1);
      odd = upper_halves(o0, o1);
      *largest = fmaxf(*largest, fmaxf(fmaxf(fabsf(e0), fabsf(e1)), fmaxf(fabsf(o0), fabsf(o1))));
    }
    // 4 bits: codes 0..3 of a half word as they come; 2 bits: codes 0, 2, 4, 6 (lower place), then 1, 3, 5, 7
    p[BITS == kBits4 ? 2 * i : i] = even;
    p[BITS == kBits4 ? 2 * i + 1 : 4 + i] = odd;
  }
  const uint32_t ones = unscale_pair(scale);
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < 2 * kSpan; ++i) sum = dot2_bf16(p[i], ones, sum);
  return sum;
}
// A quarter of a slice by a thread, four adjacent ones a slice: its numbers (x) to where its blocks start (xq, ld apart), the slice's sum
// returned to all four.  scale 0: the slice's own, which is left there.  A thread's straight run of code is a quarter of a slice's:
// cold, it is fetched line by line.
template <int BITS, bool ALIGNED>
__device__ __forceinline__ float stage_expert_x_part(uint4* xq, uint32_t ld, const uint16_t* x, uint32_t part, float& scale) {
  constexpr int kW = kPartWords<BITS>;
  uint32_t raw[kW], p[kW];
#pragma unroll
  for (int q = 0; q < kW / 4; ++q) {
    const uint4 v = load_x8<ALIGNED>(x + part * (2 * kW) + 8 * q);
    raw[4 * q] = v.x; raw[4 * q + 1] = v.y; raw[4 * q + 2] = v.z; raw[4 * q + 3] = v.w;
  }
  float largest = 0.0f, sum;
  if (scale == 0.0f) {
    scale = kRowScale;
    sum = expert_x_part<BITS, false>(raw, p, scale, &largest);
    largest = fmaxf(largest, dpp_f<0xB1>(largest));
    largest = fmaxf(largest, dpp_f<0x4E>(largest));
    scale = row_scale(largest);
  }
  if (scale != kRowScale) sum = expert_x_part<BITS, false>(raw, p, scale, &largest);
  sum += dpp_f<0xB1>(sum);
  sum += dpp_f<0x4E>(sum);
#pragma unroll
  for (int q = 0; q < kW / 4; ++q) xq[(part * (kW / 4) + q) * ld] = make_uint4(p[4 * q], p[4 * q + 1], p[4 * q + 2], p[4 * q + 3]);
  return sum;
}
// n slices by the threads of a workgroup, into the layout that load_xslice_lds reads, each at a scale of its own:
// src(i, at) gives slice i's first element and where its blocks, its sum and what takes a dot product back go.
template <int BITS, bool ALIGNED, class Src>
__device__ __forceinline__ void stage_expert_x(uint4* xq, float2* xsum, uint32_t ld, uint32_t n, Src src) {
  for (uint32_t i = threadIdx.x; i < 4 * n; i += blockDim.x) {
    uint32_t at;
    const uint16_t* x = src(i >> 2, at);
    float scale = 0.0f;
    const float sum = stage_expert_x_part<BITS, ALIGNED>(xq + at, ld, x, i & 3u, scale);
    if ((i & 3u) == 0) xsum[at] = make_float2(sum, code_unscale<BITS>(scale));
  }
}
// ... n consecutive ones at a scale that is not the ordinary one
template <int BITS>
__device__ __forceinline__ void stage_expert_x(uint4* xq, float* xsum, uint32_t ld, uint32_t n, float scale, const uint16_t* x) {
  for (uint32_t i = threadIdx.x; i < 4 * n; i += blockDim.x) {
    const uint32_t sl = i >> 2;
    const float sum = stage_expert_x_part<BITS, true>(xq + sl, ld, x + sl * Fmt<BITS>::kElemsPer16B, i & 3u, scale);
    if ((i & 3u) == 0) xsum[sl] = sum;
  }
}
// *largest is raised to the slice's largest magnitude (at that scale)
template <int BITS, bool ALIGNED>
__device__ __forceinline__ XSlice<BITS> load_expert_x(const uint16_t* x, float scale, float* largest) {
  constexpr int kQuads = Fmt<BITS>::kElemsPer16B / 8;
  uint32_t raw[kQuads * 4];
#pragma unroll
  for (int q = 0; q < kQuads; ++q) {
    const uint4 a = load_x8<ALIGNED>(x + 8 * q);
    raw[4 * q] = a.x; raw[4 * q + 1] = a.y; raw[4 * q + 2] = a.z; raw[4 * q + 3] = a.w;
  }
  XSlice<BITS> xs;
  float sum[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) sum[j] = expert_x_part<BITS, false>(raw + j * kPartWords<BITS>, xs.p + j * kPartWords<BITS>, scale, largest);
  xs.sum = (sum[0] + sum[1]) + (sum[2] + sum[3]);
  xs.unscale = code_unscale<BITS>(scale);
  return xs;
}
// a slice out of its numbers as they come, at the scale already
template <int BITS>
__device__ __forceinline__ XSlice<BITS> permuted_expert_x(const XSlice<BITS>& raw, float scale) {
  XSlice<BITS> xs;
  float sum[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) sum[j] = expert_x_part<BITS, true>(raw.p + j * kPartWords<BITS>, xs.p + j * kPartWords<BITS>, scale, nullptr);
  xs.sum = (sum[0] + sum[1]) + (sum[2] + sum[3]);
  xs.unscale = code_unscale<BITS>(scale);
  return xs;
}
// four codes of every lane against four of its values
__device__ __forceinline__ f32x4_t lane_mfma(uint32_t a0, uint32_t a1, uint32_t x0, uint32_t x1, f32x4_t c) {
  typedef __attribute__((ext_vector_type(4))) short s16x4;
  return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4, make_uint2(a0, a1)),
                                                __builtin_bit_cast(s16x4, make_uint2(x0, x1)), c, 0, 0, 0);
}
__device__ __forceinline__ float lane_diagonal(const f32x4_t& c) {
  const uint32_t i = threadIdx.x;
  const float lo = i & 1u ? c[1] : c[0], hi = i & 1u ? c[3] : c[2];
  return i & 2u ? hi : lo;
}
// sum over the lane's share of q * x.  All lanes of the wave call it (the instruction knows no inactive lanes).
template <int BITS>
__device__ __forceinline__ float expert_dot(const uint4& codes, const XSlice<BITS>& xs) {
  const uint32_t ws[4] = {codes.x, codes.y, codes.z, codes.w};
  f32x4_t c = {0.0f, 0.0f, 0.0f, 0.0f};
  if constexpr (BITS == kBits4) {
    constexpr uint32_t kMask = 0x00F000F0u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t w = ws[j];
      c = lane_mfma((w << 4) & kMask, w & kMask, xs.p[4 * j], xs.p[4 * j + 1], c);
      c = lane_mfma((w >> 4) & kMask, (w >> 8) & kMask, xs.p[4 * j + 2], xs.p[4 * j + 3], c);
    }
    return lane_diagonal(c) * xs.unscale;
  } else {
    constexpr uint32_t kHigh = 0x00C000C0u, kLow = 0x00300030u;
    f32x4_t l = c;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t w = ws[j], up = w << 4, d4 = w >> 4, d8 = w >> 8;
      l = lane_mfma(up & kLow, w & kLow, xs.p[8 * j], xs.p[8 * j + 1], l);
      c = lane_mfma(up & kHigh, w & kHigh, xs.p[8 * j + 4], xs.p[8 * j + 5], c);
      l = lane_mfma(d4 & kLow, d8 & kLow, xs.p[8 * j + 2], xs.p[8 * j + 3], l);
      c = lane_mfma(d4 & kHigh, d8 & kHigh, xs.p[8 * j + 6], xs.p[8 * j + 7], c);
    }
    return __builtin_fmaf(lane_diagonal(l), 4.0f, lane_diagonal(c)) * xs.unscale;  // (the lower place's products are q * 2^-129)
  }
}

// The lane slices of x a routed row meets (XSlice: permuted pairs + their sum) depend on the token
// only, so a workgroup builds them once in LDS instead of once per row: slice sl of token t keeps
// its pairs as 16-byte blocks xq[(t * kQ + q) * n_sl + sl] (neighbouring lanes read neighbouring
// blocks) and its sum at xsum[t * n_sl + sl].
template <int BITS>
__device__ __forceinline__ void store_xslice_lds(uint4* xq, float* xsum, uint32_t t, uint32_t n_sl, uint32_t sl,
                                                 const XSlice<BITS>& xs) {
  constexpr uint32_t kQ = XSlice<BITS>::kPairs / 4;
#pragma unroll
  for (uint32_t q = 0; q < kQ; ++q)
    xq[(t * kQ + q) * n_sl + sl] = make_uint4(xs.p[4 * q], xs.p[4 * q + 1], xs.p[4 * q + 2], xs.p[4 * q + 3]);
  xsum[t * n_sl + sl] = xs.sum;
}
template <int BITS>
__device__ __forceinline__ XSlice<BITS> load_xslice_lds(const uint4* xq, uint32_t t, uint32_t n_sl, uint32_t sl, float sum, float unscale) {
  constexpr uint32_t kQ = XSlice<BITS>::kPairs / 4;
  XSlice<BITS> xs;
#pragma unroll
  for (uint32_t q = 0; q < kQ; ++q) {
    const uint4 v = xq[(t * kQ + q) * n_sl + sl];
    xs.p[4 * q] = v.x; xs.p[4 * q + 1] = v.y; xs.p[4 * q + 2] = v.z; xs.p[4 * q + 3] = v.w;
  }
  xs.sum = sum;
  xs.unscale = unscale;
  return xs;
}

// convenience form: one row against a slice loaded on the spot
template <int BITS, bool ALIGNED>
__device__ __forceinline__ void lane_dot(const uint4& codes, const uint16_t* x, float& dot,
                                         float& sum) {
  const XSlice<BITS> xs = load_xslice<BITS, ALIGNED ? kXAligned : kXUnaligned>(x);
  dot = codes_dot<BITS>(codes, xs);
  sum = xs.sum;
}

// A lane's 64 two-bit codes as two runs of 32 (a gate projection quantized at group 32 has a
// scale / bias entry for each): sum(q x) and sum(x) of either run.
template <bool ALIGNED>
__device__ __forceinline__ void lane_dot_halves_q2(const uint4& codes, const uint16_t* x, float (&dot)[2],
                                                   float (&sum)[2]) {
  uint32_t raw[32];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const uint4 a = load_x8<ALIGNED>(x + 8 * q);
    raw[4 * q] = a.x; raw[4 * q + 1] = a.y; raw[4 * q + 2] = a.z; raw[4 * q + 3] = a.w;
  }
  const uint32_t ws[4] = {codes.x, codes.y, codes.z, codes.w};
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    float s = 0.0f, d = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) s = dot2_bf16(raw[16 * half + i], kOnes, s);
#pragma unroll
    for (int j = 2 * half; j < 2 * half + 2; ++j) {
      const uint32_t w = ws[j];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        // code i of the word pairs with code i + 8: raw pairs (x_2i', x_2i'+1) regrouped as (x_i, x_i+8)
        const uint32_t lo = raw[8 * j + (i >> 1)], hi = raw[8 * j + 4 + (i >> 1)];
        const uint32_t xp = (i & 1) ? __builtin_amdgcn_perm(hi, lo, 0x07060302u) : __builtin_amdgcn_perm(hi, lo, 0x05040100u);
        const uint32_t cw = i < 3 ? w << (5 - 2 * i) : w >> (2 * i - 5);
        d = dot2_bf16(and_or(cw, 0x00600060u, kMagic4), xp, d);
      }
    }
    sum[half] = s;
    dot[half] = __builtin_fmaf(-4.0f, s, d);  // sum((4 + q) x) -> sum(q x)
  }
}

// scale / bias of the group that holds element e0 of a row whose tables start
// at srow / brow; ternary rows carry no bias table (bias = -scale).
template <int BITS>
__device__ __forceinline__ void load_scale_bias(const uint16_t* srow, const uint16_t* brow,
                                                uint32_t e0, float& s, float& b) {
  const uint32_t g = e0 / kGroup;
  s = bf16_to_f(srow[g]);
  if constexpr (BITS == kBitsTernary) b = -s;
  else b = bf16_to_f(brow[g]);
}

}  // namespace mf
