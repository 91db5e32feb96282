// tp_encode.hip -- page encoder: polar keys + grouped int8 values.
//
// Restates PolarQuantEncoder.encode_block (rfsn_v11/quant/polar/encoder.py:24-98)
// and GroupedVQuantizer.quantize_block (rfsn_v11/quant/v_quant/encoder.py:16-30)
// bit-exactly (see tp_common.h for the fp16 rules).
//
// One workgroup encodes one page (64 tokens of one (batch, kv head)); a thread
// owns NP key pairs of one token and the 2 NP values beside them.  NP = 16 (256
// threads; a thread's 32 values are one value group) has the fewest instructions
// per value, NP = 4 (1024 threads) the shortest chain per page, for launches that
// leave CUs idle anyway (launch_encode).  fp16 and fp32 input, the two layouts of
// the runtime with their code widths as constants and any other layout with its
// code rows packed through LDS share the kernel.
#include <type_traits>

#include "tp_common.h"

namespace tp {

struct EncodeArgs {
  const void* k;
  const void* v;
  int64_t in_tokens;
  int64_t token_begin;
  int64_t n_tokens;
  int32_t int8_radii;
  int32_t l1_bits;
  int32_t deep_bits;
  int32_t split_half;
  int32_t l1_row;
  int32_t deep_row;
  uint32_t l1_magic;  // ceil(2^20 / row bytes), 0 for an empty row
  uint32_t deep_magic;
  float l1_levels;    // 2^bits - 1
  float deep_levels;
  void* radii;
  uint16_t* radii_scales;
  uint8_t* angle_l1;
  uint8_t* angle_deep;
  int8_t* v_codes;
  uint16_t* v_scales;
  int64_t capacity;
  int64_t page_begin;
  // Append launches (tp_append_pages; flag NULL otherwise): a non-finite value
  // anywhere in the input stores epoch + 1 into the pinned host word `flag`.
  // The workgroups past the n_pages pages take each row's tokens outside them,
  // [0, n_head) and [rem_begin, in_tokens): checked, and copied to the dense
  // tail (head rows at tail_pos, the others at row 0 if copy_rem).
  uint32_t* flag;
  uint32_t epoch;
  int32_t n_pages;
  int64_t n_head;
  int64_t rem_begin;
  void* tail_k;
  void* tail_v;
  int64_t tail_tokens;
  int64_t tail_pos;
  int32_t copy_rem;
};

__device__ __forceinline__ void report_nonfinite(const EncodeArgs& a) {  // every writer stores the same value
  __hip_atomic_store(a.flag, a.epoch + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// True if any element of a 16-byte chunk is NaN or inf.
template <bool kF32>
__device__ __forceinline__ bool any_nonfinite(uint4 w) {
  const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
  bool bad = false;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (kF32)
      bad = bad || (ws[i] & 0x7f800000u) == 0x7f800000u;
    else
      bad = bad || (ws[i] & 0x7c00u) == 0x7c00u || (ws[i] & 0x7c000000u) == 0x7c000000u;
  }
  return bad;
}

// The tokens of row blockIdx.y outside the launch's whole pages, by one workgroup of
// the launch (256 or 1024 threads): at most 126 rows, a 16-byte chunk of k and of v
// at a time.
template <bool kF32>
__device__ __forceinline__ void edge_tokens(const EncodeArgs& a) {
  constexpr int kChunks = kHeadDim * (kF32 ? 4 : 2) / 16;  // per token row
  const int64_t bh = blockIdx.y;
  const int n_head = (int)a.n_head;
  const int n_rows = n_head + (int)(a.in_tokens - a.rem_begin);
  bool bad = false;
  for (int c = threadIdx.x; c < n_rows * kChunks; c += blockDim.x) {
    const int r = c / kChunks;
    const int part = c - r * kChunks;
    const bool head = r < n_head;
    const int64_t src = (bh * a.in_tokens + (head ? r : a.rem_begin + (r - n_head))) * kChunks + part;
    const uint4 kw = static_cast<const uint4*>(a.k)[src];
    const uint4 vw = static_cast<const uint4*>(a.v)[src];
    bad = bad || any_nonfinite<kF32>(kw) || any_nonfinite<kF32>(vw);
    if (head || a.copy_rem) {
      const int64_t dst = (bh * a.tail_tokens + (head ? a.tail_pos + r : r - n_head)) * kChunks + part;
      static_cast<uint4*>(a.tail_k)[dst] = kw;
      static_cast<uint4*>(a.tail_v)[dst] = vw;
    }
  }
  if (bad) report_nonfinite(a);
}

// N consecutive input values of one token row as they are in memory.
template <bool kF32, int N>
struct RawRow {
  uint4 w[N * (kF32 ? 4 : 2) / 16];
};

template <bool kF32, int N>
__device__ __forceinline__ void load_row(const void* base, int64_t off, RawRow<kF32, N>& r) {
  const uint4* p = kF32 ? reinterpret_cast<const uint4*>(static_cast<const float*>(base) + off)
                        : reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(base) + off);
#pragma unroll
  for (int i = 0; i < N * (kF32 ? 4 : 2) / 16; ++i) r.w[i] = p[i];
}

// Tokens past the end of the input were read from its last token: they encode as
// zeros (the zero padding of _maybe_encode_partial, turbo_polar_cache.py:280-285).
template <bool kF32, int N>
__device__ __forceinline__ void zero_row(RawRow<kF32, N>& r, bool valid) {
#pragma unroll
  for (int i = 0; i < N * (kF32 ? 4 : 2) / 16; ++i) {
    r.w[i].x = valid ? r.w[i].x : 0u;
    r.w[i].y = valid ? r.w[i].y : 0u;
    r.w[i].z = valid ? r.w[i].z : 0u;
    r.w[i].w = valid ? r.w[i].w : 0u;
  }
}

// Dword i of a raw row, and value i.
template <bool kF32, int N>
__device__ __forceinline__ uint32_t raw_word(const RawRow<kF32, N>& r, int i) {
  const uint4 w = r.w[i >> 2];
  return (i & 3) == 0 ? w.x : (i & 3) == 1 ? w.y : (i & 3) == 2 ? w.z : w.w;
}
template <bool kF32, int N>
__device__ __forceinline__ float raw_val(const RawRow<kF32, N>& r, int i) {
  if constexpr (kF32) return __uint_as_float(raw_word(r, i));
  const uint32_t w = raw_word(r, i >> 1);
  return h2f((uint16_t)((i & 1) ? (w >> 16) : (w & 0xffffu)));
}

// The largest bit pattern of |value| over a raw row: orders finite values and inf
// as fmaxf does and puts every NaN above inf (kInfBits<kF32> and above: not finite).
template <bool kF32>
constexpr uint32_t kInfBits = kF32 ? 0x7f800000u : 0x7c00u;
template <bool kF32, int N>
__device__ __forceinline__ uint32_t row_max_bits(const RawRow<kF32, N>& r) {
  if constexpr (kF32) {
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) m = max(m, raw_word(r, i) & 0x7fffffffu);
    return m;
  }
  u16x2 m = {0, 0};  // both halves of each word at once (v_pk_max_u16)
#pragma unroll
  for (int i = 0; i < N / 2; ++i)
    m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, raw_word(r, i) & 0x7fff7fffu));
  return max((uint32_t)m[0], (uint32_t)m[1]);
}

// Packs the codes of pairs [pair0, pair0 + npairs) of all 64 tokens into rows
// of `row_bytes` bytes (low bits first, zero padded: encoder.py:101-130).
// magic = ceil(2^20 / row_bytes): (i * magic) >> 20 = i / row_bytes for the byte
// indexes i < 64 row_bytes <= 4096 of a page (their error term i (row_bytes - 1)
// stays below 2^20).
__device__ __forceinline__ void pack_rows(uint8_t* dst, int row_bytes, uint32_t magic, int bits, int pair0,
                                          int npairs, const uint8_t* codes, int tid, int threads) {
  const int words = (kPageTokens * row_bytes) >> 2;
  const int per = 8 / bits;  // codes per byte
  for (int w = tid; w < words; w += threads) {
    uint32_t word = 0;
    int tt = (int)(((uint32_t)(4 * w) * magic) >> 20);
    int bb = 4 * w - tt * row_bytes;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const uint8_t* cr = codes + tt * kPairs + pair0;
      for (int s = 0; s < per; ++s) {
        const int i = per * bb + s;
        if (i < npairs) word |= (uint32_t)cr[i] << (8 * b + bits * s);
      }
      if (++bb == row_bytes) bb = 0, ++tt;
    }
    reinterpret_cast<uint32_t*>(dst)[w] = word;
  }
}

// The page's max |lr| over the workgroup's threads (NP fp16 values each) as the
// reference's reduction takes it: NaN propagates (a NaN log radius makes the
// maximum NaN, and with it the page scale and every radius code).  An integer
// maximum of the |lr| fp16 bit patterns orders finite values and inf as fmaxf
// does and puts every NaN above inf.  s_max: a word of LDS per wave.
template <int NP>
__device__ __forceinline__ float page_abs_max(const uint16_t (&lr)[NP], uint32_t* s_max, int tid) {
  constexpr int kWaves = kPageTokens / NP;
  uint32_t m = 0;
#pragma unroll
  for (int j = 0; j < NP; ++j) m = max(m, (uint32_t)(lr[j] & 0x7fffu));
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, off, 64));
  if ((tid & 63) == 0) s_max[tid >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kWaves; ++i) m = max(m, s_max[i]);
  return h2f((uint16_t)m);
}

// ---- fast arithmetic, exact where it cannot vouch for itself ------------------
//
// Every fp32 step whose rounding is in doubt only sets a per-lane flag; flagged
// pairs and value groups are redone exactly after the main loop, so codes and
// scales are those of the reference's operation sequence, bit for bit.  The
// byte conversion v_cvt_pk_u8_f32 rounds half to even, saturates and places the
// byte in one instruction.

// The runtime's two layouts (4-bit level-1 and deep angles, split 64, fp16 radii;
// 8-bit deep angles, split 0, int8 log radii), and any other by its radii.
enum EncodeLayout { kEncDefault = 0, kEncFast = 1, kEncAnyF16 = 2, kEncAnyI8 = 3 };

// x (an fp32 value holding an fp16 number) times s in fp32, rounded once: an
// explicit FMA with a +0 addend, which the backend takes as one mixed-precision
// FMA (v_fma_mix_f32) reading the fp16 operand directly.  A -0 product reads
// as +0; the callers only test the result's distance from fp16 rounding
// midpoints, which the sign of zero does not change.
__device__ __forceinline__ float mul_f16_f32(float x, float s) { return __builtin_fmaf(x, s, 0.0f); }

// fp16 (a16 + pi) as fp32, the numerator of the angle code (encoder.py:46-50).
__device__ __forceinline__ float code_numerator(uint16_t a16) { return h2f(f2h(h2f(a16) + h2f(kF16Pi))); }

// The fast path's angle code of an fp16 pair (x, y), as the argument of the byte
// conversion, and whether it cannot be trusted: the fp32 atan2 lies near an
// fp16 rounding midpoint or is NaN (a NaN x or y, whose code is the NaN
// angle's 0, or two infinite components, an odd multiple of pi/4; atan2_poly
// propagates both as NaN).  An angle below 2^-14
// leaves fp16(a + pi) = fp16(pi) whichever way it rounds, so the guard needs
// no subnormal test, and atan2(+-0, x >= 0) = +-0 comes out of atan2_poly
// exactly.  The quotient needs no guard: for every fp16 numerator s1 the fp32
// product s1 * fp32(1 / fp16(2 pi)), rounded once, rounds to the same fp16 as
// the fp16 division s1 / fp16(2 pi) (checked over all 65536 fp16 values by
// tests/test_oracle_pins.py and, through this function, by
// atan2_exhaustive_kernel).  It needs no clamp: a non-NaN atan2 lies in [-pi,
// pi], whose fp16 rounding lies in [-fp16(pi), fp16(pi)] (pi is below the
// midpoint between fp16(pi) and the next fp16 value), so the shifted angle lies
// in [0, fp16(2 pi)] and its quotient in [0, 1].
// xy: the pair's raw fp16 word (y in the high half), whose top bit is the
// sign of y that the angle takes (one bit-field insert).  levels: 2^bits - 1, one
// mixed-precision FMA reading the fp16 quotient.
__device__ __forceinline__ float angle_arg_fast(float x, float y, uint32_t xy, float levels, bool* flag) {
  const float a = __uint_as_float((__float_as_uint(atan2_poly_mag(y, x)) & 0x7fffffffu) | (xy & 0x80000000u));
  const float q = mul_f16_f32(code_numerator(f2h(a)), kF32InvF16TwoPi);
  *flag = near_f16_midpoint_code<kGuardAtan2>(a) | __builtin_isnan(a);
  return __builtin_fmaf(h2f(f2h(q)), levels, 0.0f);
}

// Exact angle code of an fp16 pair (x, y): correctly rounded fp16 atan2, except that
// the float64 atan2 runs only when the two fp16 candidates around the fast
// result's rounding midpoint give different codes.  A NaN x or y gives the
// NaN angle's code, 0 (angle_code_f16); two infinite components take the
// float64 atan2.
__device__ __forceinline__ uint32_t exact_angle_code(float y, float x, int bits) {
  if (__builtin_isunordered(x, y)) return 0u;
  const float a = atan2_poly(y, x);
  if (__builtin_isnan(a)) return angle_code_f16(atan2_f16_slow(y, x), bits);
  const uint16_t a16 = f2h(a);
  const uint32_t c0 = angle_code_f16(a16, bits);
  if (!near_f16_midpoint_code<kGuardAtan2>(a)) return c0;
  // The fast fp32 angle lies within kGuardAtan2 ulps of the midpoint between
  // a16 and the neighbour on its side; the correctly rounded value is one of
  // the two.
  const float d = a - h2f(a16);
  const uint16_t nb = (uint16_t)(a16 + ((d > 0.0f) == !(a16 & 0x8000u) ? 1 : -1));
  if ((a16 & 0x7fffu) == 0 || angle_code_f16(nb, bits) != c0) return angle_code_f16(atan2_f16_slow(y, x), bits);
  return c0;
}

// The same for fp32 pairs, whose angle stays fp32 (encoder.py:47-55).  Within
// 2^-30 <= max(|x|, |y|) <= 2^120 (outside: flagged, with every NaN and inf) the
// ratio and the polynomial err by a few fp32 ulps of the angle, less than 6 ulps
// of pi together (1.5e-6); the turn and its product with 255 levels add two
// roundings, so the argument errs by less than 1e-4: it is trusted 2^-12 or more
// from a half-integer, and a turn below the wrap to 0 at 1 - 1e-6 by 2.8e-6.
constexpr float kInvF32TwoPi = 0.159154936671257019f;  // fp32(1 / fp32(2 pi))
__device__ __forceinline__ float angle_arg_f32(float x, float y, float levels, bool* flag) {
  const float mx = fmaxf(fabsf(x), fabsf(y));
  const float n = (atan2_poly(y, x) + kF32Pi) * kInvF32TwoPi;
  const float arg = n * levels;
  *flag = !(mx >= 0x1p-30f && mx <= 0x1p120f) | !(fabsf(__builtin_amdgcn_fractf(arg) - 0.5f) > 0x1p-12f) |
          (n > 1.0f - 0x1p-18f);
  return arg;
}
__device__ inline __attribute__((noinline)) float atan2_f32_slow(float y, float x) {
  return (float)atan2((double)y, (double)x);
}
__device__ __forceinline__ uint32_t exact_angle_code_f32(float y, float x, int bits) {
  // On the axis (zero pairs above all) the angle needs no arctangent.
  if (y == 0.0f && x == x) return angle_code_f32(__builtin_signbit(x) ? __builtin_copysignf(kF32Pi, y) : y, bits);
  return angle_code_f32(atan2_f32_slow(y, x), bits);
}

// fp32 pairs' radius (encoder.py:33): f16(sqrt(x*x + y*y)) with fp32 ops.  v_sqrt_f32
// is within 1 ulp, so its fp16 rounding is the correctly rounded root's unless it
// lies next to an fp16 midpoint (roots below 2^-14 included: fp16's subnormal
// midpoints are not 2^13 apart); then the correctly rounded root decides.
__device__ __forceinline__ uint16_t radius_f32_fast(float x, float y) {
  const float xx = x * x;
  const float yy = y * y;
  const float ss = xx + yy;
  const float r = __builtin_amdgcn_sqrtf(ss);
  return near_f16_midpoint<kGuardDiv>(r) ? f2h(sqrtf(ss)) : f2h(r);
}

// Biased byte (code + 128) of value v with scale s = 1/rs by the fast path,
// written into byte `sel` of `old`, and whether the fp32 quotient is too close
// to an fp16 midpoint to trust.
// one: 1.0f, which the caller hides from the compiler (an empty asm that
// yields it in an SGPR) so that fp16(q) * 1 + 128 stays one mixed-precision FMA
// reading the fp16 value instead of a conversion and an add; x * 1 is exact,
// so it rounds as the fp32 sum does.
__device__ __forceinline__ uint32_t vcode_fast_byte(float v, float rs, float one, uint32_t sel, uint32_t old,
                                                    bool* near) {
  const float q = mul_f16_f32(v, rs);
  *near = near_f16_midpoint_code<kGuardDiv>(q);
  return __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(h2f(f2h(q)), one, 128.0f), sel, old);
}
// 1.0f in an SGPR, opaque to the compiler's constant folding.
__device__ __forceinline__ float opaque_one() {
  float one;
  asm volatile("s_mov_b32 %0, 1.0" : "=s"(one));
  return one;
}
// The same byte from the correctly rounded quotient, NaN -> code 0.
__device__ __forceinline__ uint32_t vcode_exact_byte(float v, float s) {
  const float qn = h2f(f2h(v / s));
  return __builtin_amdgcn_cvt_pk_u8_f32((qn == qn ? qn : 0.0f) + 128.0f, 0u, 0u);
}

// fp32 values: the quotient stays fp32, so the code is rint(fp32(v / s)).  One FMA
// v * rs + 128 is within 2^-15 of v / s + 128 where the code is not clipped (the
// reciprocal 2^-23 relative, the sum 2^-17), trusted 2^-13 or more from a half-integer.
__device__ __forceinline__ uint32_t vcode_f32_fast_byte(float v, float rs, uint32_t sel, uint32_t old, bool* near) {
  const float qb = __builtin_fmaf(v, rs, 128.0f);
  *near = fabsf(__builtin_amdgcn_fractf(qb) - 0.5f) <= 0x1p-13f;
  return __builtin_amdgcn_cvt_pk_u8_f32(qb, sel, old);
}
__device__ __forceinline__ uint32_t vcode_f32_exact_byte(float v, float s) {
  return (uint32_t)(to_int8_rne(v / s) & 0xff) ^ 0x80u;
}

// Biased byte (code + 128) of the int8 log-radius code rint(lr / ls) of the
// fp16 log radius lr16 by the fast path, rl = 1 / ls by v_rcp_f32, written
// into byte `sel` of `old`, and whether it must be redone.  The fast path
// forms lr * rl + 128 in one FMA: the reciprocal is within 1 ulp, so for
// |lr / ls| < 127.1 (lr is at most the page's max |lr| and ls its fp16 / 127)
// the product is within 2^-16 of the exact quotient and the rounded sum within
// 1.5 * 2^-16 of quotient + 128; rint agrees with the reference's unless the
// sum lies within 2^-13 of a half-integer.  The sum is positive, and the byte
// conversion rounds half to even.
__device__ __forceinline__ uint32_t lcode_fast_byte(uint16_t lr16, float rl, uint32_t sel, uint32_t old,
                                                    bool* near) {
  const float qb = __builtin_fmaf(h2f(lr16), rl, 128.0f);
  // v_fract_f32 is qb - floor(qb) here (0 < qb < 256; it caps just below 1).
  *near = fabsf(__builtin_amdgcn_fractf(qb) - 0.5f) <= 0x1p-13f;
  return __builtin_amdgcn_cvt_pk_u8_f32(qb, sel, old);
}
// The same byte from the correctly rounded fp32 quotient lr / ls (NaN -> code
// 0).  The quotient of two fp16 values is a half-integer exactly or lies at
// least 2^-13 from one, so adding 128 (one rounding at 2^-16) keeps rint's
// answer, and a tie stays a tie whose even neighbour is shifted by 128.
__device__ __forceinline__ uint32_t lcode_exact_byte(uint16_t lr16, float ls) {
  const float qd = h2f(lr16) / ls;
  return __builtin_amdgcn_cvt_pk_u8_f32((qd == qd ? qd : 0.0f) + 128.0f, 0u, 0u);
}

// Per-lane masks of the items the fast path cannot vouch for are built most
// significant first: push_flag shifts the mask up and ORs the new item's flag
// in (a 0/1 select and a shift-or, where a bit of its own per item would need
// a 32-bit constant in a register for every item past the sixth), so item j
// of n sits in bit n - 1 - j.
__device__ __forceinline__ uint32_t push_flag(uint32_t m, bool f) { return (m << 1) | (f ? 1u : 0u); }

// N words to consecutive addresses, as wide as they are.
template <int N>
__device__ __forceinline__ void store_words(void* p, const uint32_t* w) {
  if constexpr (N >= 4) {
#pragma unroll
    for (int i = 0; i < N / 4; ++i)
      static_cast<uint4*>(p)[i] = make_uint4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
  } else if constexpr (N == 2) {
    *static_cast<uint2*>(p) = make_uint2(w[0], w[1]);
  } else {
    *static_cast<uint32_t*>(p) = w[0];
  }
}

// The page encoder.  Bound by instruction issue on large launches (NP = 16) and by
// the length of one page's chain on small ones (NP = 4).
//
// The non-finite check of an append (a.flag) rides on the values in registers:
// a packed maximum of the key words, and the value groups' maxima that the
// scales need anyway.  A check kernel of its own read the whole input a second
// time (24 us for 32,773 tokens of 8 heads beside 39 of encoding).
//
// kPart: the last page is partial.  A launch of whole pages has no test of the
// token, whose join would hold the first products back until every row has come.
template <bool kF32, int L, int NP, bool kPart>
__global__ __launch_bounds__(kPageTokens * kPairs / NP) void encode_kernel(EncodeArgs a) {
  constexpr bool kAny = L == kEncAnyF16 || L == kEncAnyI8;
  constexpr bool kI8 = L == kEncFast || L == kEncAnyI8;
  constexpr bool kNibbles = L == kEncDefault;     // code words hold nibbles, else bytes
  constexpr int kThreads = kPageTokens * kPairs / NP;
  constexpr int kPer = kPairs / NP;               // threads per token
  constexpr int NV = 2 * NP;                      // values per thread
  constexpr int kCodeWords = kNibbles ? (NP + 7) / 8 : NP / 4;
  __shared__ uint32_t s_max[kThreads / 64];
  __shared__ uint32_t s_codes[kAny ? kPageTokens * kPairs / 4 : 1];

  if (a.flag && (int)blockIdx.x == a.n_pages) {
    edge_tokens<kF32>(a);
    return;
  }
  const int page = blockIdx.x;
  const int64_t bh = blockIdx.y;
  const int tid = threadIdx.x;
  const int t = tid / kPer;
  const int qq = tid % kPer;
  const int p0 = NP * qq;  // the thread's first pair
  const int64_t local_tok = (int64_t)page * kPageTokens + t;
  const bool valid = !kPart || local_tok < a.n_tokens;
  const int64_t tok = valid ? local_tok : a.n_tokens - 1;
  const int64_t in_off = (bh * a.in_tokens + a.token_begin + tok) * kHeadDim + NV * qq;
  const int64_t slot = bh * a.capacity + a.page_begin + page;
  const int64_t row = slot * kPageTokens + t;
  // A launch without keys or without values reads the other's in their place.
  const void* k_in = kAny && !a.k ? a.v : a.k;
  const void* v_in = kAny && !a.v ? a.k : a.v;
  bool bad = false;

  RawRow<kF32, NV> kraw, vraw;
  load_row(k_in, in_off, kraw);
  // On large launches early value rows cost more in occupancy than their latency.
  if constexpr (NP == 4) load_row(v_in, in_off, vraw);

  if (!kAny || a.k) {
    if constexpr (kPart) zero_row(kraw, valid);
    bad = row_max_bits(kraw) >= kInfBits<kF32>;
    auto pair_bits = [&](int j) {  // angle bits of pair p0 + j
      if constexpr (L == kEncDefault) return 4;
      if constexpr (L == kEncFast) return 8;
      return p0 + j < a.split_half ? a.l1_bits : a.deep_bits;
    };
    uint16_t r16[NP];
    uint32_t cw[kCodeWords];
#pragma unroll
    for (int i = 0; i < kCodeWords; ++i) cw[i] = 0u;
    uint32_t fixa = 0;  // pairs whose angle code the fast path cannot vouch for
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      float levels;
      if constexpr (kAny)
        levels = p0 + j < a.split_half ? a.l1_levels : a.deep_levels;
      else
        levels = kNibbles ? 15.0f : 255.0f;
      bool flag;
      float arg;
      if constexpr (kF32) {
        const float x = raw_val(kraw, 2 * j), y = raw_val(kraw, 2 * j + 1);
        r16[j] = radius_f32_fast(x, y);
        arg = angle_arg_f32(x, y, levels, &flag);
      } else {
        const uint32_t w = raw_word(kraw, j);
        const half2v xy = __builtin_bit_cast(half2v, w);
        const half2v sq = xy * xy;  // fp16 products, as the reference squares in fp16 (no FMA)
        r16[j] = __builtin_bit_cast(uint16_t, __builtin_sqrtf16((f16)(sq[0] + sq[1])));  // correctly rounded
        arg = angle_arg_fast((float)xy[0], (float)xy[1], w, levels, &flag);
      }
      fixa = push_flag(fixa, flag);
      if constexpr (kNibbles)
        cw[j >> 3] |= __builtin_amdgcn_cvt_pk_u8_f32(arg, 0u, 0u) << (4 * (j & 7));
      else
        cw[j >> 2] = __builtin_amdgcn_cvt_pk_u8_f32(arg, (uint32_t)(j & 3), cw[j >> 2]);
    }
    // Exact redo of the flagged codes (padding tokens read as zeros).
    while (fixa) {
      const int j = NP - 1 - __builtin_ctz(fixa);
      fixa &= fixa - 1u;
      uint32_t c;
      if constexpr (kF32) {
        const float* kin = static_cast<const float*>(k_in) + in_off + 2 * j;
        c = exact_angle_code_f32(valid ? kin[1] : 0.0f, valid ? kin[0] : 0.0f, pair_bits(j));
      } else {
        const uint32_t w = valid ? *reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(k_in) + in_off + 2 * j) : 0u;
        c = exact_angle_code(h2f((uint16_t)(w >> 16)), h2f((uint16_t)(w & 0xffffu)), pair_bits(j));
      }
      constexpr int kBitsPer = kNibbles ? 4 : 8, kInWord = 32 / kBitsPer;
      const uint32_t sh = (uint32_t)(kBitsPer * (j & (kInWord - 1)));
      const uint32_t mask = ((1u << kBitsPer) - 1u) << sh;
#pragma unroll
      for (int k2 = 0; k2 < kCodeWords; ++k2) cw[k2] = k2 == j / kInWord ? (cw[k2] & ~mask) | (c << sh) : cw[k2];
    }
    if constexpr (L == kEncDefault) {
      uint8_t* crow = (p0 < 32 ? a.angle_l1 : a.angle_deep) + row * 16 + (p0 & 31) / 2;
      if constexpr (NP == 16)
        store_words<2>(crow, cw);
      else
        *reinterpret_cast<uint16_t*>(crow) = (uint16_t)cw[0];
    } else if constexpr (L == kEncFast) {
      store_words<kCodeWords>(a.angle_deep + row * kPairs + p0, cw);
    } else {
      store_words<kCodeWords>(&s_codes[(t * kPairs + p0) / 4], cw);
    }

    if constexpr (kI8) {
      // encoder.py:34-42: lr = f32(f16 log(max(r, fp16(1e-6)))); per-page scale
      // f16(max|lr| / 127); codes rint(lr / scale).
      // The log radii stay fp16 (the reference's f16 log, widened exactly
      // wherever it is used).
      uint16_t lr[NP];
      uint32_t lfix = 0;
#pragma unroll
      for (int j = 0; j < NP; ++j) {
        const uint16_t rb = r16[j] > kF16RadiusFloor ? r16[j] : kF16RadiusFloor;
        bool exact;
        lr[j] = log_f16_fast(h2f(rb), &exact);
        lfix = push_flag(lfix, !exact);
      }
      while (lfix) {
        const int j = NP - 1 - __builtin_ctz(lfix);
        lfix &= lfix - 1u;
        uint16_t rb = 0;
#pragma unroll
        for (int k2 = 0; k2 < NP; ++k2) rb = k2 == j ? r16[k2] : rb;
        rb = rb > kF16RadiusFloor ? rb : kF16RadiusFloor;
        const uint16_t exact_lr = log_f16_slow(h2f(rb));
#pragma unroll
        for (int k2 = 0; k2 < NP; ++k2) lr[k2] = k2 == j ? exact_lr : lr[k2];
      }
      const float mx = page_abs_max<NP>(lr, s_max, tid);  // also orders s_codes' writes
      const float ls = mx == 0.0f ? 1e-6f : mx;
      const uint16_t ls16 = f2h(ls / 127.0f);
      const float lsf = h2f(ls16);
      // code = int8(clip(rint(f32(lr / ls)))) by lcode_fast_byte, the flagged
      // ones redone by lcode_exact_byte.  NaN quotients give code 0, and they
      // come only from a scale that is 0 (every lr is 0: 0 / 0), inf (lr / inf
      // is 0 or NaN) or NaN (a NaN lr): then every code of the page is 0, and
      // otherwise every lr is finite.
      const float rl = __builtin_amdgcn_rcpf(lsf);
      const bool zero_codes = !(lsf != 0.0f && fabsf(lsf) < INFINITY);  // uniform over the page
      uint32_t packed[NP / 4];
#pragma unroll
      for (int i = 0; i < NP / 4; ++i) packed[i] = 0x80808080u;
      uint32_t dfix = 0;
      if (!zero_codes) {
#pragma unroll
        for (int j = 0; j < NP; ++j) {
          bool near;
          packed[j >> 2] = lcode_fast_byte(lr[j], rl, (uint32_t)(j & 3), packed[j >> 2], &near);
          dfix = push_flag(dfix, near);
        }
      }
      while (dfix) {
        const int j = NP - 1 - __builtin_ctz(dfix);
        dfix &= dfix - 1u;
        uint16_t lj = 0;
#pragma unroll
        for (int k2 = 0; k2 < NP; ++k2) lj = k2 == j ? lr[k2] : lj;
        const uint32_t b = lcode_exact_byte(lj, lsf);
        const uint32_t sh = 8u * (uint32_t)(j & 3);
#pragma unroll
        for (int k2 = 0; k2 < NP / 4; ++k2)
          packed[k2] = k2 == (j >> 2) ? (packed[k2] & ~(0xffu << sh)) | (b << sh) : packed[k2];
      }
#pragma unroll
      for (int k2 = 0; k2 < NP / 4; ++k2) packed[k2] ^= 0x80808080u;  // biased bytes -> int8
      store_words<NP / 4>(static_cast<int8_t*>(a.radii) + row * kPairs + p0, packed);
      if (tid == 0) a.radii_scales[slot] = ls16;
    } else {
      uint32_t w[NP / 2];
#pragma unroll
      for (int i = 0; i < NP / 2; ++i) w[i] = (uint32_t)r16[2 * i] | ((uint32_t)r16[2 * i + 1] << 16);
      store_words<NP / 2>(static_cast<uint16_t*>(a.radii) + row * kPairs + p0, w);
    }
    if constexpr (kAny) {
      if constexpr (!kI8) __syncthreads();
      const uint8_t* codes = reinterpret_cast<const uint8_t*>(s_codes);
      if (a.l1_row > 0)
        pack_rows(a.angle_l1 + slot * kPageTokens * a.l1_row, a.l1_row, a.l1_magic, a.l1_bits, 0, a.split_half, codes,
                  tid, kThreads);
      if (a.deep_row > 0)
        pack_rows(a.angle_deep + slot * kPageTokens * a.deep_row, a.deep_row, a.deep_magic, a.deep_bits, a.split_half,
                  kPairs - a.split_half, codes, tid, kThreads);
    }
  }

  if (!kAny || a.v) {
    // Values (v_quant/encoder.py:21-25): s = f16(max|v| / 127) (1e-4 if zero),
    // code = int8(clip(rint(v / s), -128, 127)), the quotient rounded to fp16
    // first for fp16 input.  A NaN makes the group's maximum NaN (row_max_bits),
    // so the scale is NaN and every code 0.
    if constexpr (NP != 4) load_row(v_in, in_off, vraw);
    if constexpr (kPart) zero_row(vraw, valid);
    uint32_t mbits = row_max_bits(vraw);
    if constexpr (NP == 4) {  // a group is the values of four neighbouring threads
      mbits = max(mbits, (uint32_t)__shfl_xor((int)mbits, 1, 64));
      mbits = max(mbits, (uint32_t)__shfl_xor((int)mbits, 2, 64));
    }
    // inf or NaN in the group: exact path (v / inf and NaN quotients give code 0).
    const bool nonfinite = mbits >= kInfBits<kF32>;
    bad = bad || nonfinite;
    const float m = kF32 ? __uint_as_float(mbits) : h2f((uint16_t)mbits);
    uint16_t s16 = f2h(m / 127.0f);
    if ((s16 & 0x7fffu) == 0) s16 = kF16VScaleFloor;
    const float s = h2f(s16);
    const float rs = __builtin_amdgcn_rcpf(s);
    const float one = opaque_one();
    uint32_t vw[NV / 4];
    uint32_t vfix = 0;  // values whose quotient the fast path cannot vouch for
#pragma unroll
    for (int i = 0; i < NV / 4; ++i) vw[i] = 0u;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      bool near;
      if constexpr (kF32)
        vw[i >> 2] = vcode_f32_fast_byte(raw_val(vraw, i), rs, (uint32_t)(i & 3), vw[i >> 2], &near);
      else
        vw[i >> 2] = vcode_fast_byte(raw_val(vraw, i), rs, one, (uint32_t)(i & 3), vw[i >> 2], &near);
      vfix = push_flag(vfix, near);
    }
    if (nonfinite) vfix = NV == 32 ? 0xffffffffu : (1u << (NV & 31)) - 1u;
    while (vfix) {  // exact quotients of the flagged values, reloaded
      const int i = NV - 1 - __builtin_ctz(vfix);
      vfix &= vfix - 1u;
      uint32_t b;
      if constexpr (kF32)
        b = vcode_f32_exact_byte(valid ? static_cast<const float*>(v_in)[in_off + i] : 0.0f, s);
      else
        b = vcode_exact_byte(valid ? h2f(static_cast<const uint16_t*>(v_in)[in_off + i]) : 0.0f, s);
      const uint32_t sh = 8u * (uint32_t)(i & 3);
#pragma unroll
      for (int k2 = 0; k2 < NV / 4; ++k2) vw[k2] = k2 == (i >> 2) ? (vw[k2] & ~(0xffu << sh)) | (b << sh) : vw[k2];
    }
#pragma unroll
    for (int i = 0; i < NV / 4; ++i) vw[i] ^= 0x80808080u;  // biased bytes -> int8
    store_words<NV / 4>(a.v_codes + row * kHeadDim + NV * qq, vw);
    if (NP == 16 || (qq & 3) == 0) a.v_scales[row * kVGroups + NV * qq / 32] = s16;
  }
  if (a.flag && bad) report_nonfinite(a);
}

// ---- codec entry points for shapes outside the page encoder ----------------------
//
// GroupedVQuantizer.quantize_block for any group size dividing the row and any
// row length, and the int8 log radii of an L-token block with one scale per
// (b, h) row (PolarQuantEncoder.encode_block with use_int8_radii and L != 64).
// Off the decode path: plain, exact per-element arithmetic, no fast paths.

// One thread per group of `group` values of a row of `dim` (v_quant/encoder.py:
// 16-30): s = f16(max|v| / 127) (fp16(1e-4) if zero), code = int8(clip(rint(v
// / s))), the quotient rounded to fp16 first for fp16 input.  A NaN in the
// group makes the maximum NaN (nan_max), as in the page encoder.
template <bool F32IN>
__global__ __launch_bounds__(256) void quantize_groups_kernel(const void* v, int64_t n_groups, int32_t group,
                                                              int8_t* codes, uint16_t* scales) {
  const int64_t gi = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (gi >= n_groups) return;
  const int64_t base = gi * group;
  auto val = [&](int i) -> float {
    if constexpr (F32IN) return static_cast<const float*>(v)[base + i];
    else return h2f(static_cast<const uint16_t*>(v)[base + i]);
  };
  float m = 0.0f;
  for (int i = 0; i < group; ++i) m = max_abs_nan(m, val(i));
  uint16_t s16 = f2h(m / 127.0f);
  if ((s16 & 0x7fffu) == 0) s16 = kF16VScaleFloor;
  const float s = h2f(s16);
  for (int i = 0; i < group; ++i) {
    const float q = F32IN ? val(i) / s : h2f(f2h(val(i) / s));
    codes[base + i] = (int8_t)to_int8_rne(q);
  }
  scales[gi] = s16;
}

// One workgroup per (b, h) row of n fp16 radii (encoder.py:34-42): lr =
// f32(f16 log(max(r, fp16(1e-6)))), scale = f16(max|lr| / 127) (max 0 ->
// 1e-6), code = int8(clip(rint(lr / scale))).  A NaN log radius makes the
// maximum NaN (nan_max), as in the page encoder.
__global__ __launch_bounds__(256) void log_radii_rows_kernel(const uint16_t* radii, int64_t n, int8_t* codes,
                                                             uint16_t* scales) {
  __shared__ float s_max[256];
  const int64_t row = blockIdx.x;
  const uint16_t* r = radii + row * n;
  auto log_r = [&](int64_t i) -> float {
    const uint16_t rb = r[i] > kF16RadiusFloor ? r[i] : kF16RadiusFloor;
    return h2f(log_f16(h2f(rb)));
  };
  float m = 0.0f;
  for (int64_t i = threadIdx.x; i < n; i += 256) m = max_abs_nan(m, log_r(i));
  s_max[threadIdx.x] = m;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s_max[threadIdx.x] = nan_max(s_max[threadIdx.x], s_max[threadIdx.x + w]);
    __syncthreads();
  }
  const float mx = s_max[0];
  const uint16_t ls16 = f2h((mx == 0.0f ? 1e-6f : mx) / 127.0f);
  const float ls = h2f(ls16);
  for (int64_t i = threadIdx.x; i < n; i += 256) codes[row * n + i] = (int8_t)to_int8_rne(log_r(i) / ls);
  if (threadIdx.x == 0) scales[row] = ls16;
}

// ---- self-test kernels -------------------------------------------------------

__global__ __launch_bounds__(256) void f16_tables_kernel(uint16_t* sqrt_out, uint16_t* log_out,
                                                         uint8_t* codes_out) {
  const uint32_t b = blockIdx.x * 256u + threadIdx.x;
  const uint16_t hb = (uint16_t)b;
  sqrt_out[b] = sqrt_f16(h2f(hb));
  const uint16_t rb = (hb < 0x8000u && hb < kF16RadiusFloor) ? kF16RadiusFloor : hb;
  log_out[b] = log_f16(h2f(rb));
  codes_out[3 * b + 0] = (uint8_t)angle_code_f16(hb, 2);
  codes_out[3 * b + 1] = (uint8_t)angle_code_f16(hb, 4);
  codes_out[3 * b + 2] = (uint8_t)angle_code_f16(hb, 8);
}

__global__ __launch_bounds__(256) void atan2_exhaustive_kernel(unsigned long long* mismatches,
                                                               int32_t x_begin) {
  const uint32_t xb = (uint32_t)(x_begin + (int32_t)blockIdx.y) & 0xffffu;
  const uint32_t yb = blockIdx.x * 256u + threadIdx.x;
  uint32_t bad = 0;
  if ((xb & 0x7c00u) != 0x7c00u && (yb & 0x7c00u) != 0x7c00u) {
    const float x = h2f((uint16_t)xb);
    const float y = h2f((uint16_t)yb);
    const uint16_t fast = atan2_f16(y, x);
    const uint16_t ref = d2h(atan2((double)y, (double)x));
    bad = fast != ref ? 1u : 0u;
    // The specialised encoder's codes: the fast path where it vouches for its
    // result, else exact_angle_code (which skips the float64 atan2 when both
    // fp16 candidates give one code).
    bool f4, f8;
    const float g4 = angle_arg_fast(x, y, (yb << 16) | xb, 15.0f, &f4);
    const float g8 = angle_arg_fast(x, y, (yb << 16) | xb, 255.0f, &f8);
    const uint32_t c4 = f4 ? exact_angle_code(y, x, 4) : __builtin_amdgcn_cvt_pk_u8_f32(g4, 0u, 0u);
    const uint32_t c8 = f8 ? exact_angle_code(y, x, 8) : __builtin_amdgcn_cvt_pk_u8_f32(g8, 0u, 0u);
    bad |= c4 != angle_code_f16(ref, 4) ? 1u : 0u;
    bad |= c8 != angle_code_f16(ref, 8) ? 1u : 0u;
  }
  const unsigned long long ballot = __ballot(bad);
  if ((threadIdx.x & 63) == 0 && ballot) atomicAdd(mismatches, (unsigned long long)__popcll(ballot));
}

__global__ __launch_bounds__(256) void div_exhaustive_kernel(unsigned long long* mismatches, int32_t s_begin) {
  const uint32_t sb = (uint32_t)(s_begin + (int32_t)blockIdx.y) & 0x7fffu;
  const uint32_t vb = blockIdx.x * 256u + threadIdx.x;
  uint32_t bad = 0;
  if (sb != 0 && (sb & 0x7c00u) != 0x7c00u && (vb & 0x7c00u) != 0x7c00u) {
    const float s = h2f((uint16_t)sb);
    const float v = h2f((uint16_t)vb);
    const uint16_t fast = f2h(div_f16(v, s, __builtin_amdgcn_rcpf(s)));
    const uint16_t ref = f2h(v / s);
    bad = fast != ref ? 1u : 0u;
  }
  const unsigned long long ballot = __ballot(bad);
  if ((threadIdx.x & 63) == 0 && ballot) atomicAdd(mismatches, (unsigned long long)__popcll(ballot));
}

// Every finite value v against one positive finite scale per blockIdx.y: the
// fast V code byte (with its exact fallback) against the exact one.
__global__ __launch_bounds__(256) void vcode_exhaustive_kernel(unsigned long long* mismatches, int32_t s_begin) {
  const uint32_t sb = (uint32_t)(s_begin + (int32_t)blockIdx.y) & 0x7fffu;
  const uint32_t vb = blockIdx.x * 256u + threadIdx.x;
  uint32_t bad = 0;
  if (sb != 0 && (sb & 0x7c00u) != 0x7c00u && (vb & 0x7c00u) != 0x7c00u) {
    const float s = h2f((uint16_t)sb);
    const float v = h2f((uint16_t)vb);
    bool near;
    uint32_t fast = vcode_fast_byte(v, __builtin_amdgcn_rcpf(s), opaque_one(), 0u, 0u, &near);
    if (near) fast = vcode_exact_byte(v, s);
    const int32_t ref = to_int8_rne(h2f(f2h(v / s)));
    bad = (int32_t)(int8_t)(uint8_t)(fast ^ 0x80u) != ref ? 1u : 0u;
  }
  const unsigned long long ballot = __ballot(bad);
  if ((threadIdx.x & 63) == 0 && ballot) atomicAdd(mismatches, (unsigned long long)__popcll(ballot));
}

// Every finite fp16 log radius lr against one positive finite fp16 scale ls
// per blockIdx.y, over the quotients the encoder forms (|lr / ls| < 127.1):
// the fast log-radius code byte (with its exact fallback) against
// int8(clip(rint(f32(lr / ls)), -128, 127)).
__global__ __launch_bounds__(256) void lcode_exhaustive_kernel(unsigned long long* mismatches, int32_t s_begin) {
  const uint32_t sb = (uint32_t)(s_begin + (int32_t)blockIdx.y) & 0x7fffu;
  const uint32_t lb = blockIdx.x * 256u + threadIdx.x;
  uint32_t bad = 0;
  if (sb != 0 && (sb & 0x7c00u) != 0x7c00u && (lb & 0x7c00u) != 0x7c00u) {
    const float ls = h2f((uint16_t)sb);
    const float lr = h2f((uint16_t)lb);
    if (fabsf(lr) < 127.1f * ls) {
      bool near;
      uint32_t fast = lcode_fast_byte((uint16_t)lb, __builtin_amdgcn_rcpf(ls), 0u, 0u, &near);
      if (near) fast = lcode_exact_byte((uint16_t)lb, ls);
      const int32_t ref = to_int8_rne(lr / ls);
      bad = (int32_t)(int8_t)(uint8_t)(fast ^ 0x80u) != ref ? 1u : 0u;
    }
  }
  const unsigned long long ballot = __ballot(bad);
  if ((threadIdx.x & 63) == 0 && ballot) atomicAdd(mismatches, (unsigned long long)__popcll(ballot));
}

}  // namespace tp

using namespace tp;

// Checks one encode launch's arguments and fills `a` (no launch).
static int32_t fill_encode(EncodeArgs& a, const void* k, const void* v, int32_t in_dtype, int64_t bh,
                           int64_t in_tokens, int64_t token_begin, int64_t n_tokens,
                           const tp_page_layout* layout, const tp_pages* pages, int64_t page_begin) {
  int l1_row = 0, deep_row = 0;
  if (!check_layout(layout, &l1_row, &deep_row)) return TP_ERR_UNSUPPORTED;
  if (!pages) {
    set_error("pages is NULL");
    return TP_ERR_INVALID;
  }
  if (in_dtype != 0 && in_dtype != 1) {
    set_error("in_dtype must be 0 (float16) or 1 (float32), got %d", in_dtype);
    return TP_ERR_INVALID;
  }
  if (!k && !v) {
    set_error("k and v are both NULL");
    return TP_ERR_INVALID;
  }
  if (n_tokens == 0) return TP_OK;  // nothing to launch
  if (bh < 1 || bh > 65535 || n_tokens < 0 || token_begin < 0 || in_tokens < 0 ||
      token_begin + n_tokens > in_tokens) {
    set_error("bad token range: bh=%lld in_tokens=%lld token_begin=%lld n_tokens=%lld",
              (long long)bh, (long long)in_tokens, (long long)token_begin, (long long)n_tokens);
    return TP_ERR_INVALID;
  }
  const int64_t n_pages = (n_tokens + kPageTokens - 1) / kPageTokens;
  if (page_begin < 0 || page_begin + n_pages > pages->capacity || n_pages > 0x7fffffff) {
    set_error("page slots [%lld, %lld) exceed capacity %lld", (long long)page_begin,
              (long long)(page_begin + n_pages), (long long)pages->capacity);
    return TP_ERR_INVALID;
  }
  if (k) {
    if (!pages->radii || (l1_row > 0 && !pages->angle_l1) || (deep_row > 0 && !pages->angle_deep) ||
        (layout->int8_radii && !pages->radii_scales)) {
      set_error("key page buffers missing for this layout");
      return TP_ERR_INVALID;
    }
    if (((uintptr_t)k & 15u) || ((uintptr_t)pages->radii & 15u) ||
        ((uintptr_t)pages->angle_l1 & 3u) || ((uintptr_t)pages->angle_deep & 3u)) {
      set_error("k / key page buffers are not 16-byte aligned");
      return TP_ERR_INVALID;
    }
  }
  if (v) {
    if (!pages->v_codes || !pages->v_scales) {
      set_error("value page buffers missing");
      return TP_ERR_INVALID;
    }
    if (((uintptr_t)v & 15u) || ((uintptr_t)pages->v_codes & 15u) ||
        ((uintptr_t)pages->v_scales & 1u)) {
      set_error("v / value page buffers are not aligned");
      return TP_ERR_INVALID;
    }
  }
  a = EncodeArgs{};
  a.k = k;
  a.v = v;
  a.in_tokens = in_tokens;
  a.token_begin = token_begin;
  a.n_tokens = n_tokens;
  a.int8_radii = layout->int8_radii;
  a.l1_bits = layout->l1_bits;
  a.deep_bits = layout->deep_bits;
  a.split_half = layout->split_dim / 2;
  a.l1_row = l1_row;
  a.deep_row = deep_row;
  a.l1_magic = l1_row ? ((1u << 20) + l1_row - 1) / l1_row : 0;
  a.deep_magic = deep_row ? ((1u << 20) + deep_row - 1) / deep_row : 0;
  a.l1_levels = (float)((1 << layout->l1_bits) - 1);
  a.deep_levels = (float)((1 << layout->deep_bits) - 1);
  a.radii = pages->radii;
  a.radii_scales = static_cast<uint16_t*>(pages->radii_scales);
  a.angle_l1 = pages->angle_l1;
  a.angle_deep = pages->angle_deep;
  a.v_codes = pages->v_codes;
  a.v_scales = static_cast<uint16_t*>(pages->v_scales);
  a.capacity = pages->capacity;
  a.page_begin = page_begin;
  a.n_pages = (int32_t)n_pages;
  return TP_OK;
}

template <int L, int NP>
static void launch_encode_layout(const EncodeArgs& a, bool f32, dim3 grid, hipStream_t s) {
  const dim3 block(kPageTokens * kPairs / NP);
  const bool part = a.n_tokens % kPageTokens != 0;
  if (f32) {
    if (part)
      hipLaunchKernelGGL((encode_kernel<true, L, NP, true>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((encode_kernel<true, L, NP, false>), grid, block, 0, s, a);
  } else {
    if (part)
      hipLaunchKernelGGL((encode_kernel<false, L, NP, true>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((encode_kernel<false, L, NP, false>), grid, block, 0, s, a);
  }
}

// The page encoder's instance for a launch.  Pairs per thread (NP): launches that
// leave CUs without a page take the short chain (NP = 4), the others the one with
// fewer instructions.  Measured, NP = 16 / 4 and the kernels before (8 heads, us):
//   fp16 default   1 page 4.8 / 4.3 (4.9)    31 pages 7.1 / 6.1 (7.2)    512 pages 42.0 / 45.1 (42.5)
//   fp16 fast      1 page 7.1 / 6.3 (7.2)    31 pages 9.1 / 8.1 (9.1)    512 pages 50.7 / 65.9 (50.9)
//   fp16 2-bit     1 page 7.6 / 6.6 (11.1)   40 pages 11.6 / 11.2 (15.4) 512 pages 44.7 / 61.1 (56.9)
//   fp32 default   1 page 6.2 / 4.5 (10.3)   64 pages 12.9 / 11.2 (18.9) 512 pages 71.9 / 63.3 (87.7)
//   fp32 fast      1 page 8.4 / 6.4 (13.7)   64 pages 15.7 / 14.4 (23.1) 512 pages 70.9 / 75.6 (102.7)
// The lines at 256 and 512 pages are where a CU has one 1024-thread workgroup and
// two; fp32 pairs in the default layout stay ahead at NP = 4 (90 VGPRs at 16).
static void launch_encode(const EncodeArgs& a, int32_t in_dtype, int64_t bh, bool edge, hipStream_t s) {
  const dim3 grid((unsigned)(a.n_pages + (edge ? 1 : 0)), (unsigned)bh);  // `edge`: the tokens outside the pages
  const bool f32 = in_dtype != 0;
  // The runtime's two layouts store their code words straight to the rows.
  const bool both = a.k && a.v;
  const bool is_default = both && !a.int8_radii && a.l1_bits == 4 && a.deep_bits == 4 && a.split_half == 32 &&
                          !(((uintptr_t)a.angle_l1 | (uintptr_t)a.angle_deep) & 7u);
  const bool is_fast =
      both && a.int8_radii && a.deep_bits == 8 && a.split_half == 0 && !((uintptr_t)a.angle_deep & 15u);
  const bool short_chain = bh * a.n_pages <= (f32 ? 512 : 256) || (f32 && is_default);
  auto launch = [&](auto np) {
    constexpr int NP = decltype(np)::value;
    if (is_default)
      launch_encode_layout<kEncDefault, NP>(a, f32, grid, s);
    else if (is_fast)
      launch_encode_layout<kEncFast, NP>(a, f32, grid, s);
    else if (a.int8_radii)
      launch_encode_layout<kEncAnyI8, NP>(a, f32, grid, s);
    else
      launch_encode_layout<kEncAnyF16, NP>(a, f32, grid, s);
  };
  if (short_chain)
    launch(std::integral_constant<int, 4>());
  else
    launch(std::integral_constant<int, 16>());
}

extern "C" {

int32_t tp_encode_pages(const void* k, const void* v, int32_t in_dtype, int64_t bh,
                        int64_t in_tokens, int64_t token_begin, int64_t n_tokens,
                        const tp_page_layout* layout, const tp_pages* pages, int64_t page_begin,
                        void* stream) {
  clear_error();
  EncodeArgs a{};
  const int32_t st = fill_encode(a, k, v, in_dtype, bh, in_tokens, token_begin, n_tokens, layout, pages, page_begin);
  if (st != TP_OK || a.n_pages == 0) return st;
  launch_encode(a, in_dtype, bh, false, static_cast<hipStream_t>(stream));
  return launch_status("tp_encode_pages");
}

int32_t tp_append_pages(const void* k, const void* v, int32_t in_dtype, int64_t bh, int64_t in_tokens,
                        int64_t n_head, void* tail_k, void* tail_v, int64_t tail_tokens, int64_t tail_pos,
                        int32_t copy_rem, const tp_page_layout* layout, const tp_pages* pages, int64_t page_begin,
                        uint32_t* flag, uint32_t epoch, void* stream) {
  clear_error();
  if (!k || !v || n_head < 0 || n_head >= kPageTokens || in_tokens - n_head < kPageTokens) {
    set_error("bad input: k=%p v=%p, %lld tokens with %lld before the first whole page", k, v, (long long)in_tokens,
              (long long)n_head);
    return TP_ERR_INVALID;
  }
  if (!flag || (epoch & 1u)) {
    set_error("a pinned host flag and an even epoch are needed");
    return TP_ERR_INVALID;
  }
  const int64_t n_full = (in_tokens - n_head) / kPageTokens;
  EncodeArgs a{};
  const int32_t st =
      fill_encode(a, k, v, in_dtype, bh, in_tokens, n_head, n_full * kPageTokens, layout, pages, page_begin);
  if (st != TP_OK) return st;
  a.flag = flag;
  a.epoch = epoch;
  a.n_head = n_head;
  a.rem_begin = n_head + n_full * kPageTokens;
  const int64_t rem = in_tokens - a.rem_begin;
  if (n_head + rem > 0) {
    const bool copies = n_head > 0 || (copy_rem && rem > 0);
    if (copies && (!tail_k || !tail_v || (((uintptr_t)tail_k | (uintptr_t)tail_v) & 15u) || tail_pos < 0 ||
                   tail_pos + n_head > tail_tokens || (copy_rem && rem > tail_tokens) || (copy_rem && n_head > 0))) {
      set_error("tail buffers missing, misaligned or too small: %lld tokens at %lld and %lld at 0 of %lld",
                (long long)n_head, (long long)tail_pos, (long long)(copy_rem ? rem : 0), (long long)tail_tokens);
      return TP_ERR_INVALID;
    }
    a.tail_k = tail_k;
    a.tail_v = tail_v;
    a.tail_tokens = tail_tokens;
    a.tail_pos = tail_pos;
    a.copy_rem = copy_rem != 0;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  launch_encode(a, in_dtype, bh, n_head + rem > 0, s);
  const int32_t ls = launch_status("tp_append_pages");
  if (ls != TP_OK) return ls;
  return wait_verdict(flag, epoch, s, false, "tp_append_pages");
}

int32_t tp_selftest_f16_tables(uint16_t* sqrt_out, uint16_t* log_out, uint8_t* codes_out,
                               void* stream) {
  clear_error();
  if (!sqrt_out || !log_out || !codes_out) {
    set_error("output buffers must not be NULL");
    return TP_ERR_INVALID;
  }
  hipLaunchKernelGGL(f16_tables_kernel, dim3(256), dim3(256), 0, static_cast<hipStream_t>(stream),
                     sqrt_out, log_out, codes_out);
  return launch_status("tp_selftest_f16_tables");
}

int32_t tp_selftest_atan2_exhaustive(unsigned long long* mismatches, int32_t x_begin,
                                     int32_t x_count, void* stream) {
  clear_error();
  if (!mismatches || x_begin < 0 || x_count < 1 || x_begin + x_count > 65536 || x_count > 65535) {
    set_error("bad self-test range");
    return TP_ERR_INVALID;
  }
  hipLaunchKernelGGL(atan2_exhaustive_kernel, dim3(256, (unsigned)x_count), dim3(256), 0,
                     static_cast<hipStream_t>(stream), mismatches, x_begin);
  return launch_status("tp_selftest_atan2_exhaustive");
}

int32_t tp_quantize_v_groups(const void* v, int32_t in_dtype, int64_t rows, int32_t dim, int32_t group_size,
                             int8_t* codes, uint16_t* scales, void* stream) {
  clear_error();
  if (in_dtype != 0 && in_dtype != 1) {
    set_error("in_dtype must be 0 (float16) or 1 (float32), got %d", in_dtype);
    return TP_ERR_INVALID;
  }
  if (!v || !codes || !scales || rows < 1 || dim < 1 || group_size < 1 || dim % group_size) {
    set_error("bad arguments: rows=%lld dim=%d group_size=%d (the group size must divide dim)", (long long)rows,
              dim, group_size);
    return TP_ERR_INVALID;
  }
  const int64_t n_groups = rows * (dim / group_size);
  const unsigned blocks = (unsigned)((n_groups + 255) / 256);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (in_dtype)
    hipLaunchKernelGGL(quantize_groups_kernel<true>, dim3(blocks), dim3(256), 0, s, v, n_groups, group_size, codes,
                       scales);
  else
    hipLaunchKernelGGL(quantize_groups_kernel<false>, dim3(blocks), dim3(256), 0, s, v, n_groups, group_size, codes,
                       scales);
  return launch_status("tp_quantize_v_groups");
}

int32_t tp_log_radii_rows(const void* radii, int64_t rows, int64_t n, int8_t* codes, uint16_t* scales,
                          void* stream) {
  clear_error();
  if (!radii || !codes || !scales || rows < 1 || rows > INT32_MAX || n < 1) {
    set_error("bad arguments: rows=%lld n=%lld", (long long)rows, (long long)n);
    return TP_ERR_INVALID;
  }
  hipLaunchKernelGGL(log_radii_rows_kernel, dim3((unsigned)rows), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint16_t*>(radii), n, codes, scales);
  return launch_status("tp_log_radii_rows");
}

int32_t tp_selftest_vcode_exhaustive(unsigned long long* mismatches, int32_t s_begin, int32_t s_count,
                                     void* stream) {
  clear_error();
  if (!mismatches || s_begin < 0 || s_count < 1 || s_begin + s_count > 32768 || s_count > 65535) {
    set_error("bad self-test range");
    return TP_ERR_INVALID;
  }
  hipLaunchKernelGGL(vcode_exhaustive_kernel, dim3(256, (unsigned)s_count), dim3(256), 0,
                     static_cast<hipStream_t>(stream), mismatches, s_begin);
  return launch_status("tp_selftest_vcode_exhaustive");
}

int32_t tp_selftest_lcode_exhaustive(unsigned long long* mismatches, int32_t s_begin, int32_t s_count,
                                     void* stream) {
  clear_error();
  if (!mismatches || s_begin < 0 || s_count < 1 || s_begin + s_count > 32768 || s_count > 65535) {
    set_error("bad self-test range");
    return TP_ERR_INVALID;
  }
  hipLaunchKernelGGL(lcode_exhaustive_kernel, dim3(256, (unsigned)s_count), dim3(256), 0,
                     static_cast<hipStream_t>(stream), mismatches, s_begin);
  return launch_status("tp_selftest_lcode_exhaustive");
}

int32_t tp_selftest_div_f16_exhaustive(unsigned long long* mismatches, int32_t s_begin, int32_t s_count,
                                       void* stream) {
  clear_error();
  if (!mismatches || s_begin < 0 || s_count < 1 || s_begin + s_count > 32768) {
    set_error("bad self-test range");
    return TP_ERR_INVALID;
  }
  hipLaunchKernelGGL(div_exhaustive_kernel, dim3(256, (unsigned)s_count), dim3(256), 0,
                     static_cast<hipStream_t>(stream), mismatches, s_begin);
  return launch_status("tp_selftest_div_f16_exhaustive");
}

}  // extern "C"
