// tp_qjl.hip -- QJL residual sign sketches and the sketch score estimate.
//
// QJLResidualEncoder.compute_residual_sketch (rfsn_v11/quant/qjl/encoder.py:
// 30-44): proj = E @ W (W [dim][P] fp32, unit columns), bit p of a token's
// sketch = proj[p] >= 0, packed little-endian (bit i of byte j is projection
// 8j + i), and the residual norm f16(sqrt(sum E^2)).  Rows of 128 (the head
// size) take the matrix-core kernel, any other length one wave per row: lane p
// computes projection p (64 at a time) from the row and W staged in LDS, and one
// ballot yields 64 sketch bits.
//
// qjl_dot_estimate (rfsn_v11/quant/qjl/score_estimate.py:6-54): correction =
// |E| |q| sin(pi/2 * (P - 2 hamming) / P), the Hamming distance between the
// query's and the token's sketches, for every (query head, token); the query
// head reads the sketches of kv head h / g.  fp32 throughout.

#include "tp_common.h"

namespace tp {

constexpr int kQjlMaxDim = 256;
constexpr int kQjlMaxProj = 256;

template <bool F32IN>
__global__ __launch_bounds__(256) void qjl_sketch_kernel(const void* e, int64_t rows, int32_t dim, const float* w,
                                                         int32_t proj, uint8_t* packed, uint16_t* norms) {
  extern __shared__ float sm[];  // W [dim][proj], then one row of E per wave
  float* sw = sm;
  float* srow = sm + dim * proj + (threadIdx.x >> 6) * dim;
  for (int i = threadIdx.x; i < dim * proj; i += 256) sw[i] = w[i];
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int64_t waves = (int64_t)gridDim.x * 4;
  for (int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); row < rows; row += waves) {
    float ss = 0.0f;
    for (int d = lane; d < dim; d += 64) {
      const float x = F32IN ? static_cast<const float*>(e)[row * dim + d]
                            : h2f(static_cast<const uint16_t*>(e)[row * dim + d]);
      srow[d] = x;
      ss = __builtin_fmaf(x, x, ss);
    }
    wave_lds_sync();  // the row is in LDS for every lane of the wave
    for (int p0 = 0; p0 < proj; p0 += 64) {
      const int p = p0 + lane;
      float acc = 0.0f;
      if (p < proj) {
        for (int d = 0; d < dim; ++d) acc = __builtin_fmaf(srow[d], sw[d * proj + p], acc);
      }
      const uint64_t bits = __builtin_amdgcn_ballot_w64(p < proj && acc >= 0.0f);
      const int nbytes = min(8, (proj - p0) >> 3);
      if (lane < nbytes) packed[row * (proj >> 3) + (p0 >> 3) + lane] = (uint8_t)(bits >> (8 * lane));
    }
    if (norms) {
      for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
      if (lane == 0) norms[row] = f2h(sqrtf(ss));
    }
    wave_lds_sync();  // every lane is done with the row before the next overwrites it
  }
}

// fp32 rows of 128 values on v_mfma_f32_16x16x4_f32 (fp32 products and sums, as the
// scalar kernel's FMAs): a wave takes 16 rows x 16 projections, with its 32 W
// values per lane in registers for every row tile it walks, so nothing goes
// through LDS.  The k order is free as long as both operands follow it: lane
// group l4 holds k = 32 l4 .. +31, 128 contiguous bytes of its row.  The accumulator
// of lane (l16, l4) holds rows 4 l4 + i, projection l16, so one ballot per i yields
// 16 sketch bits of four rows.  Measured at 65,536 rows and 64 bits: 22.8 us (the
// scalar kernel above: 123).
constexpr int kSketchDim = 128;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Lane l16 < 4 of group l4 stores the two bytes of projections 16 ct .. +15 of
// row first + 4 l4 + l16 (nb sketch bytes a row; one byte past an odd row's end).
__device__ __forceinline__ void store_sketch(uint8_t* packed, int64_t first, int64_t rows, int nb, int ct, int l16, int l4,
                                             uint32_t bits) {
  const int64_t row = first + 4 * l4 + l16;
  if (l16 >= 4 || row >= rows) return;
  uint8_t* dst = packed + row * nb + 2 * ct;
  if ((nb & 1) == 0) {
    *reinterpret_cast<uint16_t*>(dst) = (uint16_t)bits;
  } else {
    dst[0] = (uint8_t)bits;
    if (2 * ct + 1 < nb) dst[1] = (uint8_t)(bits >> 8);
  }
}

// The norm of row first + l16 from its four lanes' sums of squares.
__device__ __forceinline__ void store_norm(uint16_t* norms, int64_t first, int64_t rows, int l16, int l4, float ss) {
  ss += __shfl_xor(ss, 16, 64);
  ss += __shfl_xor(ss, 32, 64);
  if (l4 == 0 && first + l16 < rows) norms[first + l16] = f2h(sqrtf(ss));
}

__global__ __launch_bounds__(256) void qjl_sketch_f32_kernel(const float* e, int64_t rows, const float* w, int32_t proj,
                                                              uint8_t* packed, uint16_t* norms) {
  const int lane = threadIdx.x & 63;
  const int l16 = lane & 15;
  const int l4 = lane >> 4;
  const int ct = __builtin_amdgcn_readfirstlane(blockIdx.y * 4 + (threadIdx.x >> 6));  // projections 16 ct .. +15
  if (16 * ct >= proj) return;
  const int col = 16 * ct + l16;
  float wb[32];
#pragma unroll
  for (int k = 0; k < 32; ++k) wb[k] = w[(32 * l4 + k) * proj + min(col, proj - 1)];
  const int nb = proj >> 3;  // sketch bytes per row
  const bool want_norms = norms && ct == 0;
  // Row tile rt of this lane: 32 values of row 16 rt + l16 (rows past the end
  // reread the last one and store nothing).
  auto load = [&](int64_t rt, float4v* raw) {
    const int64_t row = min(rt * 16 + l16, rows - 1);
    const float4v* src = reinterpret_cast<const float4v*>(e + row * kSketchDim + 32 * l4);
#pragma unroll
    for (int i = 0; i < 8; ++i) raw[i] = src[i];
  };
  const int64_t tiles = (rows + 15) / 16;
  float4v raw[8];
  load(blockIdx.x, raw);
  for (int64_t rt = blockIdx.x; rt < tiles; rt += gridDim.x) {
    float x[32];
#pragma unroll
    for (int k = 0; k < 32; ++k) x[k] = raw[k >> 2][k & 3];
    load(min(rt + gridDim.x, tiles - 1), raw);  // the next tile's rows travel under this one's products
    // Two chains of 16 products each: a chain's next product waits for its last.
    float4v acc = {0.0f, 0.0f, 0.0f, 0.0f}, acc2 = acc;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[k], wb[k], acc, 0, 0, 0);
      acc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(x[16 + k], wb[16 + k], acc2, 0, 0, 0);
    }
    acc += acc2;
    uint32_t bits = 0;  // lane l16 = i < 4: the 16 bits of row 4 l4 + i
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint64_t b = __builtin_amdgcn_ballot_w64(acc[i] >= 0.0f && col < proj);
      bits = l16 == i ? (uint32_t)(b >> (16 * l4)) & 0xffffu : bits;
    }
    store_sketch(packed, 16 * rt, rows, nb, ct, l16, l4, bits);
    if (want_norms) {
      float ss = 0.0f;
#pragma unroll
      for (int k = 0; k < 32; ++k) ss = __builtin_fmaf(x[k], x[k], ss);
      store_norm(norms, 16 * rt, rows, l16, l4, ss);
    }
  }
}

// The same for fp16 rows, on v_mfma_f32_16x16x32_f16, sixteen times the fp32
// matrix rate: the rows are operands as they are, and every W value, scaled by
// its column's power of two (which moves no sign), is the exact sum of three
// fp16 pieces of 11 bits each, w = p1 + 2^-11 p2 + 2^-22 p3 (33 bits; below
// 2^-39 of the column's largest the last ones go).  Each piece has sums of its
// own in fp32, so a projection errs as an fp32 chain over exact products does.
//
// Bound by latency and then by the rows' bytes, so the rows in flight count: a
// wave takes 32 rows against all 64 projections of its workgroup, whose pieces
// sit in LDS in operand order (48 KiB, one conflict-free 16-byte read per product
// operand, shared by both row tiles), and its first rows travel while the pieces
// are built.  (Each wave with 16 projections in registers and the workgroup on
// one row tile had a quarter of the bytes in flight: 13.5 us at 65,536 rows.)
constexpr float kPiece = 2048.0f;
constexpr int kSketchRows = 32;  // rows a wave takes at a time

__global__ __launch_bounds__(256) void qjl_sketch_f16_kernel(const uint16_t* e, int64_t rows, const float* w,
                                                             int32_t proj, uint8_t* packed, uint16_t* norms,
                                                             int32_t by_column) {
  __shared__ half8v s_w[4 * 3 * 4 * 64];  // [column tile][piece][k-step][lane]
  const int lane = threadIdx.x & 63;
  const int l16 = lane & 15;
  const int l4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // k-step ks of lane (l16, l4): k = 32 ks + 8 l4 .. +7, of both operands.
  auto load = [&](int64_t first, u32x4 (&raw)[2][4]) {
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int64_t row = min(first + 16 * m + l16, rows - 1);  // rows past the end reread the last one
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        raw[m][ks] = *reinterpret_cast<const u32x4*>(e + row * kSketchDim + 32 * ks + 8 * l4);
    }
  };
  u32x4 raw[2][4];
  const int64_t stride = (int64_t)gridDim.x * (by_column ? 1 : 4) * kSketchRows;
  int64_t first = (by_column ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * 4 + wave) * kSketchRows;
  load(first, raw);
  {  // wave w builds the pieces of column tile w
    const int col = min(64 * (int)blockIdx.y + 16 * wave + l16, proj - 1);
    float wv[32];
#pragma unroll
    for (int k = 0; k < 32; ++k) wv[k] = w[(32 * (k >> 3) + 8 * l4 + (k & 7)) * proj + col];
    float top = 0.0f;
#pragma unroll
    for (int k = 0; k < 32; ++k) top = fmaxf(top, fabsf(wv[k]));
    top = fmaxf(top, __shfl_xor(top, 16, 64));
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    // The column's largest value lands in [2^14, 2^15); a column of zeros or
    // with an infinity keeps its scale.
    const int shift = top > 0.0f && top < INFINITY ? 15 - __builtin_amdgcn_frexp_expf(top) : 0;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      half8v p[3];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x = __builtin_amdgcn_ldexpf(wv[8 * ks + j], shift);
        const f16 p1 = (f16)x;
        const float r1 = (x - (float)p1) * kPiece;
        const f16 p2 = (f16)r1;
        const float r2 = (r1 - (float)p2) * kPiece;
        const bool fine = fabsf((float)p1) < INFINITY;  // an infinity or NaN has no pieces below it
        p[0][j] = p1;
        p[1][j] = fine ? p2 : (f16)0.0f;
        p[2][j] = fine ? (f16)r2 : (f16)0.0f;
      }
#pragma unroll
      for (int q = 0; q < 3; ++q) s_w[((wave * 3 + q) * 4 + ks) * 64 + lane] = p[q];
    }
  }
  lds_barrier();
  const int nb = proj >> 3;  // sketch bytes per row
  for (; first < rows; first += stride) {
    half8v x[2][4];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) x[m][ks] = __builtin_bit_cast(half8v, raw[m][ks]);
    }
    if (first + stride < rows) load(first + stride, raw);  // the next rows travel under this tile's products
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (by_column && c != wave) continue;
      const int ct = 4 * (int)blockIdx.y + c;
      if (16 * ct >= proj) break;
      float4v acc[2][3];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
#pragma unroll
        for (int p = 0; p < 3; ++p) acc[m][p] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
      }
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          const half8v b = s_w[((c * 3 + p) * 4 + ks) * 64 + lane];
#pragma unroll
          for (int m = 0; m < 2; ++m) acc[m][p] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[m][ks], b, acc[m][p], 0, 0, 0);
        }
      }
      const bool live = 16 * ct + l16 < proj;
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        uint32_t bits = 0;  // lane l16 = i < 4: the 16 bits of row 4 l4 + i
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          // An infinite value makes acc[0] infinite with the projection's sign;
          // its lower pieces may have another.
          const float low = (acc[m][1][i] + acc[m][2][i] * (1.0f / kPiece)) * (1.0f / kPiece);
          const float v = fabsf(acc[m][0][i]) < INFINITY ? acc[m][0][i] + low : acc[m][0][i];
          const uint64_t b = __builtin_amdgcn_ballot_w64(v >= 0.0f && live);
          bits = l16 == i ? (uint32_t)(b >> (16 * l4)) & 0xffffu : bits;
        }
        store_sketch(packed, first + 16 * m, rows, nb, ct, l16, l4, bits);
      }
    }
    if (norms && blockIdx.y == 0 && (!by_column || wave == 0)) {
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        float ss = 0.0f;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
          for (int j = 0; j < 8; ++j) ss = __builtin_fmaf((float)x[m][ks][j], (float)x[m][ks][j], ss);
        }
        store_norm(norms, first + 16 * m, rows, l16, l4, ss);
      }
    }
  }
}

// sin(pi/2 * m / P) for the integer m = P - 2 hamming.
__device__ __forceinline__ float qjl_cos_est(int hamming, int proj) {
  return sinf(1.57079632679489662f * (float)(proj - 2 * hamming) / (float)proj);
}

__global__ __launch_bounds__(256) void qjl_estimate_kernel(const uint16_t* q, int32_t hq, int32_t g, int32_t dim,
                                                           const uint8_t* k_packed, const uint16_t* norms,
                                                           int64_t tokens, const uint8_t* q_packed, int32_t proj,
                                                           int64_t total, float* out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int64_t bhq = i / tokens;
  const int64_t t = i - bhq * tokens;
  const int64_t b = bhq / hq;
  const int64_t h = bhq - b * hq;
  const int64_t bkv = b * (hq / g) + h / g;
  float qq = 0.0f;
  for (int d = 0; d < dim; ++d) {
    const float x = h2f(q[bhq * dim + d]);
    qq = __builtin_fmaf(x, x, qq);
  }
  const int nb = proj >> 3;
  const uint8_t* ks = k_packed + (bkv * tokens + t) * nb;
  const uint8_t* qs = q_packed + bhq * nb;
  int ham = 0;
  for (int j = 0; j < nb; ++j) ham += __builtin_popcount((uint32_t)(ks[j] ^ qs[j]));
  out[i] = h2f(norms[bkv * tokens + t]) * sqrtf(qq) * qjl_cos_est(ham, proj);
}

}  // namespace tp

using namespace tp;

extern "C" {

int32_t tp_qjl_sketch(const void* e, int32_t in_dtype, int64_t rows, int32_t dim, const float* w, int32_t proj_dim,
                      uint8_t* packed, uint16_t* norms, void* stream) {
  clear_error();
  if (in_dtype != 0 && in_dtype != 1) {
    set_error("in_dtype must be 0 (float16) or 1 (float32), got %d", in_dtype);
    return TP_ERR_INVALID;
  }
  if (!e || !w || !packed || rows < 1 || dim < 1 || dim > kQjlMaxDim || proj_dim < 8 || proj_dim > kQjlMaxProj ||
      proj_dim % 8) {
    set_error("bad arguments: rows=%lld dim=%d proj_dim=%d (dim <= %d, proj_dim a multiple of 8 up to %d)",
              (long long)rows, dim, proj_dim, kQjlMaxDim, kQjlMaxProj);
    return TP_ERR_INVALID;
  }
  const size_t lds = ((size_t)dim * proj_dim + 4 * (size_t)dim) * sizeof(float);
  if (lds > 160 * 1024) {
    set_error("dim x proj_dim too large for one workgroup's LDS");
    return TP_ERR_INVALID;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  // 16-byte loads of the rows and 2-byte stores of the sketches.
  if (dim == kSketchDim && !((uintptr_t)e & 15u) && !((uintptr_t)packed & 1u)) {
    const unsigned cols = (unsigned)((proj_dim + 63) / 64);
    if (in_dtype) {
      // At most 768 workgroups, three a CU, per 64 projections, which then walk several row tiles on
      // one load of W (65,536 rows, 64 bits: 256 / 512 / 768 / 1024 / 2048 workgroups 27.7 / 22.2 /
      // 22.8 / 24.5 / 29.5 us).
      const unsigned x = (unsigned)std::min<int64_t>((rows + 15) / 16, 768);
      hipLaunchKernelGGL(qjl_sketch_f32_kernel, dim3(x, cols), dim3(256), 0, s, static_cast<const float*>(e), rows, w,
                         proj_dim, packed, norms);
    } else {
      // Few rows leave most CUs idle, so a wave then takes one column tile of its workgroup's rows.
      // Whole rows / column tiles, us: 32 rows 5.6 / 4.2, 8,192 6.5 / 4.7, 16,384 6.6 / 6.5, 32,768 6.7 / 9.2.
      const int by_column = rows <= 8192;
      const int per = (by_column ? 1 : 4) * kSketchRows;  // rows of a workgroup at a time
      // At most 768 workgroups per 64 projections here too, above 98,304 rows (64 bits, 256 / 512 /
      // 768 / 1024 / 2048 workgroups, us: 131,072 rows 16.2 / 12.7 / 12.6 / 14.0 / 14.0, 262,144 rows
      // 28.5 / 21.7 / 20.3 / 22.4 / 24.9, 1,048,576 rows 101 / 77 / 69 / 73 / 74).
      const unsigned x = (unsigned)std::min<int64_t>((rows + per - 1) / per, 768);
      hipLaunchKernelGGL(qjl_sketch_f16_kernel, dim3(x, cols), dim3(256), 0, s, static_cast<const uint16_t*>(e), rows, w,
                         proj_dim, packed, norms, by_column);
    }
    return launch_status("tp_qjl_sketch");
  }
  const unsigned blocks = (unsigned)std::min<int64_t>((rows + 3) / 4, 2048);
  if (in_dtype)
    hipLaunchKernelGGL(qjl_sketch_kernel<true>, dim3(blocks), dim3(256), lds, s, e, rows, dim, w, proj_dim, packed,
                       norms);
  else
    hipLaunchKernelGGL(qjl_sketch_kernel<false>, dim3(blocks), dim3(256), lds, s, e, rows, dim, w, proj_dim, packed,
                       norms);
  return launch_status("tp_qjl_sketch");
}

int32_t tp_qjl_dot_estimate(const void* q, int64_t batch, int32_t hq, int32_t hkv, int32_t dim, const void* k_packed,
                            const void* norms, int64_t tokens, const void* q_packed, int32_t proj_dim, float* out,
                            void* stream) {
  clear_error();
  if (!q || !k_packed || !norms || !q_packed || !out || batch < 1 || hq < 1 || hkv < 1 || hq % hkv || dim < 1 ||
      tokens < 1 || proj_dim < 8 || proj_dim % 8) {
    set_error("bad arguments: batch=%lld hq=%d hkv=%d dim=%d tokens=%lld proj_dim=%d", (long long)batch, hq, hkv, dim,
              (long long)tokens, proj_dim);
    return TP_ERR_INVALID;
  }
  const int64_t total = batch * hq * tokens;
  if ((total + 255) / 256 > INT32_MAX) {
    set_error("batch * hq * tokens too large for one launch");
    return TP_ERR_INVALID;
  }
  hipLaunchKernelGGL(qjl_estimate_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(q), hq, hq / hkv, dim,
                     static_cast<const uint8_t*>(k_packed), static_cast<const uint16_t*>(norms), tokens,
                     static_cast<const uint8_t*>(q_packed), proj_dim, total, out);
  return launch_status("tp_qjl_dot_estimate");
}

}  // extern "C"
