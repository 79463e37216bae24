// Producer side of the AutoAWQ format on the GPU: group-wise asymmetric int4 quantization
// of a float weight and the AWQ-order int4 packer (the reference's quantize_awq_weight and
// _pack_int4, llmserve/quantization/awq_calibration.py:19-62).  HBM-bound byte/integer work:
// the weight is read once and 0.5 byte per weight (plus scales and zeros) is written.
//
// quantize_kernel: one workgroup per (64 output features, one group of gs <= 128 inputs).
// The 64 x gs slice of W [out, in] (rows of gs contiguous values) is read coalesced into LDS
// as fp32 (at most 33 KiB); four threads per row reduce its min and max; the row's scale and
// zero follow the reference's fp32 arithmetic exactly
//   s = max(max - min, 1e-5) / 15      z = clamp(-rint(min / s), 0, 15)
//   q = clamp(rint(w / s) + z, 0, 15)  (rint = round half to even, as torch.round;
//                                        / is the correctly rounded IEEE division)
// and the transposed AutoAWQ words qweight[k, o / 8] are written 8 consecutive words (32
// bytes) per input row k.
#include "w4a16_common.h"
#include "w4a16_launch.h"

namespace w4a16 {

constexpr int kQuantRows = 64;  // output features per workgroup
constexpr int kQuantThreads = 256;

__device__ __forceinline__ float load_weight(const uint16_t* p, int dtype, size_t i) {
  const uint16_t b = p[i];
  if (dtype == kDtypeF16) return static_cast<float>(__builtin_bit_cast(_Float16, b));
  return bf16_bits_to_f32(b);
}

__global__ __launch_bounds__(kQuantThreads) void quantize_kernel(const void* __restrict__ weight, int dtype,
                                                                 uint32_t* __restrict__ qweight,
                                                                 uint32_t* __restrict__ qzeros,
                                                                 void* __restrict__ scales, int out_f, int in_f,
                                                                 int gs, bool vec) {
  extern __shared__ float tile[];  // [kQuantRows][gs + 1]
  __shared__ float row_s[kQuantRows];
  __shared__ float row_z[kQuantRows];
  const int pitch = gs + 1;  // odd pitch: the eight rows one packed word reads sit in distinct banks
  const int o0 = blockIdx.x * kQuantRows;
  const int g = blockIdx.y;
  const int rows = out_f - o0 < kQuantRows ? out_f - o0 : kQuantRows;  // a multiple of 8
  const int tid = threadIdx.x;

  if (vec) {
    // 16-byte loads: 8 values of a 16-bit type or 4 floats per load (gs a multiple of
    // either, weight 16-byte aligned; checked on the host).
    const int per = dtype == kDtypeF32 ? 4 : 8;
    const int cpr = gs / per;  // chunks per row
    for (int e = tid; e < rows * cpr; e += kQuantThreads) {
      const int r = e / cpr;
      const int c = (e - r * cpr) * per;
      const size_t i = static_cast<size_t>(o0 + r) * in_f + static_cast<size_t>(g) * gs + c;
      float* dst = tile + r * pitch + c;
      if (dtype == kDtypeF32) {
        const float4 v = *reinterpret_cast<const float4*>(static_cast<const float*>(weight) + i);
        dst[0] = v.x; dst[1] = v.y; dst[2] = v.z; dst[3] = v.w;
      } else {
        const uint4 v = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(weight) + i);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const uint16_t lo = static_cast<uint16_t>(w[h] & 0xFFFFu), hi = static_cast<uint16_t>(w[h] >> 16);
          dst[2 * h] = dtype == kDtypeF16 ? static_cast<float>(__builtin_bit_cast(_Float16, lo)) : bf16_bits_to_f32(lo);
          dst[2 * h + 1] = dtype == kDtypeF16 ? static_cast<float>(__builtin_bit_cast(_Float16, hi)) : bf16_bits_to_f32(hi);
        }
      }
    }
  } else {
    for (int e = tid; e < rows * gs; e += kQuantThreads) {
      const int r = e / gs;
      const int c = e - r * gs;
      const size_t i = static_cast<size_t>(o0 + r) * in_f + static_cast<size_t>(g) * gs + c;
      tile[r * pitch + c] = dtype == kDtypeF32 ? static_cast<const float*>(weight)[i]
                                               : load_weight(static_cast<const uint16_t*>(weight), dtype, i);
    }
  }
  __syncthreads();

  // Min and max of row r = tid / 4 over its quarter of the group; NaN propagates as in
  // torch's amin / amax.
  static_assert(kQuantThreads == 4 * kQuantRows, "four threads per row");
  {
    const int r = tid >> 2;
    const int h = tid & 3;
    const int part = (gs + 3) >> 2;
    const int c_end = (h + 1) * part < gs ? (h + 1) * part : gs;
    float mn = __builtin_inff(), mx = -__builtin_inff();
    if (r < rows) {
      for (int c = h * part; c < c_end; ++c) {
        const float v = tile[r * pitch + c];
        mn = (v < mn || v != v) ? v : mn;
        mx = (v > mx || v != v) ? v : mx;
      }
    }
#pragma unroll
    for (int d = 1; d <= 2; d <<= 1) {
      const float mn2 = __shfl_xor(mn, d);
      const float mx2 = __shfl_xor(mx, d);
      mn = (mn2 < mn || mn2 != mn2) ? mn2 : mn;
      mx = (mx2 > mx || mx2 != mx2) ? mx2 : mx;
    }
    if (h == 0 && r < rows) {
      float d = mx - mn;
      d = d < 1e-5f ? 1e-5f : d;  // torch clamp(min=): NaN stays NaN
      const float s = d / 15.0f;
      float z = -__builtin_rintf(mn / s);
      z = z < 0.f ? 0.f : (z > 15.f ? 15.f : z);
      row_s[r] = s;
      row_z[r] = z;
      const size_t si = static_cast<size_t>(g) * out_f + o0 + r;
      if (dtype == kDtypeF32) static_cast<float*>(scales)[si] = s;
      else if (dtype == kDtypeF16) static_cast<_Float16*>(scales)[si] = static_cast<_Float16>(s);
      else static_cast<uint16_t*>(scales)[si] = f32_to_bf16_bits(s);
    }
  }
  __syncthreads();

  const int W = rows / 8;     // packed words per input row in this workgroup
  const int C8 = out_f / 8;   // packed words per input row
  if (tid < W) {
    uint32_t word = 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) word |= (static_cast<uint32_t>(row_z[8 * tid + c]) & 0xFu) << awq_shift(c);
    qzeros[static_cast<size_t>(g) * C8 + o0 / 8 + tid] = word;
  }
  for (int e = tid; e < gs * W; e += kQuantThreads) {
    const int k = e / W;
    const int j = e - k * W;
    uint32_t word = 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int r = 8 * j + c;
      float q = __builtin_rintf(tile[r * pitch + k] / row_s[r]) + row_z[r];
      q = q < 0.f ? 0.f : (q > 15.f ? 15.f : q);
      word |= (static_cast<uint32_t>(q) & 0xFu) << awq_shift(c);
    }
    qweight[(static_cast<size_t>(g) * gs + k) * C8 + o0 / 8 + j] = word;
  }
}

// Fast path for GS in {32, 64, 128} (the same results, bit for bit): 128 output rows per
// workgroup, four threads per row, each holding its GS / 4 consecutive values in registers
// (16-byte loads); the row's min and max come from two lane shuffles.  Only the 4-bit codes
// go through LDS, one byte each, for the transposed packing: a thread reads four consecutive
// input positions of eight rows as eight words, merges them nibble by nibble and transposes
// the four bytes by permutes into four output words (12 vector instructions for 32 codes);
// 16 threads write the 64 consecutive bytes of an input row's words.
//
// Bound: the weight's read and the code's write once the arithmetic is out of the way.  An
// IEEE division per weight (11 instructions), NaN-aware compares and the packing of single
// bytes made about 32 vector instructions per weight, 64 us of issue for 24576 x 4096 bf16,
// where the 254 MB take 50 us at the copy rate.  Here w / s is w times the row's reciprocal,
// and the quotient is divided out only where that could round differently (below): about 10.
constexpr int kFastRows = 128;
constexpr int kFastThreads = 4 * kFastRows;

// Which blocks an XCD takes: all in grid order, round-robin, or in strips -- each XCD a
// contiguous eighth of the blocks, in strips of kStrip row blocks that walk the groups.
//
// A block reads 256 bytes (bf16, groups of 128) of each of its rows and writes 64 bytes, half a
// cache line, of each input row's words.  In grid order the blocks in flight read one group's
// column of the weight, pieces a row pitch apart, and no L2 holds both halves of a written line.
// What decides is the pitch: 22016 rows of 4096 bf16 take 57.7 us in grid order and 49.5 in
// strips, the same rows of 4224 (3 % more data) 50.9 in either, as if the pieces a multiple of
// 4 KiB apart fell on few memory channels.  Measured over 70 shapes, grid order ->
// strips in us a call, groups of 128 / 64:
//   4 KiB pitch   64 MiB   8192 x 4096 bf16     21.3 -> 21.6 / 21.1 -> 21.2
//                 80 MiB   10240 x 4096 bf16    25.3 -> 24.7 / 25.7 -> 25.3
//                 96 MiB   12288 x 4096 bf16    32.9 -> 29.2 / 33.0 -> 29.9
//                192 MiB   24576 x 4096 bf16    64.5 -> 51.9 / 69.1 -> 54.8
//                448 MiB   28672 x 8192 bf16   173.3 -> 119.7 / 199.9 -> 122.4
//                340 MiB   17408 x 5120 fp32    97.7 -> 90.1 / 99.2 -> 83.8
//   others       130 MiB   26624 x 2560 bf16    40.1 -> 38.8 / 39.8 -> 39.2
//                170 MiB   17408 x 5120 bf16    48.9 -> 49.6 / 49.2 -> 49.7
//                170 MiB   5120 x 17408 bf16    50.5 -> 52.2 / 49.3 -> 51.3
//                172 MiB   8192 x 11008 bf16    58.3 -> 52.2 / 58.6 -> 53.1
//                190 MiB   19456 x 2560 fp32    50.6 -> 52.4 / 47.4 -> 48.1
//                340 MiB   34816 x 5120 bf16    95.9 -> 92.0 / 95.0 -> 94.9
// With a pitch of 4 KiB multiples strips gain up to 39 % from 80 MiB on (at worst +4 %: 5120 x
// 17408 fp32); with other pitches nothing below 128 MiB, and -10 to +4 % from there on, where the
// gains outweigh the losses.  Hence the two sizes.  (24576 x 4096 bf16 in strips of 1, 2, 8 and
// all row blocks: 1 - 5 % slower than 4; non-temporal loads or stores 26 and 4 %.)  Groups of 32
// gain nothing at any size and keep the grid order.
constexpr size_t kStripPitch = 4096;
constexpr size_t kStripBytes = size_t{80} << 20;
constexpr size_t kStripBytesOther = size_t{128} << 20;
constexpr int kStrip = 4;

struct QuantGrid {
  int strips;                           // else grid order
  int row_blocks, groups;
  int per, rem;                         // the blocks of an XCD: per, the first rem XCDs one more
  uint32_t strip_mul, strip_shift;      // n / (kStrip groups) = n strip_mul >> strip_shift, n < 2^31
};

static QuantGrid quant_grid(bool strips, int row_blocks, int groups) {
  const uint32_t d = static_cast<uint32_t>(kStrip) * groups;
  uint32_t shift = 31;
  while ((1ull << (shift - 31)) < d) ++shift;
  const int total = row_blocks * groups;
  return QuantGrid{strips, row_blocks, groups, total >> 3, total & 7,
                   static_cast<uint32_t>(((1ull << shift) + d - 1) / d), shift};
}

// No division: the index arithmetic runs ahead of the first load, and three divisions there
// took 4 us of the 55.4 that the call then took.
__device__ __forceinline__ void quant_block(const QuantGrid& q, int& row_block, int& group) {
  if (!q.strips) {
    row_block = blockIdx.x;
    group = blockIdx.y;
    return;
  }
  const int b = blockIdx.y * q.row_blocks + blockIdx.x;
  const int xcd = b & 7;
  const uint32_t n = xcd * q.per + (xcd < q.rem ? xcd : q.rem) + (b >> 3);
  const int strip = static_cast<int>((static_cast<uint64_t>(n) * q.strip_mul) >> q.strip_shift);
  const uint32_t at = n - strip * kStrip * q.groups;
  const int width = q.row_blocks - strip * kStrip;  // row blocks of the last strip
  if (width >= kStrip) group = at / kStrip;
  else if (width == 3) group = at / 3;
  else group = at / (width == 2 ? 2 : 1);
  row_block = strip * kStrip + at - group * (width < kStrip ? width : kStrip);
}

// Smaller / larger of two, NaN if either is (torch's amin / amax), one instruction each.
__device__ __forceinline__ float min_nan(float a, float b) { return __builtin_elementwise_minimum(a, b); }
__device__ __forceinline__ float max_nan(float a, float b) { return __builtin_elementwise_maximum(a, b); }

// clamp(n + z, 0, 15) as byte `E` of `word` (n, z whole numbers).  The conversion clamps below
// at 0 and takes NaN to 0, so the minimum has to keep NaN: the quotients of a group with a NaN
// or an infinity are code 0 here as in quantize_kernel.
template <int E>
__device__ __forceinline__ uint32_t put_code(uint32_t word, float n, float z) {
  return __builtin_amdgcn_cvt_pk_u8_f32(min_nan(n + z, 15.f), E, word);
}

template <int GS, int DTYPE>
__global__ __launch_bounds__(kFastThreads) void quantize_rows_kernel(const void* __restrict__ weight,
                                                                     uint32_t* __restrict__ qweight,
                                                                     uint32_t* __restrict__ qzeros,
                                                                     void* __restrict__ scales, int out_f, int in_f,
                                                                     QuantGrid grid) {
  constexpr int PART = GS / 4;       // values per thread
  constexpr int QP = GS + 4;         // LDS row pitch of the codes, bytes
  constexpr int PER = DTYPE == kDtypeF32 ? 4 : 8;  // values per 16-byte load
  static_assert(PART % PER == 0 && PART % 8 == 0, "a thread's values must split into 16-byte loads");
  __shared__ __attribute__((aligned(16))) uint8_t codes[kFastRows * QP];
  __shared__ float row_z[kFastRows];
  int row_block, g;
  quant_block(grid, row_block, g);
  const int o0 = row_block * kFastRows;
  const int rows = out_f - o0 < kFastRows ? out_f - o0 : kFastRows;  // a multiple of 8
  const int tid = threadIdx.x;
  const int r = tid >> 2;  // the four threads of row r are adjacent lanes of one wave
  const int h = tid & 3;
  const bool live = r < rows;

  float v[PART];
  const size_t base = static_cast<size_t>(o0 + (live ? r : 0)) * in_f + static_cast<size_t>(g) * GS + h * PART;
#pragma unroll
  for (int c = 0; c < PART; c += PER) {
    if constexpr (DTYPE == kDtypeF32) {
      const float4 w = *reinterpret_cast<const float4*>(static_cast<const float*>(weight) + base + c);
      v[c] = w.x; v[c + 1] = w.y; v[c + 2] = w.z; v[c + 3] = w.w;
    } else {
      const uint4 w = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(weight) + base + c);
      const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (DTYPE == kDtypeF16) {
          v[c + 2 * e] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(ww[e] & 0xFFFFu)));
          v[c + 2 * e + 1] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(ww[e] >> 16)));
        } else {
          v[c + 2 * e] = __uint_as_float(ww[e] << 16);
          v[c + 2 * e + 1] = __uint_as_float(ww[e] & 0xFFFF0000u);
        }
      }
    }
  }
  float mn = v[0], mx = v[0];
#pragma unroll
  for (int c = 1; c < PART; ++c) {
    mn = min_nan(mn, v[c]);
    mx = max_nan(mx, v[c]);
  }
#pragma unroll
  for (int d = 1; d <= 2; d <<= 1) {
    mn = min_nan(mn, __shfl_xor(mn, d));
    mx = max_nan(mx, __shfl_xor(mx, d));
  }
  float dd = mx - mn;
  dd = dd < 1e-5f ? 1e-5f : dd;  // torch clamp(min=): NaN stays NaN
  const float s = dd / 15.0f;
  float z = -__builtin_rintf(mn / s);
  z = z < 0.f ? 0.f : (z > 15.f ? 15.f : z);

  // Codes, eight values at a time.  t = w * (1 / s) is within 2^-23 |w / s| of w / s rounded
  // once and again, so where the code is not clamped anyway (|w / s| < 17) the two lie within
  // 4e-6 of each other and round to the same whole number unless t is that close to a half:
  // then the eight are divided out.
  const float inv = 1.0f / s;
  uint32_t* dst = reinterpret_cast<uint32_t*>(codes + r * QP + h * PART);
#pragma unroll
  for (int c = 0; c < PART; c += 8) {
    float n[8];
    float off = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float t = v[c + e] * inv;
      n[e] = __builtin_rintf(t);
      off = __builtin_fmaxf(off, __builtin_fabsf(t - n[e]));
    }
    if (off > 0.49999f) {
#pragma unroll
      for (int e = 0; e < 8; ++e) n[e] = __builtin_rintf(v[c + e] / s);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      uint32_t word = 0;
      word = put_code<0>(word, n[4 * q], z);
      word = put_code<1>(word, n[4 * q + 1], z);
      word = put_code<2>(word, n[4 * q + 2], z);
      word = put_code<3>(word, n[4 * q + 3], z);
      dst[c / 4 + q] = word;
    }
  }
  if (live && h == 0) {
    row_z[r] = z;
    const size_t si = static_cast<size_t>(g) * out_f + o0 + r;
    if constexpr (DTYPE == kDtypeF32) static_cast<float*>(scales)[si] = s;
    else if constexpr (DTYPE == kDtypeF16) static_cast<_Float16*>(scales)[si] = static_cast<_Float16>(s);
    else static_cast<uint16_t*>(scales)[si] = f32_to_bf16_bits(s);
  }
  __syncthreads();

  constexpr int W = kFastRows / 8;  // packed words per input row in this workgroup
  const int words = rows / 8;       // those inside the weight
  const int C8 = out_f / 8;         // packed words per input row
  if (tid < words) {
    uint32_t word = 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) word |= (static_cast<uint32_t>(row_z[8 * tid + c]) & 0xFu) << awq_shift(c);
    qzeros[static_cast<size_t>(g) * C8 + o0 / 8 + tid] = word;
  }
#pragma unroll
  for (int e = tid; e < GS / 4 * W; e += kFastThreads) {
    const int k4 = e / W;
    const int j = e % W;
    if (j >= words) continue;
    // Row c's codes of positions 4 k4 .. + 3; columns 0, 2, 4, 6 of an AutoAWQ word are the
    // nibbles of its low half, 1, 3, 5, 7 those of its high half.
    uint32_t row[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) row[c] = *reinterpret_cast<const uint32_t*>(codes + (8 * j + c) * QP + 4 * k4);
    const uint32_t b0 = row[0] | (row[2] << 4), b1 = row[4] | (row[6] << 4);
    const uint32_t b2 = row[1] | (row[3] << 4), b3 = row[5] | (row[7] << 4);
    // byte i of (b0, b1, b2, b3) -> word i (v_perm_b32 selects among the 8 bytes of hi:lo)
    const uint32_t lo01 = __builtin_amdgcn_perm(b1, b0, 0x05010400u), hi01 = __builtin_amdgcn_perm(b1, b0, 0x07030602u);
    const uint32_t lo23 = __builtin_amdgcn_perm(b3, b2, 0x05010400u), hi23 = __builtin_amdgcn_perm(b3, b2, 0x07030602u);
    uint32_t* out = qweight + (static_cast<size_t>(g) * GS + 4 * k4) * C8 + o0 / 8 + j;
    out[0] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
    out[C8] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
    out[2 * static_cast<size_t>(C8)] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
    out[3 * static_cast<size_t>(C8)] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
  }
}

// One thread per packed word: out[r, c8] = sum_c (v[r, 8 c8 + c] & 15) << awq_shift(c).
__global__ __launch_bounds__(256) void pack_int4_kernel(const int32_t* __restrict__ values,
                                                        uint32_t* __restrict__ packed, int rows, int c8) {
  const size_t idx = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= static_cast<size_t>(rows) * c8) return;
  const int4* src = reinterpret_cast<const int4*>(values + idx * 8);
  const int4 a = src[0], b = src[1];
  const int v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  uint32_t word = 0;
#pragma unroll
  for (int c = 0; c < 8; ++c) word |= (static_cast<uint32_t>(v[c]) & 0xFu) << awq_shift(c);
  packed[idx] = word;
}

size_t quantize_lds_bytes(int group_size) {
  return static_cast<size_t>(kQuantRows) * (group_size + 1) * sizeof(float);
}

template <int GS>
static hipError_t launch_quantize_rows(const void* weight, int dtype, uint32_t* qweight, uint32_t* qzeros,
                                       void* scales, int out_f, int in_f, hipStream_t stream) {
  const size_t pitch = static_cast<size_t>(in_f) * (dtype == kDtypeF32 ? 4 : 2);
  const bool strips = GS >= 64 && out_f * pitch >= (pitch % kStripPitch == 0 ? kStripBytes : kStripBytesOther);
  const QuantGrid grid = quant_grid(strips, (out_f + kFastRows - 1) / kFastRows, in_f / GS);
  const dim3 blocks(grid.row_blocks, grid.groups);
  switch (dtype) {
    case kDtypeF32:
      quantize_rows_kernel<GS, kDtypeF32><<<blocks, kFastThreads, 0, stream>>>(weight, qweight, qzeros, scales, out_f,
                                                                                  in_f, grid);
      break;
    case kDtypeF16:
      quantize_rows_kernel<GS, kDtypeF16><<<blocks, kFastThreads, 0, stream>>>(weight, qweight, qzeros, scales, out_f,
                                                                                  in_f, grid);
      break;
    default:
      quantize_rows_kernel<GS, kDtypeBF16><<<blocks, kFastThreads, 0, stream>>>(weight, qweight, qzeros, scales, out_f,
                                                                                  in_f, grid);
  }
  return hipGetLastError();
}

hipError_t launch_quantize(const void* weight, int dtype, uint32_t* qweight, uint32_t* qzeros, void* scales,
                           int out_f, int in_f, int group_size, hipStream_t stream) {
  const dim3 grid((out_f + kQuantRows - 1) / kQuantRows, in_f / group_size);
  // Fast path: 16-byte aligned weight (every row segment a thread loads is then aligned).
  if (reinterpret_cast<uintptr_t>(weight) % 16 == 0) {
    switch (group_size) {
      case 128: return launch_quantize_rows<128>(weight, dtype, qweight, qzeros, scales, out_f, in_f, stream);
      case 64: return launch_quantize_rows<64>(weight, dtype, qweight, qzeros, scales, out_f, in_f, stream);
      case 32: return launch_quantize_rows<32>(weight, dtype, qweight, qzeros, scales, out_f, in_f, stream);
      default: break;
    }
  }
  const bool vec = reinterpret_cast<uintptr_t>(weight) % 16 == 0 && group_size % (dtype == kDtypeF32 ? 4 : 8) == 0;
  quantize_kernel<<<grid, kQuantThreads, quantize_lds_bytes(group_size), stream>>>(
      weight, dtype, qweight, qzeros, scales, out_f, in_f, group_size, vec);
  return hipGetLastError();
}

hipError_t launch_pack_int4(const int32_t* values, uint32_t* packed, int rows, int cols, hipStream_t stream) {
  const size_t words = static_cast<size_t>(rows) * (cols / 8);
  const unsigned blocks = static_cast<unsigned>((words + 255) / 256);
  pack_int4_kernel<<<blocks, 256, 0, stream>>>(values, packed, rows, cols / 8);
  return hipGetLastError();
}

}  // namespace w4a16
