// BC4 post-training encoder on the GPU (gfx950): one launch per matrix.
//
// Same search as texelator_amd/encoder.py (reference: texelator/encoder.py:35-157), which runs it as
// torch operations, and the same bytes as those operations give on the GPU: every product, quotient
// and comparison is the same fp32 operation in the same order, and the sums over a block's sixteen
// positions are taken as torch takes them there (pairs, then pairs of pairs: sum16).
//
// A workgroup encodes one row: its threads take the row's maximum (the row scale), then each
// encodes whole 16-value blocks in registers. As torch operations a 5120 x 5120 matrix took 26.1 ms:
// about 1500 launches, each a pass over [blocks][16] arrays in memory. Here the weights are read once
// from HBM (the second read of a row hits the caches) and only the blocks are written. What is left
// is VALU work: nine candidate palettes of eight values against sixteen weights, ~4000 instructions a
// block; 174 us for that matrix, launches back to back (the best of ten cold ones in a trace 191), its issue floor
// being ~165. Five waves per SIMD (96 registers, 120 bytes spilled in the least squares) hide the palette gathers
// better than three without spills (238 us).
#include "bc4_device.h"
#include "kernels.h"

namespace tx {

namespace {

constexpr int kEncodeMaxThreads = 512;

// torch's sum over a contiguous last dimension of sixteen on the GPU: neighbours, then neighbouring
// pairs, and so on.
__device__ __forceinline__ float sum16(const float (&v)[16]) {
  float s[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) s[i] = v[2 * i] + v[2 * i + 1];
#pragma unroll
  for (int i = 0; i < 4; ++i) s[i] = s[2 * i] + s[2 * i + 1];
  return (s[0] + s[1]) + (s[2] + s[3]);
}

__device__ __forceinline__ float clamp_nan(float v, float lo, float hi) {  // NaN stays NaN, as torch.clamp
  return v != v ? v : fminf(fmaxf(v, lo), hi);
}

// torch.round then a conversion to int16 of a value within [-127, 127] (NaN becomes 0).
__device__ __forceinline__ int round_endpoint(float v) { return v != v ? 0 : (int)rintf(v); }

struct Row8 {
  float p[8];
};

// Palette row of (e0, e1) in the 255 x 255 x 8 table.
__device__ __forceinline__ Row8 palette_of(const float4 *lut, int e0, int e1) {
  const float4 *row = lut + 2 * ((e1 + 127) * 255 + (e0 + 127));
  const float4 a = row[0], b = row[1];
  return Row8{{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}};
}

// Selector of the nearest palette value, the lowest among equals (0 if no distance is below infinity).
__device__ __forceinline__ uint32_t nearest_index(float v, const Row8 &row) {
  float best = INFINITY;
  uint32_t index = 0;
#pragma unroll
  for (uint32_t s = 0; s < 8; ++s) {
    const float d = fabsf(v - row.p[s]);
    index = d < best ? s : index;
    best = d < best ? d : best;
  }
  return index;
}

// Sixteen weights of a block (32 or 64 bytes from a 16-byte aligned address) as fp32.
template <int DT>
__device__ __forceinline__ void load16(const void *w, size_t first, float (&v)[16]) {
  constexpr int kWords = DT == kF32 ? 4 : 2;
  const uint4 *src = reinterpret_cast<const uint4 *>(static_cast<const char *>(w) + first * (DT == kF32 ? 4 : 2));
  uint4 q[kWords];
#pragma unroll
  for (int i = 0; i < kWords; ++i) q[i] = src[i];
#pragma unroll
  for (int i = 0; i < kWords; ++i) {
    const uint32_t word[4] = {q[i].x, q[i].y, q[i].z, q[i].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (DT == kF32) {
        v[4 * i + e] = __uint_as_float(word[e]);
      } else if constexpr (DT == kBF16) {
        v[8 * i + 2 * e] = __uint_as_float(word[e] << 16);
        v[8 * i + 2 * e + 1] = __uint_as_float(word[e] & 0xFFFF0000u);
      } else {
        v[8 * i + 2 * e] = (float)__builtin_bit_cast(_Float16, (uint16_t)(word[e] & 0xFFFFu));
        v[8 * i + 2 * e + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(word[e] >> 16));
      }
    }
  }
}

// The larger of two maxima, NaN if either is (torch.amax).
__device__ __forceinline__ float max_nan(float a, float b) { return a != a ? a : (b > a || b != b ? b : a); }

// Weights of q = a*u + b*z + c by mode (6 values, 8 values) and selector, as {a, b, c, 0}: a copy in
// LDS, read by the selector (selecting among constants took 22 VALU instructions a weight).
__constant__ const float kCoefficients[2][8][4] = {
    {{1.f, 0.f, 0.f, 0.f}, {0.f, 1.f, 0.f, 0.f}, {(float)(4.0 / 5), (float)(1.0 / 5), 0.f, 0.f},
     {(float)(3.0 / 5), (float)(2.0 / 5), 0.f, 0.f}, {(float)(2.0 / 5), (float)(3.0 / 5), 0.f, 0.f},
     {(float)(1.0 / 5), (float)(4.0 / 5), 0.f, 0.f}, {0.f, 0.f, -1.f, 0.f}, {0.f, 0.f, 1.f, 0.f}},
    {{1.f, 0.f, 0.f, 0.f}, {0.f, 1.f, 0.f, 0.f}, {(float)(6.0 / 7), (float)(1.0 / 7), 0.f, 0.f},
     {(float)(5.0 / 7), (float)(2.0 / 7), 0.f, 0.f}, {(float)(4.0 / 7), (float)(3.0 / 7), 0.f, 0.f},
     {(float)(3.0 / 7), (float)(4.0 / 7), 0.f, 0.f}, {(float)(2.0 / 7), (float)(5.0 / 7), 0.f, 0.f},
     {(float)(1.0 / 7), (float)(6.0 / 7), 0.f, 0.f}}};

// One block: values v (weight / scale clamped to [-1, 1]) and importances h -> its 8 bytes.
__device__ __forceinline__ uint2 encode_one(const float (&v)[16], const float (&h)[16], const float4 *lut,
                                            const float4 (&coefficients)[2][8]) {
  // 1. start: endpoints at the largest and smallest value, selectors nearest
  float hi = v[0], lo = v[0];
#pragma unroll
  for (int i = 1; i < 16; ++i) {
    hi = max_nan(hi, v[i]);
    lo = lo != lo ? lo : (v[i] < lo || v[i] != v[i] ? v[i] : lo);
  }
  const int start0 = round_endpoint(clamp_nan(rintf(hi * 127.f), -127.f, 127.f));
  const int start1 = round_endpoint(clamp_nan(rintf(lo * 127.f), -127.f, 127.f));
  const bool eight = start0 > start1;
  int best0 = start0, best1 = start1;
  float u, z;
  {
    const Row8 row = palette_of(lut, start0, start1);
    // 2. weighted least squares for (u, z) = (e0 / 127, e1 / 127) with these selectors
    float aa[16], bb[16], ab[16], ay[16], by[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float4 w = coefficients[eight][nearest_index(v[i], row)];
      const float ha = h[i] * w.x, hb = h[i] * w.y, target = v[i] - w.z;
      aa[i] = ha * w.x;
      bb[i] = hb * w.y;
      ab[i] = ha * w.y;
      ay[i] = ha * target;
      by[i] = hb * target;
    }
    const float saa = sum16(aa), sbb = sum16(bb), sab = sum16(ab), say = sum16(ay), sby = sum16(by);
    float det = saa * sbb - sab * sab;
    const bool singular = fabsf(det) < 1e-12f;
    det = det < 1e-12f ? 1e-12f : det;
    u = clamp_nan((say * sbb - sby * sab) / det, -1.f, 1.f);
    z = clamp_nan((sby * saa - say * sab) / det, -1.f, 1.f);
    constexpr float kInv127 = 1.0f / 127.0f;  // torch divides a tensor by a number as a product on the GPU
    u = singular ? (float)start0 * kInv127 : u;
    z = singular ? (float)start1 * kInv127 : z;
  }
  const int center0 = round_endpoint(u * 127.f), center1 = round_endpoint(z * 127.f);

  // 3. the 3 x 3 neighbourhood: weighted squared error, the first strict improvement wins. Only
  // the distance to the nearest value is needed here; the selectors are found once, at the end.
  float best_error = INFINITY;
#pragma unroll 1
  for (int d0 = -1; d0 <= 1; ++d0) {
    const int c0 = min(max(center0 + d0, -127), 127);
#pragma unroll 1
    for (int d1 = -1; d1 <= 1; ++d1) {
      const int c1 = min(max(center1 + d1, -127), 127);
      const Row8 row = palette_of(lut, c0, c1);
      float e[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float d = INFINITY;
#pragma unroll
        for (int s = 0; s < 8; ++s) d = fminf(d, fabsf(v[i] - row.p[s]));
        e[i] = h[i] * (d * d);
      }
      const float error = sum16(e);
      const bool improved = error < best_error;
      best_error = improved ? error : best_error;
      best0 = improved ? c0 : best0;
      best1 = improved ? c1 : best1;
    }
  }
  const Row8 row = palette_of(lut, best0, best1);
  uint64_t word = (uint64_t)(uint8_t)best0 | ((uint64_t)(uint8_t)best1 << 8);
#pragma unroll
  for (int i = 0; i < 16; ++i) word |= (uint64_t)nearest_index(v[i], row) << (16 + 3 * i);
  return make_uint2((uint32_t)word, (uint32_t)(word >> 32));
}

template <int DT>
__global__ __launch_bounds__(kEncodeMaxThreads, 5) void encode_rows_kernel(const void *weight, int K, const float *hdiag,
                                                                        const float4 *lut, uint2 *blocks, float *scales) {
  __shared__ float wave_max_[kEncodeMaxThreads / 64];
  __shared__ float4 coefficients[2][8];
  const size_t row = blockIdx.x;
  const int nblk = K / 16, tid = threadIdx.x, threads = blockDim.x;
  if (tid < 64) reinterpret_cast<float *>(coefficients)[tid] = reinterpret_cast<const float *>(kCoefficients)[tid];
  float v[16];
  float m = 0.f;
  for (int b = tid; b < nblk; b += threads) {
    load16<DT>(weight, row * K + (size_t)b * 16, v);
#pragma unroll
    for (int i = 0; i < 16; ++i) m = max_nan(m, fabsf(v[i]));
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) m = max_nan(m, __shfl_xor(m, off));
  if ((tid & 63) == 0) wave_max_[tid >> 6] = m;
  __syncthreads();
  m = wave_max_[0];
  for (int w = 1; w < threads / 64; ++w) m = max_nan(m, wave_max_[w]);
  const float scale = m < 1e-12f ? 1e-12f : m;  // NaN stays
  if (tid == 0) scales[row] = scale;
  for (int b = tid; b < nblk; b += threads) {
    load16<DT>(weight, row * K + (size_t)b * 16, v);
    float h[16];
    load16<kF32>(hdiag, (size_t)b * 16, h);
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = clamp_nan(v[i] / scale, -1.f, 1.f);
    // A block that holds a NaN keeps its start, as every torch error of it is NaN. The search's minima skip NaN,
    // and negative importances would turn the infinity they leave into an improvement: positive ones never do.
    if (!(scale < INFINITY)) {  // NaN or infinite weights in the row: the same for the workgroup
      bool nan = false;
#pragma unroll
      for (int i = 0; i < 16; ++i) nan |= v[i] != v[i];
#pragma unroll
      for (int i = 0; i < 16; ++i) h[i] = nan ? 1.f : h[i];
    }
    blocks[row * nblk + b] = encode_one(v, h, lut, coefficients);
  }
}

}  // namespace

hipError_t launch_encode(const void *weight, int dtype, int64_t rows, int K, const float *hdiag, const float4 *lut,
                         uint2 *blocks, float *scales, hipStream_t stream) {
  // Threads: as few passes over the row as 512 threads allow, then as few idle lanes as that leaves.
  const int nblk = K / 16, passes = (nblk + kEncodeMaxThreads - 1) / kEncodeMaxThreads;
  const int threads = ((nblk + passes - 1) / passes + 63) / 64 * 64;
  const dim3 grid((unsigned)rows);
  if (dtype == kF32) hipLaunchKernelGGL(encode_rows_kernel<kF32>, grid, dim3(threads), 0, stream, weight, K, hdiag, lut, blocks, scales);
  else if (dtype == kBF16) hipLaunchKernelGGL(encode_rows_kernel<kBF16>, grid, dim3(threads), 0, stream, weight, K, hdiag, lut, blocks, scales);
  else hipLaunchKernelGGL(encode_rows_kernel<kF16>, grid, dim3(threads), 0, stream, weight, K, hdiag, lut, blocks, scales);
  return hipGetLastError();
}

}  // namespace tx
