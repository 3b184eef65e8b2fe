// Causal self-attention of a prompt (gfx950): query tokens 0..T-1 against keys 0..T-1 (the prompt's
// own cache rows), grouped-query, head_dim 128.
//
// No reference counterpart: the reference runs attention as the Hugging Face module's sdpa call.
//
// A workgroup takes 32 * QW queries of one head with QW * KW waves: wave (kw, qw) owns 32 queries and
// every KW-th block of KB keys up to the diagonal (KW > 1 shortens the chain of dependent key
// blocks where the grid is too small to fill the chip; the KW partial results meet in LDS at the end).
//   * scores are computed transposed, S^T = K q^T (v_mfma_f32_32x32x16_bf16: A = 32 keys, B = the
//     wave's 32 queries, held in registers): a lane then holds 16 scores of ONE query, so the row
//     maximum is an in-lane reduction plus one v_permlane32_swap, the rescale factor of the output
//     is a scalar of the lane, and the probabilities, rounded to bf16 pairs in place, already are
//     the B operand of O^T = V^T P^T (its K slots take the keys in the accumulator's order): no
//     probability passes through LDS and no wave waits for another's;
//   * keys and values reach LDS by direct buffer loads one block ahead, as they lie in the caches
//     ([key][128], 256-byte rows, 16-byte chunk c of row r at c ^ (r % 16) for keys and
//     c ^ 4 (r % 4) for values, so that the operand reads hit distinct banks); the values'
//     transpose is done by the read itself (ds_read_b64_tr_b16). The descriptors end at the last token:
//     rows past it read as zeros, so stale cache rows never reach a sum;
//   * one barrier per key block.
// Online softmax in fp32 with exp2 (running maximum m and sum l per query). Probabilities are rounded
// to bf16 and their rounded values are what l sums.
//
// Bound: the chain of key blocks of the last queries. By the slope over 1000 to 1536 tokens at 16/2 heads a block of 64
// keys takes a wave alone on its SIMD 1.42 us, two waves of a SIMD 2.24 us for a block each; the launch, the first
// block's loads and the end take 4 us (<4, 1>) to 6 (<4, 2>, with its merge). A block is 32 products (1024
// matrix cycles), ~300 VALU instructions (32 of them exponentials, 4 issue slots each) and 32 KiB of LDS operand
// reads, none dominant (copies without the staging, the exponentials, either product or either operand read were
// each 4-20% faster). At 1000 tokens and 40/8 heads <4, 2> has 320 workgroups, one a CU (LDS): eight turns and
// the fixed 6 us are 24 of its 25.1 us. Measured and level: the next block's score products woven into this block's
// exponentials, and its scaling into the value products, by hand. Letting the maximum lag until it has grown by
// 2^8 saved most rescaling (62.7 against 67.7 us at 2048 tokens and 40/8 heads, 27.1 against 27.6 at 1000), but
// tied a query's rounding to the others of its wave and raised the error against 64 bits (2.06e-3 against 2.01e-3).
// Kernel this replaced (16x16x32 products, 16 queries per wave, probabilities through LDS, three barriers per key
// block, values transposed by the stores), launches back to back: 72.9 us at 1000 tokens and 40/8 heads, 210 at
// 2048, 314 at 4096 and 16/2 heads; this one 27.6, 67.7 and 99.
#include <math.h>

#include <type_traits>

#include "elementwise.h"
#include "kernels.h"

namespace tx {

namespace {

constexpr int kDim = 128;            // head_dim
constexpr int kRowBytes = kDim * 2;  // one cached key or value
constexpr int kXcds = 8;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The larger (or the sum) of a lane's value and that of the lane 32 away.
__device__ __forceinline__ float halves_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halves_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Two waves per SIMD, but for <1, 4, 32>, whose four waves hold all of a CU's LDS.
template <int QW, int KW, int KB>
__global__ __launch_bounds__(64 * QW * KW, QW * KW * KB == 128 ? 1 : 2) __attribute__((amdgpu_num_vgpr(256))) void prompt_attention_kernel(
    const uint16_t *q, int64_t q_stride, const uint16_t *k_cache, const uint16_t *v_cache, int tokens, int heads,
    int group, int64_t max_ctx, float scale, uint16_t *out, int64_t out_stride, int direct) {
  constexpr int kTile = KB * kRowBytes;  // bytes of a key (or value) block
  constexpr int kLoads = KB / 4;         // 1 KiB direct loads per block and array
  constexpr int kPer = kLoads / QW;      // of them this wave issues
  constexpr int kSubs = KB / 32;
  // Two buffers, separate LDS objects (the compiler then knows that reads of one do not wait for the
  // direct loads that fill the other): per key group its key block, then its value block.
  __shared__ __attribute__((aligned(1024))) char buf0[KW * 2 * kTile];
  __shared__ __attribute__((aligned(1024))) char buf1[KW * 2 * kTile];
  __shared__ float stats[KW > 1 ? KW : 1][QW][2][KW > 1 ? 64 : 1];  // (m, l) of every wave, for the merge

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int qw = wave % QW, kw = wave / QW;
  const int n = lane & 31, h = lane >> 5;
  // Heads fastest, so that the heaviest query tiles (the last) start first; where the head count
  // allows, an XCD (workgroups arrive round-robin) gets neighbouring heads, which share keys.
  const int hx = blockIdx.x;
  const int head = heads % kXcds == 0 ? (hx % kXcds) * (heads / kXcds) + hx / kXcds : hx;
  const int kv = head / group;
  const int tile = (int)gridDim.y - 1 - (int)blockIdx.y;
  const int q0 = (tile * QW + qw) * 32;  // this wave's first query

  // q as MFMA B operands: column n = query q0 + n (clamped into the prompt), dimensions 16 st + 8 h ...
  const float sl2 = scale * 1.44269504088896340736f;  // scores in log2 units
  u32x4 qb[8];
  {
    const uint16_t *qr = q + (size_t)min(q0 + n, tokens - 1) * q_stride + (size_t)head * kDim;
#pragma unroll
    for (int st = 0; st < 8; ++st) qb[st] = *reinterpret_cast<const u32x4 *>(qr + 16 * st + 8 * h);
  }

  const char *kg = reinterpret_cast<const char *>(k_cache + (size_t)kv * max_ctx * kDim);
  const char *vg = reinterpret_cast<const char *>(v_cache + (size_t)kv * max_ctx * kDim);
  // Load i of a block brings rows 4i .. 4i + 3, lane l landing in chunk l % 16 of row 4i + l / 16.
  const uint32_t row_off = (uint32_t)(lane >> 4) * kRowBytes;
  const uint32_t k_off = row_off + 16u * (uint32_t)((lane & 15) ^ (lane >> 4));
  const uint32_t v_off = row_off + 16u * (uint32_t)((lane & 15) ^ (4 * (lane >> 4)));
  auto stage = [&](char *buf, int kb) __attribute__((always_inline)) {
    const int64_t first = (int64_t)kb * KB;
    const int bytes = (int)min((int64_t)kTile, max((int64_t)0, (tokens - first) * kRowBytes));
    const char *kf = kg + first * kRowBytes, *vf = vg + first * kRowBytes;
    char *kd = buf + kw * 2 * kTile, *vd = kd + kTile;
    if (direct) {
      const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(kf), (short)0, bytes, 0x00020000);
      const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(vf), (short)0, bytes, 0x00020000);
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int i = qw + QW * u;
        const uint32_t at = (uint32_t)i * 1024u;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(kr, (__attribute__((address_space(3))) void *)(kd + at), 16,
                                                 at + (k_off ^ (64u * (uint32_t)(i & 3))), 0, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(vr, (__attribute__((address_space(3))) void *)(vd + at), 16, at + v_off, 0, 0, 0);
      }
    } else {  // caches off a 16-byte boundary: the same bytes through registers
#pragma unroll 1
      for (int u = 0; u < kPer; ++u) {
        const int i = qw + QW * u;
        const uint32_t at = (uint32_t)i * 1024u, ko = at + (k_off ^ (64u * (uint32_t)(i & 3))), vo = at + v_off;
        u32x4 a = {0, 0, 0, 0}, b = {0, 0, 0, 0};
        if ((int)ko < bytes) __builtin_memcpy(&a, kf + ko, 16);
        if ((int)vo < bytes) __builtin_memcpy(&b, vf + vo, 16);
        *reinterpret_cast<u32x4 *>(kd + at + 16 * lane) = a;
        *reinterpret_cast<u32x4 *>(vd + at + 16 * lane) = b;
      }
    }
  };

  float m = -INFINITY, l = 0.f;  // running maximum (log2 units) and this lane's share of the sum, query q0 + n
  f32x16 o[4];                   // o[t][r] = O[query q0 + n][dimension 32 t + 8 (r / 4) + 4 h + r % 4]
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] = 0.f;

  // Byte offsets of this lane's operands in a tile: of key row n, dimensions 16 st + 8 h (chunk 2 st + h) at
  // k_at ^ 32 st; and, for the transposing reads, of key 4 h + (lane % 16) / 4, dimensions
  // 32 t + 16 ((lane / 16) % 2) + 4 (lane % 4) at v_at ^ 64 t.
  const uint32_t x4 = (lane >> 2) & 3;
  const uint32_t k_at = (uint32_t)n * kRowBytes + 16u * (uint32_t)(h ^ (n & 15));
  const uint32_t v_at = (4u * h + x4) * kRowBytes + 32u * ((lane >> 4) & 1) + 8u * (lane & 3) + 64u * x4;

  // NS sub-blocks of 32 keys at once (their score chains are independent); DIAG: the last of them holds
  // the queries' own positions and is masked.
  auto block = [&](const char *buf, int kb, auto ns_c, auto diag_c) __attribute__((always_inline)) {
    constexpr int NS = decltype(ns_c)::value;
    constexpr bool DIAG = decltype(diag_c)::value;
    const char *kt = buf + kw * 2 * kTile, *vt = kt + kTile;
    f32x16 sc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[s][r] = 0.f;
#pragma unroll
    for (int st = 0; st < 8; ++st)
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const u32x4 a = *reinterpret_cast<const u32x4 *>(kt + 32 * s * kRowBytes + (k_at ^ (32u * st)));
        sc[s] = mfma32(a, qb[st], sc[s]);
      }
    // sc[s][r] = score of key 32 s + 8 (r / 4) + 4 h + r % 4 of the block and query q0 + n
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        sc[s][r] *= sl2;
        if (DIAG && s == NS - 1) sc[s][r] = 8 * (r >> 2) + 4 * h + (r & 3) > n ? -INFINITY : sc[s][r];
      }
    float mx = fmaxf(sc[0][0], sc[0][1]);
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int r = s == 0 ? 2 : 0; r < 16; r += 2) mx = fmaxf(fmaxf(mx, sc[s][r]), sc[s][r + 1]);
    // The running maximum is each query's own: a query that finds no larger score scales by exactly 1, so
    // its output does not depend on which other queries share the wave. (m is finite from a query's first block
    // on, where its scores are: every query has a key <= itself in every block it reaches.)
    const float mnew = fmaxf(m, halves_max(mx));
    if (__builtin_amdgcn_ballot_w64(mnew > m) != 0) {
      const float alpha = __builtin_amdgcn_exp2f(m - mnew);
      l *= alpha;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] *= alpha;
      m = mnew;
    }
    uint32_t pb[NS][8];
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const bf16x2 pair = {(__bf16)__builtin_amdgcn_exp2f(sc[s][r] - m), (__bf16)__builtin_amdgcn_exp2f(sc[s][r + 1] - m)};
        pb[s][r / 2] = __builtin_bit_cast(uint32_t, pair);
        l = __builtin_amdgcn_fdot2_f32_bf16(pair, bf16x2{(__bf16)1.0f, (__bf16)1.0f}, l, false);
      }
    // O^T += V^T P^T, sixteen keys at a time: slots 0-3 of half h are keys 4 h .. + 3, slots 4-7 the keys 8 on
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const u32x4 b = {pb[s][4 * j], pb[s][4 * j + 1], pb[s][4 * j + 2], pb[s][4 * j + 3]};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const char *at = vt + (32 * s + 16 * j) * kRowBytes + (v_at ^ (64u * t));
          const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)at);
          const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(at + 8 * kRowBytes));
          const u32x2 lw = __builtin_bit_cast(u32x2, lo), hw = __builtin_bit_cast(u32x2, hi);
          o[t] = mfma32(u32x4{lw[0], lw[1], hw[0], hw[1]}, b, o[t]);
        }
      }
  };
  // A key block against this wave's queries (k0 and q0 are multiples of 32): the sub-blocks up to the
  // diagonal; a wave whose queries end before the block has nothing to do.
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  auto visit = [&](const char *buf, int kb) __attribute__((always_inline)) {
    const int k0 = kb * KB;
    if (k0 > q0) return;
    if constexpr (kSubs == 2) {
      if (k0 + 32 < q0) block(buf, kb, Two{}, std::false_type{});
      else if (k0 + 32 == q0) block(buf, kb, Two{}, std::true_type{});
      else block(buf, kb, One{}, std::true_type{});
    } else {
      if (k0 < q0) block(buf, kb, One{}, std::false_type{});
      else block(buf, kb, One{}, std::true_type{});
    }
  };

  // Blocks of this key group: kw, kw + KW, ... up to the workgroup's diagonal; every wave runs every
  // turn (the barriers are workgroup-wide). A turn's loads were issued a turn before; the barrier
  // that ends their wait also says that the other buffer is no longer read.
  const int last = (min((tile * QW + QW) * 32, tokens) - 1) / KB;  // last block any query of the tile reaches
  const int turns = last / KW + 1;
  auto turn = [&](int it, char *cur, char *next) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int kb = it * KW + kw;
    if (kb + KW <= last) stage(next, kb + KW);
    if (kb <= last) visit(cur, kb);
  };
  if (kw <= last) stage(buf0, kw);
  int it = 0;
  for (; it + 2 <= turns; it += 2) {
    turn(it, buf0, buf1);
    turn(it + 1, buf1, buf0);
  }
  if (it < turns) turn(it, buf0, buf1);

  l = halves_sum(l);
  if constexpr (KW > 1) {
    // The groups' (m, l) meet in LDS; with M = max m, every group scales its O by exp2(m - M), and group
    // t % KW sums the output tile t of all (a group that took no block has m = -inf, l = 0, O = 0 and
    // weighs nothing; m of group 0, which took key block 0, is finite).
    static_assert(KW * QW * 2 * 4096 <= KW * 2 * kTile, "two output tiles of every wave in a buffer");
    stats[kw][qw][0][lane] = m;
    stats[kw][qw][1][lane] = l;
    __syncthreads();  // every tile read is done, too
    float mm = m, total = 0.f;
#pragma unroll
    for (int g = 0; g < KW; ++g) mm = fmaxf(mm, stats[g][qw][0][lane]);
#pragma unroll
    for (int g = 0; g < KW; ++g) total += stats[g][qw][1][lane] * __builtin_amdgcn_exp2f(stats[g][qw][0][lane] - mm);
    l = total;
    const float alpha = __builtin_amdgcn_exp2f(m - mm);
    auto at = [&](int g, int t) {
      return reinterpret_cast<float *>(t < 2 ? buf0 : buf1) + ((g * QW + qw) * 2 + (t & 1)) * 1024 + lane;
    };
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float *mine = at(kw, t);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        o[t][r] *= alpha;
        if (t % KW != kw) mine[r * 64] = o[t][r];
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (t % KW != kw) continue;
#pragma unroll
      for (int g = 0; g < KW; ++g) {
        if (g == kw) continue;
        const float *theirs = at(g, t);
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] += theirs[r * 64];
      }
    }
  }
  const int query = q0 + n;
  if (query >= tokens) return;
  const float inv = 1.0f / l;
  uint16_t *dst = out + (size_t)query * out_stride + (size_t)head * kDim + 4 * h;
  const bool vec = (reinterpret_cast<uintptr_t>(out) & 7) == 0 && (out_stride & 3) == 0;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if (KW > 1 && t % KW != kw) continue;
#pragma unroll
    for (int rq = 0; rq < 4; ++rq) {
      const uint16_t e0 = to_bf(o[t][4 * rq] * inv), e1 = to_bf(o[t][4 * rq + 1] * inv), e2 = to_bf(o[t][4 * rq + 2] * inv),
                     e3 = to_bf(o[t][4 * rq + 3] * inv);
      uint16_t *at = dst + 32 * t + 8 * rq;
      if (vec) {
        *reinterpret_cast<uint2 *>(at) = make_uint2((uint32_t)e0 | ((uint32_t)e1 << 16), (uint32_t)e2 | ((uint32_t)e3 << 16));
      } else {
        at[0] = e0;
        at[1] = e1;
        at[2] = e2;
        at[3] = e3;
      }
    }
  }
}

}  // namespace

bool prefill_attention_supported(int heads, int kv_heads, int head_dim) {
  return head_dim == kDim && kv_heads > 0 && heads % kv_heads == 0;
}

hipError_t launch_prefill_attention(const uint16_t *q, int64_t q_stride, const uint16_t *k_cache,
                                    const uint16_t *v_cache, int64_t tokens, int heads, int kv_heads, int64_t max_ctx,
                                    float scale, uint16_t *out, int64_t out_stride, hipStream_t stream) {
  int device = 0, cus = 0;
  if (hipGetDevice(&device) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
    return hipGetLastError();
  const int direct = ((reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache)) & 15) == 0;
  auto launch = [&](auto kernel, int queries, int waves) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)heads, (unsigned)((tokens + queries - 1) / queries)), dim3(64 * waves), 0,
                       stream, q, q_stride, k_cache, v_cache, (int)tokens, heads, heads / kv_heads, max_ctx, scale, out, out_stride, direct);
  };
  // Which split of the waves: by how many workgroups of 128, 64 and 32 queries there are. Measured at
  // 17 .. 4096 tokens and 40/8, 32/8, 28/4 and 16/2 heads (us, graph replays):
  //   <4, 1> from 2.25 workgroups of 128 queries a CU (two are resident): 2048 tokens, 40 heads 61.6 against 71.9
  //          of <4, 2> (at 1.7 to 2 of them 37.0 - 57.3 against 37.9 - 52.3); and for up to 64 tokens, where there
  //          is no chain to shorten (4.2 - 5.0 against 5.7 - 7.4);
  //   <4, 2> from 1.6 workgroups of 64 queries a CU: 1000 tokens, 40 heads 25.1 against 29.3 of <4, 1> and
  //          35.6 of <2, 4>;
  //   <1, 4> while workgroups of 32 queries fit the CUs at once: 512 tokens, 16 heads 12.0 against 12.8 of
  //          <2, 4> and 15.5 of <4, 1>; <2, 4> between: 1000 tokens, 16 heads 18.7 against 24.0 - 26.7.
  const int64_t tiles128 = (tokens + 127) / 128 * heads, tiles64 = (tokens + 63) / 64 * heads,
                tiles32 = (tokens + 31) / 32 * heads;
  if (tokens <= 64 || 4 * tiles128 >= 9 * (int64_t)cus) launch(prompt_attention_kernel<4, 1, 64>, 128, 4);
  else if (5 * tiles64 >= 8 * (int64_t)cus) launch(prompt_attention_kernel<4, 2, 64>, 128, 8);
  else if (tiles32 <= cus) launch(prompt_attention_kernel<1, 4, 32>, 32, 4);
  else launch(prompt_attention_kernel<2, 4, 32>, 64, 8);
  return hipGetLastError();
}

}  // namespace tx
