// Causal prompt attention, out[b, i, hq] = softmax_j<=i(q[b, hq, i] . k[b, hq / G, j] / sqrt(128)) . v
// (the prefill attention of the sparse layer, models/attention/shadow.py:12-19, which the decode state
// is built beside), bf16 inputs and output, every sum and probability in fp32.
//
// Bound: the matrix cores, and beside them the VALU work of the softmax. One pass (flash attention),
// the scores never leave the registers. Both products are taken transposed: S^T = K Q^T on
// v_mfma_f32_32x32x16_bf16 leaves a query per lane with its keys along the registers, which is (up
// to the order of the keys inside a group of 16) the B operand of O^T = V^T P^T: no cross-lane move
// and no LDS round trip of P, one maximum and one sum per lane. The values are transposed once per
// call by vt_kernel into exactly that key order.
//
// Probabilities keep their fp32 value: p is cut by truncation into three bf16 parts (8 + 8 + 8
// significant bits, an exact sum) and P.V is three MFMAs into one fp32 accumulator, so nothing is
// rounded to 16 bits before the output. A part may be zero, and its product with an infinite value
// NaN, where the whole p gives the infinity: where the keys' values hold an infinity or a NaN (vt_kernel
// says so per tile) the second and third products take them as zeros. The maximum that the exponentials are taken against is only
// moved when a score passes it by 2^8 (the ratio of the sums does not depend on it), which leaves
// the 64 accumulators of a lane alone in most tiles.
//
// A workgroup of 4 waves owns 128 queries of one head (32 per wave) and walks the keys in tiles of
// 64 (two workgroups per CU: 64 KB of LDS, 209 VGPRs), K and V^T tiles double-buffered in LDS by direct global-to-LDS loads (K's 16-byte chunks
// swizzled by the row at the source, so that operand reads have no bank conflicts).
//
// MI355X, 32 query heads: 8 kv heads x 8192 tokens 0.93 ms (591 TFLOP/s of the causal 4 L^2 D / 2 count,
// 1180 with the three-part P.V that is issued: the rate of a large bf16 GEMM here is 1120) against
// 11.5 ms for fp32 torch operations over 1024-query blocks; 2 kv heads x 19333 tokens 4.8 ms against 58.
#include <type_traits>

#include "skv_common.h"

namespace {

using skv::u32x4;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kD = 128;
constexpr int kTileKeys = 64;
constexpr int kWaves = 4;
constexpr int kQWave = 32;
constexpr int kQBlock = kWaves * kQWave;
constexpr int kTile16 = kTileKeys * kD * 2 / 16;  // 16-byte chunks of a K or V^T tile
constexpr int kXcds = 8;

// vt[row][key / 16][dim][16 keys], the keys of a group of 16 in the order 0-3, 8-11, 4-7, 12-15; zeros past L.
// odd[row][key / 64]: whether the tile holds an infinity or a NaN.
__global__ void __launch_bounds__(256) vt_kernel(const uint16_t* __restrict__ v, int64_t sb, int64_t sh, int64_t ss,
                                                 int H, int L, u32x4* __restrict__ vt, int groups,
                                                 int* __restrict__ odd) {
  __shared__ uint16_t t[64][kD + 2];
  const int row = blockIdx.y, b = row / H, h = row - b * H;
  const int k0 = blockIdx.x * 64;
  const uint16_t* src = v + b * sb + h * sh;
  bool not_finite = false;
  for (int i = threadIdx.x; i < 64 * 16; i += 256) {
    const int r = i >> 4, c = i & 15;
    const u32x4 x = skv::load16_or_zero(src + static_cast<int64_t>(min(k0 + r, L - 1)) * ss + 8 * c, k0 + r < L);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      *reinterpret_cast<uint32_t*>(&t[r][8 * c + 2 * e]) = x[e];
      not_finite |= (x[e] & 0x7f80u) == 0x7f80u || (x[e] & 0x7f800000u) == 0x7f800000u;
    }
  }
  not_finite = __syncthreads_or(not_finite);
  if (threadIdx.x == 0) odd[row * gridDim.x + blockIdx.x] = not_finite;
  // 16-byte chunk i: group i / 256, dim (i % 256) / 2, half i % 2
  for (int i = threadIdx.x; i < 4 * 256; i += 256) {
    const int g = i >> 8, d = (i >> 1) & 127, hf = i & 1;
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int j = 16 * g + 4 * hf + (e >> 1) * 8 + (e & 1) * 2;
      o[e] = static_cast<uint32_t>(t[j][d]) | (static_cast<uint32_t>(t[j + 1][d]) << 16);
    }
    vt[(static_cast<int64_t>(row) * groups + blockIdx.x * 4 + g) * 256 + (i & 255)] = o;
  }
}

struct PrefillArgs {
  const uint16_t* q;
  int64_t q_sb, q_sh, q_ss;
  const uint16_t* k;
  int64_t k_sb, k_sh, k_ss;
  const u32x4* vt;
  const int* odd;
  uint16_t* out;
  int64_t o_sb, o_sh, o_ss;
  int Hq, Hkv, G, L, qblocks, rows;  // rows = B * Hkv
  float scale_log2e;
};

// Copies 1 KB: lane l's 16 bytes at src go to dst + 16 l (dst wave-uniform).
__device__ __forceinline__ void load_lds(const void* src, u32x4* dst) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// Infinities and NaNs of bf16 pairs as zeros.
__device__ __forceinline__ u32x4 finite_part(u32x4 x) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if ((x[e] & 0x7f80u) == 0x7f80u) x[e] &= 0xffff0000u;
    if ((x[e] & 0x7f800000u) == 0x7f800000u) x[e] &= 0x0000ffffu;
  }
  return x;
}

__device__ __forceinline__ float other_half_max(float x) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}

__global__ void __launch_bounds__(kWaves * 64, 2) prefill_attn_kernel(PrefillArgs a) {
  __shared__ u32x4 ka[kTile16], kb[kTile16], va[kTile16], vb[kTile16];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 31, half = lane >> 5;

  // Work item -> (kv row, query head of its group, query block), longest query blocks first. The
  // dispatcher hands workgroup w to XCD w mod 8: where the kv rows divide among the XCDs (or the XCDs
  // among the rows), a row's workgroups share one XCD's L2 (or few).
  int bh, g, qb;
  {
    const int w = blockIdx.x, per = a.G * a.qblocks;
    int item;
    if (a.rows % kXcds == 0) {
      const int x = w % kXcds, j = w / kXcds, n = a.rows / kXcds;  // rows of this XCD
      bh = x + kXcds * (j % n);
      item = j / n;
    } else if (kXcds % a.rows == 0) {
      const int x = w % kXcds, j = w / kXcds;
      bh = x % a.rows;
      item = j * (kXcds / a.rows) + x / a.rows;
      if (item >= per) return;  // workgroup-uniform
    } else {
      bh = w % a.rows;
      item = w / a.rows;
    }
    qb = a.qblocks - 1 - item / a.G;
    g = item % a.G;
  }
  const int b = bh / a.Hkv, h = bh - b * a.Hkv;
  const int hq = h * a.G + g;
  const int q0 = qb * kQBlock + wave * kQWave;  // the wave's first query
  const int query = q0 + li;

  const uint16_t* kbase = a.k + b * a.k_sb + h * a.k_sh;
  const int row_tiles = (a.L + kTileKeys - 1) / kTileKeys;
  const u32x4* vbase = a.vt + static_cast<int64_t>(bh) * row_tiles * kTile16;
  const int tiles = (min(a.L, qb * kQBlock + kQBlock) + kTileKeys - 1) / kTileKeys;
  const int krow = wave * 16 + (lane >> 4);  // + 4 i: this lane's K rows of a tile
  auto issue = [&](int t, u32x4* kd, u32x4* vd) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = krow + 4 * i;
      const int chunk = (lane & 15) ^ (r & 15);
      load_lds(kbase + static_cast<int64_t>(min(t * kTileKeys + r, a.L - 1)) * a.k_ss + 8 * chunk,
               kd + (wave * 16 + 4 * i) * 16);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      load_lds(vbase + static_cast<int64_t>(t) * kTile16 + (wave * 4 + i) * 64 + lane, vd + (wave * 4 + i) * 64);
  };

  u32x4 qf[8];
  const uint16_t* qrow = a.q + b * a.q_sb + hq * a.q_sh + static_cast<int64_t>(min(query, a.L - 1)) * a.q_ss + 8 * half;
#pragma unroll
  for (int s = 0; s < 8; ++s) qf[s] = *reinterpret_cast<const u32x4*>(qrow + 16 * s);

  f32x16 o[4];
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.f;
  float m = -INFINITY;  // the reference the exponentials are taken against, in units of log2
  float l = 0.f;        // this lane's share of the row sum

  auto compute = [&](auto special, int t, const u32x4* kt, const u32x4* vt) __attribute__((always_inline)) {
    const int k0 = t * kTileKeys;
    if (k0 > q0 + kQWave - 1) return;  // wave-uniform: all keys after the wave's last query
    f32x16 s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[u][r] = 0.f;
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        s[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            __builtin_bit_cast(bf16x8, kt[(32 * u + li) * 16 + ((2 * c + half) ^ (li & 15))]),
            __builtin_bit_cast(bf16x8, qf[c]), s[u], 0, 0, 0);
    if (k0 + kTileKeys - 1 > q0) {  // wave-uniform: the diagonal tiles
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (k0 + 32 * u + 8 * (r / 4) + 4 * half + (r % 4) > query) s[u][r] = -INFINITY;
    }
    float mx = s[0][0];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[u][r]);
    mx = other_half_max(mx) * a.scale_log2e;
    if (__any(mx > m + 8.f)) {  // wave-uniform
      const float mn = fmaxf(m, mx);
      const float f = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= f;
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] *= f;
    }
    const float mref = m == -INFINITY ? 0.f : m;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[u][r] = __builtin_amdgcn_exp2f(fmaf(s[u][r], a.scale_log2e, -mref));
        l += s[u][r];
      }
#pragma unroll
    for (int gk = 0; gk < 4; ++gk) {
      u32x4 p[3];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x0 = s[gk >> 1][8 * (gk & 1) + 2 * e], x1 = s[gk >> 1][8 * (gk & 1) + 2 * e + 1];
        const uint32_t a0 = __float_as_uint(x0), a1 = __float_as_uint(x1);
        const float r0 = x0 - __uint_as_float(a0 & 0xffff0000u), r1 = x1 - __uint_as_float(a1 & 0xffff0000u);
        const uint32_t b0 = __float_as_uint(r0), b1 = __float_as_uint(r1);
        const float t0 = r0 - __uint_as_float(b0 & 0xffff0000u), t1 = r1 - __uint_as_float(b1 & 0xffff0000u);
        p[0][e] = __builtin_amdgcn_perm(a1, a0, 0x07060302u);
        p[1][e] = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
        p[2][e] = __builtin_amdgcn_perm(__float_as_uint(t1), __float_as_uint(t0), 0x07060302u);
      }
      u32x4 vf[4];
#pragma unroll
      for (int d = 0; d < 4; ++d) vf[d] = vt[gk * 256 + (32 * d + li) * 2 + half];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        if (decltype(special)::value && i == 1)
#pragma unroll
          for (int d = 0; d < 4; ++d) vf[d] = finite_part(vf[d]);
#pragma unroll
        for (int d = 0; d < 4; ++d)
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vf[d]),
                                                         __builtin_bit_cast(bf16x8, p[i]), o[d], 0, 0, 0);
      }
    }
  };

  auto walk = [&](auto special) __attribute__((always_inline)) {
    for (int t = 0; t < tiles; t += 2) {
      // Tile t is in ka / va (every wave has waited for its own loads into LDS, which __syncthreads
      // alone does not do), and every wave is past tile t - 1 in kb / vb.
      skv::drain_and_barrier();
      if (t + 1 < tiles) issue(t + 1, kb, vb);
      compute(special, t, ka, va);
      if (t + 1 < tiles) {
        skv::drain_and_barrier();
        if (t + 2 < tiles) issue(t + 2, ka, va);
        compute(special, t + 1, kb, vb);
      }
    }
  };
  issue(0, ka, va);
  bool odd = false;
  for (int t = threadIdx.x; t < tiles; t += kWaves * 64) odd |= a.odd[bh * row_tiles + t] != 0;
  if (__syncthreads_or(odd)) walk(std::true_type{});  // workgroup-uniform
  else walk(std::false_type{});

  if (query < a.L) {
    const auto ls = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    const float inv = 1.f / (__uint_as_float(ls[0]) + __uint_as_float(ls[1]));
    uint16_t* dst = a.out + b * a.o_sb + hq * a.o_sh + static_cast<int64_t>(query) * a.o_ss + 4 * half;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *reinterpret_cast<uint32_t __attribute__((ext_vector_type(2)))*>(dst + 32 * d + 8 * r) = {
            skv::f2bf2(o[d][4 * r] * inv, o[d][4 * r + 1] * inv),
            skv::f2bf2(o[d][4 * r + 2] * inv, o[d][4 * r + 3] * inv)};
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

extern "C" int64_t skv_prefill_attn_workspace_bytes(int batch_size, int kv_heads, int len) {
  if (batch_size < 1 || kv_heads < 1 || len < 1) return 0;
  return static_cast<int64_t>(batch_size) * kv_heads * ((len + kTileKeys - 1) / kTileKeys) * (kTile16 * 16 + 4);
}

extern "C" int skv_prefill_attn(const uint16_t* q, int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_s,
                                const uint16_t* k, int64_t k_stride_b, int64_t k_stride_h, int64_t k_stride_s,
                                const uint16_t* v, int64_t v_stride_b, int64_t v_stride_h, int64_t v_stride_s,
                                uint16_t* out, int64_t o_stride_b, int64_t o_stride_s, int64_t o_stride_h,
                                int batch_size, int q_heads, int kv_heads, int len, float scale, void* workspace,
                                int64_t workspace_bytes, void* stream) {
  const char* what = "prefill_attn";
  if (!q || !k || !v || !out || !workspace) {
    skv_set_error("%s: null pointer", what);
    return SKV_EINVAL;
  }
  if (batch_size < 1 || kv_heads < 1 || q_heads < kv_heads || q_heads % kv_heads || len < 1) {
    skv_set_error("%s: batch=%d q_heads=%d kv_heads=%d len=%d", what, batch_size, q_heads, kv_heads, len);
    return SKV_EINVAL;
  }
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(workspace) || (reinterpret_cast<uintptr_t>(out) & 7) ||
      q_stride_b % 8 || q_stride_h % 8 || q_stride_s % 8 || k_stride_b % 8 || k_stride_h % 8 || k_stride_s % 8 ||
      v_stride_b % 8 || v_stride_h % 8 || v_stride_s % 8 || o_stride_b % 4 || o_stride_s % 4 || o_stride_h % 4) {
    skv_set_error("%s: q, k and v rows must be 16-byte aligned, out rows 8-byte", what);
    return SKV_EINVAL;
  }
  if (workspace_bytes < skv_prefill_attn_workspace_bytes(batch_size, kv_heads, len)) {
    skv_set_error("%s: workspace of %lld bytes (%lld needed)", what, (long long)workspace_bytes,
                  (long long)skv_prefill_attn_workspace_bytes(batch_size, kv_heads, len));
    return SKV_EINVAL;
  }
  const int64_t rows = static_cast<int64_t>(batch_size) * kv_heads;
  const int tiles = (len + kTileKeys - 1) / kTileKeys;
  const int qblocks = (len + kQBlock - 1) / kQBlock;
  const int G = q_heads / kv_heads;
  const int64_t per = static_cast<int64_t>(G) * qblocks;
  int64_t grid = rows * per;
  if (rows % kXcds && kXcds % rows == 0) grid = (per + kXcds / rows - 1) / (kXcds / rows) * kXcds;
  if (rows > 65535 || grid > (int64_t{1} << 30)) {
    skv_set_error("%s: batch=%d q_heads=%d kv_heads=%d len=%d", what, batch_size, q_heads, kv_heads, len);
    return SKV_EUNSUPPORTED;
  }
  const hipStream_t s = static_cast<hipStream_t>(stream);
  u32x4* vt = static_cast<u32x4*>(workspace);
  int* odd = reinterpret_cast<int*>(vt + rows * tiles * kTile16);
  hipLaunchKernelGGL(vt_kernel, dim3(tiles, static_cast<unsigned>(rows)), dim3(256), 0, s, v, v_stride_b, v_stride_h,
                     v_stride_s, kv_heads, len, vt, tiles * 4, odd);
  PrefillArgs a{q, q_stride_b, q_stride_h, q_stride_s, k, k_stride_b, k_stride_h, k_stride_s, vt, odd, out,
                o_stride_b, o_stride_h, o_stride_s, q_heads, kv_heads, G, len, qblocks, static_cast<int>(rows),
                scale * 1.44269504088896340736f};
  hipLaunchKernelGGL(prefill_attn_kernel, dim3(static_cast<unsigned>(grid)), dim3(kWaves * 64), 0, s, a);
  return skv_check_launch(what);
}
