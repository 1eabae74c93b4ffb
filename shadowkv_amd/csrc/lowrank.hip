// The two passes over a prompt's pre-RoPE keys that its low-rank factors take (get_svd,
// models/kvcache/shadow.py:411-444), straight from the bf16 keys in the layout the model has them in:
//
//   gram_kernel     G = K^T K, K [rows, H * 128]: bf16 products are exact in fp32, sums in fp32 per share
//   gram_sum_kernel of the rows, the shares added in fp64, G [n, n] fp32, both triangles.
//   factors_split_kernel  the eigenvectors as three bf16 parts (an exact sum of 8 + 8 + 8 bits),
//                         and SV = diag(s) V^T per head in bf16.
//   project_kernel  U = K V / s, the fp32 V multiplied exactly as its three parts, one rounding.
//
// Bound: the matrix cores and the reads of K. The fp32 path converted K (twice its size written and read
// back twice), multiplied on the fp32 matrix pipe (a sixteenth of the bf16 rate) and rounded in further
// passes.
//
// gram_kernel: a workgroup of 8 waves owns a 256 x 256 tile of the lower triangle and a share of the rows.
// The contraction runs over rows, so both operands need 8 rows of one column side by side: a thread reads
// an 8 x 8 block (8 rows, 16 bytes each), transposes it with 32 byte permutes and writes 8 columns to
// LDS as [8-row group][column], the columns of a group of 8 in the order c ^ group, so that writes and
// operand reads are free of bank conflicts. Each wave multiplies 128 x 64 on v_mfma_f32_32x32x16_bf16.
// project_kernel: a workgroup of 4 waves owns 256 rows and NT * 32 vectors, both operands by direct
// loads into LDS (swizzled at the source), double-buffered in blocks of 32 columns.
//
// MI355X, 122880 x 1024 keys, rank 160 (rank 64, 128, 192: factors 59, 114, 150): Gram matrix 385 us (671 TFLOP/s; conversion and fp32 product 2480),
// factors 156 us (774 TFLOP/s issued; product, division, roundings and transposed copies 450); 3001 rows: 47
// and 27 us against 70 and 43. Error of G against fp64 1e-7, at most 5e-7 in
// large batches (fp32 product: 2e-5); of U the same.
#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "skv_common.h"

namespace {

using skv::u32x4;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kD = 128;
constexpr int kTile = 256;     // Gram tile
constexpr int kStage = 64;     // rows per stage
constexpr int kMaxN = 1024;
constexpr int kGramThreads = 512;

struct Keys {
  const uint16_t* k;
  int64_t sb, sh, ss;  // (batch, head, row) strides, elements
  int rows, n;         // n = heads * 128
  __device__ __forceinline__ const uint16_t* at(int b, int row, int col) const {
    return k + b * sb + static_cast<int64_t>(row) * ss + (col >> 7) * sh + (col & 127);
  }
};

__device__ __forceinline__ f32x16 mfma(const u32x4& a, const u32x4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                 0);
}

__device__ __forceinline__ void tile_of(int t, int& ti, int& tj) {  // lower triangle, row-major
  ti = 0;
  while (t > ti) t -= ++ti;
  tj = t;
}

// part[b][share][tile][256][256]
__global__ void __launch_bounds__(kGramThreads, 2) gram_kernel(Keys x, float* __restrict__ part, int tiles, int shares,
                                                               int share_rows) {
  __shared__ u32x4 buf0[8 * 2 * kTile], buf1[8 * 2 * kTile];  // [8-row group][A columns | B columns]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 31, half = lane >> 5;
  // Share s and its tiles on one XCD (workgroup w runs on XCD w mod 8): the tiles read the same rows. The next
  // sequence's shares begin on the XCD after this one's last (batch 13 of 122880 x 1024 keys: 20.0 -> 2.8 ms).
  const int b = blockIdx.y;
  const int w = blockIdx.x, g8 = w / (8 * tiles), r8 = w - g8 * 8 * tiles;
  const int share = 8 * g8 + ((r8 - (b % 8) * shares) & 7), tile = r8 / 8;
  if (share >= shares) return;  // workgroup-uniform
  int ti, tj;
  tile_of(tile, ti, tj);
  const bool diag = ti == tj;
  const int row0 = share * share_rows, row1 = min(x.rows, row0 + share_rows);

  // This thread's 8 x 8 block of a stage: rows 8 rg .., columns 8 cg .. of [A panel | B panel].
  const int cg = lane, rg = wave;
  const int col = cg < 32 ? ti * kTile + 8 * cg : tj * kTile + 8 * (cg - 32);
  const bool want = col < x.n && (cg < 32 || !diag);
  const int lcol = want ? col : 0;
  u32x4 in[8];
  int at = 0;
  auto load = [&](int r0) {  // (unconditional, clamped loads; masked as they are stored)
    at = r0 + 8 * rg;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      in[e] = *reinterpret_cast<const u32x4*>(x.at(b, min(at + e, x.rows - 1), lcol));
  };
  auto store = [&](u32x4* buf) {
    if (cg >= 32 && diag) return;
    u32x4* dst = buf + rg * 2 * kTile + 8 * cg;
    const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int e = 0; e < 8; ++e) in[e] = want && at + e < row1 ? in[e] : zero;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t sel = e & 1 ? 0x07060302u : 0x05040100u;
      u32x4 o;
#pragma unroll
      for (int p = 0; p < 4; ++p) o[p] = __builtin_amdgcn_perm(in[2 * p + 1][e >> 1], in[2 * p][e >> 1], sel);
      dst[e ^ (cg & 7)] = o;
    }
  };
  const int wi = (wave >> 2) * 128, wj = (wave & 3) * 64;  // the wave's part of the tile
  f32x16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  auto place = [](int c) { return (c & ~7) | ((c ^ (c >> 3)) & 7); };
  const int bcol = diag ? 0 : kTile;
  auto compute = [&](const u32x4* buf) {
#pragma unroll
    for (int ks = 0; ks < kStage / 16; ++ks) {
      const u32x4* src = buf + (2 * ks + half) * 2 * kTile;
      u32x4 af[4], bf[2];
#pragma unroll
      for (int i = 0; i < 4; ++i) af[i] = src[place(wi + 32 * i + li)];
#pragma unroll
      for (int j = 0; j < 2; ++j) bf[j] = src[place(bcol + wj + 32 * j + li)];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma(af[i], bf[j], acc[i][j]);
    }
  };
  load(row0);
  store(buf0);
  for (int r = row0; r < row1; r += 2 * kStage) {
    __syncthreads();
    if (r + kStage < row1) load(r + kStage);
    compute(buf0);
    if (r + kStage < row1) {
      store(buf1);
      __syncthreads();
      if (r + 2 * kStage < row1) load(r + 2 * kStage);
      compute(buf1);
      if (r + 2 * kStage < row1) store(buf0);
    }
  }
  float* dst = part + ((static_cast<int64_t>(b) * shares + share) * tiles + tile) * kTile * kTile;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        dst[(wi + 32 * i + 8 * (r / 4) + 4 * half + (r % 4)) * kTile + wj + 32 * j + li] = acc[i][j][r];
}

// One 32 x 32 block of G per workgroup (256 threads), its shares added in order in fp64.
__global__ void __launch_bounds__(256) gram_sum_kernel(const float* __restrict__ part, float* __restrict__ gram, int n,
                                                       int tiles, int shares) {
  __shared__ float t[32][33];
  const int b = blockIdx.z, bi = blockIdx.y, bj = blockIdx.x;
  if (bj > bi) return;
  const int ti = bi / 8, tj = bj / 8, tile = ti * (ti + 1) / 2 + tj;
  const int c = threadIdx.x & 31;
  const float* src = part + (static_cast<int64_t>(b) * shares * tiles + tile) * kTile * kTile;
  float* g = gram + static_cast<int64_t>(b) * n * n;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = (threadIdx.x >> 5) + 8 * q;
    const float* p = src + ((bi % 8) * 32 + r) * kTile + (bj % 8) * 32 + c;
    double s = 0.0;
    for (int u = 0; u < shares; ++u) s += static_cast<double>(p[static_cast<int64_t>(u) * tiles * kTile * kTile]);
    t[r][c] = static_cast<float>(s);
    if (32 * bi + r < n && 32 * bj + c < n) g[static_cast<int64_t>(32 * bi + r) * n + 32 * bj + c] = t[r][c];
  }
  if (bi == bj) return;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = (threadIdx.x >> 5) + 8 * q;
    if (32 * bj + r < n && 32 * bi + c < n) g[static_cast<int64_t>(32 * bj + r) * n + 32 * bi + c] = t[c][r];
  }
}

// v3[b][part][rpad][n] (rows past the rank zero), sv[b][h][d][r] = bf16(s_r vt[r][128 h + d]).
__global__ void __launch_bounds__(256) factors_split_kernel(const float* __restrict__ w, const float* __restrict__ vt,
                                                            int rank, int rpad, int n, uint16_t* __restrict__ v3,
                                                            uint16_t* __restrict__ sv, int64_t sv_sb) {
  const int b = blockIdx.z;
  const int c = blockIdx.x * 32 + (threadIdx.x & 31), r = blockIdx.y * 8 + (threadIdx.x >> 5);
  if (c >= n || r >= rpad) return;
  const float x = r < rank ? vt[(static_cast<int64_t>(b) * rank + r) * n + c] : 0.f;
  uint16_t* dst = v3 + (static_cast<int64_t>(b) * 3 * rpad + r) * n + c;
  const uint32_t u0 = __float_as_uint(x) & 0xffff0000u;
  const float x1 = x - __uint_as_float(u0);
  const uint32_t u1 = __float_as_uint(x1) & 0xffff0000u;
  const float x2 = x1 - __uint_as_float(u1);
  dst[0] = static_cast<uint16_t>(u0 >> 16);
  dst[static_cast<int64_t>(rpad) * n] = static_cast<uint16_t>(u1 >> 16);
  dst[2 * static_cast<int64_t>(rpad) * n] = static_cast<uint16_t>(__float_as_uint(x2) >> 16);
  if (r < rank) {
    const float s = sqrtf(fmaxf(w[b * rank + r], 0.f));
    sv[b * sv_sb + static_cast<int64_t>(c) * rank + r] = skv::f2bf(s * x);
  }
}

__device__ __forceinline__ void load_lds(const void* src, u32x4* dst) {  // 1 KB: lane l's 16 bytes to dst + 16 l
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

constexpr int kPRows = 256, kPCols = 32;  // rows of a workgroup, columns of a block

template <int NT>
__global__ void __launch_bounds__(256, 1) project_kernel(Keys x, const uint16_t* __restrict__ v3, int rpad,
                                                         const float* __restrict__ w, int rank,
                                                         uint16_t* __restrict__ u, int64_t u_sb) {
  constexpr int kVRows = 3 * NT * 32;
  constexpr int kBuf = (kPRows + kVRows) * 4;  // 16-byte chunks: rows of 4
  __shared__ u32x4 buf0[kBuf], buf1[kBuf];
  __shared__ float4 inv[NT * 8];  // 1 / s of the workgroup's vectors
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 31, half = lane >> 5;
  const int b = blockIdx.z, row0 = blockIdx.x * kPRows, rt0 = blockIdx.y * NT * 32;
  const uint16_t* vb = v3 + static_cast<int64_t>(b) * 3 * rpad * x.n;
  // 16 rows of 4 chunks per load; chunk q of row r in slot q ^ (r / 4 % 4).
  const int lr = lane >> 2, lq = (lane & 3) ^ ((lane >> 4) & 3);
  auto issue = [&](int c0, u32x4* buf) {
    const int col = c0 + 8 * lq;
#pragma unroll
    for (int i = 0; i < kPRows / 16 / 4; ++i) {
      const int r = 16 * (wave + 4 * i);
      load_lds(x.at(b, min(row0 + r + lr, x.rows - 1), col), buf + 4 * r);
    }
    for (int i = wave; i < kVRows / 16; i += 4) {
      const int r = 16 * i + lr, part = r / (NT * 32), rr = r - part * NT * 32;
      load_lds(vb + (static_cast<int64_t>(part) * rpad + rt0 + rr) * x.n + col, buf + 4 * (kPRows + 16 * i));
    }
  };
  f32x16 acc[2][NT];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][t][r] = 0.f;
  const int swz = (li >> 2) & 3;
  auto compute = [&](const u32x4* buf) {
#pragma unroll
    for (int ks = 0; ks < kPCols / 16; ++ks) {
      const int q = (2 * ks + half) ^ swz;
      u32x4 kf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) kf[i] = buf[4 * (64 * wave + 32 * i + li) + q];
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const u32x4 vf = buf[4 * (kPRows + (p * NT + t) * 32 + li) + q];
#pragma unroll
          for (int i = 0; i < 2; ++i) acc[i][t] = mfma(vf, kf[i], acc[i][t]);
        }
    }
  };
  issue(0, buf0);
  if (threadIdx.x < NT * 32) {
    const int r = rt0 + static_cast<int>(threadIdx.x);
    const float e = r < rank ? w[b * rank + r] : 0.f;
    reinterpret_cast<float*>(inv)[threadIdx.x] = 1.f / fmaxf(sqrtf(fmaxf(e, 0.f)), 1e-30f);
  }
  for (int c = 0; c < x.n; c += 2 * kPCols) {  // (n is a multiple of 128)
    skv::drain_and_barrier();  // block c is in buf0 (each wave has waited for its own loads), buf1 is free
    issue(c + kPCols, buf1);
    compute(buf0);
    skv::drain_and_barrier();
    if (c + 2 * kPCols < x.n) issue(c + 2 * kPCols, buf0);
    compute(buf1);
  }
  // acc: lane (row li of its tile), vectors 8 (r / 4) + 4 half + r % 4.
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = rt0 + 32 * t + 8 * q + 4 * half;
      if (r >= rank) continue;  // (the rank is a multiple of 4)
      const float4 f = inv[8 * t + 2 * q + half];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = row0 + 64 * wave + 32 * i + li;
        if (row < x.rows)
          *reinterpret_cast<uint32_t __attribute__((ext_vector_type(2)))*>(u + b * u_sb +
                                                                           static_cast<int64_t>(row) * rank + r) = {
              skv::f2bf2(acc[i][t][4 * q] * f.x, acc[i][t][4 * q + 1] * f.y),
              skv::f2bf2(acc[i][t][4 * q + 2] * f.z, acc[i][t][4 * q + 3] * f.w)};
      }
    }
}

bool aligned(const void* p, unsigned n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }

// Shares of the rows: enough workgroups for the 256 CUs (one each, 128 KB of LDS), at least four stages each and at
// most kShareRows rows, whatever the batch: the error of a share's fp32 sums grows with its rows (122880 x 1024 keys,
// relative to float64: 1.0e-7 in shares of 4928 rows, 2.2e-7 of 15360, 2.2e-6 in one; torch's fp32 product 2.1e-5).
constexpr int kShareRows = 16384;
void gram_plan(int rows, int n, int batch, int* tiles, int* shares, int* share_rows) {
  const int nt = (n + kTile - 1) / kTile;
  *tiles = nt * (nt + 1) / 2;
  const int fill = std::min(256 / (*tiles * batch), (rows + 4 * kStage - 1) / (4 * kStage));
  const int want = std::max({1, fill, (rows + kShareRows - 1) / kShareRows});
  *share_rows = ((rows + want - 1) / want + kStage - 1) / kStage * kStage;
  *shares = (rows + *share_rows - 1) / *share_rows;
}

bool shape_ok(const char* what, const uint16_t* keys, int64_t sb, int64_t sh, int64_t ss, int batch, int rows,
              int heads) {
  if (batch < 1 || batch > 65535 || rows < 1 || rows > (1 << 30) || heads < 1 || heads * kD > kMaxN) {
    skv_set_error("%s: batch=%d rows=%d heads=%d (at most %d columns)", what, batch, rows, heads, kMaxN);
    return false;
  }
  if (!aligned(keys, 16) || sb % 8 || sh % 8 || ss % 8) {
    skv_set_error("%s: key rows must be 16-byte aligned", what);
    return false;
  }
  return true;
}

// Forms of project_kernel: a workgroup of `tiles` vector tiles (of 32) reads its rows of the keys once for all of
// them, but is more work for one CU; 256 of them are a round of `us` at 1024 columns (further rounds take as long to
// within a fifth), and the form whose rounds take least in all is taken. Measured with 1 / 2 / 3 / 4 / 5 / 6 tiles, us:
// 122880 rows, rank 128 196 / 119 / 154 / 127, rank 160 242 / 163 / 154 / 214 / 141, rank 192 288 / 170 / 161 / 220 / 252 / 165;
// 50000 rows, rank 128 75 / 52 / 67 / 59; 32768 rows, rank 160 52 / 49 / 47 / 55 / 64; 8192 rows, rank 160
// 22 / 28 / 43 / 52 / 62: 4 and 6 tiles gain nowhere.
struct ProjectForm {
  int tiles, us;
};
constexpr ProjectForm kProjectForms[] = {{1, 19}, {2, 27}, {3, 40}, {5, 66}};

int project_tiles(int rtiles, int64_t row_blocks) {
  // (Three one-tile workgroups fit on a CU, so two rounds of them are little more than one: 19333 rows, rank 160
  // 30 us against 35 with two tiles.)
  if (row_blocks * rtiles <= 2 * 256) return 1;
  int best = 1;
  int64_t least = INT64_MAX;
  for (const ProjectForm& f : kProjectForms) {
    const int64_t us = (row_blocks * ((rtiles + f.tiles - 1) / f.tiles) + 255) / 256 * f.us;
    if (f.tiles <= rtiles && us < least) {
      least = us;
      best = f.tiles;
    }
  }
  return best;
}

// Rows of a part of v3: whole groups of any form.
int padded_rank(int rank) {
  const int rtiles = (rank + 31) / 32;
  int most = 0;
  for (const ProjectForm& f : kProjectForms) most = std::max(most, (rtiles + f.tiles - 1) / f.tiles * f.tiles);
  return 32 * most;
}

}  // namespace

extern "C" int64_t skv_keys_gram_workspace_bytes(int batch, int rows, int heads) {
  if (batch < 1 || rows < 1 || heads < 1 || heads * kD > kMaxN) return 0;
  int tiles, shares, share_rows;
  gram_plan(rows, heads * kD, batch, &tiles, &shares, &share_rows);
  return static_cast<int64_t>(batch) * shares * tiles * kTile * kTile * 4;
}

extern "C" int skv_keys_gram(const uint16_t* keys, int64_t stride_b, int64_t stride_h, int64_t stride_s, int batch,
                             int rows, int heads, float* gram, void* workspace, int64_t workspace_bytes,
                             void* stream) {
  const char* what = "keys_gram";
  if (!keys || !gram || !workspace) {
    skv_set_error("%s: null pointer", what);
    return SKV_EINVAL;
  }
  if (!shape_ok(what, keys, stride_b, stride_h, stride_s, batch, rows, heads)) return SKV_EUNSUPPORTED;
  if (!aligned(workspace, 16) || workspace_bytes < skv_keys_gram_workspace_bytes(batch, rows, heads)) {
    skv_set_error("%s: workspace of %lld bytes, 16-byte aligned (%lld needed)", what, (long long)workspace_bytes,
                  (long long)skv_keys_gram_workspace_bytes(batch, rows, heads));
    return SKV_EINVAL;
  }
  const int n = heads * kD;
  int tiles, shares, share_rows;
  gram_plan(rows, n, batch, &tiles, &shares, &share_rows);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const Keys x{keys, stride_b, stride_h, stride_s, rows, n};
  float* part = static_cast<float*>(workspace);
  hipLaunchKernelGGL(gram_kernel, dim3((shares + 7) / 8 * 8 * tiles, batch), dim3(kGramThreads), 0, s, x, part, tiles,
                     shares, share_rows);
  hipLaunchKernelGGL(gram_sum_kernel, dim3(n / 32, n / 32, batch), dim3(256), 0, s, part, gram, n, tiles, shares);
  return skv_check_launch(what);
}

extern "C" int64_t skv_keys_factors_workspace_bytes(int batch, int heads, int rank) {
  if (batch < 1 || heads < 1 || heads * kD > kMaxN || rank < 1) return 0;
  return static_cast<int64_t>(batch) * 3 * padded_rank(rank) * heads * kD * 2;
}

extern "C" int skv_keys_factors(const uint16_t* keys, int64_t stride_b, int64_t stride_h, int64_t stride_s, int batch,
                                int rows, int heads, const float* w, const float* vt, int rank, uint16_t* u,
                                int64_t u_stride_b, uint16_t* sv, int64_t sv_stride_b, void* workspace,
                                int64_t workspace_bytes, void* stream) {
  const char* what = "keys_factors";
  if (!keys || !w || !vt || !u || !sv || !workspace) {
    skv_set_error("%s: null pointer", what);
    return SKV_EINVAL;
  }
  if (!shape_ok(what, keys, stride_b, stride_h, stride_s, batch, rows, heads)) return SKV_EUNSUPPORTED;
  const int n = heads * kD;
  if (rank < 1 || rank > n || rank % 4) {
    skv_set_error("%s: rank=%d (a multiple of 4 up to %d)", what, rank, n);
    return SKV_EUNSUPPORTED;
  }
  if (!aligned(u, 8) || u_stride_b % 4 || !aligned(workspace, 16) ||
      workspace_bytes < skv_keys_factors_workspace_bytes(batch, heads, rank)) {
    skv_set_error("%s: workspace of %lld bytes, 16-byte aligned (%lld needed), u rows 8-byte aligned", what,
                  (long long)workspace_bytes, (long long)skv_keys_factors_workspace_bytes(batch, heads, rank));
    return SKV_EINVAL;
  }
  const int rtiles = (rank + 31) / 32, rpad = padded_rank(rank);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const Keys x{keys, stride_b, stride_h, stride_s, rows, n};
  uint16_t* v3 = static_cast<uint16_t*>(workspace);
  hipLaunchKernelGGL(factors_split_kernel, dim3(n / 32, rpad / 8, batch), dim3(256), 0, s, w, vt, rank, rpad, n, v3, sv,
                     sv_stride_b);
  const int rb = (rows + kPRows - 1) / kPRows;
  const int nt = project_tiles(rtiles, static_cast<int64_t>(rb) * batch);
  const dim3 grid(rb, (rtiles + nt - 1) / nt, batch);
  auto go = [&](auto form) {
    hipLaunchKernelGGL(project_kernel<decltype(form)::value>, grid, dim3(256), 0, s, x, v3, rpad, w, rank, u, u_stride_b);
  };
  if (nt == 1) go(std::integral_constant<int, 1>{});
  else if (nt == 2) go(std::integral_constant<int, 2>{});
  else if (nt == 3) go(std::integral_constant<int, 3>{});
  else go(std::integral_constant<int, 5>{});
  return skv_check_launch(what);
}
