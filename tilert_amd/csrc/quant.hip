// act_quant (per 1x128 group, e4m3fn + fp32 scale), 128x128 block weight quantisation
// and weight dequantisation.
#include <type_traits>

#include "common.h"
#include "../../include/tilert_amd.h"

namespace tl {

// One thread = 8 consecutive elements; 16 threads = one 128-element group.
// Launch-bound at decode sizes (4 x 7168 1.9 us), then HBM-bound (4096 x 7168 19.1 us, 4.6 TB/s).
// Two or four chunks a thread, for fewer waves, are slower (256 x 18432 5.45 -> 5.94 / 6.90
// us): the amax, the scale's division and the encode are one chain per chunk.
__global__ __launch_bounds__(256) void act_quant_kernel(const uint16_t* __restrict__ x,
                                                        uint8_t* __restrict__ y,
                                                        float* __restrict__ s, int64_t n_groups,
                                                        int scale_mode) {
  const int64_t tid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t grp = tid >> 4;
  const bool live = grp < n_groups;
  uint4 raw = make_uint4(0, 0, 0, 0);
  if (live) raw = reinterpret_cast<const uint4*>(x)[tid];
  float v[8];
  v[0] = bf16_to_f32(raw.x & 0xffff); v[1] = bf16_to_f32(raw.x >> 16);
  v[2] = bf16_to_f32(raw.y & 0xffff); v[3] = bf16_to_f32(raw.y >> 16);
  v[4] = bf16_to_f32(raw.z & 0xffff); v[5] = bf16_to_f32(raw.z >> 16);
  v[6] = bf16_to_f32(raw.w & 0xffff); v[7] = bf16_to_f32(raw.w >> 16);
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) amax = fmaxf(amax, __builtin_fabsf(v[i]));
  amax = row16_reduce<true>(amax);  // the group's 16 lanes
  const float sc = group_scale(amax, scale_mode);
  if (live) {
    reinterpret_cast<uint2*>(y)[tid] = quant8_e4m3(v, sc);
    if ((tid & 15) == 0) s[grp] = sc;
  }
}

// One 256-thread workgroup per 128x128 block: amax, s = amax/448 (1 for all-zero
// blocks), q = e4m3(clamp(w/s)).
template <typename T>
__device__ inline float load_w(const T* p);
template <>
__device__ inline float load_w<float>(const float* p) { return *p; }
template <>
__device__ inline float load_w<uint16_t>(const uint16_t* p) { return bf16_to_f32(*p); }

typedef uint32_t u32x4n __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2n __attribute__((ext_vector_type(2)));

// NT: a non-temporal store (a run-time choice between the two would be merged into one plain store).
template <bool NT, class T>
__device__ inline void store_chunk(T* p, T v) {
  if constexpr (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// A lane's 8 weights of a 128-column block row (chunk c of 16), as fp32, by non-temporal 16-byte loads whose
// 16 lanes cover consecutive memory: bf16 columns 8c..8c+7; fp32 columns 4c..4c+3 and
// 64+4c..+3 (8 consecutive ones would leave half of every line to the second load, which a
// non-temporal line does not wait for: 128 us at 18432 x 7168, against 116 this way and 118 with
// temporal loads).
template <typename T>
struct WChunk;
template <>
struct WChunk<uint16_t> {
  static constexpr int kStep0 = 8, kOff1 = 4;  // columns: kStep0 c and kStep0 c + kOff1
  __device__ static inline void load(const uint16_t* row, int64_t c0, int64_t, float (&v)[8]) {
    const u32x4n a = __builtin_nontemporal_load(reinterpret_cast<const u32x4n*>(row + c0));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(a[i] << 16);
      v[2 * i + 1] = __uint_as_float(a[i] & 0xffff0000u);
    }
  }
};
template <>
struct WChunk<float> {
  static constexpr int kStep0 = 4, kOff1 = 64;
  __device__ static inline void load(const float* row, int64_t c0, int64_t c1, float (&v)[8]) {
    const v4f a = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(row + c0));
    const v4f b = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(row + c1));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = a[i];
      v[4 + i] = b[i];
    }
  }
};

// K % 8 == 0 and 16-byte aligned weights: HBM-bound (the weight in once, codes out).  A
// thread holds 8 rows x 8 columns of its block in registers between the amax and the
// encode, so the block is read once, by 16-byte loads that are all in flight together; rows
// and chunks past the edge repeat the last one (which leaves the amax alone) and are not stored.
// bf16 18432 x 7168 (396 MB moved): 64 us (6.2 TB/s; 74 with temporal loads) against 321 us
// with the element-wise kernel below, which reads the block twice, two bytes a lane.
template <typename T>
__global__ __launch_bounds__(256) void weight_quant_kernel(const T* __restrict__ w, uint8_t* __restrict__ q,
                                                           float* __restrict__ s, int64_t N, int64_t K) {
  __shared__ float red[4];
  constexpr int kRows = 8;  // rows per thread: r0 + 16 i
  const int64_t nb = blockIdx.y, kb = blockIdx.x;
  const int c = threadIdx.x & 15, r0 = threadIdx.x >> 4;
  using Ch = WChunk<T>;
  const int64_t col0 = kb * kBlock + Ch::kStep0 * c, col1 = col0 + Ch::kOff1;  // 4 columns each
  float v[kRows][8];
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    const int64_t n = nb * kBlock + r0 + 16 * i;
    const T* row = w + (n < N ? n : N - 1) * K;
    const int64_t tail = K - (Ch::kOff1 == 4 ? 8 : 4);  // the last whole chunk
    Ch::load(row, col0 < K ? col0 : tail, col1 < K ? col1 : tail, v[i]);
  }
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < kRows; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, __builtin_fabsf(v[i][j]));
  amax = wave_max_f32(amax);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float sc = amax > 0.f ? amax / 448.0f : 1.0f;
  if (threadIdx.x == 0) s[nb * cdiv(K, kBlock) + kb] = sc;
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    const int64_t n = nb * kBlock + r0 + 16 * i;
    const uint2 code = quant8_e4m3(v[i], sc);
    if constexpr (Ch::kOff1 == 4) {
      if (n < N && col0 < K) *reinterpret_cast<uint2*>(q + n * K + col0) = code;
    } else {
      if (n < N && col0 < K) *reinterpret_cast<uint32_t*>(q + n * K + col0) = code.x;
      if (n < N && col1 < K) *reinterpret_cast<uint32_t*>(q + n * K + col1) = code.y;
    }
  }
}

// Any K and alignment.
template <typename T>
__global__ __launch_bounds__(256) void weight_quant_any_kernel(const T* __restrict__ w, uint8_t* __restrict__ q,
                                                               float* __restrict__ s, int64_t N, int64_t K) {
  __shared__ float red[256];
  const int64_t nb = blockIdx.y, kb = blockIdx.x;
  const int64_t KB = cdiv(K, kBlock);
  const int col = threadIdx.x & 127;
  const int r0 = threadIdx.x >> 7;  // 0..1
  const int64_t c = kb * kBlock + col;
  float amax = 0.f;
  for (int r = r0; r < kBlock; r += 2) {
    const int64_t n = nb * kBlock + r;
    if (n < N && c < K) amax = fmaxf(amax, __builtin_fabsf(load_w(w + n * K + c)));
  }
  red[threadIdx.x] = amax;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (static_cast<int>(threadIdx.x) < o) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + o]);
    __syncthreads();
  }
  amax = red[0];
  const float sc = amax > 0.f ? amax / 448.0f : 1.0f;
  if (threadIdx.x == 0) s[nb * KB + kb] = sc;
  for (int r = r0; r < kBlock; r += 2) {
    const int64_t n = nb * kBlock + r;
    if (n < N && c < K) {
      float v = load_w(w + n * K + c) / sc;
      q[n * K + c] = static_cast<uint8_t>(f32_to_e4m3(fminf(fmaxf(v, -kE4m3Max), kE4m3Max)));
    }
  }
}

__device__ inline float e4m3_to_f32(uint32_t code) {
  const uint32_t sign = (code & 0x80u) << 24;
  const uint32_t e = (code >> 3) & 0xfu, m = code & 7u;
  float mag;
  if (e == 0xfu && m == 7u) return __uint_as_float(0x7fc00000u);
  if (e == 0) mag = static_cast<float>(m) * 0.001953125f;  // m * 2^-9
  else mag = __uint_as_float(((e + 120u) << 23) | (m << 20));
  return __uint_as_float(__float_as_uint(mag) | sign);
}

// Rows of a multiple of V columns, aligned, in weights of kDqWide elements: HBM-bound on the output.  A lane turns V
// codes (4 for fp32, 8 for bf16) into one 16-byte store, so a wave stores 1 KB of consecutive memory per
// instruction; a wave's kDqRows rows (4 apart, inside one 128-row scale block) are loaded
// together.  v_cvt_pk_f32_fp8 decodes two codes exactly and v_cvt_pk_bf16_f32 rounds two results (RNE): rounding in
// integer operations made the unrolled bf16 body long enough for its instruction fetch to bound small weights
// (512 x 2048 5.4 us, 3.6 this way).  18432 x 7168 to fp32 (661 MB moved): 96 us (6.9 TB/s) against 366 us with the
// one-code-per-thread kernel below, which spends its time in a 64-bit division per element and moves 1 byte per lane.
constexpr int kDqRows = 8;
// Below 1 M elements 8 rows a lane leave too few waves (us, wide / one code per thread, bf16: 128 x 128 3.6 / 2.3,
// 512 x 512 3.5 / 2.4, 512 x 1024 3.5 / 2.9, 1024 x 1024 3.6 / 3.8, 512 x 4096 3.7 / 5.8).
constexpr int64_t kDqWide = 1 << 20;
// Results that the Infinity Cache cannot hold for their reader are stored non-temporally (NT).  us, dequantise + a
// product that reads the result, NT against plain stores: bf16 2112 x 7168 (29 MB) 26.7 / 24.4, 7168 x 7168 (98 MB)
// 50.0 / 45.2, 18432 x 7168 (252 MB) 122 / 116; fp32 7168 x 7168 (196 MB) 112 / 86, 9216 x 7168 (252 MB) 141 / 142,
// 10240 x 7168 (280 MB) 153 / 161, 18432 x 7168 (504 MB) 269 / 275.
constexpr int64_t kDqNtBytes = 256 << 20;
template <bool BF16, bool NT>
__global__ __launch_bounds__(256) void weight_dequant_kernel(const uint8_t* __restrict__ q, const float* __restrict__ s,
                                                             void* __restrict__ out, int64_t N, int64_t K) {
  constexpr int V = BF16 ? 8 : 4, W = V / 4;
  const int64_t col = (static_cast<int64_t>(blockIdx.x) * 64 + (threadIdx.x & 63)) * V;
  if (col >= K) return;
  const int64_t n0 = static_cast<int64_t>(blockIdx.y) * (4 * kDqRows) + (threadIdx.x >> 6);
  uint32_t d[kDqRows][W];
#pragma unroll
  for (int i = 0; i < kDqRows; ++i) {
    const int64_t n = n0 + 4 * i;
    const uint32_t* p = reinterpret_cast<const uint32_t*>(q + (n < N ? n : N - 1) * K + col);
    if constexpr (W == 2) {
      const uint2 t = *reinterpret_cast<const uint2*>(p);
      d[i][0] = t.x; d[i][1] = t.y;
    } else {
      d[i][0] = *p;
    }
  }
  const float sc = s[(n0 / kBlock) * cdiv(K, kBlock) + col / kBlock];
#pragma unroll
  for (int i = 0; i < kDqRows; ++i) {
    const int64_t n = n0 + 4 * i;
    float f[V];
#pragma unroll
    for (int j = 0; j < W; ++j) {
      const v2f a = __builtin_amdgcn_cvt_pk_f32_fp8(d[i][j], false), b = __builtin_amdgcn_cvt_pk_f32_fp8(d[i][j], true);
      f[4 * j] = a[0] * sc; f[4 * j + 1] = a[1] * sc;
      f[4 * j + 2] = b[0] * sc; f[4 * j + 3] = b[1] * sc;
    }
    if (n >= N) continue;
    if constexpr (BF16) {
      uint32_t o[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = bf16x2_bits(v2f{f[2 * j], f[2 * j + 1]});
      store_chunk<NT>(reinterpret_cast<u32x4n*>(static_cast<uint16_t*>(out) + n * K + col), u32x4n{o[0], o[1], o[2], o[3]});
    } else {
      store_chunk<NT>(reinterpret_cast<v4f*>(static_cast<float*>(out) + n * K + col), v4f{f[0], f[1], f[2], f[3]});
    }
  }
}

// Any size, K and alignment.
__global__ __launch_bounds__(256) void weight_dequant_any_kernel(const uint8_t* __restrict__ q,
                                                                 const float* __restrict__ s,
                                                                 void* __restrict__ out, int64_t N,
                                                                 int64_t K, int out_bf16) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= N * K) return;
  const int64_t n = i / K, k = i - n * K;
  const float v = e4m3_to_f32(q[i]) * s[(n / kBlock) * cdiv(K, kBlock) + k / kBlock];
  if (out_bf16) static_cast<uint16_t*>(out)[i] = f32_to_bf16(v);
  else static_cast<float*>(out)[i] = v;
}

// RMSNorm (tilert/models/common.py:92-133, no residual): y = bf16(gamma * x * rsqrt(mean(x^2)
// + eps)) in fp32, then -- when y8/ys are given -- act_quant of those bf16 values per
// 1x128 group (rmsnorm_quant_op, ops/rmsnorm_quant.py:19-63).  rsqrt is 1 / sqrt with IEEE
// sqrt and division, as torch's.
// A row's sum of squares is taken over a fixed tree of kNormVirt virtual threads: virtual
// thread v adds the squares of chunks (8 elements) v, v + kNormVirt, ... in order, each
// 64 virtual threads are one DPP wave reduction, and the kNormVirt / 64 wave partials are
// added in order -- the same float result whatever the launch shape.  The row is then cut
// into slices of kNormSlice chunks, one 256-thread workgroup each (thread = one chunk, 16
// threads = one 128-element group): every workgroup of a row recomputes the row's sum
// (the row is 8-32 KB, read from L2 after the first) and normalises and quantises only
// its slice.  One 1024-thread workgroup per row left a decode step's 4 rows on 4 CUs,
// issue-bound on the quantisation (5.2 us at 4 x 7168).
constexpr int kNormThreads = 256;
constexpr int kNormVirt = 1024;
constexpr int kNormPerThread = kNormVirt / kNormThreads;  // virtual threads per thread
constexpr int kNormMaxChunks = 2;                           // chunks per virtual thread
constexpr int kNormSlice = kNormThreads;                    // chunks per workgroup
constexpr int kNormMaxDim = kNormMaxChunks * kNormVirt * 8;  // 16384
constexpr int kNormRowsGrid = 1024;  // workgroups of the whole-row kernel (512 and 2048 measured level)
// Rows from which whole rows beat slices, by slices per row: a row of one slice (dim <= 2048) is a
// whole row either way, without the sum's clamped loads (2.8 against 2.9 us at 1 row); up to 12288 wide the redundant
// sums of the slices cost as much as the longer chain of a whole row at 256 rows (us, whole rows / slices; dim 7168:
// 128 / 256 / 512 / 4096 rows 4.6 / 3.8, 5.0 / 5.2, 6.3 / 8.1, 28.5 / 48.8; dim 3072: 3.5 / 3.2, 3.7 / 3.7,
// 4.3 / 5.0, 15.1 / 18.5; dim 12288: 5.8 / 5.2, 6.5 / 7.8, 8.7 / 11.6, 44.3 / 108); beyond that the registers of a whole
// row (8 chunks a thread: 256 VGPRs) leave one workgroup per CU (dim 16384: 320 / 512 / 1024 / 4096 rows 13.3 / 10.7,
// 14.7 / 14.8, 26.3 / 35.5, 78.9 / 189; dim 14336: 1024 / 4096 rows 25.6 / 24.9, 74.9 / 148).
__host__ inline int64_t norm_rows_min(int64_t slices) { return slices <= 1 ? 1 : (slices <= 6 ? 256 : 1024); }

__device__ inline float sum_squares(const uint4& raw, bool in, float ss) {
  const uint32_t w4[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float lo = in ? bf16_to_f32(w4[j] & 0xffff) : 0.f;
    const float hi = in ? bf16_to_f32(w4[j] >> 16) : 0.f;
    ss = __builtin_fmaf(lo, lo, ss);
    ss = __builtin_fmaf(hi, hi, ss);
  }
  return ss;
}

__device__ inline float norm_factor(const float (&part)[kNormVirt / 64], int dim, float eps) {
  float tot = 0.f;
#pragma unroll
  for (int w = 0; w < kNormVirt / 64; ++w) tot += part[w];
  return 1.0f / __builtin_sqrtf(tot / static_cast<float>(dim) + eps);
}

// Which outputs the whole-row kernel stores non-temporally: from 3 MB of them (y and codes) both, about what the L2s
// hold and would write back at the kernel's end; smaller ones the next kernel reads from L2.  From 40 MB only y, and only
// where codes are given: what is stored non-temporally then goes to memory, where plain stores leave it in the Infinity
// Cache, and the codes are what the next GEMMs read.  us, norm + a kernel that reads the codes / that reads y,
// non-temporal against plain: 256 x 1536 5.4 / 5.5 against 5.2 / 5.4; 2048 x 1536 9.4 / 11.0 against 10.1 / 12.2;
// 8192 x 1536 23.9 / 28.5 against 24.9 / 29.1; 256 x 7168 8.0 / 8.7 against 8.1 / 9.1; 1024 x 7168 13.6 / 16.6 against
// 14.8 / 17.9; 2048 x 7168 24.0 / 30.6 against 25.0 / 29.1; 4096 x 7168 45.2 / 53.8 against 43.3 / 50.9.  4096 x 7168 with
// the index keys behind it, both / y only / plain: 32.1 / 33.0 / 35.8; with 16 FP8 GEMMs 7168 -> 2112 on its codes too
// 334.8 / 327.1 / 327.7; where y is read as well 355 / 348 / 347.
enum NormNt { kNtNone, kNtY, kNtBoth };
constexpr int64_t kNormNtMin = 3 << 20, kNormNtMax = 40 << 20;
__host__ inline NormNt norm_nt(int64_t rows, int64_t dim, bool codes) {
  const int64_t bytes = rows * dim * (codes ? 3 : 2);
  return bytes < kNormNtMin ? kNtNone : (bytes < kNormNtMax ? kNtBoth : (codes ? kNtY : kNtNone));
}

// Normalise (and quantise) chunk c of a row: 16 consecutive lanes hold a 128-element group.
template <NormNt NT>
__device__ inline void norm_chunk(const uint4& raw, const float (&gv)[8], float r, bool live, int c, int row, int dim,
                                  uint16_t* __restrict__ y, uint8_t* __restrict__ y8, float* __restrict__ ys,
                                  int scale_mode) {
  const uint32_t w4[4] = {raw.x, raw.y, raw.z, raw.w};
  uint32_t b[4];  // bf16 pairs
  float q[8];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const v2f f = {gv[2 * j] * (bf16_to_f32(w4[j] & 0xffff) * r), gv[2 * j + 1] * (bf16_to_f32(w4[j] >> 16) * r)};
    b[j] = bf16x2_bits(f);
    q[2 * j] = bf16_to_f32(b[j] & 0xffff);
    q[2 * j + 1] = bf16_to_f32(b[j] >> 16);
  }
  if (live) store_chunk<NT != kNtNone>(reinterpret_cast<u32x4n*>(y + static_cast<int64_t>(row) * dim) + c, u32x4n{b[0], b[1], b[2], b[3]});
  if (!y8) return;  // kernel-uniform
  float amax = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) amax = fmaxf(amax, __builtin_fabsf(q[j]));
  amax = row16_reduce<true>(amax);  // the group's 16 lanes
  const float sc = group_scale(amax, scale_mode);
  const uint2 code = quant8_e4m3(q, sc);
  if (live) {
    store_chunk<NT == kNtBoth>(reinterpret_cast<u32x2n*>(y8 + static_cast<int64_t>(row) * dim) + c, u32x2n{code.x, code.y});
    if ((c & 15) == 0) ys[static_cast<int64_t>(row) * (dim / kBlock) + (c >> 4)] = sc;
  }
}

// CH: chunks per virtual thread (1 up to dim 8192: no load or sum of chunks that are not there).
template <int CH>
__global__ __launch_bounds__(kNormThreads) void rmsnorm_quant_kernel(
    const uint16_t* __restrict__ x, const float* __restrict__ gamma, float eps, int dim,
    uint16_t* __restrict__ y, uint8_t* __restrict__ y8, float* __restrict__ ys, int scale_mode) {
  __shared__ float part[kNormVirt / 64];
  const int row = blockIdx.x, tid = threadIdx.x;
  const int nch = dim / 8;
  const int c = blockIdx.y * kNormSlice + tid;  // this thread's chunk
  const bool live = c < nch;
  const uint4* xr = reinterpret_cast<const uint4*>(x + static_cast<int64_t>(row) * dim);
  // every load up front (clamped, unconditional): the row for the sum, this chunk, gamma
  uint4 raw[kNormPerThread][CH];
#pragma unroll
  for (int u = 0; u < kNormPerThread; ++u)
#pragma unroll
    for (int i = 0; i < CH; ++i) raw[u][i] = xr[min(tid + u * kNormThreads + i * kNormVirt, nch - 1)];
  const int cc = min(c, nch - 1);
  const uint4 mine = xr[cc];
  const float4 g0 = reinterpret_cast<const float4*>(gamma)[2 * cc];
  const float4 g1 = reinterpret_cast<const float4*>(gamma)[2 * cc + 1];
#pragma unroll
  for (int u = 0; u < kNormPerThread; ++u) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < CH; ++i) ss = sum_squares(raw[u][i], tid + u * kNormThreads + i * kNormVirt < nch, ss);
    ss = wave_sum_f32(ss);
    if ((tid & 63) == 0) part[(tid >> 6) + u * (kNormThreads / 64)] = ss;
  }
  __syncthreads();
  const float r = norm_factor(part, dim, eps);
  const float gv[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
  norm_chunk<kNtNone>(mine, gv, r, live, c, row, dim, y, y8, ys, scale_mode);
}

// Many rows (norm_rows_min): HBM-bound.  One workgroup takes whole rows, kept in registers between the sum and the outputs (the slices above read
// and sum every row once per slice), strides over the rows with gamma held in registers -- as fp32
// it is twice a row's bytes -- and requests its next row before it works on this one.  The sum is
// the same tree: chunk tid + 256 j is virtual thread tid + 256 (j % 4)'s chunk j / 4.
// 4096 x 7168 (147 MB moved): 33 us (4.4 TB/s) against 49 us for the slices, which took 64 before the hardware
// conversions and the reciprocal quotient (quant8_e4m3).  Up to kNormRowsGrid rows a workgroup has one row and its
// request of a next one repeats the last row for nothing.
// Instances for 1, 2, 4, 5, 6 and 8 chunks a thread: registers go with the chunks (5: 158 VGPRs, three workgroups per CU;
// 10240 wide rows in the instance for 8 chunks, with one, 1024 / 4096 rows 23.5 / 76 us, in their own 11.7 / 39.3).
template <int NC, NormNt NT>  // chunks per thread: dim <= 2048 NC
__global__ __launch_bounds__(kNormThreads) void rmsnorm_quant_rows_kernel(
    const uint16_t* __restrict__ x, const float* __restrict__ gamma, float eps, int rows, int dim,
    uint16_t* __restrict__ y, uint8_t* __restrict__ y8, float* __restrict__ ys, int scale_mode) {
  __shared__ float part[2][kNormVirt / 64];
  const int tid = threadIdx.x, nch = dim / 8;
  float gv[NC][8];
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int c = min(tid + j * kNormThreads, nch - 1);
    const float4 g0 = reinterpret_cast<const float4*>(gamma)[2 * c], g1 = reinterpret_cast<const float4*>(gamma)[2 * c + 1];
    gv[j][0] = g0.x; gv[j][1] = g0.y; gv[j][2] = g0.z; gv[j][3] = g0.w;
    gv[j][4] = g1.x; gv[j][5] = g1.y; gv[j][6] = g1.z; gv[j][7] = g1.w;
  }
  uint4 cur[NC], nxt[NC];
  auto load = [&](int row, uint4 (&v)[NC]) {
    const uint4* xr = reinterpret_cast<const uint4*>(x + static_cast<int64_t>(row) * dim);
#pragma unroll
    for (int j = 0; j < NC; ++j) v[j] = xr[min(tid + j * kNormThreads, nch - 1)];
  };
  auto work = [&](int row, const uint4 (&v)[NC], float (&pt)[kNormVirt / 64]) {
#pragma unroll
    for (int u = 0; u < kNormPerThread; ++u) {
      float ss = 0.f;
#pragma unroll
      for (int j = u; j < NC; j += kNormPerThread)
        ss = sum_squares(v[j], tid + j * kNormThreads < nch, ss);
      ss = wave_sum_f32(ss);
      if ((tid & 63) == 0) pt[(tid >> 6) + u * (kNormThreads / 64)] = ss;
    }
    __syncthreads();
    const float r = norm_factor(pt, dim, eps);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int c = tid + j * kNormThreads;
      norm_chunk<NT>(v[j], gv[j], r, c < nch, c, row, dim, y, y8, ys, scale_mode);
    }
  };
  // two rows a step, so that no row is copied between register sets; the partials alternate too:
  // a row's are rewritten two rows later, after a barrier that follows every read of them
  const int step = static_cast<int>(gridDim.x);
  int row = blockIdx.x;
  load(row, cur);
  for (; row < rows; row += 2 * step) {
    load(min(row + step, rows - 1), nxt);
    work(row, cur, part[0]);
    if (row + step >= rows) break;
    load(min(row + 2 * step, rows - 1), cur);
    work(row + step, nxt, part[1]);
  }
}

}  // namespace tl

using namespace tl;

extern "C" int tl_rmsnorm_quant(const void* x_bf16, const float* gamma, float eps, int64_t rows, int64_t dim,
                                void* y_bf16, void* y_fp8, float* y_scale, int scale_mode, void* stream) {
  if (rows < 0 || dim <= 0 || dim % kBlock || dim > kNormMaxDim) {
    set_error("rmsnorm_quant: dim=%lld must be a positive multiple of 128, at most %d", (long long)dim,
              kNormMaxDim);
    return kErrArg;
  }
  if (scale_mode < 0 || scale_mode > 2) { set_error("rmsnorm_quant: bad scale_mode %d", scale_mode); return kErrArg; }
  if (!x_bf16 || !gamma || !y_bf16 || (!y_fp8) != (!y_scale)) {
    set_error("rmsnorm_quant: null pointer (y_fp8 and y_scale are given together or not at all)");
    return kErrArg;
  }
  if ((reinterpret_cast<uintptr_t>(x_bf16) | reinterpret_cast<uintptr_t>(gamma) | reinterpret_cast<uintptr_t>(y_bf16) |
       reinterpret_cast<uintptr_t>(y_fp8)) & 15) {
    set_error("rmsnorm_quant: pointers must be 16-byte aligned");
    return kErrArg;
  }
  if (rows == 0) return kOk;
  if (rows > 0x7fffffff) { set_error("rmsnorm_quant: too many rows (%lld)", (long long)rows); return kErrArg; }
  const unsigned slices = static_cast<unsigned>(cdiv(dim / 8, kNormSlice));
  if (rows < norm_rows_min(slices)) {
    const dim3 grid(static_cast<unsigned>(rows), slices);
    auto slice = [&](auto ch) {
      hipLaunchKernelGGL((rmsnorm_quant_kernel<decltype(ch)::value>), grid, dim3(kNormThreads), 0, (hipStream_t)stream,
                         (const uint16_t*)x_bf16, gamma, eps, (int)dim, (uint16_t*)y_bf16, (uint8_t*)y_fp8, y_scale, scale_mode);
    };
    if (dim <= kNormVirt * 8) slice(std::integral_constant<int, 1>{});
    else slice(std::integral_constant<int, 2>{});
    return check_launch("rmsnorm_quant");
  }
  const NormNt nt = norm_nt(rows, dim, y_fp8 != nullptr);
  auto launch = [&](auto nc) {
    constexpr int NC = decltype(nc)::value;
    const auto kern = nt == kNtNone ? rmsnorm_quant_rows_kernel<NC, kNtNone>
                                    : (nt == kNtY ? rmsnorm_quant_rows_kernel<NC, kNtY> : rmsnorm_quant_rows_kernel<NC, kNtBoth>);
    hipLaunchKernelGGL(kern,
                       dim3(static_cast<unsigned>(rows < kNormRowsGrid ? rows : kNormRowsGrid)), dim3(kNormThreads), 0,
                       (hipStream_t)stream, (const uint16_t*)x_bf16, gamma, eps, (int)rows, (int)dim, (uint16_t*)y_bf16,
                       (uint8_t*)y_fp8, y_scale, scale_mode);
  };
  if (slices <= 1) launch(std::integral_constant<int, 1>{});
  else if (slices <= 2) launch(std::integral_constant<int, 2>{});
  else if (slices <= 4) launch(std::integral_constant<int, 4>{});
  else if (slices <= 5) launch(std::integral_constant<int, 5>{});
  else if (slices <= 6) launch(std::integral_constant<int, 6>{});
  else launch(std::integral_constant<int, 8>{});
  return check_launch("rmsnorm_quant");
}

extern "C" int tl_act_quant(const void* x_bf16, void* y_fp8, float* s, int64_t rows, int64_t K,
                            int64_t group, int scale_mode, void* stream) {
  if (group != kBlock) { set_error("act_quant: only group size 128 is supported (got %lld)", (long long)group); return kErrUnsupported; }
  if (rows < 0 || K <= 0 || K % kBlock != 0) { set_error("act_quant: K=%lld must be a positive multiple of 128", (long long)K); return kErrArg; }
  if (scale_mode < 0 || scale_mode > 2) { set_error("act_quant: bad scale_mode %d", scale_mode); return kErrArg; }
  if (!x_bf16 || !y_fp8 || !s) { set_error("act_quant: null pointer"); return kErrArg; }
  if (rows == 0) return kOk;
  const int64_t n_groups = rows * (K / kBlock);
  const int64_t threads = n_groups * 16;
  hipLaunchKernelGGL(act_quant_kernel, dim3(cdiv(threads, 256)), dim3(256), 0, (hipStream_t)stream,
                     (const uint16_t*)x_bf16, (uint8_t*)y_fp8, s, n_groups, scale_mode);
  return check_launch("act_quant");
}

extern "C" int tl_weight_quant(const void* w, int w_is_bf16, void* q_fp8, float* s, int64_t N,
                               int64_t K, void* stream) {
  if (N <= 0 || K <= 0) { set_error("weight_quant: empty weight"); return kErrArg; }
  if (!w || !q_fp8 || !s) { set_error("weight_quant: null pointer"); return kErrArg; }
  const dim3 grid(cdiv(K, kBlock), cdiv(N, kBlock));
  const hipStream_t st = (hipStream_t)stream;
  // 16-byte loads and 8-byte stores need every row to start aligned
  const bool wide = K % 8 == 0 && !(reinterpret_cast<uintptr_t>(w) & 15) && !(reinterpret_cast<uintptr_t>(q_fp8) & 7);
  auto launch = [&](auto* wt) {
    using T = std::remove_pointer_t<decltype(wt)>;
    if (wide) hipLaunchKernelGGL((weight_quant_kernel<std::remove_const_t<T>>), grid, dim3(256), 0, st, wt, (uint8_t*)q_fp8, s, N, K);
    else hipLaunchKernelGGL((weight_quant_any_kernel<std::remove_const_t<T>>), grid, dim3(256), 0, st, wt, (uint8_t*)q_fp8, s, N, K);
  };
  if (w_is_bf16) launch((const uint16_t*)w);
  else launch((const float*)w);
  return check_launch("weight_quant");
}

extern "C" int tl_weight_dequant(const void* q_fp8, const float* s, void* out, int out_bf16,
                                 int64_t N, int64_t K, void* stream) {
  if (N <= 0 || K <= 0) { set_error("weight_dequant: empty weight"); return kErrArg; }
  if (!q_fp8 || !s || !out) { set_error("weight_dequant: null pointer"); return kErrArg; }
  const hipStream_t st = (hipStream_t)stream;
  const int64_t V = out_bf16 ? 8 : 4;
  const int64_t groups = cdiv(N, 4 * kDqRows);
  if (N * K >= kDqWide && K % V == 0 && !(reinterpret_cast<uintptr_t>(q_fp8) & (V - 1)) && !(reinterpret_cast<uintptr_t>(out) & 15) &&
      groups <= 65535) {  // (grid.y)
    const dim3 grid(cdiv(K, 64 * V), groups);
    const bool nt = N * K * (out_bf16 ? 2 : 4) > kDqNtBytes;
    const auto kern = out_bf16 ? (nt ? weight_dequant_kernel<true, true> : weight_dequant_kernel<true, false>)
                               : (nt ? weight_dequant_kernel<false, true> : weight_dequant_kernel<false, false>);
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, (const uint8_t*)q_fp8, s, out, N, K);
  } else {
    hipLaunchKernelGGL(weight_dequant_any_kernel, dim3(cdiv(N * K, 256)), dim3(256), 0, st, (const uint8_t*)q_fp8, s,
                       out, N, K, out_bf16);
  }
  return check_launch("weight_dequant");
}
