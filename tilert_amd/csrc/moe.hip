// MoE expert layer at one expert-parallel shard: grouped gate/up GEMM with fused SwiGLU,
// then the down GEMM with the routing-weighted combine.
//
// Numerics follow the reference MoE (BF16MMA: bf16 activations, fp8 weights dequantised
// per 128x128 block; expert_sel_up_gate_silu.py:670-692, expert_down_allreduce.py:455-468).
// Each fp8 weight is dequantised in registers exactly as the reference's golden weights
// are built (init_reference_weights, expert_sel_up_gate_silu.py:545-552:
// bf16(fp32(q) * block_scale), round-to-nearest-even) and multiplied on the bf16 MFMA
// v_mfma_f32_16x16x32_bf16 with fp32 accumulation over the whole K -- so the products
// are the reference's products and only the fp32 summation order differs.
// (v_cvt_scalef32_pk_bf16_fp8 cannot do this: it applies only the scale's exponent.)
//
// Routing is an input (token -> 8 global expert ids).  Every kernel derives the shard's
// hit-expert set on the device from topk_idx, so no host synchronisation is needed: a
// local expert hit by any token gets a "slot" (ascending expert order); only hit experts'
// weights are read.  With M <= 16 tokens the MFMA's 16 columns cover every token, so
// each hit expert is evaluated for all tokens (unrouted rows are ignored by the combine).
//
// Weight layout: the fragment-packed layout of tl_fp8_pack_weight applied to the stacked
// per-expert matrices: gate/up as w13 [E][2I rows (gate then up)][D], down as
// w2 [E][D rows][I]; scales [E][2I/128][D/128] and [E][D/128][I/128].
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "moe_common.h"
#include "../../include/tilert_amd.h"

namespace tl {

constexpr int kMoeWaves = 8;        // gate/up waves per workgroup (2 workgroups per CU)
constexpr int kDownWaves = 8;       // down waves per workgroup
constexpr int kDnSlots = 8;    // hit experts per batch of the LDS down kernel
constexpr int kDownRedBytes = sizeof(float) * kDownWaves * kDnSlots * 4 * 64;  // cross-wave partials
constexpr int kDownTermBytes = sizeof(float) * kDnSlots * 4 * 64;              // per-slot terms
constexpr int kDnHBytes = 128 * 1024;  // staged h limit of the LDS down kernel (one workgroup per CU)
constexpr int kMaxLocalExperts = 64;

// Hit-expert bitmask of this shard, computed by each wave on its own (no LDS, no
// barrier): lanes test the routed ids and the 64-bit masks are OR-reduced across the
// wave's lanes.
__device__ inline uint64_t routing_mask(const int32_t* __restrict__ topk_idx, int pairs, int e0, int n_local) {
  const int lane = threadIdx.x & 63;
  uint64_t m = 0;
  for (int i = lane; i < pairs; i += 64) {
    const int e = topk_idx[i] - e0;
    if (e >= 0 && e < n_local) m |= 1ull << e;
  }
  // wave-uniform result (read from one lane), so the hit count, expert ids and weight
  // addresses derived from it live in scalar registers
  return wave_or_u64(m);
}


// One routed (expert, weight) pair per lane, loaded at kernel start and read back with
// lane shuffles by routing_weight: no dependent loads after the weight stream.
// The loads are unconditional (lanes past `pairs` reread the last pair), so wait counts
// for loads issued after them stay exact.
__device__ inline int lane_pair_expert(const int32_t* __restrict__ topk_idx, int pairs, int e0) {
  const int lane = threadIdx.x & 63;
  const int v = topk_idx[min(lane, pairs - 1)];
  return lane < pairs ? v - e0 : -1;
}
__device__ inline float lane_pair_weight(const float* __restrict__ topk_w, int pairs) {
  const int lane = threadIdx.x & 63;
  const float v = topk_w[min(lane, pairs - 1)];
  return lane < pairs ? v : 0.f;
}

// Hit-expert bitmask from the lane-held pairs (pairs <= 64), wave-uniform.
__device__ inline uint64_t lane_pairs_mask(int my_e, int n_local) {
  return wave_or_u64((my_e >= 0 && my_e < n_local) ? (1ull << my_e) : 0ull);
}

// Routing weight of (token r, local expert e), from at most 64 lane-held pairs; 0 when the token does not use it.
__device__ inline float routing_weight(int my_e, float my_w, int topk, int r, bool tok, int e) {
  float wj = 0.f;
  for (int k = 0; k < topk; ++k) {
    const int src = (r * topk + k) & 63;
    const int ee = __shfl(my_e, src);
    const float v = __shfl(my_w, src);
    if (tok && ee == e) wj = v;
  }
  return wj;
}

constexpr int kGuDepth = 2;  // weight blocks in flight per wave (gate/up, LDS activations)
constexpr int kDnDepth = 2;  // down items in flight per wave (LDS activations)
constexpr int kLdsActBytes = 64 * 1024;  // activation staging limit (2 workgroups per CU)

// ------------------------------------------------------ gate/up, LDS activations
// Used when x [M, D] bf16 fits in 64 KB (M <= 4 at D = 7168).  The workgroup stages x in
// LDS once; the waves then stream only weight fragments, kGuDepth blocks ahead through
// ring_pipeline, and read their activation operands from LDS, so nothing but the weight
// stream is waited on.  Work item = (slot, 16-channel tile); a persistent grid strides over n_hit * I/16 items, and
// an item's partials are summed in wave order.
__global__ __launch_bounds__(kMoeWaves * 64, 4) void moe_gate_up_lds_kernel(
    const uint16_t* __restrict__ x, const uint8_t* __restrict__ w13, const float* __restrict__ s13,
    const int32_t* __restrict__ topk_idx, int M, int topk, int e0, int n_local, int D, int I,
    uint16_t* __restrict__ h) {
  extern __shared__ __align__(16) uint16_t xl[];  // [M][D]
  __shared__ v4f red[kMoeWaves - 1][2][64];
  // the routing and the x staging loads are in flight together (one round trip)
  const int pairs = M * topk;
  const int lane = threadIdx.x & 63;
  const int raw_e = topk_idx[min(lane, pairs - 1)];
  // x is copied straight into LDS (global_load_lds: no registers) once the hit set is
  // known, and the first weight fetches are requested right after it, before it has
  // landed; it is waited for just before the first compute.  (Issued before the routing
  // load is consumed, the copies would be waited for there: the compiler does not count
  // direct-to-LDS loads, so its wait for the routing load is a full vmcnt(0).)  Every
  // thread issues the same kStageChunks copies; sources past x repeat its last chunk and
  // their LDS destinations lie in the unused tail of the 64 KB allocation.
  const uint64_t mask = lane_pairs_mask(lane < pairs ? raw_e - e0 : -1, n_local);
  const int x16 = M * D / 8;
  copy_to_lds_fixed<kStageChunks>(x, x16, xl);
  const int n_hit = __builtin_popcountll(mask);
  const int KB = D >> 7;
  const int tiles = I >> 4;
  const int rows_e = 2 * I;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int r = lane & 15, g = lane >> 4;
  const uint16_t* xrow = xl + min(r, M - 1) * D;
  const int n = wave < KB ? (KB - wave + kMoeWaves - 1) / kMoeWaves : 0;  // K blocks wave + i*8
  bool staged = false;

  for (int item = blockIdx.x; item < n_hit * tiles; item += gridDim.x) {
    const int slot = item / tiles, rt = item - slot * tiles;
    const int e = nth_set_bit(mask, slot);
    const uint8_t* gate = w13 + (static_cast<size_t>(e) * (rows_e >> 4) + rt) * KB * 2048;
    const uint8_t* up = gate + static_cast<size_t>(tiles) * KB * 2048;
    const float* gs = s13 + (static_cast<size_t>(e) * (rows_e >> 7) + ((rt * 16) >> 7)) * KB;
    const float* us = s13 + (static_cast<size_t>(e) * (rows_e >> 7) + ((I + rt * 16) >> 7)) * KB;
    v4f ag = {0.f, 0.f, 0.f, 0.f}, au = {0.f, 0.f, 0.f, 0.f};
    struct Ops {
      v8i wg, wu;
      float gs, us;
    };
    Ops buf[kGuDepth];
    ring_pipeline(
        n, buf,
        [&](int i, Ops& o) {
          const int kb = wave + i * kMoeWaves;
          o.wg = load_fragment(gate + static_cast<size_t>(kb) * 2048, lane);
          o.wu = load_fragment(up + static_cast<size_t>(kb) * 2048, lane);
          o.gs = load_f32_vector(gs + kb);
          o.us = load_f32_vector(us + kb);
        },
        [&](int i, const Ops& o) {
          const int kb = wave + i * kMoeWaves;
          const uint16_t* xk = xrow + kb * kBlock;
          const int off[4] = {16 * g, 16 * g + 8, 64 + 16 * g, 64 + 16 * g + 8};
#pragma unroll
          for (int j = 0; j < 4; ++j) {  // one 32-wide K step at a time: few live registers
            const v8bf xa = *reinterpret_cast<const v8bf*>(xk + off[j]);
            ag = __builtin_amdgcn_mfma_f32_16x16x32_bf16(dequant8_bf16(o.wg[2 * j], o.wg[2 * j + 1], o.gs), xa, ag, 0, 0, 0);
            au = __builtin_amdgcn_mfma_f32_16x16x32_bf16(dequant8_bf16(o.wu[2 * j], o.wu[2 * j + 1], o.us), xa, au, 0, 0, 0);
          }
        },
        [&] {  // first item: x has landed (this wave's copies) and is visible (barrier)
          if (!staged) {
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            staged = true;
          }
        });
    if (wave > 0) {
      red[wave - 1][0][lane] = ag;
      red[wave - 1][1][lane] = au;
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int w = 0; w < kMoeWaves - 1; ++w) {
        ag += red[w][0][lane];
        au += red[w][1][lane];
      }
      if (r < M) {
        uint16_t o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = f32_to_bf16(silu(ag[j]) * au[j]);
        uint16_t* dst = h + (static_cast<size_t>(slot) * M + r) * I + rt * 16 + 4 * g;
        *reinterpret_cast<uint2*>(dst) = make_uint2(o[0] | (static_cast<uint32_t>(o[1]) << 16),
                                                    o[2] | (static_cast<uint32_t>(o[3]) << 16));
      }
    }
    __syncthreads();
  }
  if (!staged) __builtin_amdgcn_s_waitcnt(0);  // no item: the LDS copies land before the workgroup ends
}

// ------------------------------------------------------ gate/up, register activations
// Small layers whose x or routing the LDS kernel above does not hold (gate_up_from_registers): work items, reduction
// and output are the same, the activation operands come from L2.  <= 128 VGPRs (4 waves per SIMD): two workgroups
// per CU where the kernel of the larger batches below has one; with few items, or little K, that one's longer start
// and its rounds of 256 items cost more than the activation loads here.
__global__ __launch_bounds__(kMoeWaves * 64, 4) void moe_gate_up_kernel(
    const uint16_t* __restrict__ x, const uint8_t* __restrict__ w13, const float* __restrict__ s13,
    const int32_t* __restrict__ topk_idx, int M, int topk, int e0, int n_local, int D, int I,
    uint16_t* __restrict__ h) {
  __shared__ v4f red[kMoeWaves - 1][2][64];
  const uint64_t mask = routing_mask(topk_idx, M * topk, e0, n_local);
  const int n_hit = __builtin_popcountll(mask);
  const int KB = D >> 7;
  const int tiles = I >> 4;
  const int rows_e = 2 * I;  // gate rows then up rows
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const bool tok = r < M;
  const uint16_t* xrow = x + static_cast<size_t>(tok ? r : 0) * D;

  for (int item = blockIdx.x; item < n_hit * tiles; item += gridDim.x) {
    const int slot = item / tiles, rt = item - slot * tiles;
    const int e = nth_set_bit(mask, slot);
    const uint8_t* gate = w13 + (static_cast<size_t>(e) * (rows_e >> 4) + rt) * KB * 2048;
    const uint8_t* up = gate + static_cast<size_t>(tiles) * KB * 2048;
    const float* gs = s13 + (static_cast<size_t>(e) * (rows_e >> 7) + ((rt * 16) >> 7)) * KB;
    const float* us = s13 + (static_cast<size_t>(e) * (rows_e >> 7) + ((I + rt * 16) >> 7)) * KB;
    // Every operand of the next K block (both fragments, the activation block, both
    // scales) is requested one iteration ahead.  Vector loads retire in issue order, so a
    // current-iteration load issued after a prefetch would make the wait cover the
    // prefetch too; here the loop body only consumes registers loaded earlier.
    v4f ag = {0.f, 0.f, 0.f, 0.f}, au = {0.f, 0.f, 0.f, 0.f};
    int kb = wave;
    v8i wg_n = zero_v8i(), wu_n = zero_v8i();
    ActOperand xa_n = {};
    float gs_n = 0.f, us_n = 0.f;
    if (kb < KB) {
      wg_n = load_fragment(gate + static_cast<size_t>(kb) * 2048, lane);
      wu_n = load_fragment(up + static_cast<size_t>(kb) * 2048, lane);
      xa_n = load_act(xrow + kb * kBlock, g, tok);
      gs_n = gs[kb];
      us_n = us[kb];
    }
    for (; kb < KB; kb += kMoeWaves) {
      const v8i wg = wg_n, wu = wu_n;
      const ActOperand xa = xa_n;
      const float gsc = gs_n, usc = us_n;
      const int kn = kb + kMoeWaves;
      if (kn < KB) {
        wg_n = load_fragment(gate + static_cast<size_t>(kn) * 2048, lane);
        wu_n = load_fragment(up + static_cast<size_t>(kn) * 2048, lane);
        xa_n = load_act(xrow + kn * kBlock, g, tok);
        gs_n = gs[kn];
        us_n = us[kn];
      }
      ag = mfma_block_bf16(wg, gsc, xa, ag);
      au = mfma_block_bf16(wu, usc, xa, au);
    }
    if (wave > 0) {
      red[wave - 1][0][lane] = ag;
      red[wave - 1][1][lane] = au;
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int w = 0; w < kMoeWaves - 1; ++w) {
        ag += red[w][0][lane];
        au += red[w][1][lane];
      }
      if (tok) {
        uint16_t o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = f32_to_bf16(silu(ag[j]) * au[j]);
        uint16_t* dst = h + (static_cast<size_t>(slot) * M + r) * I + rt * 16 + 4 * g;
        *reinterpret_cast<uint2*>(dst) = make_uint2(o[0] | (static_cast<uint32_t>(o[1]) << 16),
                                                    o[2] | (static_cast<uint32_t>(o[3]) << 16));
      }
    }
    __syncthreads();
  }
}

// ------------------------------------------------------ down, LDS activations
// For few tokens (down_from_lds) whose one hit expert's h rows [M, I] fit in kDnHBytes.  A workgroup covers two 16-row
// output tiles (D % 128 == 0 makes their count even) with 8 waves each, so the staged h rows serve both.  Hit experts
// are taken `sb` at a time (sb * M * I * 2 <= 128 KB); the batch's h rows are staged in LDS and
// each tile's (slot, K block) items, dealt round-robin to its 8 waves, are streamed
// kDnDepth ahead through ring_pipeline, one fp32 accumulator per slot.  After the stream
// the same LDS holds the cross-wave partials: local wave j of a tile reduces slot j over
// the tile's waves in order and rounds its weighted term to bf16, as the golden rounds each
// term; local wave 0 adds the terms in slot order.
constexpr int kDnTiles = 2;  // output tiles per workgroup
__global__ __launch_bounds__(kDownWaves * 64 * kDnTiles, 4) void moe_down_lds_kernel(
    const uint16_t* __restrict__ h, const uint8_t* __restrict__ w2, const float* __restrict__ s2,
    const int32_t* __restrict__ topk_idx, const float* __restrict__ topk_w, int M, int topk, int e0,
    int n_local, int D, int I, int sb, uint16_t* __restrict__ y) {
  extern __shared__ __align__(16) uint8_t smem[];
  uint16_t* hl = reinterpret_cast<uint16_t*>(smem);  // [sb][M][I] during the stream
  v4f(*red)[kDnSlots][64] = reinterpret_cast<v4f(*)[kDnSlots][64]>(smem);  // after it
  v4f(*term)[kDnSlots][64] = reinterpret_cast<v4f(*)[kDnSlots][64]>(smem + kDnTiles * kDownRedBytes);
  const int pairs = M * topk;
  const int my_e = lane_pair_expert(topk_idx, pairs, e0);
  const float my_w = lane_pair_weight(topk_w, pairs);
  // The hit set first (the routing loads are waited for here), then the first batch's h
  // rows are copied straight into LDS (global_load_lds, no registers) and the first weight
  // fetches requested behind them; the copy is waited for just before the first compute.
  // (Issued before the routing loads are consumed, the copies would be waited for there:
  // the compiler does not count direct-to-LDS loads, so its wait for them is a vmcnt(0).)
  const uint64_t mask = lane_pairs_mask(my_e, n_local);
  const int n_hit = __builtin_popcountll(mask);
  {
    const int ln = threadIdx.x & 63;
    const int c_end = min(n_hit, sb) * M * I / 8;
    for (int c0 = threadIdx.x - ln; c0 < c_end; c0 += blockDim.x)  // c0: this wave's first chunk
      if (c0 + ln < c_end)
        __builtin_amdgcn_global_load_lds(reinterpret_cast<const u32x4*>(h) + c0 + ln,
                                         (lds_ptr)(smem + static_cast<size_t>(c0) * 16), 16, 0, 0);
  }
  const int KB = I >> 7;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int tt = wave / kDownWaves, wl = wave % kDownWaves;           // tile in group, local wave
  const int r = lane & 15, g = lane >> 4;
  const bool tok = r < M;
  const int row = min(r, M - 1);
  const int rt = blockIdx.x * kDnTiles + tt;
  v4f yacc = {0.f, 0.f, 0.f, 0.f};

  for (int s0 = 0; s0 < n_hit; s0 += sb) {
    const int ns = min(sb, n_hit - s0);
    const int h16 = ns * M * I / 8;
    v4f acc[kDnSlots];
#pragma unroll
    for (int j = 0; j < kDnSlots; ++j) acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
    const int items = ns * KB;  // item = (slot it / KB, K block it % KB)
    const int n = wl < items ? (items - wl + kDownWaves - 1) / kDownWaves : 0;
    struct Ops {
      v8i w;
      float sc;
    };
    Ops buf[kDnDepth];
    float wj = 0.f;  // routing weight of (token r, slot s0 + wl): local wave j reduces slot j
    ring_pipeline(
        n, buf,
        [&](int i, Ops& o) {
          const int it = wl + i * kDownWaves;
          const int j = it / KB, kb = it - j * KB;
          const int e = nth_set_bit(mask, s0 + j);  // scalar bit arithmetic (no indexed array)
          const uint8_t* f = w2 + (static_cast<size_t>(e) * (D >> 4) + rt) * KB * 2048;
          const float* sp = s2 + (static_cast<size_t>(e) * (D >> 7) + ((rt * 16) >> 7)) * KB;
          o.w = load_fragment(f + static_cast<size_t>(kb) * 2048, lane);
          o.sc = load_f32_vector(sp + kb);
        },
        [&](int i, const Ops& o) {
          const int it = wl + i * kDownWaves;
          const int j = it / KB, kb = it - j * KB;
          const ActOperand xa = lds_act(hl + (j * M + row) * I + kb * kBlock, g);
#pragma unroll
          for (int jj = 0; jj < kDnSlots; ++jj)
            if (jj == j) acc[jj] = mfma_block_bf16(o.w, o.sc, xa, acc[jj]);
        },
        [&] {  // the batch's h rows into LDS while the first weight fetches are in flight
          if (s0 > 0) stage_commit(hl, stage_issue(h + static_cast<size_t>(s0) * M * I, h16), h16);
          if (wl < ns)
            wj = routing_weight(my_e, my_w, topk, r, tok, nth_set_bit(mask, s0 + wl));
          if (s0 == 0) __builtin_amdgcn_s_waitcnt(0);  // this wave's part of the direct copy has landed
          __syncthreads();
        });
    __syncthreads();  // every wave is done with hl before it becomes the partials
#pragma unroll
    for (int j = 0; j < kDnSlots; ++j)
      if (j < ns) red[wave][j][lane] = acc[j];  // (slots past the batch hold nothing)
    __syncthreads();
    if (wl < ns) {
      v4f t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < kDownWaves; ++w) t += red[tt * kDownWaves + w][wl][lane];
      v4f tw;
#pragma unroll
      for (int q = 0; q < 4; ++q) tw[q] = bf16_to_f32(f32_to_bf16(t[q] * wj));
      term[tt][wl][lane] = tw;
    }
    __syncthreads();
    if (wl == 0) {
      for (int j = 0; j < ns; ++j) yacc += term[tt][j][lane];
    }
    __syncthreads();
  }
  if (wl == 0 && tok) {
    uint16_t* dst = y + static_cast<size_t>(r) * D + rt * 16 + 4 * g;
    *reinterpret_cast<uint2*>(dst) =
        make_uint2(f32_to_bf16(yacc[0]) | (static_cast<uint32_t>(f32_to_bf16(yacc[1])) << 16),
                   f32_to_bf16(yacc[2]) | (static_cast<uint32_t>(f32_to_bf16(yacc[3])) << 16));
  }
}

// ------------------------------------------------------ larger batches
// x [M, D] no longer fits beside the weight stream (64 KB at M = 5, D = 7168), and reading the
// activation operands from L2 into registers costs more than the weights: 16 rows of 32-byte
// pieces per load, a quarter of the contiguous rate.  Here every wave streams its own K
// blocks through a private ring of two LDS stages (kBigStage: the block of two weight tiles, 4 KB,
// and of 4 MQ tokens, MQ KB), all by load-to-LDS copies of 1 KB: a weight fragment half
// is consecutive memory, an activation copy is 4 rows of 256 bytes.  A stage is read into
// registers at once and refilled before its block is multiplied, so nearly both stages
// of all 8 waves (one workgroup per CU) stay in flight, and no wave waits for another until the
// sums of a tile are combined.  Activation chunk c of row r lands at chunk c ^ r (16 chunks
// of 16 bytes): the operand reads of 16 rows hit 16 different chunks.  Block scales are
// scalar loads one block ahead.
// D = 7168, I = 2048, M = 16, 11.4 hit experts: gate/up 66.6 us (5.0 TB/s of weights), down 35.8
// (4.7 TB/s), where the kernels with register activations and four slots a batch took
// 75.3 and 82.3.
constexpr int kBigWaves = 8;
constexpr int kBigStage(int MQ) { return 4096 + MQ * 1024; }
constexpr int kBigRing(int MQ) { return kBigWaves * 2 * kBigStage(MQ); }
constexpr int kBigRedGu = 2 * kBigWaves * 2 * 1024;             // gate/up partials, two items
constexpr int kBigRedDn = 2 * (kBigWaves * 2 - 2) * 1024;       // down partials, two slot pairs
constexpr int kBigWeights = kMaxLocalExperts * 16 * 4;          // routing weights [slot][token]

// Block scales through the constant address space: the copies' memory clobbers would otherwise make
// these uniform loads vector loads, counted with the copies.
typedef const __attribute__((address_space(4))) float* scales_ptr;
__device__ inline scales_ptr as_scales(const float* p) { return (scales_ptr)p; }

// One K block of a wave: two weight fragments, the activation operand.
struct BigOps {
  v8i w0, w1;
  v8bf x[4];
};

template <int MQ>
struct BigRing {
  const uint8_t* base;  // this wave's stages
  uint32_t lds;         // their LDS address
  int lane, r, g;

  __device__ inline BigRing(const uint8_t* smem, int wave, int lane_) : lane(lane_), r(lane_ & 15), g(lane_ >> 4) {
    base = smem + wave * 2 * kBigStage(MQ);
    lds = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_u8_ptr)base)));
  }
  // this lane's source in a 16-token activation block [16, ...] of row pitch `pitch` bytes (rows past M: row M - 1)
  __device__ inline void rows(const uint8_t* x, size_t pitch, int M, const uint8_t* (&src)[MQ]) const {
#pragma unroll
    for (int i = 0; i < MQ; ++i) {
      const int row = 4 * i + (lane >> 4);
      src[i] = x + static_cast<size_t>(min(row, M - 1)) * pitch + (((lane & 15) ^ row) << 4);
    }
  }
  // copies of one block into stage b: 4 + MQ (the weights, read once, leave the L2 to the activations)
  __device__ inline void issue(const uint8_t* f0, const uint8_t* f1, const uint8_t* (&src)[MQ], size_t xoff, int b) const {
    const uint32_t st = lds + b * kBigStage(MQ);
    dma_lds16<true>(f0 + lane * 16, st);
    dma_lds16<true>(f0 + 1024 + lane * 16, st + 1024);
    dma_lds16<true>(f1 + lane * 16, st + 2048);
    dma_lds16<true>(f1 + 1024 + lane * 16, st + 3072);
#pragma unroll
    for (int i = 0; i < MQ; ++i) dma_lds16(src[i] + xoff, st + 4096 + i * 1024);
  }
  // stage b has landed (at most the other stage's copies are in flight, none past the last block)
  __device__ inline void wait(bool more) const {
    if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 + MQ) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  __device__ inline void read(int b, BigOps& o) const {
    const uint8_t* st = base + b * kBigStage(MQ);
    const u32x4* w = reinterpret_cast<const u32x4*>(st);
    const u32x4 a = w[lane], c = w[64 + lane], d = w[128 + lane], e = w[192 + lane];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o.w0[i] = a[i]; o.w0[4 + i] = c[i];
      o.w1[i] = d[i]; o.w1[4 + i] = e[i];
    }
    // chunks 2g, 2g + 1, 8 + 2g, 9 + 2g of row r (rows past the copied ones: the last, their columns are not stored)
    const int row = min(r, 4 * MQ - 1);
    const uint8_t* xr = st + 4096 + row * 256;
    const int ch[4] = {2 * g, 2 * g + 1, 8 + 2 * g, 9 + 2 * g};
#pragma unroll
    for (int j = 0; j < 4; ++j) o.x[j] = *reinterpret_cast<const v8bf*>(xr + ((ch[j] ^ row) << 4));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the stage may be refilled
  }
  __device__ static inline void mma(const BigOps& o, float s0, float s1, v4f& a0, v4f& a1) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(dequant8_bf16(o.w0[2 * j], o.w0[2 * j + 1], s0), o.x[j], a0, 0, 0, 0);
      a1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(dequant8_bf16(o.w1[2 * j], o.w1[2 * j + 1], s1), o.x[j], a1, 0, 0, 0);
    }
  }
};

// This wave's LDS writes are visible after the barrier (its copies in flight stay in flight).
__device__ inline void big_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Gate/up: work item = (slot, 16-channel tile), a gate and an up tile; a persistent grid of one
// workgroup per CU strides over the items, and each wave's stream of K blocks (wave + 8 i) runs on
// across them.  An item's partials go to one of two LDS buffers; after the barrier one
// wave, another for each item, adds them in wave order.
template <int MQ>
__global__ __launch_bounds__(kBigWaves * 64, 2) void moe_gate_up_big_kernel(
    const uint16_t* __restrict__ x, const uint8_t* __restrict__ w13, const float* __restrict__ s13,
    const int32_t* __restrict__ topk_idx, int M, int topk, int e0, int n_local, int D, int I,
    uint16_t* __restrict__ h) {
  extern __shared__ __align__(16) uint8_t smem[];
  v4f(*red)[kBigWaves][2][64] = reinterpret_cast<v4f(*)[kBigWaves][2][64]>(smem + kBigRing(MQ));
  const uint64_t mask = routing_mask(topk_idx, M * topk, e0, n_local);
  const int n_hit = __builtin_popcountll(mask);
  const int KB = D >> 7, tiles = I >> 4, items = n_hit * tiles;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const BigRing<MQ> ring(smem, wave, lane);
  const uint8_t* xs[MQ];
  ring.rows(reinterpret_cast<const uint8_t*>(x), static_cast<size_t>(D) * 2, M, xs);
  const int n = wave < KB ? (KB - wave + kBigWaves - 1) / kBigWaves : 0;  // this wave's K blocks of an item
  const int mine = static_cast<int>(blockIdx.x) < items ? (items - blockIdx.x + gridDim.x - 1) / gridDim.x : 0;
  const int total = n * mine;

  struct Cursor {  // the stream's position: its item's tiles and this wave's block of it
    const uint8_t *gate, *up;
    scales_ptr gs, us;
    int item, j;
  };
  auto at_item = [&](int item, Cursor& c) {
    const int slot = item / tiles, rt = item - slot * tiles;
    const int e = nth_set_bit(mask, slot);
    c.gate = w13 + (static_cast<size_t>(e) * (2 * tiles) + rt) * KB * 2048;
    c.up = c.gate + static_cast<size_t>(tiles) * KB * 2048;
    c.gs = as_scales(s13) + (static_cast<size_t>(e) * ((2 * I) >> 7) + ((rt * 16) >> 7)) * KB;
    c.us = as_scales(s13) + (static_cast<size_t>(e) * ((2 * I) >> 7) + ((I + rt * 16) >> 7)) * KB;
    c.item = item;
    c.j = 0;
  };
  auto next = [&](Cursor& c) {
    if (++c.j == n) at_item(min(c.item + static_cast<int>(gridDim.x), items - 1), c);
  };
  Cursor cur{};
  float gs_q[2] = {0.f, 0.f}, us_q[2] = {0.f, 0.f};  // scales of the two stages
  auto issue = [&](int b) {
    const int kb = wave + cur.j * kBigWaves;
    ring.issue(cur.gate + static_cast<size_t>(kb) * 2048, cur.up + static_cast<size_t>(kb) * 2048, xs,
               static_cast<size_t>(kb) * 256, b);
    gs_q[b] = cur.gs[kb];
    us_q[b] = cur.us[kb];
    next(cur);
  };
  if (total > 0) {
    at_item(blockIdx.x, cur);
    issue(0);
    if (total > 1) issue(1);
  }
  int i = 0;
  auto block = [&](int b, v4f& ag, v4f& au) {  // b: i % 2
    BigOps o;
    ring.wait(i + 1 < total);
    ring.read(b, o);
    const float gs = gs_q[b], us = us_q[b];
    if (i + 2 < total) issue(b);
    BigRing<MQ>::mma(o, gs, us, ag, au);
    ++i;
  };
  for (int k = 0; k < mine; ++k) {
    v4f ag = {0.f, 0.f, 0.f, 0.f}, au = {0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < n; ++j) {
      if (i & 1) block(1, ag, au);
      else block(0, ag, au);
    }
    const int rb = k & 1;
    red[rb][wave][0][lane] = ag;
    red[rb][wave][1][lane] = au;
    big_barrier();
    if (wave == (k & (kBigWaves - 1))) {
      ag = red[rb][0][0][lane];
      au = red[rb][0][1][lane];
#pragma unroll
      for (int w = 1; w < kBigWaves; ++w) {
        ag += red[rb][w][0][lane];
        au += red[rb][w][1][lane];
      }
      const int item = blockIdx.x + k * gridDim.x;
      const int slot = item / tiles, rt = item - slot * tiles;
      if (ring.r < M) {
        uint16_t o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = f32_to_bf16(silu(ag[j]) * au[j]);
        uint16_t* dst = h + (static_cast<size_t>(slot) * M + ring.r) * I + rt * 16 + 4 * ring.g;
        *reinterpret_cast<uint2*>(dst) = make_uint2(o[0] | (static_cast<uint32_t>(o[1]) << 16),
                                                    o[2] | (static_cast<uint32_t>(o[3]) << 16));
      }
    }
  }
}

// Down + combine: one workgroup per two 16-row output tiles, over all hit experts two slots at a time:
// waves 0-3 take the even slot of a pair, waves 4-7 the odd one, K blocks (wave % 4) + 4 i.  A
// pair's partials go to one of two LDS buffers; after the barrier waves 0 and 1 (one tile
// each) add a slot's four in wave order, apply the routing weight, round the term to bf16 and add it to
// the output in slot order, while the streams run on.
template <int MQ>
__global__ __launch_bounds__(kBigWaves * 64, 2) void moe_down_big_kernel(
    const uint16_t* __restrict__ h, const uint8_t* __restrict__ w2, const float* __restrict__ s2,
    const int32_t* __restrict__ topk_idx, const float* __restrict__ topk_w, int M, int topk, int e0,
    int n_local, int D, int I, uint16_t* __restrict__ y) {
  extern __shared__ __align__(16) uint8_t smem[];
  constexpr int kParts = kBigWaves * 2 - 2;  // (wave, tile) partials but waves 0's and 1's own
  v4f(*red)[kParts][64] = reinterpret_cast<v4f(*)[kParts][64]>(smem + kBigRing(MQ));
  float(*wgt)[16] = reinterpret_cast<float(*)[16]>(smem + kBigRing(MQ) + kBigRedDn);
  const uint64_t mask = routing_mask(topk_idx, M * topk, e0, n_local);
  const int n_hit = __builtin_popcountll(mask);
  const int KB = I >> 7;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = wave >> 2, wk = wave & 3;
  const int rt = blockIdx.x * 2;
  const BigRing<MQ> ring(smem, wave, lane);
  const uint8_t* hs[MQ];
  ring.rows(reinterpret_cast<const uint8_t*>(h), static_cast<size_t>(I) * 2, M, hs);
  const int n = wk < KB ? (KB - wk + 3) / 4 : 0;  // this wave's K blocks of a slot
  const int slots = (n_hit - half + 1) / 2;       // its slots: half, half + 2, ...
  const int total = n * slots;
  const size_t tile_bytes = static_cast<size_t>(KB) * 2048;
  const size_t slot_bytes = static_cast<size_t>(M) * I * 2;

  const uint8_t* f = nullptr;  // the stream's position: its slot's first tile and scales, this wave's block
  scales_ptr sc = nullptr;
  int cs = half, cj = 0;
  auto at_slot = [&](int slot) {
    const int e = nth_set_bit(mask, slot);
    f = w2 + (static_cast<size_t>(e) * (D >> 4) + rt) * tile_bytes;
    sc = as_scales(s2) + (static_cast<size_t>(e) * (D >> 7) + ((rt * 16) >> 7)) * KB;  // both tiles lie in one 128-row block
  };
  float sc_q[2] = {0.f, 0.f};
  auto issue = [&](int b) {
    const int kb = wk + cj * 4;
    const uint8_t* f0 = f + static_cast<size_t>(kb) * 2048;
    ring.issue(f0, f0 + tile_bytes, hs, cs * slot_bytes + static_cast<size_t>(kb) * 256, b);
    sc_q[b] = sc[kb];
    if (++cj == n) {
      cj = 0;
      cs += 2;
      if (cs < n_hit) at_slot(cs);
    }
  };
  if (total > 0) {
    at_slot(half);
    issue(0);
    if (total > 1) issue(1);
  }
  // routing weights [slot][token], 0 where the token does not use the expert (visible to waves 0 and 1 after
  // the first pair's barrier)
  for (int t = threadIdx.x; t < n_hit * 16; t += kBigWaves * 64) {
    const int tok = t & 15, e = e0 + nth_set_bit(mask, t >> 4);
    float w = 0.f;
    if (tok < M)
      for (int k = 0; k < topk; ++k)
        if (topk_idx[tok * topk + k] == e) w = topk_w[tok * topk + k];
    wgt[t >> 4][tok] = w;
  }
  v4f yacc = {0.f, 0.f, 0.f, 0.f};
  int i = 0;
  auto block = [&](int b, v4f& a0, v4f& a1) {
    BigOps o;
    ring.wait(i + 1 < total);
    ring.read(b, o);
    const float s = sc_q[b];
    if (i + 2 < total) issue(b);
    BigRing<MQ>::mma(o, s, s, a0, a1);
    ++i;
  };
  for (int p = 0; 2 * p < n_hit; ++p) {
    v4f a0 = {0.f, 0.f, 0.f, 0.f}, a1 = {0.f, 0.f, 0.f, 0.f};
    if (2 * p + half < n_hit)
      for (int j = 0; j < n; ++j) {
        if (i & 1) block(1, a0, a1);
        else block(0, a0, a1);
      }
    const int rb = p & 1;
    // partial (w, t) at 2 w + t - 1 before (1, 1), - 2 after it
    if (wave != 0) red[rb][2 * wave - (wave > 1 ? 2 : 1)][lane] = a0;
    if (wave != 1) red[rb][2 * wave + 1 - (wave > 1 ? 2 : 1)][lane] = a1;
    big_barrier();
    if (wave < 2) {
      v4f t = wave == 0 ? a0 : red[rb][0][lane];  // waves 0 and 1 of this tile: (0, 1) is partial 0, (1, 0) partial 1
      t += wave == 0 ? red[rb][1][lane] : a1;
      t += red[rb][2 + wave][lane];
      t += red[rb][4 + wave][lane];
      const float wa = wgt[2 * p][ring.r];
#pragma unroll
      for (int q = 0; q < 4; ++q) yacc[q] += bf16_to_f32(f32_to_bf16(t[q] * wa));
      if (2 * p + 1 < n_hit) {
        t = red[rb][6 + wave][lane];
#pragma unroll
        for (int w = 1; w < 4; ++w) t += red[rb][6 + 2 * w + wave][lane];
        const float wb = wgt[2 * p + 1][ring.r];
#pragma unroll
        for (int q = 0; q < 4; ++q) yacc[q] += bf16_to_f32(f32_to_bf16(t[q] * wb));
      }
    }
  }
  if (wave < 2 && ring.r < M) {
    uint16_t* dst = y + static_cast<size_t>(ring.r) * D + (rt + wave) * 16 + 4 * ring.g;
    *reinterpret_cast<uint2*>(dst) =
        make_uint2(f32_to_bf16(yacc[0]) | (static_cast<uint32_t>(f32_to_bf16(yacc[1])) << 16),
                   f32_to_bf16(yacc[2]) | (static_cast<uint32_t>(f32_to_bf16(yacc[3])) << 16));
  }
}

// MQ = groups of 4 token rows
template <class F>
static int by_token_rows(int64_t M, F&& f) {
  switch (cdiv(M, 4)) {
    case 1: return f(std::integral_constant<int, 1>{});
    case 2: return f(std::integral_constant<int, 2>{});
    case 3: return f(std::integral_constant<int, 3>{});
    default: return f(std::integral_constant<int, 4>{});
  }
}

// Gate/up of x or routing that the LDS kernel does not hold: the register kernel up to these sizes, else the kernel of
// the larger batches.  n_local I M stands for the number of work items (us, register / larger batches, 8 experts of 256
// a token; 32 local: D = 512, I = 512, M = 16 5.4 / 6.2; D = 1024, I = 2048, M = 16 14.8 / 16.2; D = 2048, I = 1024, M = 10
// 11.5 / 12.7, M = 14 14.7 / 15.1, M = 16 15.5 / 15.0; D = 2048, I = 2048, M = 10 18.9 / 21.0, M = 14 23.9 / 23.7; D = 4096,
// I = 512, M = 9 10.1 / 10.7, M = 14 level; D = 7168, I = 512, M = 8 12.1 / 12.4, M = 12 19.0 / 18.3; D = 7168, I = 1024, M = 6
// 20.7 / 20.3; 16 local: D = 4096, I = 512, M = 11 8.7 / 9.2; D = 6144, I = 768, M = 9 10.5 / 11.1; D = 7168, I = 1024, M = 10
// 0.98).
static bool gate_up_from_registers(int64_t M, int64_t n_local, int64_t D, int64_t I) {
  const int64_t items = n_local * I * M;
  return D <= 1024 || (D <= 2048 && (M < 14 || items <= 1 << 19)) || items <= 5 << 15;
}

// Down of 6 to 8 tokens: the LDS kernel takes h rows of up to 8 K blocks that fill the larger batches' two rounds of 4
// waves a slot badly, as at up to 5 tokens.
static bool down_from_lds(int64_t M, int64_t I) {
  const int64_t KB = I / kBlock;
  return M <= 5 || (M <= 8 && KB < 8 && (KB % 4 == 1 || KB % 4 == 2));
}

static int check_moe(const char* who, int64_t M, int64_t topk, int64_t n_local, int64_t D, int64_t I) {
  if (M < 1 || M > 16) { set_error("%s: M=%lld must be in [1, 16]", who, (long long)M); return kErrUnsupported; }
  if (topk < 1 || topk > 64) { set_error("%s: topk=%lld must be in [1, 64]", who, (long long)topk); return kErrArg; }
  if (n_local < 1 || n_local > kMaxLocalExperts) { set_error("%s: n_local=%lld must be in [1, %d]", who, (long long)n_local, kMaxLocalExperts); return kErrUnsupported; }
  if (D <= 0 || I <= 0 || D % kBlock || I % kBlock) { set_error("%s: D=%lld and I=%lld must be positive multiples of 128", who, (long long)D, (long long)I); return kErrArg; }
  if (D > (1 << 20) || I > (1 << 20)) { set_error("%s: D or I too large", who); return kErrArg; }
  return kOk;
}

}  // namespace tl

using namespace tl;

extern "C" int tl_moe_gate_up_swiglu(const void* x_bf16, const void* w13_packed, const float* s13,
                                     const int32_t* topk_idx, int64_t M, int64_t topk,
                                     int64_t expert_begin, int64_t n_local, int64_t D, int64_t I,
                                     void* h_bf16, void* stream) {
  int rc = check_moe("moe_gate_up_swiglu", M, topk, n_local, D, I);
  if (rc) return rc;
  if (!x_bf16 || !w13_packed || !s13 || !topk_idx || !h_bf16) { set_error("moe_gate_up_swiglu: null pointer"); return kErrArg; }
  if ((reinterpret_cast<uintptr_t>(x_bf16) | reinterpret_cast<uintptr_t>(w13_packed)) & 15) { set_error("moe_gate_up_swiglu: x and weights must be 16-byte aligned"); return kErrArg; }
  // enough workgroups for the largest possible hit set, capped at 4 per CU
  const int64_t max_items = n_local * (I / 16);
  const int grid = static_cast<int>(max_items < 512 ? max_items : 512);  // 2 x 8 waves per CU
  const int64_t x_bytes = M * D * 2;
  // x staged in LDS, routing in lanes, where both fit: 2-7 % ahead of the stream with x in it at
  // D = 4096, M = 5..8 and D = 6144, 7168, M <= 5
  if (x_bytes <= kLdsActBytes && M * topk <= 64) {
    rc = allow_dynamic_lds(reinterpret_cast<const void*>(moe_gate_up_lds_kernel), kLdsActBytes, "moe_gate_up_swiglu");
    if (rc) return rc;
    hipLaunchKernelGGL(moe_gate_up_lds_kernel, dim3(grid), dim3(kMoeWaves * 64), static_cast<size_t>(kLdsActBytes),
                       (hipStream_t)stream, (const uint16_t*)x_bf16, (const uint8_t*)w13_packed, s13, topk_idx,
                       (int)M, (int)topk, (int)expert_begin, (int)n_local, (int)D, (int)I, (uint16_t*)h_bf16);
  } else if (gate_up_from_registers(M, n_local, D, I)) {
    hipLaunchKernelGGL(moe_gate_up_kernel, dim3(grid), dim3(kMoeWaves * 64), 0, (hipStream_t)stream,
                       (const uint16_t*)x_bf16, (const uint8_t*)w13_packed, s13, topk_idx, (int)M, (int)topk,
                       (int)expert_begin, (int)n_local, (int)D, (int)I, (uint16_t*)h_bf16);
  } else {
    auto launch = [&](auto mq_tag) -> int {
      constexpr int MQ = decltype(mq_tag)::value, lds = kBigRing(MQ) + kBigRedGu;
      if (const int rc2 = allow_dynamic_lds(reinterpret_cast<const void*>(moe_gate_up_big_kernel<MQ>), lds, "moe_gate_up_swiglu")) return rc2;
      hipLaunchKernelGGL((moe_gate_up_big_kernel<MQ>), dim3(std::min<int64_t>(max_items, 256)), dim3(kBigWaves * 64), lds,
                         (hipStream_t)stream, (const uint16_t*)x_bf16, (const uint8_t*)w13_packed, s13, topk_idx,
                         (int)M, (int)topk, (int)expert_begin, (int)n_local, (int)D, (int)I, (uint16_t*)h_bf16);
      return 0;
    };
    rc = by_token_rows(M, launch);
    if (rc) return rc;
  }
  return check_launch("moe_gate_up_swiglu");
}

extern "C" int tl_moe_down_combine(const void* h_bf16, const void* w2_packed, const float* s2,
                                   const int32_t* topk_idx, const float* topk_w, int64_t M,
                                   int64_t topk, int64_t expert_begin, int64_t n_local, int64_t D,
                                   int64_t I, void* y_bf16, void* stream) {
  int rc = check_moe("moe_down_combine", M, topk, n_local, D, I);
  if (rc) return rc;
  if (!h_bf16 || !w2_packed || !s2 || !topk_idx || !topk_w || !y_bf16) { set_error("moe_down_combine: null pointer"); return kErrArg; }
  if ((reinterpret_cast<uintptr_t>(h_bf16) | reinterpret_cast<uintptr_t>(w2_packed)) & 15) { set_error("moe_down_combine: h and weights must be 16-byte aligned"); return kErrArg; }
  const int64_t h_bytes = M * I * 2;  // one hit expert's h rows
  // Up to 5 tokens: h staged in LDS, sb hit experts per batch, two tiles' 16 waves on it; above, the
  // batches' staging and reductions cost more than streaming h beside the weights (D = 7168, I =
  // 2048, M = 4 / 5 / 6 / 8: 15.1 / 14.6 / 19.9 / 28.9 against 15.1 / 14.8 / 17.7 / 23.8 us;
  // D = 6144, I = 1408: 10.9 / 11.1 / 14.6 / 21.3 against 11.7 / 11.7 / 13.9 / 18.6).  Where h has 1, 2, 5 or 6 K blocks,
  // which the stream deals to 4 waves a slot, staging pays up to 8 tokens (D = 7168, M = 7 / 8: I = 128 7.2 / 7.9 against
  // 7.9 / 8.7, I = 640 10.8 / 12.2 against 11.4 / 12.8; I = 512 10.1 / 11.3 against 9.4 / 10.3).
  if (down_from_lds(M, I) && h_bytes <= kDnHBytes && M * topk <= 64) {
    // (the later batches are staged through registers: kStageChunks x 16 B per thread, 128 KB)
    const int sb = static_cast<int>(std::min<int64_t>(kDnSlots, kDnHBytes / h_bytes));
    const size_t lds = std::max<size_t>(static_cast<size_t>(sb) * h_bytes, kDnTiles * (kDownRedBytes + kDownTermBytes));
    rc = allow_dynamic_lds(reinterpret_cast<const void*>(moe_down_lds_kernel), static_cast<int>(lds), "moe_down_combine");
    if (rc) return rc;
    hipLaunchKernelGGL(moe_down_lds_kernel, dim3(D / 16 / kDnTiles), dim3(kDownWaves * 64 * kDnTiles), lds,
                       (hipStream_t)stream, (const uint16_t*)h_bf16, (const uint8_t*)w2_packed, s2, topk_idx, topk_w,
                       (int)M, (int)topk, (int)expert_begin, (int)n_local, (int)D, (int)I, sb, (uint16_t*)y_bf16);
  } else {
    auto launch = [&](auto mq_tag) -> int {
      constexpr int MQ = decltype(mq_tag)::value, lds = kBigRing(MQ) + kBigRedDn + kBigWeights;
      if (const int rc2 = allow_dynamic_lds(reinterpret_cast<const void*>(moe_down_big_kernel<MQ>), lds, "moe_down_combine")) return rc2;
      hipLaunchKernelGGL((moe_down_big_kernel<MQ>), dim3(D / 32), dim3(kBigWaves * 64), lds, (hipStream_t)stream,
                         (const uint16_t*)h_bf16, (const uint8_t*)w2_packed, s2, topk_idx, topk_w, (int)M, (int)topk,
                         (int)expert_begin, (int)n_local, (int)D, (int)I, (uint16_t*)y_bf16);
      return 0;
    };
    rc = by_token_rows(M, launch);
    if (rc) return rc;
  }
  return check_launch("moe_down_combine");
}
