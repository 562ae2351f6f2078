// Projections of few rows: out[M][N] = x[M][K] W[N][K]^T for the M <= 64 tokens of a decode step,
// with the steps either side of each projection done in the same launch.
//
// At these sizes a projection is one pass over its weights (2 flop per weight byte and row), so
// the kernel is built to keep as much of W in flight as the chip can hold:
//   * A tile is 16 rows of W.  A work-group's 8 waves split K, at most 8 steps of 32 each (longer K
//     is split over work-groups), so a wave issues all its loads of a tile at once, and the next
//     tile's as each arrives.  x stays in registers for all the tiles of a work-group.
//   * W is the A operand of v_mfma_f32_16x16x32 straight from its row-major [N][K] layout: lane
//     (n, g) reads 16 bytes of row n, and a wave's steps read whole cache lines of 16 rows, so no
//     transposed or repacked copy of the weights is needed.  x is the B operand, 16 tokens per
//     MFMA, MT of them.
//   * The waves' sums meet in LDS and are added in wave order by one wave, a different one from
//     tile to tile, while the others go on; with K split over work-groups, the last of a tile's
//     work-groups to arrive adds their sums in split order.  The result does not depend on the
//     order of arrival.
//   * Loads go through buffer resources: tokens past M, steps past a wave's share and tiles past a
//     work-group's share read as zeros, with no branch around the loads.
//
// Before the product (NORM): x is RMS-normalised (model.py:49-55) in registers.  The 8 waves hold
// each token's whole row between them, so the sum of squares is one LDS exchange, and it runs while
// the first tile's weight loads, issued before, are on their way.
// After it:
//   kOut:  + bias, rounded; + residual (model.py:128-138), rounded.
//   kSilu: a tile is the gate and the up rows of 8 features; out = silu(gate) * up
//          (model.py:112-120).
//   kRope: a tile is the 8 + 8 features of 8 rotation pairs of one head: + bias, rotary embedding
//          (model.py:58-65), rotated q to q_out, rotated k and v to their cache slots
//          (kv_cache.py:108-115).
// Every intermediate is rounded to the tensor dtype where the reference's separate tensor ops
// round it; all sums are fp32.
//
// Bound by the weight stream.  Measured (bf16, 16 tokens, weights cold, one launch in a graph, of
// which about 2 us are the launch): gate/up + SwiGLU + norm 17920 x 1536 14.5 us (3.8 TB/s; library
// GEMM 23.0, norm and SwiGLU 5 each), down 1536 x 8960 10 us (21), q/k/v + norm + RoPE 2048 x 1536
// 6.5 us (7.1 + 5 + 5), 151936 x 1536 87 us (5.3 TB/s; 121).  A contiguous stream of the same bytes
// reads at 5.9 and 6.9 TB/s: the rest is the 64-byte pieces of 16 rows each load takes.
#include "linear_rows.h"

#include <algorithm>

namespace mi_fa2 {

namespace {

constexpr int kLrWaves = 8;
constexpr int kLrThreads = 64 * kLrWaves;
constexpr int kLrNone = 0x7ffffff0;   // a byte offset past every resource: reads zeros
constexpr int kLrSteps = 8;   // 32-wide steps of K per wave and tile, at most


template <typename E>
__device__ __forceinline__ float lr_f(uint32_t x16) {
  return E::lo(x16);
}
template <typename E>
__device__ __forceinline__ uint32_t lr_r(float x) {
  return E::pack2(x, 0.f) & 0xffffu;
}
// a value rounded to the tensor dtype; opaque, so that what follows cannot be contracted with what
// came before
template <typename E>
__device__ __forceinline__ float lr_round(float x) {
  float r = lr_f<E>(lr_r<E>(x));
  asm volatile("" : "+v"(r));
  return r;
}

// s_waitcnt operand: at most n vector loads outstanding, other counters not waited for
constexpr int lr_vmcnt(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0F70; }

}  // namespace

// MT: 16-token tiles of x; NS: steps of K per wave and tile, at most.
template <typename E, int MT, int NS, int EPI, bool NORM>
__global__ __launch_bounds__(kLrThreads, 2) void linear_rows_kernel(
    const LinearParams p) {
  static_assert(EPI != kRope || MT == 1, "one tile of tokens is rotated");
  static_assert(!NORM || MT == 1, "one tile of tokens is normalised");
  // Tiles in flight per work-group.  With one work-group per CU and a few tiles each, a second one
  // is worth 2% (17920 x 1536: 14.6 -> 14.3 us); with many tiles, or two work-groups per CU, nothing.
  constexpr int D = EPI == kSilu && MT == 1 ? 2 : 1;
  __shared__ f32x4 red[2][kLrWaves][MT][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;

  // counters the next launch of the sequence uses
  if (p.zero && blockIdx.x == 0)
    for (int i = tid; i < p.n_zero; i += kLrThreads) p.zero[i] = 0;

  // This work-group's share: split `split` of K, tiles grp, grp + groups, ... (at any time the
  // chip's work-groups read neighbouring tiles: 87 us against 94 for a contiguous range of tiles
  // each, 151,936 x 1536 bf16).
  const int groups = gridDim.x / p.splits;
  const int grp = blockIdx.x / p.splits, split = blockIdx.x - grp * p.splits;
  // this wave's steps of K
  const int steps = p.K >> 5, parts = p.splits * kLrWaves, part = split * kLrWaves + wave;
  const int lo = part * steps / parts, hi = (part + 1) * steps / parts;
  const int n_steps = hi - lo;

  // Tile t's 16 rows of W: [base(t), + 16 rows), rows 8 .. 15 `far` rows further on for kSilu and
  // kRope (the up features; the upper halves of the rotation pairs).
  const int row_bytes = p.K * 2;
  const auto base_row = [&](int t) -> int64_t {
    if constexpr (EPI == kSilu) return 8 * t;
    if constexpr (EPI == kRope) return (int64_t)(t >> 3) * kHeadDim + 8 * (t & 7);
    return (int64_t)16 * t;
  };
  const int far = EPI == kSilu ? p.N - 8 : EPI == kRope ? kHeadDim / 2 - 8 : 0;
  const int extent = (16 + far) * row_bytes;
  const int w_off = (n + (n >= 8 ? far : 0)) * row_bytes + 16 * g + lo * 64;
  // Step i of the share of tile t.
  const auto load_w = [&](int t, u32x4 (&d)[NS], int i) {
    const __amdgpu_buffer_rsrc_t r =
        make_rsrc(p.w + base_row(t < p.tiles ? t : grp) * p.K, t < p.tiles ? extent : 0);
    // default cache policy: two steps share a cache line, which a non-temporal load may drop
    // between them (151,936 x 1536: 96 us against 102)
    d[i] = ld16_buf(r, i < n_steps ? w_off + i * 64 : kLrNone);
  };
  // x as the B operand: token 16j + n, k = 32 (lo + i) + 8g .. +7.
  u32x4 xb[NS][MT];
  if (p.x_frag) {
    // already in operand order, [MT][steps][64 lanes][8]: whole contiguous loads
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(p.x, MT * steps * 1024);
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int i = 0; i < NS; ++i)
        xb[i][j] = ld16_buf(xr, i < n_steps ? ((j * steps + lo + i) * 64 + lane) * 16 : kLrNone);
  } else {
    const __amdgpu_buffer_rsrc_t xr =
        make_rsrc(p.x, (int)(((int64_t)(p.M - 1) * p.x_st + p.K) * 2));
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int i = 0; i < NS; ++i)
        xb[i][j] = ld16_buf(xr, i < n_steps && 16 * j + n < p.M
                                    ? (16 * j + n) * (int)p.x_st * 2 + 16 * g + (lo + i) * 64
                                    : kLrNone);
  }

  u32x4 wb[D][NS];
#pragma unroll
  for (int d = 0; d < D; ++d)
#pragma unroll
    for (int i = 0; i < NS; ++i) load_w(grp + d * groups, wb[d], i);
  // x, issued first, is here: told to the compiler, which would otherwise keep waiting for it in
  // every pass of the tile loop, and with it for weight loads that are still on their way
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(lr_vmcnt(D * NS));

  if constexpr (NORM) {
    __shared__ float ssq[kLrWaves][16];
    __shared__ u32x4 nw[kLrWaves * kLrSteps * 4];
    if (tid < (p.K >> 3)) nw[tid] = ld16(p.norm_w + 8 * tid);
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NS; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float a = E::lo(xb[i][0][j]), b = E::hi(xb[i][0][j]);
        ss = __builtin_fmaf(a, a, ss);
        ss = __builtin_fmaf(b, b, ss);
      }
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    if (g == 0) ssq[wave][n] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int u = 0; u < kLrWaves; ++u) tot += ssq[u][n];
    const float inv = rsqrtf(tot / (float)p.K + p.eps);
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const u32x4 wv = nw[min(lo + i, steps - 1) * 4 + g];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float a = lr_round<E>(E::lo(xb[i][0][j]) * inv);
        const float b = lr_round<E>(E::hi(xb[i][0][j]) * inv);
        xb[i][0][j] = E::pack2(E::lo(wv[j]) * a, E::hi(wv[j]) * b);
      }
    }
  }

  const auto one_tile = [&](int tile, int it, u32x4 (&w)[NS]) {
    
    f32x4 acc[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NS; ++i) {
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[j] = E::mfma16(w[i], xb[i][j], acc[j]);
      load_w(tile + D * groups, w, i);
    }
    // The waves' sums: lane (n, g) holds rows 4g .. 4g + 3 of the tile for token 16j + n.  One
    // barrier per tile: the other buffer's readers are past it when they meet this one.
#pragma unroll
    for (int j = 0; j < MT; ++j) red[it & 1][wave][j][lane] = acc[j];
    __syncthreads();
    for (int j = 0; j < MT; ++j) {
      if (((it * MT + j) & (kLrWaves - 1)) != wave) continue;
      f32x4 v = red[it & 1][0][j][lane];
#pragma unroll
      for (int u = 1; u < kLrWaves; ++u) v += red[it & 1][u][j][lane];
      const int m = 16 * j + n;

      if constexpr (EPI == kRope) {
        const int head = tile >> 3;
        // this lane's 4 dims of the head: lower halves of the pairs in g = 0, 1, upper in g = 2, 3
        const int d = 8 * (tile & 7) + 4 * (g & 1) + 64 * (g >> 1);
        if (p.bias) {
          const u32x2 bv = *reinterpret_cast<const u32x2*>(p.bias + head * kHeadDim + d);
          v += f32x4{E::lo(bv[0]), E::hi(bv[0]), E::lo(bv[1]), E::hi(bv[1])};
        }
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = lr_round<E>(v[r]);
        const bool live = m < p.M;
        if (head < p.Hq + p.Hkv) {
          const int64_t at = (int64_t)(live ? m : 0) * p.cs_st + d;
          const u32x2 cv = *reinterpret_cast<const u32x2*>(p.cos + at);
          const u32x2 sv = *reinterpret_cast<const u32x2*>(p.sin + at);
          const float cs[4] = {E::lo(cv[0]), E::hi(cv[0]), E::lo(cv[1]), E::hi(cv[1])};
          const float sn[4] = {E::lo(sv[0]), E::hi(sv[0]), E::lo(sv[1]), E::hi(sv[1])};
          float other[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) other[r] = __shfl_xor(o[r], 32);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            // d < 64: x[d] cos[d] + (-x[d + 64]) sin[d];  d >= 64: x[d] cos[d] + x[d - 64] sin[d]
            const float a = lr_round<E>(o[r] * cs[r]);
            const float b = lr_round<E>((g < 2 ? -other[r] : other[r]) * sn[r]);
            o[r] = a + b;
          }
        }
        if (!live) continue;
        uint16_t* dst;
        if (head < p.Hq) {
          dst = p.out + (int64_t)m * p.out_st + head * kHeadDim + d;
        } else {
          const int slot = p.slots[m];
          if ((unsigned)slot >= (unsigned)p.num_slots) continue;   // padding row
          const int kh = head - p.Hq;
          dst = (kh < p.Hkv ? p.k_pool + (int64_t)kh * p.pool_sh
                            : p.v_pool + (int64_t)(kh - p.Hkv) * p.pool_sh) +
                (int64_t)slot * p.pool_st + d;
        }
        *reinterpret_cast<u32x2*>(dst) = u32x2{E::pack2(o[0], o[1]), E::pack2(o[2], o[3])};
      } else if constexpr (EPI == kSilu) {
        // gate features 8t + 4g .. in g = 0, 1, the same features' up rows in g = 2, 3
        float u[4], o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) u[r] = __shfl_xor(v[r], 32);
        if (g >= 2 || m >= p.M) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float a = lr_round<E>(v[r]);
          o[r] = lr_round<E>(a / (1.f + expf(-a))) * lr_round<E>(u[r]);
        }
        // in the operand order of the next product: k = 8t .. 8t + 7 of lane (n, t % 4)
        uint16_t* dst = p.out + ((int64_t)(j * (p.N >> 5) + (tile >> 2)) * 64 + (tile & 3) * 16 + n) * 8 + 4 * g;
        *reinterpret_cast<u32x2*>(dst) = u32x2{E::pack2(o[0], o[1]), E::pack2(o[2], o[3])};
      } else {
        if (p.splits > 1) {
          // This work-group's sums go to its slot of the workspace; the last of the tile's
          // work-groups to arrive adds all of them up.  Partials and the arrival count are relaxed
          // agent-scope atomics, each coherent across the XCDs' L2s by itself (plain stores
          // published by an agent-scope fence would write back the whole L2); the wave waits for
          // its stores, so they are visible before the count is.
          uint64_t* first = p.part + ((int64_t)(tile * MT + j) * p.splits) * 128 + 2 * lane;
          const u32x4 b = __builtin_bit_cast(u32x4, v);
          __hip_atomic_store(first + split * 128, ((uint64_t)b[1] << 32) | b[0], __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(first + split * 128 + 1, ((uint64_t)b[3] << 32) | b[2],
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          uint32_t arrived = 0;
          if (lane == 0)
            arrived = __hip_atomic_fetch_add(p.count + tile * MT + j, 1u, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
          if (__builtin_amdgcn_readfirstlane(arrived) != (uint32_t)p.splits - 1) continue;
          v = f32x4{0.f, 0.f, 0.f, 0.f};
          for (int s = 0; s < p.splits; ++s) {
            const uint64_t a = __hip_atomic_load(first + s * 128, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
            const uint64_t c = __hip_atomic_load(first + s * 128 + 1, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
            v += f32x4{__uint_as_float((uint32_t)a), __uint_as_float((uint32_t)(a >> 32)),
                       __uint_as_float((uint32_t)c), __uint_as_float((uint32_t)(c >> 32))};
          }
        }
        const int f = 16 * tile + 4 * g;
        if (m >= p.M) continue;
        if (p.bias) {
          const u32x2 bv = *reinterpret_cast<const u32x2*>(p.bias + f);
          v += f32x4{E::lo(bv[0]), E::hi(bv[0]), E::lo(bv[1]), E::hi(bv[1])};
        }
        if (p.res) {
          const u32x2 rv = *reinterpret_cast<const u32x2*>(p.res + (int64_t)m * p.res_st + f);
          const float r[4] = {E::lo(rv[0]), E::hi(rv[0]), E::lo(rv[1]), E::hi(rv[1])};
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = lr_round<E>(v[e]) + r[e];
        }
        *reinterpret_cast<u32x2*>(p.out + (int64_t)m * p.out_st + f) =
            u32x2{E::pack2(v[0], v[1]), E::pack2(v[2], v[3])};
      }
    }
  };
  int it = 0;
  for (int tile = grp; tile < p.tiles; tile += D * groups) {
#pragma unroll
    for (int d = 0; d < D; ++d, ++it)
      if (tile + d * groups < p.tiles) one_tile(tile + d * groups, it, wb[d]);
  }
}

namespace {

template <typename E, int MT, int EPI, bool NORM>
hipError_t launch_rows_t(const LinearParams& p, int grid, hipStream_t stream) {
  const int per_wave = ((p.K >> 5) + p.splits * kLrWaves - 1) / (p.splits * kLrWaves);
  if (per_wave <= 6)
    hipLaunchKernelGGL((linear_rows_kernel<E, MT, 6, EPI, NORM>), dim3(grid), dim3(kLrThreads), 0,
                       stream, p);
  else
    hipLaunchKernelGGL((linear_rows_kernel<E, MT, kLrSteps, EPI, NORM>), dim3(grid),
                       dim3(kLrThreads), 0, stream, p);
  return hipGetLastError();
}

template <typename E>
hipError_t launch_rows_e(const LinearParams& p, int epi, int grid, hipStream_t stream) {
  const int mt = p.M <= 16 ? 1 : p.M <= 32 ? 2 : 4;
  if (p.norm_w) {
    if (mt > 1) return hipErrorInvalidValue;
    if (epi == kRope) return launch_rows_t<E, 1, kRope, true>(p, grid, stream);
    if (epi == kSilu) return launch_rows_t<E, 1, kSilu, true>(p, grid, stream);
    return launch_rows_t<E, 1, kOut, true>(p, grid, stream);
  }
  if (epi == kSilu) {
    if (mt == 1) return launch_rows_t<E, 1, kSilu, false>(p, grid, stream);
    if (mt == 2) return launch_rows_t<E, 2, kSilu, false>(p, grid, stream);
    return launch_rows_t<E, 4, kSilu, false>(p, grid, stream);
  }
  if (epi != kOut) return hipErrorInvalidValue;
  if (mt == 1) return launch_rows_t<E, 1, kOut, false>(p, grid, stream);
  if (mt == 2) return launch_rows_t<E, 2, kOut, false>(p, grid, stream);
  return launch_rows_t<E, 4, kOut, false>(p, grid, stream);
}

}  // namespace

// cos and sin of position x inverse frequency, in fp32 and rounded, as the reference takes them once
// per step (model.py:151-155): there about eight small launches of 2 to 4 us each, here one.
template <typename E>
__global__ __launch_bounds__(64) void rope_table_kernel(const RopeTableParams p) {
  const int token = blockIdx.x, d = threadIdx.x;
  const int row = token / p.T;
  const float a = (float)(p.starts[row] + (token - row * p.T)) * E::lo(p.inv_freq[d]);
  const uint16_t c = (uint16_t)lr_r<E>(cosf(a)), s = (uint16_t)lr_r<E>(sinf(a));
  const int64_t at = (int64_t)token * kHeadDim + d;
  p.cos[at] = c;
  p.cos[at + kHeadDim / 2] = c;
  p.sin[at] = s;
  p.sin[at + kHeadDim / 2] = s;
}

hipError_t launch_rope_table(const RopeTableParams& p, int dtype, hipStream_t stream) {
  const dim3 grid(p.rows * p.T);
  if (dtype == 0)
    hipLaunchKernelGGL((rope_table_kernel<BF16>), grid, dim3(64), 0, stream, p);
  else
    hipLaunchKernelGGL((rope_table_kernel<FP16>), grid, dim3(64), 0, stream, p);
  return hipGetLastError();
}

int linear_splits(int K) {
  const int per_group = 32 * kLrSteps * kLrWaves;
  return (K + per_group - 1) / per_group;
}

hipError_t launch_linear_rows(LinearParams p, int dtype, int epi, int n_cus, hipStream_t stream) {
  p.tiles = p.N / (epi == kSilu ? 8 : 16);
  // One work-group per CU walks the tiles with its x in registers: a second one reads x once more
  // from the L2 (17920 x 1536: 14.3 us at one per CU, 16.6 at two).  With K split, x is a slice and
  // in operand order, and two per CU are faster (1536 x 8960: 12.2 against 13.3 us).
  const int groups = std::min(p.tiles, p.splits > 1 ? std::max(1, 2 * n_cus / p.splits) : n_cus);
  const int grid = groups * p.splits;
  return dtype == 0 ? launch_rows_e<BF16>(p, epi, grid, stream)
                    : launch_rows_e<FP16>(p, epi, grid, stream);
}

}  // namespace mi_fa2
