// Fused last-position token sampler: one pass over each row's logits draws the row's next token.
//
// Replaces the reference's batched sampling (chat.py:103-107): probs = softmax(logits / T) and
// torch.multinomial(probs, 1), which on the GPU are about eight launches per step (the float cast,
// the scaled softmax's max / sum / normalise passes, the exponential draw, the divide, the argmax).
// torch.multinomial draws one sample per row by the exponential race, argmax_v probs_v / E_v with
// E_v ~ Exp(1); in log space the softmax normaliser cancels and the draw is
//
//     token = argmax_v ( logit_v / T - ln E_v ),   E_v = -ln U_v,
//
// so the logits are read once, with no max or sum pass.  T <= 0 is greedy (argmax of the logits).
// Ties go to the lowest index; NaN scores never win; a row with no candidate gets -1.
//
// Uniforms: Philox4x32-10 (Salmon et al., SC 2011), key = the 64-bit seed, counter = (v / 4, row,
// offset low, offset high); word v % 4 of that block is entry v's, mapped to
// U = (2 * (x >> 9) + 1) * 2^-24, exact in fp32 and strictly inside (0, 1).  A caller advances
// `offset` once per call, so every (row, step) draws fresh numbers, reproducibly from the seed.
//
// Work split: work-group (chunk, row) scans 8192 entries (1024 threads x 2 Philox blocks of 4
// consecutive entries; consecutive threads take consecutive blocks) and keeps the best
// (score, index).  A row that fits in one chunk is finished there; otherwise the last of the row's
// work-groups to arrive reduces the chunks' winners (or, without arrival counters, a second
// one-wave-per-row kernel).
//
// Bound by the vector ALU: Philox (32 x 32 -> 64-bit products at a quarter of the rate) and two
// logarithms per entry.  The accurate logarithms are only taken where they can matter: every entry's
// score is first taken with the hardware's log2 (1 ulp), and only entries within a margin of the
// wave's best, far wider than the difference between the two, are scored as above.  The winner is
// the same.  16 rows of 151,936 bf16: 12.1 + 3.8 us in two
// launches -> 10.0 us in one (one row: 7.0).
#include "fa2_arrival.h"
#include "fa2_common.h"

namespace mi_fa2 {

constexpr int kSmpThreads = 1024;
constexpr int kSmpBlocksPerThread = 2;                              // Philox blocks per thread
constexpr int kSmpChunk = kSmpThreads * kSmpBlocksPerThread * 4;   // 8192 entries per work-group

constexpr uint32_t kPhiloxM0 = 0xD2511F53u, kPhiloxM1 = 0xCD9E8D57u;
constexpr uint32_t kPhiloxW0 = 0x9E3779B9u, kPhiloxW1 = 0xBB67AE85u;

__device__ __forceinline__ void philox4x32_10(uint32_t (&c)[4], uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    if (r) {
      k0 += kPhiloxW0;
      k1 += kPhiloxW1;
    }
    const uint64_t p0 = (uint64_t)kPhiloxM0 * c[0], p1 = (uint64_t)kPhiloxM1 * c[2];
    const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0, n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1;
    c[0] = n0;
    c[1] = (uint32_t)p1;
    c[2] = n2;
    c[3] = (uint32_t)p0;
  }
}

template <int DT>
__device__ __forceinline__ float load_logit(const void* base, int64_t i) {
  if constexpr (DT == 0) {
    return __uint_as_float((uint32_t)static_cast<const uint16_t*>(base)[i] << 16);
  } else if constexpr (DT == 1) {
    return (float)static_cast<const _Float16*>(base)[i];
  } else {
    return static_cast<const float*>(base)[i];
  }
}

// (s, i) beats (bs, bi): higher score, or the same finite-or-+inf score at a lower index.
__device__ __forceinline__ bool better(float s, int i, float bs, int bi) {
  return s > bs || (s == bs && i >= 0 && (bi < 0 || i < bi));
}

__device__ __forceinline__ void wave_best(float& s, int& i) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    const float os = __shfl_xor(s, d);
    const int oi = __shfl_xor(i, d);
    if (better(os, oi, s, i)) {
      s = os;
      i = oi;
    }
  }
}

// Entries 4g .. 4g + 3 of a row as fp32, NaN past the end (which never wins).  `wide`: the row allows
// one load of the four.
template <int DT>
__device__ __forceinline__ void load_block(const void* base, int g, int vocab, bool wide,
                                           float (&l)[4]) {
  const int64_t v = 4 * (int64_t)g;
  if (wide && v + 4 <= vocab) {
    if constexpr (DT == 2) {
      const f32x4 t = *reinterpret_cast<const f32x4*>(static_cast<const float*>(base) + v);
#pragma unroll
      for (int e = 0; e < 4; ++e) l[e] = t[e];
    } else {
      const u32x2 t = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(base) + v);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint16_t x = (uint16_t)(t[e >> 1] >> (16 * (e & 1)));
        l[e] = DT == 0 ? __uint_as_float((uint32_t)x << 16) : (float)__builtin_bit_cast(_Float16, x);
      }
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      l[e] = v + e < vocab ? load_logit<DT>(base, v + e) : __builtin_nanf("");
  }
}

__device__ __forceinline__ float uniform_of(uint32_t w) {
  return (float)(2u * (w >> 9) + 1u) * 0x1p-24f;
}

// Best of the row's chunk winners, by one wave; `coherent`: they were left by work-groups of this
// launch.
__device__ __forceinline__ int reduce_chunks(const SampleParams& p, int row, int lane,
                                             bool coherent) {
  float best_s = -INFINITY;
  int best_i = -1;
  for (int c = lane; c < p.chunks; c += 64) {
    uint32_t* at = p.part + 2 * ((int64_t)row * p.chunks + c);
    const auto read = [&](uint32_t* a) {
      return coherent ? __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : *a;
    };
    const float s = __uint_as_float(read(at));
    const int i = (int)read(at + 1);
    if (better(s, i, best_s, best_i)) {
      best_s = s;
      best_i = i;
    }
  }
  wave_best(best_s, best_i);
  return best_i;
}

template <int DT>
__global__ __launch_bounds__(kSmpThreads) void sample_chunk_kernel(const SampleParams p) {
  const int row = blockIdx.y, chunk = blockIdx.x, tid = threadIdx.x;
  constexpr int kSize = DT == 2 ? 4 : 2;
  const void* base = static_cast<const char*>(p.logits) + (int64_t)row * p.row_stride * kSize;
  const bool wide = (reinterpret_cast<uintptr_t>(base) & (4 * kSize - 1)) == 0;
  const int g0 = chunk * (kSmpChunk / 4) + tid;   // Philox block = entries 4g .. 4g+3
  float l[kSmpBlocksPerThread][4];
#pragma unroll
  for (int j = 0; j < kSmpBlocksPerThread; ++j)
    load_block<DT>(base, g0 + j * kSmpThreads, p.vocab, wide, l[j]);

  float best_s = -INFINITY;
  int best_i = -1;
  // v increases within a thread: strict > keeps the lowest index
  const auto consider = [&](float s, int v) {
    if (s > best_s) {
      best_s = s;
      best_i = v;
    }
  };
  if (p.greedy) {
#pragma unroll
    for (int j = 0; j < kSmpBlocksPerThread; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) consider(l[j][e], 4 * (g0 + j * kSmpThreads) + e);
  } else {
    float u[kSmpBlocksPerThread][4], a[kSmpBlocksPerThread][4];
    float top = -INFINITY;
#pragma unroll
    for (int j = 0; j < kSmpBlocksPerThread; ++j) {
      uint32_t w[4] = {(uint32_t)(g0 + j * kSmpThreads), (uint32_t)row, p.off_lo, p.off_hi};
      philox4x32_10(w, p.seed_lo, p.seed_hi);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        u[j][e] = uniform_of(w[e]);
        // ln E through log2: E = -ln 2 log2(u)
        const float ln_e = kLn2 * __builtin_amdgcn_logf(-kLn2 * __builtin_amdgcn_logf(u[j][e]));
        a[j][e] = l[j][e] * p.inv_t - ln_e;
        top = fmaxf(top, a[j][e]);
      }
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) top = fmaxf(top, __shfl_xor(top, d));
    // Both logs are good to a few units in the last place and |ln E| < 17, so the two scores differ
    // by less than 1e-5 + 1e-6 of their size; NaN and -inf stay out, +inf is its own margin.
    const float cut = top - (1e-3f + 1e-4f * fabsf(top));
#pragma unroll
    for (int j = 0; j < kSmpBlocksPerThread; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (a[j][e] >= cut || a[j][e] == INFINITY)
          consider(l[j][e] * p.inv_t - logf(-logf(u[j][e])), 4 * (g0 + j * kSmpThreads) + e);
  }
  wave_best(best_s, best_i);
  __shared__ float ws_s[kSmpThreads / 64];
  __shared__ int ws_i[kSmpThreads / 64];
  const int lane = tid & 63, wave = tid >> 6;
  if (lane == 0) {
    ws_s[wave] = best_s;
    ws_i[wave] = best_i;
  }
  __syncthreads();
  if (wave != 0) return;
  best_s = lane < kSmpThreads / 64 ? ws_s[lane] : -INFINITY;
  best_i = lane < kSmpThreads / 64 ? ws_i[lane] : -1;
  wave_best(best_s, best_i);
  if (p.chunks == 1) {
    if (lane == 0) p.tokens[row] = best_i;
    return;
  }
  // The chunk's winner goes to the workspace.  With counters, the row's last work-group to arrive
  // reduces them: relaxed agent-scope accesses, each coherent by itself, the store waited for before
  // the arrival is counted.  The counter is left at zero.
  const uint32_t weight = arrival_weight(chunk, p.chunks);
  uint32_t arrived = 0;
  if (lane == 0) {
    uint32_t* at = p.part + 2 * ((int64_t)row * p.chunks + chunk);
    __hip_atomic_store(at, __float_as_uint(best_s), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(at + 1, (uint32_t)best_i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (p.count) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      arrived = __hip_atomic_fetch_add(p.count + row, weight, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (!p.count || __builtin_amdgcn_readfirstlane(arrived) + weight != 0) return;
  const int token = reduce_chunks(p, row, lane, true);
  if (lane == 0) p.tokens[row] = token;
}

__global__ __launch_bounds__(64) void sample_reduce_kernel(const SampleParams p) {
  const int token = reduce_chunks(p, blockIdx.x, threadIdx.x, false);
  if (threadIdx.x == 0) p.tokens[blockIdx.x] = token;
}

int sample_chunks(int vocab) { return (vocab + kSmpChunk - 1) / kSmpChunk; }

hipError_t launch_sample(const SampleParams& p, int dtype, hipStream_t stream) {
  const dim3 grid(p.chunks, p.batch);
  if (dtype == 0)
    hipLaunchKernelGGL((sample_chunk_kernel<0>), grid, dim3(kSmpThreads), 0, stream, p);
  else if (dtype == 1)
    hipLaunchKernelGGL((sample_chunk_kernel<1>), grid, dim3(kSmpThreads), 0, stream, p);
  else
    hipLaunchKernelGGL((sample_chunk_kernel<2>), grid, dim3(kSmpThreads), 0, stream, p);
  if (p.chunks > 1 && !p.count)
    hipLaunchKernelGGL(sample_reduce_kernel, dim3(p.batch), dim3(64), 0, stream, p);
  return hipGetLastError();
}

}  // namespace mi_fa2
