// Prefill forward for head dims 32, 64 and 256 (d = d_v) in bf16 / fp16: the organisation of the
// head-dim-128 kernel (fa2_prefill.hip) for the other sizes in wide use, padded mode.
//
//   * A work-group is RG row groups of 32 query rows of one query head by NS key streams (64-key
//     tiles NS j + s), one wave each.  S^T = K Q^T and O^T += V^T P^T on v_mfma_f32_32x32x16, so P
//     stays in registers and the softmax state is per lane.
//   * K and V tiles go straight from memory into LDS (rows of 2 d bytes, 16-byte chunks
//     XOR-swizzled so that 16 consecutive rows, and the 4 rows of a transposing read, fall on
//     different banks); V^T operands are transposing reads.  Two stages: step j reads V(j) and
//     K(j + 1) of one while the other receives V(j + 1) and K(j + 2); one barrier per step.
//   * At d <= 64 the softmax's exponentials, not the MFMAs, bound a tile (per 64 keys and wave
//     32 quarter-rate exponentials, FMAs and packing, about 770 cycles, against 16 MFMAs of 32 at
//     d = 64), so the shapes keep waves in flight: 4 x 2 (128 rows), 64 KB of LDS at d = 64, two
//     work-groups per CU; and for launches that fill the chip once, 2 x 4 (64 rows), which halves the
//     chain of a tile.  At d = 256 a wave holds 128 registers of O and 64 of Q and the tiles take
//     128 KB, so 4 x 1 has the CU.
//   * The work-groups' order is that of the head-dim-128 kernel: heads sharing a kv head on one XCD,
//     longest tiles first.
// Measured (bf16, causal, 12 heads over 2 kv heads, before on the general kernels -> here; 4 x 2
// unless said): 4 x 1000 x 64 37.7 -> 21.0 us, 1 x 1000 x 64 25.0 -> 2 x 4 13.7; 4 x 1500 x 64 67.7 ->
// 32.0, 2 x 4 53; 4 x 1200 x 32 36.3 -> 19.8; 2 x 1000 x 256 112.6 -> 55.9; 1 x 4096 x 256 586 -> 200
// (516 TFLOP/s, ten calls back to back).  The branch for large scores costs 0-2% of that at d = 64, 0-3%
// at 32, 3-4% at 256 (the exponentials of two runs of keys are no longer scheduled across it; walking the
// tile twice instead, or scaling the scores first, cost 2-3% at every size, and up to 20%).
#include "fa2_common.h"
#include "fa2_tiles.h"

namespace mi_fa2 {

namespace {

constexpr int kPdKeys = 64;

// RG row groups of 32 rows, NS key streams.
template <int D, int RG, int NS>
struct PdShape {
  static constexpr int kRows = 32 * RG;
  static constexpr int kThreads = 64 * RG * NS;
  static constexpr int kOcc = D > 64 ? 1 : NS == 2 ? 4 : 2;  // waves per SIMD
  static constexpr int kRow = 2 * D;                       // bytes of a K or V row
  static constexpr int kChunks = D / 8;                    // 16-byte chunks of it
  static constexpr int kTile = kPdKeys * kRow;
  static constexpr int kStage = 2 * NS * kTile;            // K tiles, then V tiles
  static constexpr int kLds = 2 * kStage;
  static constexpr int kLoads = kTile / 1024 / RG;         // per wave and tile, 1 KB each
  static constexpr int kLoadRows = 1024 / kRow;            // rows of one load
  static constexpr int kSlotRows = D < 128 ? 128 / D : 1;  // rows per 256 bytes of LDS
  static constexpr int kXor = kChunks < 16 ? kChunks - 1 : 15;
  // swizzles of a row's chunk index
  static __device__ __forceinline__ int k_swz(int row) { return (row / kSlotRows) & kXor; }
  static __device__ __forceinline__ int v_swz(int row) {   // of 64-byte groups of four chunks
    return D == 32 ? 0 : D == 64 ? (row >> 1) & 1 : row & 3;
  }
};

}  // namespace

template <typename E, int D, int RG, int NS>
__global__ __launch_bounds__(
    (PdShape<D, RG, NS>::kThreads),
    (PdShape<D, RG, NS>::kOcc)) void fa2_prefill_dims_kernel(const FwdParams p, int n_qt,
                                                            const ItemMap map) {
  using Sh = PdShape<D, RG, NS>;
  constexpr int kStep = kPdKeys * NS, kDB = D / 32, kDS = D / 16, kPdRows = Sh::kRows;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[Sh::kLds];
  probe_mark(p.clock_probe, blockIdx.x, false);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = wave % RG, ks = wave / RG;
  int b, h, rank;
  if (!prefill_item(blockIdx.x, map, n_qt, b, h, rank)) return;
  b = __builtin_amdgcn_readfirstlane(b);
  h = __builtin_amdgcn_readfirstlane(h);
  rank = __builtin_amdgcn_readfirstlane(rank);
  const int hk = __builtin_amdgcn_readfirstlane(fdiv(h, map.group));
  const int T = p.T;
  const int kv_len =
      __builtin_amdgcn_readfirstlane(p.kv_lens ? clamp_len(p.kv_lens[b], p.S) : p.S);
  const int q0 = (n_qt - 1 - rank) * kPdRows;
  const int off = kv_len - T;   // query i sits at key position i + off
  int kv_hi = p.causal ? min(kv_len, min(q0 + kPdRows, T) + off) : kv_len;
  kv_hi = __builtin_amdgcn_readfirstlane(max(kv_hi, 0));
  const int n_steps = (kv_hi + kStep - 1) / kStep;

  const int wq0 = q0 + rg * 32;
  const bool wave_active = wq0 < T;
  const int wave_hi = p.causal ? min(kv_len, min(wq0 + 31, T - 1) + off + 1) : kv_len;
  const int wave_full = p.causal ? min(kv_len, wq0 + off + 1) : kv_len;
  const int r32 = lane & 31, g = lane >> 5;
  const int qrow = wq0 + r32;
  const float c = p.scale_log2;
  const int lim = p.causal ? min(kv_len, qrow + off + 1) : kv_len;   // keys < lim are visible

  // Q^T as the B operand: k-step s covers d = 16 s + 8 g + [0, 8).
  u32x4 qb[kDS];
  {
    const uint16_t* qp =
        p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)min(qrow, T - 1) * p.q_st + 8 * g;
#pragma unroll
    for (int s = 0; s < kDS; ++s) qb[s] = ld16(qp + 16 * s);
  }

  // Loads: instruction i of a tile moves rows kLoadRows i .., lane l row l / kChunks of them into
  // chunk l % kChunks, which holds global chunk (l % kChunks) ^ swizzle(row).  Wave w loads its own
  // stream's tiles, instructions w % RG + RG u.
  const uint16_t* kp = p.k + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  const uint16_t* vp = p.v + (int64_t)b * p.v_sb + (int64_t)hk * p.v_sh;
  const int k_st = (int)p.k_st, v_st = (int)p.v_st;
  int k_voff[Sh::kLoads], v_voff[Sh::kLoads];
#pragma unroll
  for (int u = 0; u < Sh::kLoads; ++u) {
    const int row = (rg + RG * u) * Sh::kLoadRows + lane / Sh::kChunks, ch = lane % Sh::kChunks;
    k_voff[u] = row * k_st * 2 + 16 * (ch ^ Sh::k_swz(row));
    v_voff[u] = row * v_st * 2 + 16 * (ch ^ (4 * Sh::v_swz(row)));
  }
  const uint32_t lds_base = lds_addr_of(smem);
  const auto load_tile = [&](const uint16_t* base, int st, int ts, int lds_off,
                             const int (&voff)[Sh::kLoads]) {
    const int rows = sclamp(kv_hi - ts, 0, kPdKeys);   // rows past kv_hi read as zeros
    const uint64_t at = uniform_u64(reinterpret_cast<uint64_t>(base + (int64_t)ts * st));
    const int bytes = __builtin_amdgcn_readfirstlane(rows * st * 2);
#pragma unroll
    for (int u = 0; u < Sh::kLoads; ++u)
      lds_dma16(at, bytes,
                __builtin_amdgcn_readfirstlane(lds_base + lds_off + 1024 * (rg + RG * u)), voff[u]);
  };
  const auto tile_kt = [&](int j) { return j * kStep + ks * kPdKeys; };
  const auto k_lds = [&](int slot) { return slot * Sh::kStage + ks * Sh::kTile; };
  const auto v_lds = [&](int slot) { return slot * Sh::kStage + (NS + ks) * Sh::kTile; };
  // Stage j, in LDS slot j & 1: V(j) and K(j + 1).
  const auto load_stage = [&](int j, int slot) {
    load_tile(vp, v_st, tile_kt(j), v_lds(slot), v_voff);
    load_tile(kp, k_st, tile_kt(j + 1), k_lds(slot), k_voff);
  };
  const auto stage_ready = [&]() {
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0), for the compiler's own loads
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };
  const auto active = [&](int j) { return wave_active && j < n_steps && tile_kt(j) < wave_hi; };

  f32x16 oacc[kDB];
#pragma unroll
  for (int i = 0; i < kDB; ++i) oacc[i] = f32x16{};
  float m_run = -INFINITY, l_run = 0.f;

  // S^T of a tile, MFMA row m holding key pi(m) of its 32-key block, so that a lane's accumulators
  // are runs of 8 consecutive keys.
  const int pim = 16 * (r32 >> 4) + 8 * ((r32 >> 2) & 1) + 4 * ((r32 >> 3) & 1) + (r32 & 3);
  const int f = Sh::k_swz(pim);   // of period 16 rows: the same for pim + 32
  const int kx = pim * Sh::kRow + 16 * (g ^ (f & 1)) + 32 * (f >> 1);
  const auto scores = [&](int slot, f32x16& s0, f32x16& s1) {
    const uint8_t* kt = smem + k_lds(slot);
    s0 = f32x16{};
    s1 = f32x16{};
#pragma unroll
    for (int s = 0; s < kDS; ++s) {
      const uint8_t* a = kt + (kx ^ (32 * s));
      s0 = E::mfma32(*reinterpret_cast<const u32x4*>(a), qb[s], s0);
      s1 = E::mfma32(*reinterpret_cast<const u32x4*>(a + 32 * Sh::kRow), qb[s], s1);
    }
  };

  // Online softmax.  The exponent reference is the row's running maximum itself, so that the largest
  // weight so far is 1, which rounds to itself.  It moves once per tile; with four streams, whose
  // launches are bound by latency rather than by this arithmetic, every 32 keys, as in the split
  // kernel whose launches they take (the outputs are then as close to 64 bits as that kernel's).
  const auto mask = [&](int key0, f32x16& s) {
    if (key0 + 32 > wave_full) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (key0 + 16 * (r >> 3) + 8 * g + (r & 7) >= lim) s[r] = -INFINITY;
    }
  };
  const auto row_max = [&](const f32x16& s) {
    float mx = fmaxf(s[0], s[1]);
#pragma unroll
    for (int r = 2; r < 16; r += 2) mx = fmax3(mx, s[r], s[r + 1]);
    return mx;
  };
  constexpr float kExactScore = 0x1p24f;
  bool exact = false;   // whether some row's maximum is that large (exps)
  const auto move_max = [&](float mx) {
    mx = fmaxf(mx, __shfl_xor(mx, 32)) * c;
    if (__any(mx > m_run)) {
      const float m_new = fmaxf(m_run, mx);
      // a row that sees its first key scales its empty state by exp2(-inf) = 0; one that has seen
      // none yet keeps it
      const float alpha = mx > m_run ? exp2_fast(m_run - m_new) : 1.f;
      l_run *= alpha;
#pragma unroll
      for (int i = 0; i < kDB; ++i) oacc[i] *= alpha;
      m_run = m_new;
      exact = __any(m_run != -INFINITY && fabsf(m_run) >= kExactScore);
    }
  };
  // P^T of 32 keys as the B operand of two k-steps; the row sum adds P as rounded.  The exponents are
  // one fma each: the row's largest is then off 0 by the rounding of m_run, which cancels in the
  // division while it is small (below 1/2 up to kExactScore).  Beyond, where it would overflow, the
  // products are rounded as m_run was, so that the largest is 0.
  const auto exps = [&](const f32x16& s, u32x4 (&pb)[2]) {
    const float m_use = m_run == -INFINITY ? 0.f : m_run;
    float lt = 0.f;
    if (D > 64 ? exact : __builtin_expect(exact, false)) {
#pragma clang fp contract(off)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float x0 = s[2 * i] * c, x1 = s[2 * i + 1] * c;
        pb[i >> 2][i & 3] = E::pack2(exp2_fast(x0 - m_use), exp2_fast(x1 - m_use));
        lt = E::sum2(pb[i >> 2][i & 3], lt);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        pb[i >> 2][i & 3] = E::pack2(exp2_fast(__builtin_fmaf(s[2 * i], c, -m_use)),
                                     exp2_fast(__builtin_fmaf(s[2 * i + 1], c, -m_use)));
        lt = E::sum2(pb[i >> 2][i & 3], lt);
      }
    }
    l_run += lt;
  };
  // O^T += V^T P^T of 32 keys: lane 16 G + 4 k + q (g = G / 2) reads rows 16 kk + 8 g + 4 sec + k,
  // columns 32 db + 16 (G % 2) + 4 q .. +3.
  const int vk = (lane >> 2) & 3;
  const int vx = (8 * g + vk) * Sh::kRow + 32 * ((lane >> 4) & 1) + 8 * (lane & 3);
  const int vz = Sh::v_swz(vk);   // rows 4 apart share it
  const auto pv = [&](int slot, int key_off, const u32x4 (&pb)[2]) {
    const uint8_t* vt = smem + v_lds(slot) + vx + key_off * Sh::kRow;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int db = 0; db < kDB; ++db) {
        const uint8_t* a = vt + 64 * (db ^ vz) + 16 * kk * Sh::kRow;
        const u32x2 lo = ds_read_tr16(a), hi = ds_read_tr16(a + 4 * Sh::kRow);
        oacc[db] = E::mfma32(u32x4{lo[0], lo[1], hi[0], hi[1]}, pb[kk], oacc[db]);
      }
  };
  const auto softmax_pv = [&](int j, int slot, f32x16& s0, f32x16& s1) {
    const int kt = tile_kt(j);
    u32x4 p0[2], p1[2];
    mask(kt, s0);
    if constexpr (NS == 4) {
      move_max(row_max(s0));
      exps(s0, p0);
      pv(slot, 0, p0);
      if (kt + 32 >= wave_hi) return;
      mask(kt + 32, s1);
      move_max(row_max(s1));
      exps(s1, p1);
      pv(slot, 32, p1);
    } else {
      mask(kt + 32, s1);
      move_max(fmaxf(row_max(s0), row_max(s1)));
      exps(s0, p0);
      exps(s1, p1);
      pv(slot, 0, p0);
      pv(slot, 32, p1);
    }
  };

  f32x16 s0, s1;
  if (n_steps > 0) {
    load_tile(kp, k_st, tile_kt(0), k_lds(1), k_voff);   // stage -1 holds K(0) only
    load_stage(0, 0);
  }
  stage_ready();
  if (active(0)) scores(1, s0, s1);
  __syncthreads();   // slot 1 is rewritten during step 0
  const auto step = [&](int j, int slot) {
    if (j + 1 < n_steps) load_stage(j + 1, slot ^ 1);
    if (active(j)) softmax_pv(j, slot, s0, s1);
    if (active(j + 1)) scores(slot, s0, s1);
    stage_ready();
  };
  int j = 0;
  for (; j + 2 <= n_steps; j += 2) {
    step(j, 0);
    step(j + 1, 1);
  }
  if (j < n_steps) step(j, 0);

  // The last barrier came after every LDS read and load of the loop: the stages may be overwritten.
  constexpr int kXVals = 16 * kDB + 2;   // exchanged per lane: O, m, l
  float* red = reinterpret_cast<float*>(smem);
  if constexpr (NS > 1) {
    // streams 1 .. NS - 1 hand their state to stream 0
    float* x = red + rg * kXVals * 64 + lane;
    constexpr int kNext = RG * kXVals * 64;
    if (ks > 0) {
      float* y = x + (ks - 1) * kNext;
#pragma unroll
      for (int i = 0; i < kDB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) y[(16 * i + r) * 64] = oacc[i][r];
      y[16 * kDB * 64] = m_run;
      y[(16 * kDB + 1) * 64] = l_run;
    }
    __syncthreads();
    if (ks > 0) return;
#pragma unroll
    for (int t = 0; t < NS - 1; ++t, x += kNext) {
      const float mo = x[16 * kDB * 64], lo = x[(16 * kDB + 1) * 64];
      const float M = fmaxf(m_run, mo), M_use = M == -INFINITY ? 0.f : M;
      const float fs = exp2_fast(m_run - M_use), fo = exp2_fast(mo - M_use);
#pragma unroll
      for (int i = 0; i < kDB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          oacc[i][r] = __builtin_fmaf(oacc[i][r], fs, x[(16 * i + r) * 64] * fo);
      l_run = __builtin_fmaf(l_run, fs, lo * fo);
      m_run = M;
    }
  }
  const float l_tot = l_run + __shfl_xor(l_run, 32);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  // Rows go through LDS so that the stores write whole rows: [32 rows][d], chunks XOR-swizzled.
  // Accumulator r of block db is d = 32 db + 8 (r / 4) + 4 g + r % 4.
  constexpr int kExchange = (NS - 1) * RG * kXVals * 256;
  static_assert(kExchange + RG * 32 * Sh::kRow <= Sh::kLds, "staging fits");
  uint8_t* ot = smem + kExchange + rg * 32 * Sh::kRow;
#pragma unroll
  for (int db = 0; db < kDB; ++db)
#pragma unroll
    for (int rr = 0; rr < 4; ++rr)
      *reinterpret_cast<u32x2*>(ot + r32 * Sh::kRow + 16 * ((4 * db + rr) ^ Sh::k_swz(r32)) + 8 * g) =
          u32x2{E::pack2(oacc[db][4 * rr] * inv, oacc[db][4 * rr + 1] * inv),
                E::pack2(oacc[db][4 * rr + 2] * inv, oacc[db][4 * rr + 3] * inv)};
  __builtin_amdgcn_wave_barrier();
  uint16_t* op = p.o + (int64_t)b * p.o_sb + (int64_t)h * p.o_sh;
#pragma unroll
  for (int k = 0; k < 32 / Sh::kLoadRows; ++k) {
    const int row = k * Sh::kLoadRows + lane / Sh::kChunks, ch = lane % Sh::kChunks;
    const u32x4 val =
        *reinterpret_cast<const u32x4*>(ot + row * Sh::kRow + 16 * (ch ^ Sh::k_swz(row)));
    if (wq0 + row < T)
      *reinterpret_cast<u32x4*>(op + (int64_t)(wq0 + row) * p.o_st + 8 * ch) = val;
  }
  if (p.lse && g == 0 && qrow < T)
    p.lse[(int64_t)b * p.l_sb + (int64_t)h * p.l_sh + (int64_t)qrow * p.l_st] =
        l_tot > 0.f ? (m_run + __builtin_log2f(l_tot)) * kLn2 : -INFINITY;
  probe_mark(p.clock_probe, blockIdx.x, true);
}

template <typename E, int D, int RG, int NS>
static hipError_t launch_dims_t(const FwdParams& p, hipStream_t stream) {
  using Sh = PdShape<D, RG, NS>;
  const int n_qt = (p.T + Sh::kRows - 1) / Sh::kRows, classes = p.B * p.Hkv;
  hipLaunchKernelGGL((fa2_prefill_dims_kernel<E, D, RG, NS>),
                     dim3(prefill_grid_size(classes, p.group, n_qt, p.xcd_log2)),
                     dim3(Sh::kThreads), 0, stream, p, n_qt,
                     make_item_map(classes, p.group, p.Hkv, p.xcd_log2));
  return hipGetLastError();
}

template <typename E>
static hipError_t launch_dims_e(const FwdParams& p, int d, bool small, hipStream_t stream) {
  if (d == 32) return small ? launch_dims_t<E, 32, 2, 4>(p, stream) : launch_dims_t<E, 32, 4, 2>(p, stream);
  if (d == 64) return small ? launch_dims_t<E, 64, 2, 4>(p, stream) : launch_dims_t<E, 64, 4, 2>(p, stream);
  return launch_dims_t<E, 256, 4, 1>(p, stream);
}

// small: the 64-row shape of four key streams (d <= 64).  The calls that fit are
// fa2_general_rule.h's.
hipError_t launch_prefill_dims(const FwdParams& p, int dtype, int d, bool small,
                               hipStream_t stream) {
  return dtype == 0 ? launch_dims_e<BF16>(p, d, small, stream)
                    : launch_dims_e<FP16>(p, d, small, stream);
}

}  // namespace mi_fa2
