// Which kernel a call of the general entry point runs on: host code, without HIP.
#pragma once

#include <cstdint>

namespace mi_fa2 {

enum GeneralKernel {
  kGenStaged = 0,    // fa2_general_kernel
  kGenSplit = 1,     // fa2_general_split_kernel
  kGenDims = 2,      // fa2_prefill_dims_kernel, 128-row work-groups
  kGenDimsSmall = 3  // the same, 64-row work-groups of four key streams
};

struct GeneralCall {
  int64_t batch, heads_q, heads_kv, seqlen_q, seqlen_k, k_stride, v_stride;   // token strides
  int d, dv;
  bool bits16;
  float scale_log2;
  int n_cus, xcd_log2;
};

// Whether fa2_prefill_dims_kernel can run the call: K/V rows that neither overlap nor outgrow the
// loads' 32-bit offsets; a scale under which the largest score is the largest exponent (its masked
// scores are -inf before the scaling; the other kernels mask after it and take any); and a launch of
// one dimension that HIP and the kernel's divisions take: fewer than 2^32 threads.
inline bool prefill_dims_fit(const GeneralCall& c, bool small) {
  const auto stride_ok = [&](int64_t st) { return st >= c.d && st < (int64_t(1) << 23); };
  if (c.seqlen_k <= 0 || !stride_ok(c.k_stride) || !stride_ok(c.v_stride)) return false;
  if (!(c.scale_log2 > 0.f && c.scale_log2 < 3.0e38f)) return false;
  const int64_t rows = small ? 64 : 128, threads = c.d > 64 ? 256 : 512, X = int64_t(1) << c.xcd_log2;
  const int64_t groups = ((c.batch * c.heads_kv) | 1) * ((c.seqlen_q + rows - 1) / rows);
  return (groups + X - 1) / X * X * (c.heads_q / c.heads_kv) * threads < int64_t(1) << 32;
}

inline GeneralKernel general_kernel(const GeneralCall& c) {
  constexpr int64_t kRows = 16, kWgRows = 64;   // query rows of a wave, of a staged work-group
  const int64_t heads = c.batch * c.heads_q;
  const int64_t tiles = (c.seqlen_q + kWgRows - 1) / kWgRows * heads;
  // Fewer query rows than a work-group holds, or fewer work-groups than the device's CUs (256 on
  // MI355X): split each 16-row tile's keys over 4 waves instead (4x the work-groups, a quarter of
  // the chain).  fp32 always: its MFMAs are slow enough to cover the split kernel's loads, and
  // staging bought nothing (1 x 12 x 1500 x 128 causal: staged 217 us, split 130; 4 x 1500 x 64:
  // 246 and 197; 4096 x 128: 1,040 and 669).
  const bool split = !c.bits16 || c.seqlen_q < kWgRows || tiles < c.n_cus;
  // The sizes of fa2_prefill_dims.hip.  12 heads, causal, us:
  //  * instead of the split kernel (d <= 64; at d = 256 it is the closer one to 64 bits), where its
  //    shape of 64 rows gains: by the work, 16-row tiles x keys.  d = 64, split and 64-row: 2 x 300
  //    (137 K) 8.7 and 9.0, 4 x 200 (125 K) 8.1 and 7.8, 3 x 300 (205 K) 10.3 and 9.2, 1 x 700
  //    (370 K) 14.2 and 11.0, 1 x 1000 (756 K) 19.2 and 13.5; d = 32 the same within 0.3; and with more
  //    of those tiles than CUs: up to there the split kernel has a CU and eight waves for each (1 x 300
  //    over 4,000 keys, 228 tiles, d = 64 26.8 and 36.6, d = 32 19.5 and 27.4; 1 x 400 over 2,000, 300
  //    tiles, 25.1 and 22.0, 18.5 and 16.3);
  //  * instead of the staged kernel, from one full tile of queries on: d = 64, 4 x 64 4.8 staged and
  //    6.3, 4 x 200 9.0 and 8.3, 4 x 1000 36.7 and 20.9.
  // Of its two shapes, the 64-row one while its work-groups run at once (d = 32: two per CU) and, where
  // rows are long, a little beyond; 64-row and 128-row: d = 64, 2 x 400 9.3 and 10.5, 4 x 400 13.7 and
  // 10.8, 3 x 512 13.8 and 12.2, 1 x 1500 16.7 and 24.5, 2 x 1000 17.5 and 18.7, 2 x 1500 28.5 and 26.7;
  // d = 32, 4 x 512 8.6 and 9.2, 4 x 1000 15.9 and 15.3.
  if (c.bits16 && c.d == c.dv && (c.d == 32 || c.d == 64 || c.d == 256)) {
    const int64_t tiles16 = (c.seqlen_q + kRows - 1) / kRows * heads;
    const bool better = split ? c.d <= 64 && c.seqlen_q >= kRows && tiles16 > c.n_cus &&
                                    tiles16 * c.seqlen_k >= 150000
                              : c.seqlen_q >= 128;
    const bool small = c.d == 32   ? tiles <= 2 * c.n_cus
                       : c.d == 64 ? 4 * tiles <= 3 * c.n_cus ||
                                         (c.seqlen_k >= 1000 && 2 * tiles <= 3 * c.n_cus)
                                   : false;
    if (better && prefill_dims_fit(c, small)) return small ? kGenDimsSmall : kGenDims;
  }
  return split ? kGenSplit : kGenStaged;
}

}  // namespace mi_fa2
