// C ABI of libmi_model.so: argument checks and launches of the few-row projections.  The contract
// of every entry point is in include/mi_model.h.
#include "mi_model.h"

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdarg>
#include <cstdio>

#include "linear_rows.h"

namespace {

using mi_fa2::LinearParams;

enum Status { kOk = 0, kInvalid = 1, kUnsupported = 2, kWorkspace = 3, kLaunch = 4 };

thread_local char g_err[256] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int ok() {
  g_err[0] = '\0';
  return kOk;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// The current device's compute units, read once per device.
int compute_units(int* out) {
  static std::atomic<int> known[64];
  int dev = -1;
  hipError_t err = hipGetDevice(&dev);
  if (err == hipSuccess && dev >= 0 && dev < 64) *out = known[dev].load(std::memory_order_relaxed);
  else *out = 0;
  if (err == hipSuccess && *out == 0) {
    err = hipDeviceGetAttribute(out, hipDeviceAttributeMultiprocessorCount, dev);
    if (err == hipSuccess && dev < 64) known[dev].store(*out, std::memory_order_relaxed);
  }
  if (err != hipSuccess || *out <= 0)
    return fail(kLaunch, "reading the device's CU count failed: %s", hipGetErrorString(err));
  return kOk;
}

int check_dtype(int32_t dtype) {
  if (dtype != 0 && dtype != 1)
    return fail(kUnsupported, "dtype %d is not bf16 (0) or fp16 (1)", dtype);
  return kOk;
}

int check_sizes(int32_t rows, int32_t in, const void* norm_weight) {
  const int max_rows = norm_weight ? mi_fa2::kLrMaxNormRows : mi_fa2::kLrMaxRows;
  if (rows < 0 || rows > max_rows)
    return fail(kInvalid, "rows %d: 0 to %d%s", rows, max_rows, norm_weight ? " with a norm" : "");
  if (in <= 0 || in % 32 || in > mi_fa2::kLrMaxK)
    return fail(kInvalid, "in features %d: a multiple of 32, at most %d", in, mi_fa2::kLrMaxK);
  return kOk;
}

int check_ptr(const char* name, const void* p) {
  if (!p) return fail(kInvalid, "%s is NULL", name);
  if (!aligned16(p)) return fail(kInvalid, "%s is not 16-byte aligned", name);
  return kOk;
}

// Row offsets are 32-bit bytes: 64 rows x 2 bytes x stride < 2^30.
int check_rows(const char* name, const void* p, int64_t stride, int64_t width) {
  if (int rc = check_ptr(name, p)) return rc;
  if (stride < width || stride % 8 || stride >= int64_t(1) << 23)
    return fail(kInvalid, "%s row stride %lld: a multiple of 8 from %lld to 2^23 - 8", name,
                (long long)stride, (long long)width);
  return kOk;
}

int launch(const LinearParams& p, int dtype, int epi, void* stream) {
  int cus = 0;
  if (int rc = compute_units(&cus)) return rc;
  const hipError_t err =
      mi_fa2::launch_linear_rows(p, dtype, epi, cus, reinterpret_cast<hipStream_t>(stream));
  if (err != hipSuccess) return fail(kLaunch, "kernel launch failed: %s", hipGetErrorString(err));
  return ok();
}

// The MLP's workspace: the activation in operand order, then (when the down projection's K is split)
// its fp32 partials and arrival counts.
struct MlpSpace {
  size_t act, part, count, total;
};
MlpSpace mlp_space(int32_t rows, int32_t hidden, int32_t inter) {
  const size_t tokens = rows <= 16 ? 16 : rows <= 32 ? 32 : 64;
  const int splits = mi_fa2::linear_splits(inter);
  MlpSpace s{};
  s.act = tokens * inter * 2;
  s.part = splits > 1 ? tokens * hidden * splits * sizeof(float) : 0;
  s.count = splits > 1 ? tokens / 16 * (hidden / 16) * sizeof(uint32_t) : 0;
  s.total = s.act + s.part + s.count;
  return s;
}

}  // namespace

extern "C" {

const char* mi_model_last_error(void) { return g_err; }

int mi_model_linear(int32_t dtype, const void* x, int64_t x_stride, const void* norm_weight,
                    float eps, const void* w, const void* bias, const void* residual,
                    int64_t residual_stride, void* out, int64_t out_stride, int32_t rows,
                    int32_t out_features, int32_t in_features, void* stream) {
  if (int rc = check_dtype(dtype)) return rc;
  if (int rc = check_sizes(rows, in_features, norm_weight)) return rc;
  if (out_features <= 0 || out_features % 16)
    return fail(kInvalid, "out features %d: a multiple of 16", out_features);
  if (rows == 0) return ok();
  if (int rc = check_rows("x", x, x_stride, in_features)) return rc;
  if (int rc = check_ptr("w", w)) return rc;
  if (norm_weight && !aligned16(norm_weight)) return check_ptr("norm_weight", norm_weight);
  if (bias && !aligned16(bias)) return check_ptr("bias", bias);
  if (residual)
    if (int rc = check_rows("residual", residual, residual_stride, out_features)) return rc;
  if (int rc = check_rows("out", out, out_stride, out_features)) return rc;
  LinearParams p{};
  p.x = static_cast<const uint16_t*>(x);
  p.x_st = x_stride;
  p.norm_w = static_cast<const uint16_t*>(norm_weight);
  p.eps = eps;
  p.w = static_cast<const uint16_t*>(w);
  p.bias = static_cast<const uint16_t*>(bias);
  p.res = static_cast<const uint16_t*>(residual);
  p.res_st = residual_stride;
  p.out = static_cast<uint16_t*>(out);
  p.out_st = out_stride;
  p.M = rows;
  p.N = out_features;
  p.K = in_features;
  p.splits = 1;
  return launch(p, dtype, mi_fa2::kOut, stream);
}

int mi_model_rope_table(int32_t dtype, const int32_t* starts, const void* inv_freq, void* cos,
                        void* sin, int32_t rows, int32_t tokens_per_row, void* stream) {
  if (int rc = check_dtype(dtype)) return rc;
  if (rows < 0 || tokens_per_row < 0 || (int64_t)rows * tokens_per_row > (1 << 24))
    return fail(kInvalid, "bad sizes: rows=%d tokens_per_row=%d (at most 2^24 tokens)", rows,
                tokens_per_row);
  if (rows == 0 || tokens_per_row == 0) return ok();
  if (!starts) return fail(kInvalid, "starts is NULL");
  if (!inv_freq) return fail(kInvalid, "inv_freq is NULL");
  if (int rc = check_ptr("cos", cos)) return rc;
  if (int rc = check_ptr("sin", sin)) return rc;
  const mi_fa2::RopeTableParams p{starts, static_cast<const uint16_t*>(inv_freq),
                                  static_cast<uint16_t*>(cos), static_cast<uint16_t*>(sin), rows,
                                  tokens_per_row};
  const hipError_t err =
      mi_fa2::launch_rope_table(p, dtype, reinterpret_cast<hipStream_t>(stream));
  if (err != hipSuccess) return fail(kLaunch, "kernel launch failed: %s", hipGetErrorString(err));
  return ok();
}

size_t mi_model_mlp_workspace_size(int32_t rows, int32_t hidden, int32_t inter) {
  if (rows <= 0 || hidden <= 0 || inter <= 0) return 0;
  return mlp_space(rows, hidden, inter).total;
}

int mi_model_mlp(int32_t dtype, const void* x, int64_t x_stride, const void* norm_weight,
                 float eps, const void* gate_up_w, const void* down_w, const void* residual,
                 int64_t residual_stride, void* out, int64_t out_stride, int32_t rows,
                 int32_t hidden, int32_t inter, void* workspace, size_t workspace_bytes,
                 void* stream) {
  if (int rc = check_dtype(dtype)) return rc;
  if (int rc = check_sizes(rows, hidden, norm_weight)) return rc;
  if (inter <= 0 || inter % 32 || inter > (1 << 18))
    return fail(kInvalid, "inter %d: a multiple of 32, at most 2^18", inter);
  if (rows == 0) return ok();
  if (int rc = check_rows("x", x, x_stride, hidden)) return rc;
  if (int rc = check_ptr("gate_up_w", gate_up_w)) return rc;
  if (int rc = check_ptr("down_w", down_w)) return rc;
  if (norm_weight && !aligned16(norm_weight)) return check_ptr("norm_weight", norm_weight);
  if (residual)
    if (int rc = check_rows("residual", residual, residual_stride, hidden)) return rc;
  if (int rc = check_rows("out", out, out_stride, hidden)) return rc;
  const MlpSpace s = mlp_space(rows, hidden, inter);
  if (int rc = check_ptr("workspace", workspace)) return rc;
  if (workspace_bytes < s.total)
    return fail(kWorkspace, "workspace of %zu bytes needed, %zu given", s.total, workspace_bytes);
  char* ws = static_cast<char*>(workspace);

  LinearParams a{};
  a.x = static_cast<const uint16_t*>(x);
  a.x_st = x_stride;
  a.norm_w = static_cast<const uint16_t*>(norm_weight);
  a.eps = eps;
  a.w = static_cast<const uint16_t*>(gate_up_w);
  a.out = reinterpret_cast<uint16_t*>(ws);
  a.M = rows;
  a.N = inter;
  a.K = hidden;
  a.splits = 1;
  // the next launch's arrival counts
  a.zero = s.count ? reinterpret_cast<uint32_t*>(ws + s.act + s.part) : nullptr;
  a.n_zero = (int32_t)(s.count / sizeof(uint32_t));
  if (int rc = launch(a, dtype, mi_fa2::kSilu, stream)) return rc;

  LinearParams b{};
  b.x = a.out;
  b.x_frag = 1;
  b.w = static_cast<const uint16_t*>(down_w);
  b.res = static_cast<const uint16_t*>(residual);
  b.res_st = residual_stride;
  b.out = static_cast<uint16_t*>(out);
  b.out_st = out_stride;
  b.M = rows;
  b.N = hidden;
  b.K = inter;
  b.splits = mi_fa2::linear_splits(inter);
  b.part = reinterpret_cast<uint64_t*>(ws + s.act);
  b.count = a.zero;
  return launch(b, dtype, mi_fa2::kOut, stream);
}

int mi_model_qkv_rope(int32_t dtype, const void* x, int64_t x_stride, const void* norm_weight,
                      float eps, const void* w, const void* bias, const void* cos,
                      const void* sin, int64_t cs_stride, const int32_t* slot_mapping,
                      void* q_out, int64_t q_stride, void* k_pool, void* v_pool,
                      const int64_t* pool_strides, int32_t num_slots, int32_t rows,
                      int32_t hidden, int32_t heads_q, int32_t heads_kv, void* stream) {
  if (int rc = check_dtype(dtype)) return rc;
  if (!norm_weight) return fail(kInvalid, "norm_weight is NULL");
  if (int rc = check_sizes(rows, hidden, norm_weight)) return rc;
  if (heads_q <= 0 || heads_kv <= 0 || num_slots < 0 || heads_q > 4096 || heads_kv > 4096)
    return fail(kInvalid, "bad sizes: heads_q=%d heads_kv=%d num_slots=%d", heads_q, heads_kv,
                num_slots);
  if (rows == 0) return ok();
  const int d = mi_fa2::kHeadDim;
  if (int rc = check_rows("x", x, x_stride, hidden)) return rc;
  if (int rc = check_ptr("norm_weight", norm_weight)) return rc;
  if (int rc = check_ptr("w", w)) return rc;
  if (bias && !aligned16(bias)) return check_ptr("bias", bias);
  if (int rc = check_rows("cos", cos, cs_stride, d)) return rc;
  if (int rc = check_rows("sin", sin, cs_stride, d)) return rc;
  if (!slot_mapping) return fail(kInvalid, "slot_mapping is NULL");
  if (int rc = check_rows("q_out", q_out, q_stride, (int64_t)heads_q * d)) return rc;
  if (!pool_strides) return fail(kInvalid, "pool strides are NULL");
  if (int rc = check_ptr("k_pool", k_pool)) return rc;
  if (int rc = check_ptr("v_pool", v_pool)) return rc;
  for (int i = 0; i < 2; ++i)
    if (pool_strides[i] <= 0 || pool_strides[i] % 8)
      return fail(kInvalid, "pool stride %lld is not a positive multiple of 8",
                  (long long)pool_strides[i]);
  LinearParams p{};
  p.x = static_cast<const uint16_t*>(x);
  p.x_st = x_stride;
  p.norm_w = static_cast<const uint16_t*>(norm_weight);
  p.eps = eps;
  p.w = static_cast<const uint16_t*>(w);
  p.bias = static_cast<const uint16_t*>(bias);
  p.out = static_cast<uint16_t*>(q_out);
  p.out_st = q_stride;
  p.M = rows;
  p.N = (heads_q + 2 * heads_kv) * d;
  p.K = hidden;
  p.splits = 1;
  p.cos = static_cast<const uint16_t*>(cos);
  p.sin = static_cast<const uint16_t*>(sin);
  p.cs_st = cs_stride;
  p.slots = slot_mapping;
  p.k_pool = static_cast<uint16_t*>(k_pool);
  p.v_pool = static_cast<uint16_t*>(v_pool);
  p.pool_st = pool_strides[0];
  p.pool_sh = pool_strides[1];
  p.num_slots = num_slots;
  p.Hq = heads_q;
  p.Hkv = heads_kv;
  return launch(p, dtype, mi_fa2::kRope, stream);
}

}  // extern "C"
