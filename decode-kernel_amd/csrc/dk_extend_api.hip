// dk_extend_api.hip — the extend (prefill) attention's C ABI (include/dk_decode.h:
// dk_extend_attention): argument checks and launches.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

#include "dk_args.h"
#include "dk_decode.h"
#include "dk_extend.h"
#include "dk_launch.h"

namespace dk {
namespace {

// Workgroups per query tile (kExtendFill): 1 = the keys are not split.
int extend_split(int32_t batch, const int32_t* new_lens, const int32_t* all_lens, int32_t hkv,
                 int32_t group, int32_t window) {
  int64_t groups = 0, keys = 0;
  for (int32_t b = 0; b < batch; ++b) {
    if (new_lens[b] <= 0) continue;
    groups += ((int64_t)new_lens[b] * group + kExtendRows - 1) / kExtendRows * hkv;
    // a tile of 128 rows spans up to 128 / group + 1 positions beyond its window
    const int64_t seen = window > 0 ? (int64_t)window + kExtendRows / group + 1 : INT32_MAX;
    keys = std::max<int64_t>(keys, std::min<int64_t>(all_lens[b], seen));
  }
  if (groups == 0) return 1;
  const int64_t s = std::min<int64_t>(kExtendFill / groups, keys / kExtendSplitKeys);
  return (int)std::min<int64_t>(std::max<int64_t>(s, 1), kExtendMaxSplit);
}

template <class T>
hipError_t merge(const ExtendArgs& a, int64_t tokens, int d, hipStream_t stream) {
  MergeArgs m{};
  m.po = a.part_o;
  m.pm = a.part_m;
  m.pl = a.part_l;
  m.out = a.out;
  m.o_b = a.o_b;
  m.o_h = a.o_h;
  m.batch = (int32_t)tokens;
  m.hq = a.hkv * a.group;
  m.split = a.split;
  m.sinks = a.sinks;
  return launch_merge<T>(m, d, false, stream);
}

}  // namespace
}  // namespace dk

extern "C" size_t dk_extend_workspace_bytes(int32_t batch, const int32_t* new_lens,
                                            const int32_t* all_lens, int32_t num_q_heads,
                                            int32_t num_kv_heads, int32_t head_dim,
                                            int32_t window) {
  using namespace dk;
  if (batch <= 0 || !new_lens || !all_lens || num_q_heads <= 0 || num_kv_heads <= 0 ||
      num_q_heads % num_kv_heads != 0 || head_dim <= 0 || window < 0)
    return 0;
  const int s = extend_split(batch, new_lens, all_lens, num_kv_heads, num_q_heads / num_kv_heads,
                             window);
  if (s == 1) return 0;
  int64_t tokens = 0;
  for (int32_t b = 0; b < batch; ++b) tokens += std::max(new_lens[b], 0);
  size_t o, m, l, total;
  partials_layout_rows(tokens * num_q_heads * s, head_dim, &o, &m, &l, &total);
  return total;
}

extern "C" int dk_extend_attention(
    const void* q, const void* k_pool, const void* v_pool, const int32_t* req_to_token,
    int64_t req_stride, int64_t num_rows, const int32_t* rows, const int32_t* new_lens,
    const int32_t* all_lens, void* out, void* workspace, size_t workspace_bytes, int32_t batch,
    int64_t num_tokens, int32_t num_q_heads,
    int32_t num_kv_heads, int32_t head_dim, int64_t num_slots, int32_t dtype, int32_t kv_dtype,
    const dk_extend_strides* strides, float score_scale, float v_scale, float logit_cap,
    int32_t window, const float* sinks, void* hip_stream) {
  using namespace dk;
  clear_error();
  if (!strides) return set_error(DK_ENULL, "strides must be non-NULL");
  if (batch < 0 || num_tokens < 0 || num_tokens > INT32_MAX || num_q_heads <= 0 ||
      num_kv_heads <= 0 || num_q_heads % num_kv_heads != 0 || window < 0 || num_rows < 0 ||
      num_rows > INT32_MAX || num_slots < 0 || num_slots > INT32_MAX || req_stride < 0 ||
      req_stride >= kMaxStride)
    return set_error(DK_EINVAL, "dk_extend_attention: bad sizes");
  if (head_dim != 64 && head_dim != 128 && head_dim != 256)
    return set_error(DK_EINVAL, "head_dim must be 64, 128 or 256; got %d", head_dim);
  if (dtype != DK_F16 && dtype != DK_BF16)
    return set_error(DK_EINVAL, "dtype must be DK_F16 or DK_BF16; got %d", dtype);
  if (kv_dtype != DK_KV_SAME && kv_dtype != DK_KV_FP8_E4M3)
    return set_error(DK_EINVAL, "kv_dtype must be DK_KV_SAME or DK_KV_FP8_E4M3");
  if (!std::isfinite(score_scale) || !(score_scale > 0.f) || !std::isfinite(v_scale) ||
      !std::isfinite(logit_cap))
    return set_error(DK_EINVAL, "score_scale must be finite and > 0, v_scale and logit_cap finite");
  if (batch == 0) return DK_OK;
  if (!rows || !new_lens || !all_lens)
    return set_error(DK_ENULL, "dk_extend_attention: NULL pointer");
  const int64_t kes = kv_dtype == DK_KV_FP8_E4M3 ? 1 : 2;
  const dk_extend_strides& s = *strides;
  if (!extent_ok(num_tokens, s.q_b, num_q_heads, s.q_h, head_dim, 2) ||
      !extent_ok(num_tokens, s.o_b, num_q_heads, s.o_h, head_dim, 2) ||
      !extent_ok(num_slots, s.k_s, num_kv_heads, s.k_h, head_dim, kes) ||
      !extent_ok(num_slots, s.v_s, num_kv_heads, s.v_h, head_dim, kes))
    return set_error(DK_EUNSUPPORTED, "strides must be non-negative and below 2^40 elements");
  for (int64_t b : {s.q_b * 2, s.q_h * 2, s.o_b * 2, s.o_h * 2, s.k_s * kes, s.k_h * kes,
                    s.v_s * kes, s.v_h * kes, (int64_t)((uintptr_t)q % 16),
                    (int64_t)((uintptr_t)out % 16), (int64_t)((uintptr_t)k_pool % 16),
                    (int64_t)((uintptr_t)v_pool % 16)})
    if (b % 16 != 0)
      return set_error(DK_EUNSUPPORTED, "q, out and the pools must be 16-byte aligned, and "
                                        "their strides multiples of 16 bytes");
  if (s.k_s * kes > INT32_MAX || s.v_s * kes > INT32_MAX)
    return set_error(DK_EUNSUPPORTED, "pool slots must be less than 2^31 bytes apart");
  const int32_t group = num_q_heads / num_kv_heads;
  int64_t first = 0;
  for (int32_t b = 0; b < batch; ++b) {
    if (new_lens[b] < 0 || all_lens[b] < new_lens[b] || all_lens[b] > INT32_MAX - 1024 ||
        (int64_t)new_lens[b] * group > INT32_MAX - 1024)
      return set_error(DK_EINVAL, "request %d: %d new of %d tokens", b, new_lens[b], all_lens[b]);
    if (rows[b] < 0 || rows[b] >= num_rows || (num_rows > 1 && all_lens[b] > req_stride))
      return set_error(DK_EINVAL, "request %d: row %d or its length exceeds the map", b, rows[b]);
    first += new_lens[b];
  }
  if (first > num_tokens)
    return set_error(DK_EINVAL, "%lld new tokens in q rows for %lld", (long long)first,
                     (long long)num_tokens);
  if (first == 0) return DK_OK;
  if (!q || !k_pool || !v_pool || !req_to_token || !out)
    return set_error(DK_ENULL, "dk_extend_attention: NULL pointer");
  if (num_slots == 0) return set_error(DK_EINVAL, "the token pool is empty");

  ExtendArgs a{};
  a.q = static_cast<const uint8_t*>(q);
  a.k = static_cast<const uint8_t*>(k_pool);
  a.v = static_cast<const uint8_t*>(v_pool);
  a.req_to_token = req_to_token;
  a.out = static_cast<uint8_t*>(out);
  a.sinks = sinks;
  a.q_b = s.q_b * 2;
  a.q_h = s.q_h * 2;
  a.o_b = s.o_b * 2;
  a.o_h = s.o_h * 2;
  a.k_s = (uint32_t)(s.k_s * kes);
  a.k_h = s.k_h * kes;
  a.v_s = (uint32_t)(s.v_s * kes);
  a.v_h = s.v_h * kes;
  a.req_stride = req_stride;
  a.group = group;
  a.hkv = num_kv_heads;
  a.window = window;
  a.num_slots = (uint32_t)num_slots;
  a.kscale = kLog2e * score_scale;
  a.cap_in = logit_cap != 0.f ? score_scale / logit_cap : 0.f;
  a.cap_out = kLog2e * logit_cap;
  a.vscale = v_scale;
  // without a workspace for the partials the keys are not split
  a.split = extend_split(batch, new_lens, all_lens, num_kv_heads, group, window);
  if (a.split > 1) {
    size_t off_o, off_m, off_l, total;
    partials_layout_rows(first * num_q_heads * a.split, head_dim, &off_o, &off_m, &off_l, &total);
    if (!workspace || workspace_bytes < total || (uintptr_t)workspace % 256 != 0) {
      a.split = 1;
    } else {
      uint8_t* ws = static_cast<uint8_t*>(workspace);
      a.part_o = reinterpret_cast<float*>(ws + off_o);
      a.part_m = reinterpret_cast<float*>(ws + off_m);
      a.part_l = reinterpret_cast<float*>(ws + off_l);
    }
  }
  const bool bf16 = dtype == DK_BF16, kv8 = kes == 1, cap = logit_cap != 0.f;
  const void* fn = head_dim == 64    ? extend_symbol<64>(bf16, kv8, cap)
                   : head_dim == 128 ? extend_symbol<128>(bf16, kv8, cap)
                                     : extend_symbol<256>(bf16, kv8, cap);
  // kExtendMaxReqs requests per launch: their sizes travel as kernel arguments, so a call
  // copies nothing to the device
  int32_t b = 0;
  int64_t q0 = 0;
  while (b < batch) {
    int32_t n = 0;
    int64_t tiles = 0;
    for (; b < batch && n < kExtendMaxReqs; ++b) {
      if (new_lens[b] == 0) continue;
      const int64_t t = ((int64_t)new_lens[b] * group + kExtendRows - 1) / kExtendRows;
      if ((tiles + t) * num_kv_heads > INT32_MAX) {
        if (n == 0) return set_error(DK_EUNSUPPORTED, "request %d has too many new tokens", b);
        break;
      }
      a.req[n++] = ExtendReq{rows[b], (int32_t)q0, new_lens[b], all_lens[b], (int32_t)tiles};
      tiles += t;
      q0 += new_lens[b];
    }
    if (n == 0) break;
    a.num_reqs = n;
    a.tiles = (int32_t)tiles;
    void* args[] = {&a};
    const hipError_t e =
        hipLaunchKernel(fn, dim3((uint32_t)(tiles * num_kv_heads), a.split), dim3(kExtendThreads), args, 0,
                        static_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) return set_error((int)e, "extend launch: %s", hipGetErrorString(e));
  }
  if (a.split > 1) {
    const hipStream_t st = static_cast<hipStream_t>(hip_stream);
    const hipError_t e =
        bf16 ? merge<BF16>(a, first, head_dim, st) : merge<F16>(a, first, head_dim, st);
    if (e != hipSuccess) return set_error((int)e, "extend merge launch: %s", hipGetErrorString(e));
  }
  return DK_OK;
}
