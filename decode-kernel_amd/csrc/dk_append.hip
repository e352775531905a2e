// dk_append.hip — the cache write before a decode step (C ABI in include/dk_decode.h:
// dk_append_kv).
//
// For every sequence b the new token is the last one the page table describes: page
// kv_indices[kv_indptr[b+1] - 1], slot kv_last_page_len[b] - 1 (the caller has grown the
// table first, as a paged allocator does). Its K row (rotated) and V row are written there
// for every kv head, and q (optional) is rotated in place, all with rotary position
// embedding at the token's position:
//   rotate-half pairs (i, i + D/2) (Llama / GPT-NeoX) or interleaved pairs (2i, 2i + 1)
//   (GPT-J), angle = position * inv_freq[i], y0 = x0 cos - x1 sin, y1 = x1 cos + x0 sin,
// computed in fp32 and rounded once to the cache type. inv_freq carries any frequency
// scaling (e.g. Llama 3's); without it the rows are copied unrotated. An fp8 (OCP E4M3)
// cache stores RNE(clamp(x / scale, -448, 448)) of each fp32 value x (NaN stays NaN).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

#include "dk_args.h"
#include "dk_decode.h"

namespace dk {
namespace {

constexpr int kAppendThreads = 256;
// A thread rotates the same VEC pairs of up to kAppendHeads heads: one sincos for all of them
constexpr int kAppendHeads = 4;
template <int VEC>
constexpr int kAppendV = VEC == 1 ? 1 : 4 * VEC;   // elements of a V row that a thread copies

// the page table is read through the constant address space (scalar loads): it is not written here
__device__ __forceinline__ int32_t ld_table(const int32_t* p, int64_t i) {
  return ((const __attribute__((address_space(4))) int32_t*)p)[i];
}

struct AppendArgs {
  uint8_t* q;                 // may be null
  const uint8_t* k_new;
  const uint8_t* v_new;
  uint8_t* k_cache;
  int64_t v_off;              // bytes from a K row to the V row of the same slot
  const int32_t* indptr;
  const int32_t* indices;
  const int32_t* last_len;
  const int32_t* positions;   // may be null: position = tokens in the sequence - 1
  const float* inv_freq;      // may be null: no rotation
  int64_t q_b, q_h, n_b, n_h, kv_p, kv_s, kv_h;   // bytes
  int32_t batch, hq, hkv, d, num_indices, rope_style;
  uint32_t num_pages;
  float k_scale, v_scale;     // fp8 cache: stored = value / scale
  int32_t cols;               // VEC-pair columns of a head
  int32_t q_units, k_units, v_units;   // threads on q (0: not rotated), K and V rows
  int32_t slice0;             // first slice of the launch
};

template <class E, int N>
using Vec = E __attribute__((ext_vector_type(N)));

typedef short short2_t __attribute__((ext_vector_type(2)));

// N values in the cache's (or q's) own type, rounded once
template <class E>
struct Store {
  static constexpr int kBytes = 2;
  template <int N>
  __device__ void operator()(uint8_t* p, const float (&x)[N]) const {
    Vec<E, N> r;
#pragma unroll
    for (int i = 0; i < N; ++i) r[i] = (E)x[i];
    *reinterpret_cast<Vec<E, N>*>(p) = r;
  }
};

// OCP E4M3 of x / scale: round to nearest even, clamped to +-448 (the largest finite value)
// so that no finite input becomes NaN; NaN stays NaN.
struct Fp8Store {
  static constexpr int kBytes = 1;
  float scale;
  template <int N>
  __device__ void operator()(uint8_t* p, const float (&x)[N]) const {
    Vec<uint8_t, N> r;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      float y = x[i] / scale;
      y = y != y ? y : fminf(fmaxf(y, -448.f), 448.f);
      const short2_t w =
          __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(short2_t{0, 0}, y, 0.f, 1.f, false);
      r[i] = (uint8_t)(w[0] & 0xff);
    }
    *reinterpret_cast<Vec<uint8_t, N>*>(p) = r;
  }
};

// VEC consecutive pairs (i0, i1) of one row, from column `col`: (col*VEC + e, half + ...) in
// the rotate-half style, (2*(col*VEC + e), ... + 1) interleaved.
template <class E, int VEC>
struct Pairs {
  Vec<E, VEC> lo, hi;   // as they lie in the row: two runs of VEC elements
  static __device__ int at0(int col, int style) { return col * VEC * (style == 0 ? 1 : 2); }
  static __device__ int at1(int col, int style, int half) {
    return at0(col, style) + (style == 0 ? half : VEC);
  }
  __device__ void load(const uint8_t* row, int col, int style, int half) {
    lo = *reinterpret_cast<const Vec<E, VEC>*>(row + 2 * at0(col, style));
    hi = *reinterpret_cast<const Vec<E, VEC>*>(row + 2 * at1(col, style, half));
  }
  template <class Out>
  __device__ void rotate_to(uint8_t* row, int col, int style, int half, bool rot,
                            const float (&c)[VEC], const float (&s)[VEC], const Out& out) const {
    float x[2 * VEC], y[2 * VEC];   // in row order
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      x[e] = (float)lo[e];
      x[VEC + e] = (float)hi[e];
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float x0 = style == 0 ? x[e] : x[2 * e], x1 = style == 0 ? x[VEC + e] : x[2 * e + 1];
      const float y0 = rot ? __builtin_fmaf(x0, c[e], -(x1 * s[e])) : x0;
      const float y1 = rot ? __builtin_fmaf(x0, s[e], x1 * c[e]) : x1;
      if (style == 0) {
        y[e] = y0;
        y[VEC + e] = y1;
      } else {
        y[2 * e] = y0;
        y[2 * e + 1] = y1;
      }
    }
    float a[VEC], b[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      a[e] = y[e];
      b[e] = y[VEC + e];
    }
    out(row + Out::kBytes * at0(col, style), a);
    out(row + Out::kBytes * at1(col, style, half), b);
  }
};

// Workgroups (sequence, slice of its units). A unit is VEC pairs of kAppendHeads heads of q
// or K, or kAppendV elements of a V row; every load that does not need the page table is
// issued before the table's dependent reads. VEC 1 takes any head_dim and alignment, VEC 2
// needs whole vectors (append_impl).
// Bound by latency (kernel start, the table's two dependent reads, sincos, stores). Per call in
// a replayed graph, against one workgroup per sequence with one pair of one head per step and
// a sincos each, us: B=32 32/8/64 bf16 3.8 -> 3.0, B=1 32/8/128 fp16 5.3 -> 2.7, B=256
// 32/8/128 bf16 5.8 -> 3.2, B=32 32/8/128 into fp8 6.2 -> 3.5, B=16 128/8/256 into fp8 25.4
// -> 3.7.
template <class E, bool KV8, int VEC>
__global__ __launch_bounds__(kAppendThreads) void dk_append_kv_kernel(AppendArgs a) {
  constexpr int NV = kAppendV<VEC>;
  const int b = blockIdx.x;
  int u = (a.slice0 + (int)blockIdx.y) * kAppendThreads + (int)threadIdx.x;
  const bool is_q = u < a.q_units;
  if (!is_q) u -= a.q_units;
  const bool is_k = !is_q && u < a.k_units;
  if (!is_q && !is_k) u -= a.k_units;
  if (!is_q && !is_k && u >= a.v_units) return;

  const int half = a.d / 2, style = a.rope_style;
  const int col = u % a.cols, h0 = u / a.cols * kAppendHeads;
  const int heads = min(kAppendHeads, (is_q ? a.hq : a.hkv) - h0);
  const uint8_t* src = is_q ? a.q + (int64_t)b * a.q_b : a.k_new + (int64_t)b * a.n_b;
  const int64_t s_h = is_q ? a.q_h : a.n_h;
  Pairs<E, VEC> p[kAppendHeads];
  float f[VEC];
  Vec<E, NV> v;
  const int vh = u * NV / a.d, vi = u * NV % a.d;
  if (is_q || is_k) {
#pragma unroll
    for (int h = 0; h < kAppendHeads; ++h)
      if (h < heads) p[h].load(src + (h0 + h) * s_h, col, style, half);
#pragma unroll
    for (int e = 0; e < VEC; ++e) f[e] = a.inv_freq ? a.inv_freq[col * VEC + e] : 0.f;
  } else {
    v = *reinterpret_cast<const Vec<E, NV>*>(a.v_new + (int64_t)b * a.n_b + vh * a.n_h + 2 * vi);
  }

  const int s0 = min(max(ld_table(a.indptr, b), 0), a.num_indices);
  const int s1 = min(max(ld_table(a.indptr, b + 1), 0), a.num_indices);
  if (s1 <= s0) return;                        // a sequence without pages has no slot
  uint32_t page = (uint32_t)ld_table(a.indices, s1 - 1);
  page = page < a.num_pages ? page : 0u;
  const int slot = min(max(ld_table(a.last_len, b) - 1, 0), kPageSize - 1);
  const float pos = a.positions ? (float)ld_table(a.positions, b)
                                : (float)((s1 - s0 - 1) * kPageSize + slot);
  uint8_t* krow = a.k_cache + (int64_t)page * a.kv_p + (int64_t)slot * a.kv_s;
  if (is_q || is_k) {
    const bool rot = a.inv_freq != nullptr;
    float c[VEC], s[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) sincosf(pos * f[e], &s[e], &c[e]);
#pragma unroll
    for (int h = 0; h < kAppendHeads; ++h) {
      if (h >= heads) break;
      if (is_q)
        p[h].rotate_to(a.q + (int64_t)b * a.q_b + (h0 + h) * a.q_h, col, style, half, rot, c, s,
                       Store<E>{});
      else if constexpr (KV8)
        p[h].rotate_to(krow + (h0 + h) * a.kv_h, col, style, half, rot, c, s,
                       Fp8Store{a.k_scale});
      else
        p[h].rotate_to(krow + (h0 + h) * a.kv_h, col, style, half, rot, c, s, Store<E>{});
    }
  } else {
    uint8_t* dst = krow + a.v_off + vh * a.kv_h;
    if constexpr (KV8) {
      float x[NV];
#pragma unroll
      for (int e = 0; e < NV; ++e) x[e] = (float)v[e];
      Fp8Store{a.v_scale}(dst + vi, x);
    } else {
      *reinterpret_cast<Vec<E, NV>*>(dst + 2 * vi) = v;
    }
  }
}

template <int VEC>
const void* append_symbol(int32_t dtype, bool kv8) {
  if (kv8)
    return dtype == DK_F16 ? (const void*)dk_append_kv_kernel<_Float16, true, VEC>
                           : (const void*)dk_append_kv_kernel<__bf16, true, VEC>;
  return dtype == DK_F16 ? (const void*)dk_append_kv_kernel<_Float16, false, VEC>
                         : (const void*)dk_append_kv_kernel<__bf16, false, VEC>;
}

}  // namespace
}  // namespace dk

static int append_impl(void* q, const void* k_new, const void* v_new, int64_t new_b,
                       int64_t new_h, void* k_cache, void* v_cache,
                       const int32_t* kv_indptr, const int32_t* kv_indices,
                       const int32_t* kv_last_page_len, const int32_t* positions,
                       const float* inv_freq, int32_t rope_style, int32_t batch,
                       int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                       int32_t page_size, int64_t num_pages, int64_t num_indices,
                       int32_t dtype, bool kv8, float k_scale, float v_scale,
                       const dk_strides* strides, void* hip_stream) {
  dk::clear_error();
  if (!strides) return dk::set_error(DK_ENULL, "strides must be non-NULL");
  if (batch < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || head_dim % 2 ||
      head_dim > 1024)
    return dk::set_error(DK_EINVAL, "dk_append_kv: bad batch / head counts / head_dim");
  if (page_size != dk::kPageSize)
    return dk::set_error(DK_EINVAL, "page_size must be 16; got %d", page_size);
  if (dtype != DK_F16 && dtype != DK_BF16)
    return dk::set_error(DK_EINVAL, "dtype must be DK_F16 or DK_BF16; got %d", dtype);
  if (kv8 && (!(k_scale > 0.f) || !(v_scale > 0.f) || !std::isfinite(k_scale) ||
              !std::isfinite(v_scale)))
    return dk::set_error(DK_EINVAL, "k_scale and v_scale must be finite and > 0");
  if (rope_style != 0 && rope_style != 1)
    return dk::set_error(DK_EINVAL, "rope_style must be 0 (rotate half) or 1 (interleaved)");
  if (num_indices < 0 || num_indices > INT32_MAX || num_pages < 0)
    return dk::set_error(DK_EINVAL, "dk_append_kv: bad num_indices / num_pages");
  if (num_indices > 0 && num_pages == 0)
    return dk::set_error(DK_EINVAL, "kv_indices is non-empty but the page pool is empty");
  const dk_strides& s = *strides;
  if (new_b < 0 || new_h < 0 || s.q_b < 0 || s.q_h < 0 || s.kv_p < 0 || s.kv_s < 0 ||
      s.kv_h < 0 || (!v_cache && s.kv_r < 0))
    return dk::set_error(DK_EINVAL, "strides must be non-negative");
  // every byte offset formed from the strides must fit int64 (bounded in 128-bit arithmetic)
  const int64_t kes_ = kv8 ? 1 : 2;
  if (!dk::extent_ok(batch, s.q_b, num_q_heads, s.q_h, head_dim, 2) ||
      !dk::extent_ok(batch, new_b, num_kv_heads, new_h, head_dim, 2) ||
      !dk::pool_ok(num_pages, s, v_cache ? 0 : s.kv_r, num_kv_heads, head_dim, kes_))
    return dk::set_error(DK_EUNSUPPORTED,
                         "strides must be below 2^40 elements and q, the new rows and the cache "
                         "must span less than 2^62 bytes");
  if (batch == 0) return DK_OK;
  if (!k_new || !v_new || !k_cache || !kv_indptr || !kv_last_page_len ||
      (num_indices > 0 && !kv_indices))
    return dk::set_error(DK_ENULL, "dk_append_kv: NULL pointer");
  dk::AppendArgs a{};
  a.q = static_cast<uint8_t*>(q);
  a.k_new = static_cast<const uint8_t*>(k_new);
  a.v_new = static_cast<const uint8_t*>(v_new);
  a.k_cache = static_cast<uint8_t*>(k_cache);
  const int64_t kes = kv8 ? 1 : 2;   // cache element bytes
  a.v_off = v_cache ? (int64_t)(static_cast<uint8_t*>(v_cache) - static_cast<uint8_t*>(k_cache))
                    : s.kv_r * kes;
  a.indptr = kv_indptr;
  a.indices = kv_indices;
  a.last_len = kv_last_page_len;
  a.positions = positions;
  a.inv_freq = inv_freq;
  a.q_b = s.q_b * 2;
  a.q_h = s.q_h * 2;
  a.n_b = new_b * 2;
  a.n_h = new_h * 2;
  a.kv_p = s.kv_p * kes;
  a.kv_s = s.kv_s * kes;
  a.kv_h = s.kv_h * kes;
  a.k_scale = k_scale;
  a.v_scale = v_scale;
  a.batch = batch;
  a.hq = num_q_heads;
  a.hkv = num_kv_heads;
  a.d = head_dim;
  a.num_indices = (int32_t)num_indices;
  a.rope_style = rope_style;
  a.num_pages = (uint32_t)std::min<int64_t>(num_pages, (int64_t)1 << 31);
  // whole vectors: 4 bytes of q / K and 16 of V per thread (fp8 rows half that)
  auto mult16 = [](int64_t bytes) { return bytes % 16 == 0; };
  const int64_t cw = kv8 ? 8 : 16;   // bytes of 8 cache elements
  const bool wide = head_dim % 8 == 0 && (!q || (mult16(a.q_b) && mult16(a.q_h))) &&
                    mult16(a.n_b) && mult16(a.n_h) && (uintptr_t)q % 16 == 0 &&
                    (uintptr_t)k_new % 16 == 0 && (uintptr_t)v_new % 16 == 0 &&
                    (uintptr_t)k_cache % cw == 0 && a.v_off % cw == 0 && a.kv_p % cw == 0 &&
                    a.kv_s % cw == 0 && a.kv_h % cw == 0;
  const int vec = wide ? 2 : 1;
  a.cols = head_dim / 2 / vec;
  auto groups = [](int64_t heads) { return (heads + dk::kAppendHeads - 1) / dk::kAppendHeads; };
  const int64_t qu = q && inv_freq ? groups(num_q_heads) * a.cols : 0;
  const int64_t ku = groups(num_kv_heads) * a.cols;
  const int64_t vu = (int64_t)num_kv_heads * head_dim / (wide ? dk::kAppendV<2> : dk::kAppendV<1>);
  const int64_t slices = (qu + ku + vu + dk::kAppendThreads - 1) / dk::kAppendThreads;
  a.q_units = (int32_t)qu;
  a.k_units = (int32_t)ku;
  a.v_units = (int32_t)vu;
  void* args[] = {&a};
  const void* fn = wide ? dk::append_symbol<2>(dtype, kv8) : dk::append_symbol<1>(dtype, kv8);
  for (int64_t y = 0; y < slices; y += 65535) {   // one launch but for absurdly long rows
    a.slice0 = (int32_t)y;
    const dim3 grid(batch, (uint32_t)std::min<int64_t>(slices - y, 65535));
    const hipError_t e = hipLaunchKernel(fn, grid, dim3(dk::kAppendThreads), args, 0,
                                         static_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) return dk::set_error((int)e, "append launch: %s", hipGetErrorString(e));
  }
  return DK_OK;
}

extern "C" int dk_append_kv(void* q, const void* k_new, const void* v_new, int64_t new_b,
                            int64_t new_h, void* k_cache, void* v_cache,
                            const int32_t* kv_indptr, const int32_t* kv_indices,
                            const int32_t* kv_last_page_len, const int32_t* positions,
                            const float* inv_freq, int32_t rope_style, int32_t batch,
                            int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                            int32_t page_size, int64_t num_pages, int64_t num_indices,
                            int32_t dtype, const dk_strides* strides, void* hip_stream) {
  return append_impl(q, k_new, v_new, new_b, new_h, k_cache, v_cache, kv_indptr, kv_indices,
                     kv_last_page_len, positions, inv_freq, rope_style, batch, num_q_heads,
                     num_kv_heads, head_dim, page_size, num_pages, num_indices, dtype, false,
                     0.f, 0.f, strides, hip_stream);
}

extern "C" int dk_append_kv_fp8(void* q, const void* k_new, const void* v_new, int64_t new_b,
                                int64_t new_h, void* k_cache, void* v_cache,
                                const int32_t* kv_indptr, const int32_t* kv_indices,
                                const int32_t* kv_last_page_len, const int32_t* positions,
                                const float* inv_freq, int32_t rope_style, int32_t batch,
                                int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                int32_t page_size, int64_t num_pages, int64_t num_indices,
                                int32_t dtype, float k_scale, float v_scale,
                                const dk_strides* strides, void* hip_stream) {
  return append_impl(q, k_new, v_new, new_b, new_h, k_cache, v_cache, kv_indptr, kv_indices,
                     kv_last_page_len, positions, inv_freq, rope_style, batch, num_q_heads,
                     num_kv_heads, head_dim, page_size, num_pages, num_indices, dtype, true,
                     k_scale, v_scale, strides, hip_stream);
}
