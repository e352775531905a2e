// dk_extend.h — device code of the extend (prefill) attention over a token pool (gfx950,
// wave64): causal attention of each request's new tokens over its cached prefix and
// themselves, K and V gathered token by token through a request-to-token map.
//
// A workgroup of 4 wavefronts owns kBM = 128 query rows of one kv head: rows are (new token,
// q head of the GQA group) pairs in token order, so one read of a K/V tile serves every q
// head that shares it, and a wavefront owns 32 of the rows. Tiles of BN keys are staged in
// LDS, double-buffered through registers (the next tile's global loads are in flight while a
// tile is computed; one barrier per tile).
//   * S^T = K.Q^T on v_mfma_f32_32x32x16: lane (h = lane/32, c = lane%32) holds, for query
//     row c, the scores of keys 8*(i/4) + 4h + i%4 of a 32-key block in registers i = 0..15.
//     A row's softmax is therefore in-lane but for one swap of the two halves.
//   * O^T += V^T.P^T: those registers are, as they lie, the B operand of the next MFMA, if
//     the contraction's 16 keys are taken in the order 4h..4h+3, 8+4h..8+4h+3. V^T comes in
//     that order from the row-major V tile by LDS transpose reads (ds_read_b64_tr_b16).
//     Each lane's accumulators all belong to its own query row, so rescaling is in-lane.
//   * p enters as a sum of parts of the element type, 2 in fp16 and 3 in bf16 (ExtendParts).
//     Scores, softmax, sums and accumulators are fp32.
// Bound by the MFMAs and the softmax between them: in bf16 at D = 128 the four MFMA streams (q.k
// and the 3 parts of p) run at 1100 TFLOP/s where a large library product reaches 1267, but a
// SIMD is in an MFMA only 57 % of the time; the rest is exponentials and the split of the
// weights, which the SIMD's other wavefront hides in part. 32/8/128, 2048 new of 8192 tokens,
// back to back: bf16 441 us (546 TFLOP/s of attention), fp16 376; the PyTorch path 6,200 us. 8
// requests of 33-777 new tokens over up to 500 at D = 64: 51-53 us (profiled, new inputs each
// call). 32 query rows per wavefront, so that two wavefronts fit a SIMD (241 registers at D =
// 128); 128 rows per workgroup keep the LDS reads at two thirds of the LDS rate.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dk_kernels.h"

namespace dk {

constexpr int kExtendRows = 128;      // query rows per workgroup
constexpr int kExtendThreads = 256;
// A call of fewer workgroups than fill the chip splits each query tile's keys over several, so
// that about kExtendFill run (two per CU, what a CU holds at D = 128, the only head_dim that the
// figure was measured at; it holds three at D = 64 and one at D = 256), with at least
// kExtendSplitKeys keys each for the longest request; one split for the whole call, so the
// tiles of shorter requests get ranges without keys. fp32 partials and the decode merge kernel
// put them together. 32/8/128
// bf16, us, one workgroup per tile -> split: 16 new of 8,016 tokens 246 -> 21 (split 31), 8
// requests of 16-64 new of 2,000-4,000 tokens 125 -> 64 (split 5); calls that fill the chip
// keep one (2048 new of 8192 tokens 489 both).
constexpr int kExtendFill = 512;
constexpr int kExtendSplitKeys = 256;
constexpr int kExtendMaxSplit = 32;
constexpr int kExtendMaxReqs = 128;   // requests per launch (their sizes are kernel arguments)

struct ExtendReq {
  int32_t row;     // row of the request-to-token map
  int32_t q0;      // first new token's row of q and out
  int32_t n_new;   // new tokens
  int32_t n_all;   // tokens (prefix and new)
  int32_t tile0;   // first workgroup tile of this request (over all requests)
};

struct ExtendArgs {
  const uint8_t* q;
  const uint8_t* k;
  const uint8_t* v;
  const int32_t* req_to_token;
  uint8_t* out;
  const float* sinks;                  // one fp32 logit per q head, or null
  int64_t q_b, q_h, o_b, o_h;          // bytes
  int64_t k_h, v_h;                    // bytes: kv head
  uint32_t k_s, v_s;                   // bytes: token slot
  int64_t req_stride;                  // elements
  int32_t group, hkv, num_reqs, tiles, window;
  int32_t split;                       // workgroups per query tile, each a range of its keys
  float *part_o, *part_m, *part_l;     // split > 1: row (token * q heads + head) * split + s
  uint32_t num_slots;
  float kscale;                        // log2(e) * softmax scale * K dequantisation scale (> 0)
  float cap_in, cap_out;               // soft-cap: x = cap_out * tanh(q.k * cap_in)
  float vscale;
  ExtendReq req[kExtendMaxReqs];
};

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x16 mfma32(F16, u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32(BF16, u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// 4 consecutive rows' elements of this lane's column: within 16 lanes, lane i passes the
// address of row i/4, elements 4*(i%4).., and receives column i of the 4 rows.
__device__ __forceinline__ u32x2 lds_read_tr(const uint8_t* p) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                       (__attribute__((address_space(3))) i16x4*)p));
}

// Parts of the element type that a weight p = 2^(x - reference) is split into. bf16, 3 parts: 24
// bits of every weight, as its exponents are fp32's; a row's reference follows its running
// maximum. The output's error against float64 is that of fp32 weights (1.660468e-3 of the norm
// at 2048 new of 8192 tokens, 32/8/128), 1e-6 of itself more with 2 parts, which would be 12 %
// faster.
template <class T>
struct ExtendParts {
  static constexpr int n = 3;
};
// fp16, 2 parts: 22 bits of a weight >= 2^-3, steps of 2^-24 below that. So a row's reference
// follows its tiles, up and DOWN (a first token may draw most of the attention, and the fp32
// sums have room): it moves when a tile's largest weight would leave [1, 2^kExtendTop] (fp16
// ends at 2^16), to where that weight is 2^kExtendMid, or 2^kExtendJump where it lies far above
// the tiles before it and perhaps above its neighbours too. Error of the weighted sum against
// float64 in a CPU model of this loop, 8192 keys, one of them with V = 0 and 0 / 14 / 16 / 18
// nats above the others: 3e-7 / 4e-7 / 3e-7 / 5e-7, of fp32 weights 2e-7 / 3e-7 / 4e-7 / 5e-7,
// with the running maximum as reference 3e-7 / 9e-5 / 3e-3 / 7e-2; the output's own rounding is
// 2e-4. Moves are rare but for scores of a wide spread: 2048 new of 8192 tokens, 32/8/128, us,
// running maximum vs this: scores of 1 nat 374 vs 376, of 3 nats 371 vs 388; D = 64 227 vs 229.
template <>
struct ExtendParts<F16> {
  static constexpr int n = 2;
};
constexpr float kExtendTop = 15.5f, kExtendMid = 8.f, kExtendJump = 14.f;
// The reference never moves further down than leaves the row's sum of weights at 2^kExtendRoom:
// values of up to 2^16 times that, over any number of keys, stay far from fp32's 2^128.
constexpr float kExtendRoom = 64.f;

template <class T, int D, bool KV8, bool CAP>
__global__ __launch_bounds__(kExtendThreads, (D == 64 ? 3 : D == 128 ? 2 : 1)) void dk_extend(ExtendArgs a) {
  constexpr int BN = D <= 128 ? 64 : 32;          // keys per tile
  constexpr int RB = 2 * D;                       // bytes per LDS row
  constexpr int TILE = BN * RB;
  constexpr int SCH = D * (KV8 ? 1 : 2) / 16;     // 16-byte chunks per cache row
  constexpr int RPR = kExtendThreads / SCH;       // rows per round of the workgroup's loads
  constexpr int NR = BN / RPR;
  constexpr int KSW = (RB / 16 < 16 ? RB / 16 : 16) - 1;   // K chunk c of row t at c ^ (t & KSW)
  constexpr int VSW = (RB / 32 < 8 ? RB / 32 : 8) - 1;     // V chunk c at c ^ 2 * (t & VSW)
  constexpr int NB = BN / 32;                     // 32-key blocks per tile
  constexpr int DB = D / 32;                      // 32-dim blocks
  constexpr int QK = D / 16;                      // MFMAs per 32-key block
  constexpr int NP = ExtendParts<T>::n;           // parts of p
  __shared__ __attribute__((aligned(16))) uint8_t smem[2][2][TILE];

  const int tid = threadIdx.x, lane = tid & 63, w = uniform(tid >> 6);
  const int h = lane >> 5, c = lane & 31;
  // workgroup -> (kv head, query tile): the kv head is fastest, so with 8 kv heads every XCD
  // streams one head and its L2 holds that head's K and V for all tiles of a request
  const int kvh = (int)blockIdx.x % a.hkv;
  const int t = (int)blockIdx.x / a.hkv;
  int lo = 0, hi = a.num_reqs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.req[mid].tile0 <= t) lo = mid; else hi = mid - 1;
  }
  const ExtendReq rq = a.req[lo];
  const int G = a.group, rows = rq.n_new * G;
  // the last tiles of a request see the most keys: they start first
  const int ntile = (rows + kExtendRows - 1) / kExtendRows;
  const int row0 = (ntile - 1 - (t - rq.tile0)) * kExtendRows;
  const int prefix = rq.n_all - rq.n_new;

  const int row = row0 + 32 * w + c;
  const int rr = min(row, rows - 1);
  const int tok = rr / G, head = rr - tok * G;
  const int pos = prefix + tok;                                  // of this lane's query
  // key range of the workgroup and of this wavefront (uniform)
  const int wrow = min(row0 + 32 * w, rows - 1);
  const int wpos0 = prefix + wrow / G, wpos1 = prefix + min(row0 + 32 * w + 31, rows - 1) / G;
  const bool active = row0 + 32 * w < rows;
  const int bpos0 = prefix + row0 / G, bpos1 = prefix + min(row0 + kExtendRows - 1, rows - 1) / G;
  const int win = a.window > 0 ? a.window : INT32_MAX;
  int kbeg = max(bpos0 - win + 1, 0) / BN;
  int kend = bpos1 / BN + 1;
  if (a.split > 1) {                   // this workgroup's range of key tiles (may be empty)
    const int per = (kend - kbeg + a.split - 1) / a.split;
    kbeg += (int)blockIdx.y * per;
    kend = min(kbeg + per, kend);
  }

  u32x4 qf[QK];
  {
    const uint8_t* qp = a.q + (int64_t)(rq.q0 + tok) * a.q_b + (int64_t)(kvh * G + head) * a.q_h +
                        16 * h;
#pragma unroll
    for (int i = 0; i < QK; ++i) qf[i] = *reinterpret_cast<const u32x4*>(qp + 32 * i);
  }

  const int32_t* map = a.req_to_token + (int64_t)rq.row * a.req_stride;
  const uint8_t* kbase = a.k + (int64_t)kvh * a.k_h;
  const uint8_t* vbase = a.v + (int64_t)kvh * a.v_h;
  const int srow = tid / SCH, sch = tid % SCH;
  int slot[NR];                       // of the tile whose rows are loaded next, as the map holds it
  u32x4 kr[NR], vr[NR];
  int odd;                            // some row of kr / vr is absent or outside the pool
  auto load_slots = [&](int j) {      // past the last key: its slot again
#pragma unroll
    for (int i = 0; i < NR; ++i) slot[i] = map[min(j * BN + i * RPR + srow, rq.n_all - 1)];
  };
  // a slot below 0 counts from the pool's end; outside the pool, slot 0 is read instead
  auto load_tile = [&]() {
    odd = 0;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      uint32_t s = (uint32_t)(slot[i] < 0 ? slot[i] + (int)a.num_slots : slot[i]);
      if (s >= a.num_slots) {
        s = 0u;
        odd |= 1 << i;
      }
      kr[i] = *reinterpret_cast<const u32x4*>(kbase + (uint64_t)s * a.k_s + 16 * sch);
      vr[i] = *reinterpret_cast<const u32x4*>(vbase + (uint64_t)s * a.v_s + 16 * sch);
    }
  };
  // rows of keys past the request's last are zero; a row outside the pool has K = NaN, V = 0,
  // so that every query that attends to it gives NaN
  auto fix_tile = [&](int j) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const bool absent = j * BN + i * RPR + srow >= rq.n_all, out = odd >> i & 1;
      const u32 fill = absent ? 0u : 0xffffffffu;
      kr[i] = absent || out ? u32x4{fill, fill, fill, fill} : kr[i];
      vr[i] = absent || out ? u32x4{0u, 0u, 0u, 0u} : vr[i];
    }
  };
  auto store_tile = [&](int j, uint8_t* kt, uint8_t* vt) {
    if ((j + 1) * BN > rq.n_all || __builtin_amdgcn_ballot_w64(odd != 0)) fix_tile(j);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int r = i * RPR + srow;
      if constexpr (KV8) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          u32x4 kw, vw;
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            kw[2 * x] = T::template from_fp8<false>(kr[i][2 * e + x]);
            kw[2 * x + 1] = T::template from_fp8<true>(kr[i][2 * e + x]);
            vw[2 * x] = T::template from_fp8<false>(vr[i][2 * e + x]);
            vw[2 * x + 1] = T::template from_fp8<true>(vr[i][2 * e + x]);
          }
          const int ch = 2 * sch + e;
          *reinterpret_cast<u32x4*>(kt + r * RB + ((ch ^ (r & KSW)) << 4)) = kw;
          *reinterpret_cast<u32x4*>(vt + r * RB + ((ch ^ (2 * (r & VSW))) << 4)) = vw;
        }
      } else {
        *reinterpret_cast<u32x4*>(kt + r * RB + ((sch ^ (r & KSW)) << 4)) = kr[i];
        *reinterpret_cast<u32x4*>(vt + r * RB + ((sch ^ (2 * (r & VSW))) << 4)) = vr[i];
      }
    }
  };

  f32x16 o[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[b][i] = 0.f;
  float mref = kMinit, lsum = 0.f;

  // lane offsets of the operand reads (see the layouts above)
  const uint32_t koff = (uint32_t)(c * RB + ((h ^ (c & KSW)) << 4));
  const int vi = lane & 15, vdh = (lane >> 4) & 1;
  const int vrow = 4 * h + (vi >> 2);
  uint32_t voff[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b)
    voff[b] = (uint32_t)(vrow * RB + (((4 * b + 2 * vdh + ((vi & 3) >> 1)) ^ (2 * (vrow & VSW))) << 4) +
                         8 * (vi & 1));

  auto compute = [&](int j, const uint8_t* kt, const uint8_t* vt) {
    const int k0 = j * BN;
    f32x16 s[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[n][i] = 0.f;
#pragma unroll
      for (int i = 0; i < QK; ++i) {
        const u32x4 kf =
            *reinterpret_cast<const u32x4*>(kt + 32 * n * RB + (koff ^ (uint32_t)(i << 5)));
        s[n] = mfma32(T{}, kf, qf[i], s[n]);
      }
    }
    const bool edge = k0 + BN - 1 > wpos0 || k0 <= wpos1 - win;
    float mx = kNegInf;
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if constexpr (CAP) s[n][i] = a.cap_out * tanhf(s[n][i] * a.cap_in);
      }
    if (edge) {
#pragma unroll
      for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = k0 + 32 * n + 8 * (i / 4) + 4 * h + (i % 4);
          if (key > pos || key <= pos - win) s[n][i] = kNegInf;
        }
    }
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[n][i]);
    mx = max_xor32(mx);
    if constexpr (!CAP) mx *= a.kscale;
    constexpr bool follow = NP == 2;   // the reference follows the tiles (ExtendParts<F16>)
    const bool move = follow ? fabsf(mx - (mref + kExtendTop / 2)) > kExtendTop / 2
                             : mx > mref + kSlack;
    if (__builtin_amdgcn_ballot_w64(move)) {
      float mn = fmaxf(mref, mx);
      if constexpr (follow) {
        const float to = mx - (mx > mref + kExtendTop + kExtendMid ? kExtendJump : kExtendMid);
        const float room = __builtin_amdgcn_logf(sum_xor32(lsum)) - kExtendRoom;   // log2
        mn = mx > kNegInf ? fmaxf(to, mref + room) : mref;   // no key of the tile seen: stays
      }
      const float al = __builtin_amdgcn_exp2f(mref - mn);
      lsum *= al;
#pragma unroll
      for (int b = 0; b < DB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[b][i] *= al;
      mref = mn;
    }
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        float p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float x = s[n][8 * kk + i];
          p[i] = __builtin_amdgcn_exp2f(CAP ? x - mref : __builtin_fmaf(x, a.kscale, -mref));
        }
        lsum += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        u32x4 pp[NP];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          float r0 = p[2 * x], r1 = p[2 * x + 1];
#pragma unroll
          for (int e = 0; e < NP; ++e) {
            float t0, t1;
            pp[e][x] = T::pack2(r0, r1, &t0, &t1);
            r0 -= t0;
            r1 -= t1;
          }
        }
#pragma unroll
        for (int b = 0; b < DB; ++b) {
          const uint8_t* vp = vt + (32 * n + 16 * kk) * RB + voff[b];
          const u32x2 v0 = lds_read_tr(vp), v1 = lds_read_tr(vp + 8 * RB);
          const u32x4 vf = {v0[0], v0[1], v1[0], v1[1]};
#pragma unroll
          for (int e = 0; e < NP; ++e) o[b] = mfma32(T{}, vf, pp[e], o[b]);
        }
      }
  };

  load_slots(kbeg);
  load_tile();
  load_slots(kbeg + 1);
  store_tile(kbeg, smem[0][0], smem[0][1]);
  __syncthreads();
  for (int j = kbeg; j < kend; ++j) {
    const int cur = (j - kbeg) & 1;
    if (j + 1 < kend) {
      load_tile();
      load_slots(j + 2);
    }
    // a wavefront whose rows see none of the tile's keys skips it
    if (active && j * BN <= wpos1 && j * BN + BN - 1 > wpos0 - win)
      compute(j, smem[cur][0], smem[cur][1]);
    if (j + 1 < kend) store_tile(j + 1, smem[cur ^ 1][0], smem[cur ^ 1][1]);
    __syncthreads();
  }

  lsum = sum_xor32(lsum);
  if (a.split > 1) {
    // relative to this range's reference; dk_merge_split adds the sinks and normalises
    if (row < rows) {
      const int64_t r = ((int64_t)(rq.q0 + tok) * (a.hkv * G) + kvh * G + head) * a.split +
                        blockIdx.y;
#pragma unroll
      for (int b = 0; b < DB; ++b)
#pragma unroll
        for (int x = 0; x < 4; ++x)
          *reinterpret_cast<f32x4*>(a.part_o + r * D + 32 * b + 8 * x + 4 * h) =
              f32x4{o[b][4 * x] * a.vscale, o[b][4 * x + 1] * a.vscale, o[b][4 * x + 2] * a.vscale,
                    o[b][4 * x + 3] * a.vscale};
      if (h == 0) {
        a.part_m[r] = mref * kLn2;
        a.part_l[r] = lsum;
      }
    }
    return;
  }
  if (a.sinks) lsum += __builtin_amdgcn_exp2f(a.sinks[kvh * G + head] * kLog2e - mref);
  const float inv = lsum == 0.f ? 0.f : a.vscale / lsum;
  if (row < rows) {
    uint8_t* op = a.out + (int64_t)(rq.q0 + tok) * a.o_b + (int64_t)(kvh * G + head) * a.o_h;
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        float e0, e1;
        const u32x2 v = {T::pack2(o[b][4 * x] * inv, o[b][4 * x + 1] * inv, &e0, &e1),
                         T::pack2(o[b][4 * x + 2] * inv, o[b][4 * x + 3] * inv, &e0, &e1)};
        *reinterpret_cast<u32x2*>(op + 2 * (32 * b + 8 * x + 4 * h)) = v;
      }
  }
}

// Kernel symbol of one head_dim (dk_extend.hip, compiled once per head_dim)
template <int D>
const void* extend_symbol(bool bf16, bool kv8, bool cap);
extern template const void* extend_symbol<64>(bool, bool, bool);
extern template const void* extend_symbol<128>(bool, bool, bool);
extern template const void* extend_symbol<256>(bool, bool, bool);

}  // namespace dk
