// fp32 mode of the three attention paths (decode, paged multi-query, compression-masked prefill) for gfx950.
//
// Same semantics as the bf16 kernels (decode_attn.hip, paged_prefill.hip, prefill_attn.hip), with fp32 queries,
// keys, values and outputs, fp32 accumulation in a fixed order and accurate expf/logf: the mode the reference's
// PyTorch paths run in fp32 (abridgekv/gen_compress.py:359-360, 555; compresslm_packed_kv.py:608-613;
// compress_forward.py:695-727 under FlexAttention) for tight parity checks. Every product is a fp32 matrix instruction
// (v_mfma_f32_16x16x4_f32: fp32 inputs, fp32 sums). Masked B=1, 3 x (512 + 128) rows, 200 raw prompt rows: 1546 -> 203 us
// a call against one wave per (token, KV head) of VALU dot products with the mask's predicate per key.
#include <cstring>

#include "common.h"

namespace abkv {

struct F32Args {
  const float* q;
  long q_sb, q_st, q_sh;       // masked: [B, S, 32, 128]; paged and decode: [T, 32, 128] (q_sb unused)
  // paged keys (paged and decode): [num_pages, 2, 16, 8, 128]
  const float* kv;
  int num_pages;
  const int32_t* block_table;
  long bt_stride;
  int bt_width;
  // dense keys (masked): [B, S, 8, 128]
  const float* k;
  const float* v;
  long k_sb, k_ss, k_sh, v_sb, v_ss, v_sh;
  // paged: per-request key limits
  const int32_t* tok_req;      // [T] request of every query token
  const int32_t* q_start;      // [B + 1]
  const int32_t* kv_start;     // [B]
  const int32_t* kv_limit;     // [B]
  const int32_t* kv_excluded;  // [B][2] physical [start, end) hidden from the request, or nullptr
  const int32_t* causal;       // [B] or nullptr (causal_default)
  int causal_default;
  // decode
  const int32_t* seq_lens;     // [B]
  int max_pages;
  // masked
  int batch, num_blocks, block_c, codes_k, seq_len;
  const int32_t* prompt_len;   // [B] or nullptr
  const int32_t* head_quota;   // [32] or nullptr
  int retain_tail;             // retained tail T (0: none)
  int tail_policy;             // its policy (kTailStatic, kTailRolling, kTailSticky, kTailRaw)
  int pause_xattn;             // code <-> code attention in a block (kXattn*)
  int pause_passes;            // pause passes of codes_k rows per block
  int copy_rows;               // copy-region rows at the end of the seq_len rows
  int replay_rows;             // replay rows after each block's codes
  int replay_exclude;          // the codes do not see the block's last replay_rows content rows
  int num_tokens;
  int windows, window_parts;   // paged: 16-token windows, workgroups per window and KV head
  float scale;
  float* out;
  long o_sb, o_st, o_sh;
  float* lse;                  // paged and decode: [T, 32]; masked: [B, 32, S]; or nullptr
};

// Unaligned-safe vector access (rows are 4-byte aligned at least).
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ floatx4 ldf4(const float* p) { return *reinterpret_cast<const f32x4u*>(p); }
__device__ __forceinline__ void stf4(float* p, const floatx4& x) { *reinterpret_cast<f32x4u*>(p) = x; }
__device__ __forceinline__ floatx4 mfma16x16x4(float a, float b, const floatx4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int kF32Rows = 16;             // query rows of a workgroup (MFMA columns of each of its waves)
constexpr float kF32Headroom = 8.f;      // the running max moves only when a score exceeds it by more (p <= e^8)

// Scores of 16 keys x 16 columns: s[r] = q(column m16) . k(key 4g + r). The operands' contraction order is dim
// 16c + 4g + e at step (c, e), so a lane's K and Q are 16-byte pieces; two accumulators halve the length of the sums.
__device__ __forceinline__ floatx4 f32_scores(const floatx4 (&kx)[8], const floatx4 (&q)[8]) {
  floatx4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < 8; c += 2)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s0 = mfma16x16x4(kx[c][e], q[c][e], s0);
      s1 = mfma16x16x4(kx[c + 1][e], q[c + 1][e], s1);
    }
  return s0 + s1;
}

// Online softmax of n 16-key score tiles of a wave's columns (hidden scores are -inf), in place: t becomes exp(t - m).
template <int N>
__device__ __forceinline__ void f32_softmax(floatx4 (&t)[N], float& m, float& l, floatx4 (&o)[8]) {
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) mx = fmaxf(mx, t[i][r]);
  if (__any(m == -INFINITY ? mx > -INFINITY : mx > m + kF32Headroom)) {
    const float m_new = fmaxf(m, max_xor32(max_xor16(mx)));
    const float alpha = m == -INFINITY ? 0.f : expf(m - m_new);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] *= alpha;
  }
  float sum = 0.f;                                           // summed before it meets l: short chains round less
#pragma unroll
  for (int i = 0; i < N; ++i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) t[i][r] = t[i][r] == -INFINITY ? 0.f : expf(t[i][r] - m);
    sum += (t[i][0] + t[i][1]) + (t[i][2] + t[i][3]);
  }
  l += sum;
}

// O^T += V^T . P^T over 16 keys: step r contracts the keys 4g + r, which is the order the scores lie in; o[t][r] is the
// dim 64 * (t / 4) + 16g + 4r + t % 4 of column m16. va[r], vb[r]: V row 4g + r, dims 4 * m16 .. + 3 and 64 + those.
__device__ __forceinline__ void f32_pv(const floatx4 (&va)[4], const floatx4 (&vb)[4], const floatx4& p,
                                       floatx4 (&o)[8]) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] = mfma16x16x4(va[r][e], p[r], o[e]);
      o[4 + e] = mfma16x16x4(vb[r][e], p[r], o[4 + e]);
    }
}

__device__ __forceinline__ bool f32_finite(float x) { return fabsf(x) < INFINITY; }

// z stays 0 while all x are finite (four sums: a short chain).
__device__ __forceinline__ void f32_probe(const floatx4& x, floatx4& z) {
#pragma unroll
  for (int e = 0; e < 4; ++e) z[e] = fmaf(x[e], 0.f, z[e]);
}
__device__ __forceinline__ bool f32_odd(const floatx4& z) {
  const float s = (z[0] + z[1]) + (z[2] + z[3]);
  return s != s;
}

// V elements that are infinite or NaN, apart from the product: a key that a column does not see has weight 0 there, but the
// matrix instruction multiplies every key with every column, and 0 x inf is NaN. What 16 keys' such elements give the
// columns that see them (sees(key): this lane's column sees key 0 .. 15) is added to `extra` (this lane's dims of its row,
// each 0, infinite or NaN; the caller has them set to 0 in the operands). load(key, chunk): V row `key` of the 16, dims
// 4 * chunk .. + 3. Rare, and kept low in registers: it must not cost the loop around it an occupancy step.
template <class Sees, class Load>
__device__ __forceinline__ void f32_odd_v(const floatx4& p, Sees sees, float* extra, Load load) {
  const int lane = threadIdx.x & 63, m16 = lane & 15, g = lane >> 4;
#pragma unroll 1
  for (int key = 0; key < 16; ++key) {
    const int r = key & 3;
    const float mine = r == 0 ? p[0] : r == 1 ? p[1] : r == 2 ? p[2] : p[3];
    const float pk = __shfl(mine, 16 * (key >> 2) + m16, 64);
    const bool vis = extra != nullptr && sees(key);
#pragma unroll 1
    for (int i = 0; i < 8; ++i) {                            // dims 16g + 4i .., then 64 + those
      const floatx4 x = load(key, 4 * g + (i & 3) + 16 * (i >> 2));
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (vis && !f32_finite(x[e])) extra[4 * (i & 3) + 64 * (i >> 2) + e] += pk * x[e];
    }
  }
}

// Keys a lane's column sees in a stage: key < lim, or lo <= key < lo + len.
struct F32Span {
  int lim, lo;
  unsigned len;
};
struct F32Stage {
  int k0, end;             // keys k0 .. end - 1 (one stage); rows at or past end are replaced by row end - 1 (weight 0)
  F32Span span;
};

// Stages of kKeys keys of the compression mask: SegWalk's 64-key tiles cut up.
template <int kKeys>
struct MaskedStages {
  const float* k;
  const float* v;
  long k_ss, v_ss;
  SegWalk walk;
  MaskShape g;
  RowFacts row;
  int plen, quota, u;      // u: which of the walk's two head limits is this wave's
  int k0 = 0, left = 0;    // the tile's next stage, keys left in it
  F32Span span;
  __device__ __forceinline__ bool next(F32Stage& st) {
    if (left <= 0) {
      TileMask tm;
      if (!walk.next(k0, tm, false)) return false;
      left = min(kBN, walk.end - k0);
      span = F32Span{tm.mode == 0 ? kNoKey : tm.mode == 1 ? row.q + 1 : u ? tm.limit[1] : tm.limit[0], 0, 0u};
      if (tm.mode == 3) {
        int lo = kNoKey;
        lane_span(g, row, tm.seg, tm.kb, tm.limit[0], tm.limit[1], plen, quota, span.lim, lo);
        span.lo = lo;
        span.len = (unsigned)imax(tm.limit[1] - lo, 0);
      }
    }
    st = F32Stage{k0, min(k0 + kKeys, k0 + left), span};
    k0 += kKeys;
    left -= kKeys;
    return true;
  }
  // K and V rows of half h (rows 16h .. 16h + 15) of a stage
  struct Half {
    const float* k;
    const float* v;
    long k_ss, v_ss;
  };
  __device__ __forceinline__ Half half(const F32Stage& st, int) const {
    return Half{k + (long)st.k0 * k_ss, v + (long)st.k0 * v_ss, k_ss, v_ss};
  }
  __device__ __forceinline__ static int row_of(const F32Stage& st, int row) { return min(row, st.end - 1 - st.k0); }
};

// Stages of kKeys keys of one request's paged keys [0, n_keys) (the largest limit of the rows), with an excluded range.
template <int kKeys>
struct PagedStages {
  const float* kv;         // cache base + head * 128
  const int32_t* table;
  int num_pages, n_keys, k0;
  F32Span span;
  __device__ __forceinline__ bool next(F32Stage& st) {
    if (k0 >= n_keys) return false;
    st = F32Stage{k0, min(k0 + kKeys, n_keys), span};
    k0 += kKeys;
    return true;
  }
  struct Half {
    const float* k;
    const float* v;
    static constexpr long k_ss = kSlotElems, v_ss = kSlotElems;
  };
  __device__ __forceinline__ Half half(const F32Stage& st, int h) const {
    const __attribute__((address_space(4))) int32_t* t = (const __attribute__((address_space(4))) int32_t*)table;
    const int page = min(max(t[min(st.k0 / kPage + h, (st.end - 1) / kPage)], 0), num_pages - 1);
    const float* p = kv + (long)page * kPageElems;
    return Half{p, p + kHalfElems};
  }
  __device__ __forceinline__ static int row_of(const F32Stage& st, int row) {
    return min(st.k0 + row, st.end - 1) & (kPage - 1);
  }
};

// One wave's head over the stages: 16 query rows against K and V stages that the four waves of the workgroup load
// together. The next stage's rows are on their way (in registers) while this one is multiplied. Row r's 16-byte chunk
// c lies at chunk c ^ (r & 15), so both read patterns hit all banks.
// kOdd = false returns whether V held values that are not finite (uniform; one FMA per loaded value): then the result
// holds only if every column sees every key of every stage, and f32_attend walks again with kOdd = true. That one keeps such
// values out of the product and returns whether extra (this lane's dims 16g .. of its output row; nullptr: no row) holds
// sums of f32_odd_v to be added. As a branch of the first walk they cost 5 % (masked, 3 x (512 + 128) rows); so, the look
// costs short walks 3 % (masked, 10 x (128 + 64) rows 141 -> 145 us) and long ones nothing.
template <int kKeys, bool kOdd, class Stages>
__device__ __forceinline__ bool f32_walk(Stages src, float* lds, const floatx4 (&q)[8], float scale, float* extra,
                                           float& m, float& l, floatx4 (&o)[8]) {
  const int tid = threadIdx.x, lane = tid & 63, m16 = lane & 15, g = lane >> 4;
  const int r0 = tid >> 5, chunk = tid & 31;
  constexpr int kHalves = kKeys / 16, kStageElems = kKeys * kHeadDim;
  floatx4 kr[2 * kHalves], vr[2 * kHalves];
  auto load = [&](const F32Stage& st) {
#pragma unroll
    for (int h = 0; h < kHalves; ++h) {
      const auto base = src.half(st, h);
#pragma unroll
      for (int i = 2 * h; i < 2 * h + 2; ++i) {
        const int row = Stages::row_of(st, 8 * i + r0);
        kr[i] = ldf4(base.k + row * base.k_ss + 4 * chunk);
        vr[i] = ldf4(base.v + row * base.v_ss + 4 * chunk);
      }
    }
  };
  floatx4 z = {0.f, 0.f, 0.f, 0.f};                          // 0 while all V values of this thread were finite, else a NaN
  bool dirty = false;                                        // (kOdd) extra holds sums
  auto store = [&](int n) {                                  // buffer n: K rows, then V rows
    if constexpr (!kOdd) {
#pragma unroll
      for (int i = 0; i < 2 * kHalves; ++i) f32_probe(vr[i], z);
    }
    float* kb = lds + 2 * n * kStageElems;
    float* vb = kb + kStageElems;
#pragma unroll
    for (int i = 0; i < 2 * kHalves; ++i) {
      const int row = 8 * i + r0, at = row * kHeadDim + 4 * (chunk ^ (row & 15));
      *reinterpret_cast<floatx4*>(kb + at) = kr[i];
      *reinterpret_cast<floatx4*>(vb + at) = vr[i];
    }
  };
  F32Stage cur, nxt;
  if (!src.next(cur)) return false;
  load(cur);
  store(0);
  __syncthreads();
  for (int n = 0;; n ^= 1) {
    const bool more = src.next(nxt);
    if (more) load(nxt);
    const float* kb = lds + 2 * n * kStageElems;
    float* vb = lds + (2 * n + 1) * kStageElems;
    floatx4 t[kHalves];
    auto sees = [&](int key) {
      return key < cur.end && (key < cur.span.lim || (unsigned)(key - cur.span.lo) < cur.span.len);
    };
#pragma unroll
    for (int i = 0; i < kHalves; ++i) {
      floatx4 kx[8];
#pragma unroll
      for (int c = 0; c < 8; ++c)
        kx[c] = *reinterpret_cast<const floatx4*>(kb + (16 * i + m16) * kHeadDim + 4 * ((4 * c + g) ^ m16));
      t[i] = f32_scores(kx, q);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        t[i][r] = sees(cur.k0 + 16 * i + 4 * g + r) ? t[i][r] * scale : -INFINITY;
      }
    }
    f32_softmax(t, m, l, o);
    if constexpr (kOdd) {
      for (int i = 0; i < 32 && !dirty && extra != nullptr; ++i) extra[(i & 15) + 64 * (i >> 4)] = 0.f;
      dirty = true;
#pragma unroll
      for (int i = 0; i < kHalves; ++i)
        f32_odd_v(t[i], [&](int key) { return sees(cur.k0 + 16 * i + key); }, extra, [&](int key, int c) {
          return *reinterpret_cast<const floatx4*>(vb + (16 * i + key) * kHeadDim + 4 * (c ^ key));
        });
      __syncthreads();                                       // every wave has seen them
      for (int i = tid; i < kStageElems; i += 256) vb[i] = f32_finite(vb[i]) ? vb[i] : 0.f;
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < kHalves; ++i) {
      floatx4 va[4], vb4[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 4 * g + r;
        const float* p = vb + (16 * i + row) * kHeadDim;
        va[r] = *reinterpret_cast<const floatx4*>(p + 4 * (m16 ^ row));
        vb4[r] = *reinterpret_cast<const floatx4*>(p + 4 * ((16 + m16) ^ row));
      }
      f32_pv(va, vb4, t[i], o);
    }
    if (!more) break;
    store(n ^ 1);                            // read last before the barrier that closed the previous stage
    __syncthreads();
    cur = nxt;
  }
  l = sum_xor32(sum_xor16(l));
  return kOdd ? dirty : __syncthreads_or(f32_odd(z)) != 0;
}

template <int kKeys, class Stages>
__device__ __forceinline__ bool f32_attend(const Stages& src, float* lds, const floatx4 (&q)[8], float scale, float* extra,
                                           float& m, float& l, floatx4 (&o)[8]) {
  if (!f32_walk<kKeys, false>(src, lds, q, scale, extra, m, l, o)) return false;
  m = -INFINITY;
  l = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  return f32_walk<kKeys, true>(src, lds, q, scale, extra, m, l, o);
}

__device__ __forceinline__ void f32_load_q(const float* row, int g, bool ok, floatx4 (&q)[8]) {
#pragma unroll
  for (int c = 0; c < 8; ++c) q[c] = ok ? ldf4(row + 16 * c + 4 * g) : floatx4{0.f, 0.f, 0.f, 0.f};
}

// add: the row holds sums of f32_odd_v.
__device__ __forceinline__ void f32_store(float* row, int g, float l, const floatx4 (&o)[8], bool add) {
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float* at = row + 64 * h + 16 * g + 4 * r;
      floatx4 x = floatx4{o[4 * h][r], o[4 * h + 1][r], o[4 * h + 2][r], o[4 * h + 3][r]} * inv;
      if (add) x += ldf4(at);
      stf4(at, x);
    }
}

// The sum in 64 bits: m lies up to the headroom below the largest score, so log(l) alone would round more coarsely.
__device__ __forceinline__ float f32_lse(float m, float l) {
  return l > 0.f ? (float)((double)m + log((double)l)) : -INFINITY;
}

__device__ const float kZeroRow[kHeadDim] = {};

// A wave's share of paged keys, pages w, w + kWaves, ... straight into operand registers (the next page's K loads while this
// page is multiplied). kSpan: the columns see keys of `span`, which may differ; otherwise all of them. Returns (kSpan)
// whether this lane met a V value that is not finite: the sums then hold only if every column sees every key.
template <int kWaves, bool kSpan>
__device__ __forceinline__ bool f32_pages(const float* kv, const int32_t* block_table, int num_pages, int n_keys,
                                           const F32Span& span, float scale, int w, const floatx4 (&q)[8], float& m,
                                           float& l, floatx4 (&o)[8]) {
  const int lane = threadIdx.x & 63, m16 = lane & 15, g = lane >> 4;
  const int n_pages = (n_keys + kPage - 1) / kPage;
  const __attribute__((address_space(4))) int32_t* table = (const __attribute__((address_space(4))) int32_t*)block_table;
  floatx4 kx[8], z = {0.f, 0.f, 0.f, 0.f};
  m = -INFINITY;
  l = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto page_of = [&](int p) { return kv + (long)min(max(table[p], 0), num_pages - 1) * kPageElems; };
  auto load_k = [&](const float* page, int p) {              // rows past the end: the last row (not seen)
    const float* r = page + min(m16, n_keys - 1 - p * kPage) * kSlotElems + 4 * g;
#pragma unroll
    for (int c = 0; c < 8; ++c) kx[c] = ldf4(r + 16 * c);
  };
  if (w < n_pages) {
    const float* page = page_of(w);
    load_k(page, w);
    for (int p = w; p < n_pages; p += kWaves) {
      floatx4 va[4], vb[4], t[1];
#pragma unroll
      for (int r = 0; r < 4; ++r) {                          // rows past the end: zeros (0 x inf is NaN)
        const float* vr = 4 * g + r < n_keys - p * kPage ? page + kHalfElems + (4 * g + r) * kSlotElems : kZeroRow;
        va[r] = ldf4(vr + 4 * m16);
        vb[r] = ldf4(vr + 4 * m16 + 64);
        if constexpr (kSpan) {
          f32_probe(va[r], z);
          f32_probe(vb[r], z);
        }
      }
      t[0] = f32_scores(kx, q);
      if (p + kWaves < n_pages) {
        page = page_of(p + kWaves);
        load_k(page, p + kWaves);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = p * kPage + 4 * g + r;
        const bool vis = kSpan ? key < span.lim || (unsigned)(key - span.lo) < span.len : key < n_keys;
        t[0][r] = vis ? t[0][r] * scale : -INFINITY;
      }
      f32_softmax(t, m, l, o);
      f32_pv(va, vb, t[0], o);
    }
  }
  l = sum_xor32(sum_xor16(l));
  return f32_odd(z);
}

// A lane's sums to a row of 128 dims.
__device__ __forceinline__ void f32_put(float* row, int g, const floatx4 (&o)[8]) {
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *reinterpret_cast<floatx4*>(row + 64 * h + 16 * g + 4 * r) =
          floatx4{o[4 * h][r], o[4 * h + 1][r], o[4 * h + 2][r], o[4 * h + 3][r]};
}

// Up to kNarrowRows rows of one request against a KV head, by the four waves of a workgroup: the 16 columns are 4 heads x 4
// rows, and the waves share the request's pages instead of the heads. A tile of 16 rows by head would leave 12 of 16
// columns empty (16 requests of one row over 5000 keys, one after the other in both forms: 7700 us by head, 2320 so; a wave
// of dot products per token and KV head took 2967). Writes the rows and returns false, or returns true (uniform) and writes
// nothing if V held values that are not finite. lds: 4 x 16 x (128 + 2) floats.
constexpr int kNarrowRows = 4;
__device__ __forceinline__ bool f32_narrow(const F32Args& a, float* lds, const F32Span& span, int n_keys, int b, int kvh,
                                           int t, int t1) {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, m16 = lane & 15, g = lane >> 4;
  const int row = t + (m16 & 3);
  floatx4 q[8], o[8];
  float m, l;
  f32_load_q(a.q + (long)min(row, t1 - 1) * a.q_st + (long)(kvh * kGroup + (m16 >> 2)) * a.q_sh, g, row < t1, q);
  const bool odd = f32_pages<4, true>(a.kv + kvh * kHeadDim, a.block_table + (long)b * a.bt_stride, a.num_pages, n_keys,
                                      span, a.scale, w, q, m, l, o);
  float* ml = lds + 4 * 16 * kHeadDim;
  f32_put(lds + (w * 16 + m16) * kHeadDim, g, o);
  if (g == 0) *reinterpret_cast<float2*>(ml + 2 * (w * 16 + m16)) = make_float2(m, l);
  if (__syncthreads_or(odd)) return true;
  const int col = threadIdx.x >> 4, d = 8 * (threadIdx.x & 15), out_row = t + (col & 3);
  float M = -INFINITY, L = 0.f;
  floatx4 x = {0.f, 0.f, 0.f, 0.f}, y = x;
  float2 rec[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    rec[i] = *reinterpret_cast<const float2*>(ml + 2 * (i * 16 + col));
    M = fmaxf(M, rec[i].x);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float f = rec[i].x == M ? 1.f : expf(rec[i].x - M);          // (both -inf: sums of 0 or of NaN)
    const float* p = lds + (i * 16 + col) * kHeadDim + d;
    L += rec[i].y * f;
    x += *reinterpret_cast<const floatx4*>(p) * f;
    y += *reinterpret_cast<const floatx4*>(p + 4) * f;
  }
  if (out_row < t1) {
    const int head = kvh * kGroup + (col >> 2);
    const float inv = L > 0.f ? 1.f / L : 0.f;
    float* out = a.out + (long)out_row * a.o_st + (long)head * a.o_sh + d;
    stf4(out, x * inv);
    stf4(out + 4, y * inv);
    if (a.lse != nullptr && d == 0) a.lse[(long)out_row * kHeadsQ + head] = f32_lse(M, L);
  }
  return false;
}

// Multi-query attention, masked (kMasked) or paged: a workgroup of 4 waves takes 16 query rows of one KV head, one query
// head per wave. Bound by the fp32 matrix rate (16x16x4: 256 flop per clock and CU). Matrix instructions, LDS stages
// shared by the four heads and the segment walk instead of VALU dot products per key with the mask's predicate per
// element: masked, B=1, 3 x (512 + 128) rows 1546 -> 203 us; a code step of 256 rows over 4000 keys 1909 -> 397 us.
template <bool kMasked, int kKeys>
__global__ __launch_bounds__(256, kKeys == 16 ? 3 : 2) void attn_f32_rows_kernel(F32Args a) {
  static_assert(kMasked || 4 * kKeys * kHeadDim >= 4 * 16 * (kHeadDim + 2), "f32_narrow");
  __shared__ __attribute__((aligned(16))) float lds[4 * kKeys * kHeadDim];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, m16 = lane & 15, g = lane >> 4;
  const int kvh = blockIdx.x % kHeadsKV;
  const int head = kvh * kGroup + w;
  floatx4 q[8], o[8];
  float m = -INFINITY, l = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  if constexpr (kMasked) {
    const int rank = blockIdx.x / kHeadsKV;                  // later (costlier) rows first, every sequence of a rank
    const int b = rank % a.batch;
    const int q0 = ((a.seq_len + kF32Rows - 1) / kF32Rows - 1 - rank / a.batch) * kF32Rows;
    const int qrow = q0 + m16;
    const int plen = a.prompt_len ? a.prompt_len[b] : 0;
    int qmin = kNoKey, qmax = 0, quota = 0;
#pragma unroll
    for (int u = 0; u < kGroup; ++u) {
      const int x = a.head_quota ? a.head_quota[kvh * kGroup + u] : a.codes_k;
      qmin = min(qmin, x);
      qmax = max(qmax, x);
      if (u == w) quota = x;
    }
    const MaskShape g_ = {a.seq_len, a.block_c, a.codes_k, a.pause_passes, a.replay_rows, a.copy_rows,
                          a.block_c + a.pause_passes * a.codes_k + a.replay_rows, a.num_blocks, a.retain_tail,
                          a.tail_policy, a.pause_xattn, a.replay_exclude != 0};
    f32_load_q(a.q + (long)b * a.q_sb + (long)min(qrow, a.seq_len - 1) * a.q_st + (long)head * a.q_sh, g,
               qrow < a.seq_len, q);
    MaskedStages<kKeys> src{a.k + (long)b * a.k_sb + (long)kvh * a.k_sh, a.v + (long)b * a.v_sb + (long)kvh * a.v_sh,
                     a.k_ss, a.v_ss,
                     SegWalk(g_, q0, min(q0 + kF32Rows, a.seq_len) - 1, plen, qmin, qmax, quota, quota), g_,
                     row_facts(g_, qrow), plen, quota, 0};
    float* out = a.out + (long)b * a.o_sb + (long)qrow * a.o_st + (long)head * a.o_sh;
    const bool add = f32_attend<kKeys>(src, lds, q, a.scale, qrow < a.seq_len ? out + 16 * g : nullptr, m, l, o);
    if (qrow >= a.seq_len) return;
    f32_store(out, g, l, o, add);
    if (a.lse != nullptr && g == 0) a.lse[((long)b * kHeadsQ + head) * a.seq_len + qrow] = f32_lse(m, l);
  } else {
    // windows of 16 consecutive tokens; a window's requests go to window_parts workgroups in turn (all uniform)
    const int window = blockIdx.x / kHeadsKV % a.windows, part = blockIdx.x / kHeadsKV / a.windows;
    const int t0 = window * kF32Rows, t_end = min(t0 + kF32Rows, a.num_tokens);
    const int my_req = a.tok_req[min(t0 + m16, t_end - 1)];
    for (int t = t0, t1, turn = 0; t < t_end; t = t1, ++turn) {
      const int b = __builtin_amdgcn_readlane(my_req, t - t0);
      // tokens of this request from t on (lanes 0 .. 15 hold the window's requests)
      const unsigned differs = (unsigned)__ballot(my_req != b) & 0xffffu & (~0u << (t - t0));
      t1 = min(differs ? t0 + __ffs(differs) - 1 : t_end, t_end);
      if (turn % a.window_parts != part) continue;
      const int n = t1 - t;
      const int pos = a.kv_start[b] + t - a.q_start[b];      // position of row t
      const int limit = min(a.kv_limit[b], a.bt_width * kPage);
      const bool causal = a.causal ? a.causal[b] != 0 : a.causal_default != 0;
      const int n_keys = causal ? min(limit, pos + n) : limit;
      auto span_of = [&](int i) {                            // keys that row t + i sees
        const int lim = i >= n ? 0 : causal ? min(limit, pos + i + 1) : limit;
        F32Span span{lim, 0, 0u};
        if (a.kv_excluded != nullptr) {
          const int lo = a.kv_excluded[2 * b], hi = a.kv_excluded[2 * b + 1];
          if (lo < hi) span = F32Span{min(lim, lo), hi, (unsigned)max(lim - hi, 0)};
        }
        return span;
      };
      if (n > kNarrowRows || f32_narrow(a, lds, span_of(m16 & 3), n_keys, b, kvh, t, t1)) {
        const int row = t + m16;                             // this lane's token (valid below t1)
        f32_load_q(a.q + (long)min(row, t1 - 1) * a.q_st + (long)head * a.q_sh, g, row < t1, q);
        PagedStages<kKeys> src{a.kv + kvh * kHeadDim, a.block_table + (long)b * a.bt_stride, a.num_pages, n_keys, 0,
                               span_of(m16)};
        float* out = a.out + (long)row * a.o_st + (long)head * a.o_sh;
        const bool add = f32_attend<kKeys>(src, lds, q, a.scale, row < t1 ? out + 16 * g : nullptr, m, l, o);
        if (row < t1) {
          f32_store(out, g, l, o, add);
          if (a.lse != nullptr && g == 0) a.lse[(long)row * kHeadsQ + head] = f32_lse(m, l);
        }
        m = -INFINITY;
        l = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
      __syncthreads();                                       // the next request's first stage overwrites this one's
    }
  }
}

// Decode: a workgroup of 8 waves per (sequence, KV head); the waves share the pages (f32_pages) and their partial results
// meet in LDS. The four heads fill the 16 columns four times over: the path is bound by memory, not by the matrix rate. 32
// sequences of 900 .. 9500 rows 7014 -> 286 us (4.8 TB/s), one of 5000 rows 2102 -> 108 us, against the VALU form of one
// wave each.
constexpr int kDecWaves = 8;
__global__ __launch_bounds__(64 * kDecWaves, 2) void decode_f32_kernel(F32Args a) {
  __shared__ __attribute__((aligned(16))) float po[kDecWaves][kGroup][kHeadDim];
  __shared__ float pm[kDecWaves][kGroup], pl[kDecWaves][kGroup];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, m16 = lane & 15, g = lane >> 4;
  const int kvh = blockIdx.x % kHeadsKV, b = blockIdx.x / kHeadsKV;
  const int n_keys = max(min(a.seq_lens[b], a.max_pages * kPage), 0);
  floatx4 q[8], o[8];
  f32_load_q(a.q + (long)b * a.q_st + (long)(kvh * kGroup + (m16 & 3)) * a.q_sh, g, true, q);
  float m, l;
  f32_pages<kDecWaves, false>(a.kv + kvh * kHeadDim, a.block_table + (long)b * a.bt_stride, a.num_pages, n_keys, F32Span{},
                              a.scale, w, q, m, l, o);
  if (m16 < kGroup) {
    f32_put(po[w][m16], g, o);
    if (g == 0) {
      pm[w][m16] = m;
      pl[w][m16] = l;
    }
  }
  __syncthreads();
  const int u = threadIdx.x / kHeadDim, d = threadIdx.x % kHeadDim;   // 512 threads: 4 heads x 128 dims
  float M = -INFINITY, L = 0.f, acc = 0.f;
#pragma unroll
  for (int i = 0; i < kDecWaves; ++i) M = fmaxf(M, pm[i][u]);
#pragma unroll
  for (int i = 0; i < kDecWaves; ++i) {
    if (pl[i][u] == 0.f && pm[i][u] == -INFINITY) continue;           // a wave that had no page
    const float f = expf(pm[i][u] - M);
    L += pl[i][u] * f;
    acc += po[i][u][d] * f;
  }
  const int head = kvh * kGroup + u;
  a.out[(long)b * a.o_st + (long)head * a.o_sh + d] = acc * (L > 0.f ? 1.f / L : 0.f);   // (sums of NaN stay NaN)
  if (a.lse != nullptr && d == 0) a.lse[(long)b * kHeadsQ + head] = f32_lse(M, L);
}

// Workgroups of the row kernels: 8 KV heads x (16-row tiles); 0 when the work items would not fit the grid.
static unsigned f32_grid(long tiles) {
  const long n = tiles * kHeadsKV;
  return n <= 0 || n * 256 > 0xFFFFFFFFL ? 0u : (unsigned)n;
}

static F32Args f32_defaults() {
  F32Args a;
  memset(&a, 0, sizeof(a));
  return a;
}

}  // namespace abkv

extern "C" {

int abkv_decode_attn_f32(const float* q, long q_stride_seq, long q_stride_head, const float* kv_cache, int num_pages,
                         const int32_t* block_table, long block_table_stride, const int32_t* seq_lens, int num_seqs,
                         int max_pages_per_seq, float scale, float* out, long out_stride_seq, long out_stride_head,
                         float* lse, hipStream_t stream) {
  using namespace abkv;
  if (num_seqs <= 0) return 0;
  if (q == nullptr || kv_cache == nullptr || block_table == nullptr || seq_lens == nullptr || out == nullptr ||
      num_pages <= 0 || max_pages_per_seq <= 0 || block_table_stride < max_pages_per_seq)
    return (int)hipErrorInvalidValue;
  F32Args a = f32_defaults();
  a.q = q;
  a.q_st = q_stride_seq;
  a.q_sh = q_stride_head;
  a.kv = kv_cache;
  a.num_pages = num_pages;
  a.block_table = block_table;
  a.bt_stride = block_table_stride;
  a.seq_lens = seq_lens;
  a.max_pages = max_pages_per_seq;
  a.num_tokens = num_seqs;
  a.scale = scale;
  a.out = out;
  a.o_st = out_stride_seq;
  a.o_sh = out_stride_head;
  a.lse = lse;
  if ((long)num_seqs * kHeadsKV * 64 * kDecWaves > 0xFFFFFFFFL) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(decode_f32_kernel, dim3((unsigned)num_seqs * kHeadsKV), dim3(64 * kDecWaves), 0, stream, a);
  return (int)hipGetLastError();
}

int abkv_paged_prefill_attn_f32(const float* q, long q_stride_t, long q_stride_h, const float* kv_cache, int num_pages,
                                const int32_t* block_table, long block_table_stride, int block_table_width,
                                const int32_t* q_start, const int32_t* kv_start, const int32_t* kv_limit,
                                const int32_t* kv_excluded, const int32_t* tok_req, int num_tokens,
                                const int32_t* causal, int causal_default, float scale, float* out, long out_stride_t,
                                long out_stride_h, float* lse, hipStream_t stream) {
  using namespace abkv;
  if (num_tokens <= 0) return 0;
  if (q == nullptr || kv_cache == nullptr || block_table == nullptr || q_start == nullptr || kv_start == nullptr ||
      kv_limit == nullptr || tok_req == nullptr || out == nullptr || num_pages <= 0 || block_table_width <= 0)
    return (int)hipErrorInvalidValue;
  F32Args a = f32_defaults();
  a.q = q;
  a.q_st = q_stride_t;
  a.q_sh = q_stride_h;
  a.kv = kv_cache;
  a.num_pages = num_pages;
  a.block_table = block_table;
  a.bt_stride = block_table_stride;
  a.bt_width = block_table_width;
  a.q_start = q_start;
  a.kv_start = kv_start;
  a.kv_limit = kv_limit;
  a.kv_excluded = kv_excluded;
  a.tok_req = tok_req;
  a.causal = causal;
  a.causal_default = causal_default;
  a.num_tokens = num_tokens;
  a.scale = scale;
  a.out = out;
  a.o_st = out_stride_t;
  a.o_sh = out_stride_h;
  a.lse = lse;
  // A window may hold rows of up to 16 requests, which one workgroup would walk one after the other: 16 workgroups a window
  // where windows are few, 4 where they fill the GPU anyway. A workgroup that finds no request left ends at once: a code
  // step and a prompt of 2000 rows take the same with 1, 4 or 16. us with 16 / 4 / 1: 16 requests of one row over 5000
  // keys 159 / - / 2320, 256 over 2000 500 / - / 991, 1024 over 500 548 / 528 / 525, 2048 over 300 688 / 656 / 645.
  const long windows = ((long)num_tokens + kF32Rows - 1) / kF32Rows;
  a.windows = (int)windows;
  a.window_parts = windows <= 32 ? 16 : f32_grid(4 * windows) != 0 ? 4 : 1;
  const unsigned grid = f32_grid(windows * a.window_parts);
  if (grid == 0) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL((attn_f32_rows_kernel<false, 32>), dim3(grid), dim3(256), 0, stream, a);
  return (int)hipGetLastError();
}

int abkv_prefill_masked_attn_f32(const float* q, long q_sb, long q_ss, long q_sh, const float* k, long k_sb,
                                 long k_ss, long k_sh, const float* v, long v_sb, long v_ss, long v_sh, int batch,
                                 int block_c, int codes_k, int num_blocks, int seq_len, const int32_t* prompt_len,
                                 const int32_t* head_quota, int retain_tail, int tail_policy, int pause_xattn,
                                 int pause_passes, int copy_rows, int replay_rows, int replay_exclude, float scale,
                                 float* out, long o_sb, long o_ss, long o_sh, float* lse,
                                 hipStream_t stream) {
  using namespace abkv;
  if (batch <= 0 || seq_len <= 0) return 0;
  if (q == nullptr || k == nullptr || v == nullptr || out == nullptr || block_c <= 0 || codes_k < 0 ||
      num_blocks <= 0 || pause_passes <= 0 || copy_rows < 0 || (codes_k == 0 && (pause_passes != 1 || copy_rows)) ||
      replay_rows < 0 || replay_rows > block_c || (replay_rows && (retain_tail || codes_k == 0)) ||
      (replay_exclude && (replay_rows <= 0 || replay_rows >= block_c)) ||
      (long)seq_len != (long)num_blocks * (block_c + (long)pause_passes * codes_k + replay_rows) + copy_rows ||
      retain_tail < 0 ||
      retain_tail > block_c || (retain_tail == block_c && tail_policy != kTailRaw) ||
      tail_policy < kTailStatic || tail_policy > kTailRaw || pause_xattn < kXattnFull ||
      pause_xattn > kXattnNone)
    return (int)hipErrorInvalidValue;
  F32Args a = f32_defaults();
  a.q = q;
  a.q_sb = q_sb;
  a.q_st = q_ss;
  a.q_sh = q_sh;
  a.k = k;
  a.v = v;
  a.k_sb = k_sb;
  a.k_ss = k_ss;
  a.k_sh = k_sh;
  a.v_sb = v_sb;
  a.v_ss = v_ss;
  a.v_sh = v_sh;
  a.block_c = block_c;
  a.codes_k = codes_k;
  a.seq_len = seq_len;
  a.prompt_len = prompt_len;
  a.head_quota = head_quota;
  a.retain_tail = retain_tail;
  a.tail_policy = tail_policy;
  a.pause_xattn = pause_xattn;
  a.pause_passes = pause_passes;
  a.copy_rows = copy_rows;
  a.replay_rows = replay_rows;
  a.replay_exclude = replay_exclude;
  a.batch = batch;
  a.num_blocks = num_blocks;
  a.scale = scale;
  a.out = out;
  a.o_sb = o_sb;
  a.o_st = o_ss;
  a.o_sh = o_sh;
  a.lse = lse;
  const unsigned grid = f32_grid(((long)seq_len + kF32Rows - 1) / kF32Rows * batch);
  if (grid == 0) return (int)hipErrorInvalidValue;
  // Stages of 16 keys (three workgroups a CU) where blocks have codes: segments are short, their last stage partly empty;
  // of 32 (two, half the barriers) for one long causal walk. 16 / 32 by events: 3 x (512 + 128) rows 209 / 229 us,
  // 6 x (200 + 2 x 40) 107 / 133; causal 1337 rows 209 / 181, and a paged code step over 4000 keys 7 % slower with 16.
  if (codes_k > 0) hipLaunchKernelGGL((attn_f32_rows_kernel<true, 16>), dim3(grid), dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((attn_f32_rows_kernel<true, 32>), dim3(grid), dim3(256), 0, stream, a);
  return (int)hipGetLastError();
}

}  // extern "C"
