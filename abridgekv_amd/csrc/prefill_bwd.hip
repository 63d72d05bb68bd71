// Backward pass (gradients of q, k, v through the same mask), the FlashAttention-2 decomposition with the forward's
// LSE: P = exp2(S * scale * log2(e) - lse * log2(e)), dS = P o (dP - rowsum(dO o O)), dQ = scale * dS K,
// dK = scale * dS^T Q, dV = P^T dO. The reference trains through FlexAttention's backward of the same mask
// (abridgekv/compress_forward.py:1134-1230 called under autograd, :1329).
//   prefill_bwd_prep_kernel  per (row, query head): lse2 = lse * log2(e) and D = sum_d dO * O, in a workspace padded
//                            to whole 64-row tiles (lse2 = +inf and D = 0 past S0, so padded rows weigh 0)
//   prefill_bwd_dq_kernel    the forward's work decomposition and tile walk (query tile x KV head; wave = 16 rows x
//                            2 heads); per key tile S^T = K Q^T and dP^T = V dO^T, dQ^T += K^T dS^T
//   prefill_bwd_dkv_kernel   roles swapped: workgroup = 64 keys of a KV head, wave = 16 keys; the (query tile, head)
//                            pairs that see the key tile are staged in LDS (Q, dO, lse2, D); S = Q K^T and
//                            dP = dO V^T as the forward's score tiles, dV^T += dO^T P and dK^T += Q^T dS as its PV step.
//                            A key is seen by at most two ranges of query rows in every layout (key_span), so one
//                            instance serves all of them and a mask test is two range tests per element: 3220 -> 583 us
//                            (layouts off the 64-row grid, B=1, 8 x (512 + 128 + 16 rows)); on the grid, where it
//                            replaced a classification per tile pair, 988 -> 965 us (B=2, 12 x (512 + 128 rows))
#include "prefill_common.h"

#include "bwd_plan.h"

namespace abkv {

struct PrefillBwdArgs {
  PrefillArgs f;                              // q, k, v, geometry, prompt_len, head_quota, scale_log2
  const __bf16* o;    long o_sb, o_ss, o_sh;  // forward output [B, S0, 32, 128]
  const __bf16* dout; long g_sb, g_ss, g_sh;  // its gradient
  const float* lse;                           // [B, 32, S0] natural log, from the forward
  float* lse2;                                // workspace [B, 32, S0p]
  float* dvec;                                // workspace [B, 32, S0p]
  int S0p;                                    // S0 rounded up to a multiple of 64
  int* seen;                                  // [key tiles x B] query tiles that see the key tile (workspace, as the next
                                              // two); nullptr: no parts, one workgroup per key tile in tile order
  int* done;                                  // [slot_cap x 8] finished parts, at the tile's first item
  float* slots;                               // [slot_cap x 8][kSlotFloats] sums of the parts
  int slot_cap;                               // partial slots per KV head
  int workers;                                // workgroups of the dK/dV kernel the GPU runs at once, per KV head
  int count_blocks;                           // workgroups of the prep kernel that count
  float scale;                                // softmax scale
  __bf16* dq; long dq_sb, dq_ss, dq_sh;       // [B, S0, 32, 128]
  __bf16* dk; long dk_sb, dk_ss, dk_sh;       // [B, S0, 8, 128]
  __bf16* dv; long dv_sb, dv_ss, dv_sh;
};

// f over the wave's lanes (uniform), in VALU (DPP inside rows of 16 lanes, then lane swaps): a TileSpan is twelve of these,
// and as chains of LDS permutes they cost 3.5 us a key tile.
template <class F>
__device__ __forceinline__ int wave_all(int v, F f) {
  v = f(v, __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xF, 0xF, false));      // quad_perm 1,0,3,2
  v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xF, 0xF, false));      // quad_perm 2,3,0,1
  v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xF, 0xF, false));     // row_half_mirror
  v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x140, 0xF, 0xF, false));     // row_mirror
  const auto r16 = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = f((int)r16[0], (int)r16[1]);
  const auto r32 = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return __builtin_amdgcn_readfirstlane(f((int)r32[0], (int)r32[1]));
}
__device__ __forceinline__ int wave_min(int v) { return wave_all(v, [](int a, int b) { return min(a, b); }); }
__device__ __forceinline__ int wave_sum(int v) { return wave_all(v, [](int a, int b) { return a + b; }); }

// Which query tiles a 64-key tile is seen by, from the query ranges of its keys (lane l: key k0 + l; wave-uniform and
// the same in every wave): a query tile outside the hulls of the ranges is hidden, one inside the common part of the
// first (or of the second) ranges of all 64 keys is visible throughout, the others take the ranges per key.
struct TileSpan {
  int a1, e1, a2, e2;        // hulls over the keys that are no codes
  int ca, ce;                // hull over the codes
  int f1, g1, f2, g2;        // [f1, g1) and [f2, g2): rows that see every key (given the quota)
  int slot_min, slot_max;    // of the codes
  __device__ __forceinline__ explicit TileSpan(const KeySpan& s) {
    const bool code = s.slot >= 0;
    const bool r1 = s.a1 < s.e1, r2 = s.a2 < s.e2;
    a1 = wave_min(!code && r1 ? s.a1 : kNoKey);
    e1 = -wave_min(!code && r1 ? -s.e1 : 0);
    a2 = wave_min(!code && r2 ? s.a2 : kNoKey);
    e2 = -wave_min(!code && r2 ? -s.e2 : 0);
    ca = wave_min(code && r1 ? s.a1 : code && r2 ? s.a2 : kNoKey);
    ce = -wave_min(code ? -max(s.e1, s.e2) : 0);
    f1 = -wave_min(-s.a1);
    g1 = wave_min(s.e1);
    f2 = -wave_min(-s.a2);
    g2 = wave_min(s.e2);
    slot_min = wave_min(code ? s.slot : kNoKey);
    slot_max = -wave_min(-s.slot);
  }
  __device__ __forceinline__ int first_row() const { return min(min(a1, a2), ca); }
  __device__ __forceinline__ int last_row() const { return max(max(e1, e2), ce); }
  // -1 hidden, 0 every pair visible, 1 per key
  __device__ __forceinline__ int mode(int q0, int q1, int quota) const {
    const bool seen = (q0 < e1 && q1 > a1) || (q0 < e2 && q1 > a2) || (slot_min < quota && q0 < ce && q1 > ca);
    if (!seen) return -1;
    return ((q0 >= f1 && q1 <= g1) || (q0 >= f2 && q1 <= g2)) && slot_max < quota ? 0 : 1;
  }
};

// Work of the dK/dV kernel. A key tile's cost is the query tiles that see it: a block's content is seen by its own block
// only, its codes and the raw prompt by all later rows, so a launch of one workgroup per key tile can wait for the first
// codes' workgroup. Tiles longer than 3/2 of a worker's even share of the launch are split into parts of at most the
// share; the parts leave fp32 sums in slots, and the last part to finish adds them up in part order. Parts and long tiles
// go first. The prep kernel counts (the raw prompt's length is not known on the host), each dK/dV workgroup finds its
// part from the counts. Backward calls in us, one workgroup per tile in tile order -> this: B=1, 8 x (512 + 128 + 16) rows
// (82 query tiles against a share of 16) 829 -> 508, 4 x (512 + 128) 277 -> 152, causal 1500 rows 267 -> 230; B=2,
// 4 x (512 + 256) with a rolling tail 466 -> 399; B=2, 12 x (512 + 128) (120 against 82: not split, only ordered)
// 1242 -> 1119, and parts of 3/4 of the share there, which lose the reuse of query tiles in L2, 4 % slower. A least part of
// 8 instead of 12 query tiles: causal 1500 rows 6 % slower.
static_assert(kSlotFloats == 2 * kBN * kHeadDim && kHeadsQ == 32 && kHeadsKV == 8, "bwd_plan.h");
// One part: parts == 1: the whole tile.
struct DkvItem {
  int tile;                  // key tile * B + sequence
  int z, parts, seen;        // part z of parts; query tiles that see the tile
  int first;                 // the tile's first slot
};

// Largest code quota of all heads.
__device__ __forceinline__ int quota_max(const PrefillArgs& f) {
  return f.head_quota ? -wave_min(-f.head_quota[threadIdx.x & (kHeadsQ - 1)]) : f.K;
}

// The query tiles qt0 .. qt0 + 63 that see the key tile for some head (bit i: tile qt0 + i).
__device__ __forceinline__ unsigned long long seen_mask(const PrefillArgs& f, const TileSpan& span, int qt0, int quota) {
  const int qt = qt0 + (int)(threadIdx.x & 63);
  return __ballot(qt * kBN < f.S0 && span.mode(qt * kBN, min(qt * kBN + kBN, f.S0), quota) >= 0);
}

// Sum of v over the workgroup's 256 threads (uniform).
__device__ __forceinline__ int block_sum(int v, int* lds) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  return lds[0] + lds[1] + lds[2] + lds[3];
}

// Order of issue: 0 the split tiles' parts, then whole tiles by length: 1 over the share, 2 over half of it, 3 the rest.
__device__ __forceinline__ int dkv_class(int seen, int share) {
  return dkv_parts(seen, share) > 1 ? 0 : seen > share ? 1 : 2 * seen > share ? 2 : 3;
}

// Item i of a KV head (workgroup of 256 threads; uniform), by class and tile; false past the last. With no tile over the
// share there is no tail to shorten, and the items are the tiles in their order, which reuses query tiles in L2: B=4,
// 16 x (512 + 128) rows 3345 us a backward against 3430 by class.
__device__ __forceinline__ bool dkv_item(const int* seen, int tiles, int workers, int i, DkvItem& item) {
  __shared__ int lds[4];
  __shared__ int2 whole[4];
  __shared__ DkvItem found;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  int v = 0, longest = 0;
  for (int e = tid; e < tiles; e += 256) {
    v += seen[e];
    longest = max(longest, seen[e]);
  }
  v = wave_sum(v);
  longest = -wave_min(-longest);
  if (lane == 0) whole[w] = make_int2(v, longest);
  __syncthreads();
  const int share = dkv_share(whole[0].x + whole[1].x + whole[2].x + whole[3].x, workers);
  if (max(max(whole[0].y, whole[1].y), max(whole[2].y, whole[3].y)) <= share) {
    item = DkvItem{i, 0, 1, 0, 0};
    return i < tiles;
  }
  int at = 0, cls = 0, n = 0;                                // the class that item i lies in: items at .. at + n - 1
  for (; cls < 4; ++cls) {
    v = 0;
    for (int e = tid; e < tiles; e += 256) v += dkv_class(seen[e], share) == cls ? dkv_parts(seen[e], share) : 0;
    n = block_sum(v, lds);
    if (i < at + n) break;                                   // uniform
    at += n;
  }
  if (cls == 4) return false;
  for (int e0 = 0; e0 < tiles; e0 += 256) {
    const int e = e0 + tid;
    const int mine = e < tiles && dkv_class(seen[e], share) == cls ? dkv_parts(seen[e], share) : 0;
    int scan = mine;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
      const int up = __shfl_up(scan, m, 64);
      scan += lane >= m ? up : 0;
    }
    __syncthreads();
    if (lane == 63) lds[w] = scan;
    __syncthreads();
    int before = at + scan - mine;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      before += k < w ? lds[k] : 0;
      at += lds[k];
    }
    if (i >= before && i < before + mine) found = DkvItem{e, i - before, mine, seen[e], before};
    if (i < at) break;                                      // uniform
  }
  __syncthreads();
  item = found;
  return true;
}

// Prep's part of it: four key tiles a workgroup, one per wave.
__device__ __forceinline__ void dkv_count(const PrefillBwdArgs& a, int block) {
  const PrefillArgs& f = a.f;
  const int lane = threadIdx.x & 63;
  const int e = 4 * block + (threadIdx.x >> 6);
  if (block == 0)
    for (int i = threadIdx.x; i < a.slot_cap * kHeadsKV; i += 256) a.done[i] = 0;
  if (e >= f.num_q_tiles * f.B) return;
  const int b = e % f.B, k0 = e / f.B * kBN;
  const TileSpan span(key_span(mask_shape(f), k0 + lane, f.prompt_len ? f.prompt_len[b] : 0));
  const int quota = quota_max(f);
  int n = 0;
  for (int qt = span.first_row() / kBN; qt * kBN < span.last_row(); qt += 64)
    n += __popcll(seen_mask(f, span, qt, quota));
  if (lane == 0) a.seen[e] = n;
}

__global__ __launch_bounds__(256) void prefill_bwd_prep_kernel(PrefillBwdArgs a) {
  // 16 lanes per (row, query head): lane c takes dims 8c .. 8c + 7 of O and dO (one 16-byte load each, so a wave reads
  // four whole 256-byte rows), and the 16 partial dot products are summed by lane shuffles inside the group
  if ((int)blockIdx.x < a.count_blocks) return dkv_count(a, blockIdx.x);
  const long idx = ((long)((int)blockIdx.x - a.count_blocks) * 256 + threadIdx.x) >> 4;
  const int c = threadIdx.x & 15;
  if (idx >= (long)a.f.B * kHeadsQ * a.S0p) return;         // uniform over the 16 lanes of a row
  const int i = (int)(idx % a.S0p);
  const long bh = idx / a.S0p;
  const int h = (int)(bh % kHeadsQ), b = (int)(bh / kHeadsQ);
  float d = 0.f;
  if (i < a.f.S0) {
    const __bf16* op = a.o + (long)b * a.o_sb + (long)i * a.o_ss + (long)h * a.o_sh;
    const __bf16* gp = a.dout + (long)b * a.g_sb + (long)i * a.g_ss + (long)h * a.g_sh;
    const u32x4 x = ld16g(op + 8 * c), y = ld16g(gp + 8 * c);
#pragma unroll
    for (int e = 0; e < 4; ++e) d += bf16_lo(x[e]) * bf16_lo(y[e]) + bf16_hi(x[e]) * bf16_hi(y[e]);
  }
#pragma unroll
  for (int m = 1; m < 16; m <<= 1) d += __shfl_xor(d, m, 64);
  if (c != 0) return;
  a.lse2[idx] = i < a.f.S0 ? a.lse[bh * a.f.S0 + i] * 1.4426950408889634f : INFINITY;
  a.dvec[idx] = d;
}

// acc[t][u] += A^T . B^T over one 64-row tile: A^T operands by LDS transpose reads of the tile, B^T the packed bf16
// operands (the forward's PV step without its row sums). acc[t][u][r] = dim 32j + 4 * acc_tile(t, j) + r of column
// (u, m16), j = lane >> 4.
template <int H>
__device__ __forceinline__ void tile_acc(const __bf16* buf, const bf16x8 (&op)[2][H], floatx4 (&acc)[8][H], int lane) {
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const bf16x8 a = vt_operand(buf, 32 * kk, t, lane);
#pragma unroll
      for (int u = 0; u < H; ++u) acc[t][u] = mfma16x16x32(a, op[kk][u], acc[t][u]);
    }
}

// bf16 MFMA operand of a 64-row score tile x[kk][t][u][r] (row 32kk + 16t + 4j + r): k-index e < 4 is row
// 32kk + 4j + e, e >= 4 row 32kk + 16 + 4j + e - 4 (the order vt_operand reads the tile in).
template <int H>
__device__ __forceinline__ void pack_tile_op(const floatx4 (&x)[2][2][H], bf16x8 (&op)[2][H]) {
#pragma unroll
  for (int u = 0; u < H; ++u)
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      u32x4 pw;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        pw[2 * t] = pack_bf16x2(x[kk][t][u][0], x[kk][t][u][1]);
        pw[2 * t + 1] = pack_bf16x2(x[kk][t][u][2], x[kk][t][u][3]);
      }
      op[kk][u] = __builtin_bit_cast(bf16x8, pw);
    }
}

template <int N>
struct Buf {
  static constexpr int value = N;
};

template <bool kAligned, bool kTail, bool kWindow>
__global__ __launch_bounds__(512, 1) void prefill_bwd_dq_kernel(PrefillBwdArgs a) {
  constexpr int H = 2, kWaves = 8;
  __shared__ __attribute__((aligned(16))) __bf16 K0[kTileElems], K1[kTileElems], V0[kTileElems], V1[kTileElems];
  __bf16* const Kb[2] = {K0, K1};
  __bf16* const Vb[2] = {V0, V1};
  const PrefillArgs& f = a.f;
  const GridPos gp = grid_pos(f.B);
  const int qt = f.num_q_tiles - 1 - gp.rank;               // heavier (later) query tiles first
  const int kvh = gp.kvh;
  const int b = gp.b;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int m16 = lane & 15, j = lane >> 4;
  const int rg = w / 2, hbase = H * (w % 2);
  const int q0 = qt * kBM;
  const int qrow = q0 + 16 * rg + m16;
  const int plen = f.prompt_len ? f.prompt_len[b] : 0;
  int quota_all[4];
  int qmin = 1 << 30, qmax = 0;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    quota_all[u] = f.head_quota ? f.head_quota[kvh * kGroup + u] : f.K;
    qmin = min(qmin, quota_all[u]);
    qmax = max(qmax, quota_all[u]);
  }
  bf16x8 qop[H][4], gop[H][4];
  float l2[H], dd[H];
  {
    const bool ok = qrow < f.S0;
    const int r = min(qrow, f.S0 - 1);
#pragma unroll
    for (int u = 0; u < H; ++u) {
      const int head = kvh * kGroup + hbase + u;
      const __bf16* qp = f.q + (long)b * f.q_sb + (long)r * f.q_ss + (long)head * f.q_sh;
      const __bf16* gp = a.dout + (long)b * a.g_sb + (long)r * a.g_ss + (long)head * a.g_sh;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        u32x4 x = ld16g(qp + 8 * (4 * i + j)), y = ld16g(gp + 8 * (4 * i + j));
        if (!ok) x = y = u32x4{0, 0, 0, 0};
        qop[u][i] = __builtin_bit_cast(bf16x8, x);
        gop[u][i] = __builtin_bit_cast(bf16x8, y);
      }
      const long wi = ((long)b * kHeadsQ + head) * a.S0p + qrow;      // qrow < S0p
      l2[u] = a.lse2[wi];
      dd[u] = a.dvec[wi];
    }
  }
  floatx4 dq[8][H];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int u = 0; u < H; ++u) dq[i][u] = floatx4{0.f, 0.f, 0.f, 0.f};

  const DenseRows<kAligned> rows{f.k + (long)b * f.k_sb + (long)kvh * f.k_sh, f.v + (long)b * f.v_sb + (long)kvh * f.v_sh,
                                 f.k_ss, f.v_ss};
  const int wq0 = hbase ? quota_all[2] : quota_all[0], wq1 = hbase ? quota_all[3] : quota_all[1];
  const int q_last = min(q0 + kBM, f.S0) - 1;
  typedef MaskWalk<kAligned, kTail, kWindow> MW;
  MW mw(f, q0, q_last, qrow, plen, qmin, qmax, wq0, wq1);
  auto& walk = mw.walk;

  int tc = 0;
  TileMask mc;
  if (walk.next(tc, mc, true)) {
    {
      const auto s0 = rows.template src<2>(tc, w, f.S0);
      issue_half<kWaves, false>(rows, s0, f.S0, Kb[0], w, lane);
      issue_half<kWaves, true>(rows, s0, f.S0, Vb[0], w, lane);
    }
    // Double buffer: iteration n waits for tile n (every wave's DMAs, then a barrier, which also ends all reads of
    // the other buffer), issues tile n+1 (or re-loads tile n past the end) into the other buffer, computes tile n.
    auto step = [&](auto buf_c) -> bool {
      constexpr int sl = decltype(buf_c)::value;
      int tn = tc;
      TileMask mn;
      const bool hn = walk.next(tn, mn, false);
      const auto src = rows.template src<2>(hn ? tn : tc, w, f.S0);
      __asm__ volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      issue_half<kWaves, false>(rows, src, f.S0, Kb[1 - sl], w, lane);
      issue_half<kWaves, true>(rows, src, f.S0, Vb[1 - sl], w, lane);
      floatx4 s[2][2][H], dp[2][2][H];
      tile_scores<H>(Kb[sl], qop, s, m16, j);
      tile_scores<H>(Vb[sl], gop, dp, m16, j);
      tile_mask<H, typename MW::Walk>(s, tc, mc, mw.lane, j);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int u = 0; u < H; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float pr = fast_exp2(fmaf(s[kk][t][u][r], f.scale_log2, -l2[u]));
              s[kk][t][u][r] = pr * (dp[kk][t][u][r] - dd[u]);
            }
      bf16x8 dsop[2][H];
      pack_tile_op<H>(s, dsop);
      tile_acc<H>(Kb[sl], dsop, dq, lane);
      if (!hn) return false;
      tc = tn;
      mc = mn;
      return true;
    };
    for (;;) {
      if (!step(Buf<0>{})) break;
      if (!step(Buf<1>{})) break;
    }
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  if (qrow >= f.S0) return;
#pragma unroll
  for (int u = 0; u < H; ++u) {
    __bf16* dp = a.dq + (long)b * a.dq_sb + (long)qrow * a.dq_ss + (long)(kvh * kGroup + hbase + u) * a.dq_sh + 32 * j;
#pragma unroll
    for (int p = 0; p < 4; ++p) store_acc_bf16x8(dp + 8 * p, dq[2 * p][u], dq[2 * p + 1][u], j, a.scale);
  }
}

// S = Q K^T and dP = dO V^T of a wave's 16 keys over one staged tile (32 ds_read_b128, 32 MFMAs). The two products
// are interleaved and the reads run eight ahead of the MFMAs: at 2 waves per SIMD the other wave alone cannot cover
// an LDS round trip per MFMA.
__device__ __forceinline__ void dkv_scores(const __bf16* Qbuf, const __bf16* Gbuf, const bf16x8 (&kop)[4],
                                           const bf16x8 (&vop)[4], floatx4 (&s)[2][2][1], floatx4 (&dp)[2][2][1],
                                           int m16, int j) {
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int t = 0; t < 2; ++t) s[kk][t][0] = dp[kk][t][0] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const bf16x8 qa = __builtin_bit_cast(bf16x8, lds16(Qbuf, 32 * kk + 16 * t + m16, 4 * i + j));
        const bf16x8 ga = __builtin_bit_cast(bf16x8, lds16(Gbuf, 32 * kk + 16 * t + m16, 4 * i + j));
        s[kk][t][0] = mfma16x16x32(qa, kop[i], s[kk][t][0]);
        dp[kk][t][0] = mfma16x16x32(ga, vop[i], dp[kk][t][0]);
      }
  // scheduling groups (mask 0x100 LDS reads, 0x008 MFMA): 8 reads, then one MFMA per read, then the last 8 MFMAs
  __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
  for (int n = 0; n < 24; ++n) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
  }
  __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
}

// dV^T += dO^T P and dK^T += Q^T dS over one staged tile (the forward's PV step twice, interleaved; 64 transposed
// reads, 32 MFMAs), the reads running ahead of the MFMAs as in dkv_scores.
__device__ __forceinline__ void dkv_acc(const __bf16* Qbuf, const __bf16* Gbuf, const bf16x8 (&pop)[2][1],
                                        const bf16x8 (&dsop)[2][1], floatx4 (&dk)[8][1], floatx4 (&dv)[8][1],
                                        int lane) {
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const bf16x8 ga = vt_operand(Gbuf, 32 * kk, t, lane);
      const bf16x8 qa = vt_operand(Qbuf, 32 * kk, t, lane);
      dv[t][0] = mfma16x16x32(ga, pop[kk][0], dv[t][0]);
      dk[t][0] = mfma16x16x32(qa, dsop[kk][0], dk[t][0]);
    }
  __builtin_amdgcn_sched_group_barrier(0x100, 8, 1);
#pragma unroll
  for (int n = 0; n < 28; ++n) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
    __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
  }
  __builtin_amdgcn_sched_group_barrier(0x008, 4, 1);
}

__global__ __launch_bounds__(256, 2) void prefill_bwd_dkv_kernel(PrefillBwdArgs a) {
  constexpr int kWaves = 4;
  __shared__ __attribute__((aligned(16))) __bf16 Q0[kTileElems], Q1[kTileElems], G0[kTileElems], G1[kTileElems];
  __shared__ __attribute__((aligned(16))) float L0[kBN], L1[kBN], E0[kBN], E1[kBN];
  __shared__ KeySpan key_spans[kBN];
  __bf16* const Qb[2] = {Q0, Q1};
  __bf16* const Gb[2] = {G0, G1};
  float* const Lb[2] = {L0, L1};
  float* const Eb[2] = {E0, E1};
  const PrefillArgs& f = a.f;
  const int kvh = blockIdx.x % kHeadsKV;                    // a KV head's workgroups on one XCD, as grid_pos
  DkvItem item{(int)(blockIdx.x / kHeadsKV), 0, 1, 0, 0};
  if (a.seen != nullptr && !dkv_item(a.seen, f.num_q_tiles * f.B, a.workers, item.tile, item)) return;
  const int kt = item.tile / f.B;
  const int b = item.tile - kt * f.B;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int m16 = lane & 15, j = lane >> 4;
  const int k0 = kt * kBN;
  const int key = k0 + 16 * w + m16;                        // this lane's column
  const int plen = f.prompt_len ? f.prompt_len[b] : 0;
  // the four heads' code quotas, two to a register pair (an indexed array would live in scratch memory)
  auto quota_of = [&](int u) { return f.head_quota ? f.head_quota[kvh * kGroup + u] : f.K; };
  auto pair_of = [&](int u) { return (uint64_t)(uint32_t)quota_of(u) | (uint64_t)(uint32_t)quota_of(u + 1) << 32; };
  const uint64_t quota01 = pair_of(0), quota23 = pair_of(2);
  auto head_quota = [&](int u) { return (int)(uint32_t)((u & 2 ? quota23 : quota01) >> (32 * (u & 1))); };

  bf16x8 kop[4], vop[4];
  {
    const bool ok = key < f.S0;
    const int r = min(key, f.S0 - 1);
    const __bf16* kp = f.k + (long)b * f.k_sb + (long)r * f.k_ss + (long)kvh * f.k_sh;
    const __bf16* vp = f.v + (long)b * f.v_sb + (long)r * f.v_ss + (long)kvh * f.v_sh;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u32x4 x = ld16g(kp + 8 * (4 * i + j)), y = ld16g(vp + 8 * (4 * i + j));
      if (!ok) x = y = u32x4{0, 0, 0, 0};
      kop[i] = __builtin_bit_cast(bf16x8, x);
      vop[i] = __builtin_bit_cast(bf16x8, y);
    }
  }
  floatx4 dk[8][1], dv[8][1];
#pragma unroll
  for (int i = 0; i < 8; ++i) dk[i][0] = dv[i][0] = floatx4{0.f, 0.f, 0.f, 0.f};

  // (query tile, head) pairs that can see this key tile, head fastest
  const MaskShape shape = mask_shape(f);
  const KeySpan lane_key = key_span(shape, k0 + lane, plen);
  if (w == 0) key_spans[lane] = lane_key;                   // read by masked tiles (held in registers it spills);
                                                            // published by the first step's barrier
  const TileSpan span(lane_key);
  int qt_end = (span.last_row() + kBN - 1) / kBN;
  int qt = span.first_row() / kBN, h = -1, mode = 0;
  if (item.parts > 1) {                                     // this part's share of the query tiles
    const int quota = quota_max(f);
    auto nth = [&](int n) {                                 // the n-th query tile that sees the key tile
      for (int t = span.first_row() / kBN; t < qt_end; t += 64) {
        unsigned long long m = seen_mask(f, span, t, quota);
        if (n < __popcll(m)) {
          for (; n > 0; --n) m &= m - 1;
          return t + __ffsll(m) - 1;
        }
        n -= __popcll(m);
      }
      return qt_end;
    };
    qt = nth((int)((long)item.seen * item.z / item.parts));
    qt_end = nth((int)((long)item.seen * (item.z + 1) / item.parts));
  }
  auto next_pair = [&]() -> bool {
    for (;;) {
      if (++h == kGroup) {
        h = 0;
        ++qt;
      }
      if (qt >= qt_end) return false;
      mode = span.mode(qt * kBN, min(qt * kBN + kBN, f.S0), head_quota(h));
      if (mode >= 0) return true;
    }
  };
  // Q / dO rows of (qt, head) as the tile rows, lse2 / D rows beside them (waves 0 and 1, 4 bytes per lane)
  auto issue = [&](int pq, int ph, int sl_dst) {
    const int head = kvh * kGroup + ph;
    const DenseRows<false> rows{f.q + (long)b * f.q_sb + (long)head * f.q_sh,
                                a.dout + (long)b * a.g_sb + (long)head * a.g_sh, f.q_ss, a.g_ss};
    const auto src = rows.template src<4>(pq * kBN, w, f.S0);
    issue_half<kWaves, false>(rows, src, f.S0, Qb[sl_dst], w, lane);
    issue_half<kWaves, true>(rows, src, f.S0, Gb[sl_dst], w, lane);
    const long wi = ((long)b * kHeadsQ + head) * a.S0p + pq * kBN + lane;
    if (w == 0) __builtin_amdgcn_global_load_lds((const void*)(a.lse2 + wi), ABKV_LDS(Lb[sl_dst]), 4, 0, 0);
    if (w == 1) __builtin_amdgcn_global_load_lds((const void*)(a.dvec + wi), ABKV_LDS(Eb[sl_dst]), 4, 0, 0);
  };
  if (next_pair()) {
    issue(qt, h, 0);
    auto step = [&](auto buf_c) -> bool {
      constexpr int sl = decltype(buf_c)::value;
      const int cq = qt, ch = h, cmode = mode;
      const bool hn = next_pair();
      __asm__ volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      if (hn) issue(qt, h, 1 - sl);
      floatx4 s[2][2][1], dp[2][2][1];
      dkv_scores(Qb[sl], Gb[sl], kop, vop, s, dp, m16, j);
      if (cmode == 0) {                                     // wave-uniform: every pair of the tile visible
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const int r0 = 32 * kk + 16 * t + 4 * j;
            const floatx4 l4 = *reinterpret_cast<const floatx4*>(Lb[sl] + r0);
            const floatx4 e4 = *reinterpret_cast<const floatx4*>(Eb[sl] + r0);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float pr = fast_exp2(fmaf(s[kk][t][0][r], f.scale_log2, -l4[r]));
              s[kk][t][0][r] = pr;
              dp[kk][t][0][r] = pr * (dp[kk][t][0][r] - e4[r]);
            }
          }
      } else {                                              // the rows that see this lane's key
        const KeySpan ks = key_spans[16 * w + m16];
        const bool slot_ok = ks.slot < head_quota(ch);
        const unsigned m1 = slot_ok ? ks.e1 - ks.a1 : 0, m2 = slot_ok ? ks.e2 - ks.a2 : 0;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const int r0 = 32 * kk + 16 * t + 4 * j;
            const floatx4 l4 = *reinterpret_cast<const floatx4*>(Lb[sl] + r0);
            const floatx4 e4 = *reinterpret_cast<const floatx4*>(Eb[sl] + r0);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int qrow = cq * kBN + r0 + r;
              const bool vis = (unsigned)(qrow - ks.a1) < m1 || (unsigned)(qrow - ks.a2) < m2;
              const float pr = vis ? fast_exp2(fmaf(s[kk][t][0][r], f.scale_log2, -l4[r])) : 0.f;
              s[kk][t][0][r] = pr;
              dp[kk][t][0][r] = pr * (dp[kk][t][0][r] - e4[r]);
            }
          }
      }
      bf16x8 pop[2][1], dsop[2][1];
      pack_tile_op<1>(s, pop);
      pack_tile_op<1>(dp, dsop);
      dkv_acc(Qb[sl], Gb[sl], pop, dsop, dk, dv, lane);
      return hn;
    };
    for (;;) {
      if (!step(Buf<0>{})) break;
      if (!step(Buf<1>{})) break;
    }
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  if (item.parts > 1) {
    // sums of this part to its slot (lane order: whole 1 KiB runs); the part that finishes last adds the parts up in
    // order. Every slot's stores are released before the count and read after it is acquired (agent scope: the parts
    // may run on different XCDs). No part waits for another.
    __shared__ int finished;
    floatx4* slot = reinterpret_cast<floatx4*>(a.slots) +
                    ((long)(item.first * kHeadsKV + kvh) * kWaves + w) * (16 * 64) + lane;
    constexpr long kSlotStep = (long)kHeadsKV * kSlotFloats / 4;    // between the parts of a tile
    floatx4* mine = slot + item.z * kSlotStep;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      mine[64 * i] = dk[i][0];
      mine[64 * (8 + i)] = dv[i][0];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __syncthreads();
    if (threadIdx.x == 0)
      finished = __hip_atomic_fetch_add(a.done + item.first * kHeadsKV + kvh, 1, __ATOMIC_ACQ_REL,
                                        __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (finished != item.parts - 1) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      dk[i][0] = slot[64 * i];
      dv[i][0] = slot[64 * (8 + i)];
    }
    for (int z = 1; z < item.parts; ++z) {
      slot += kSlotStep;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        dk[i][0] += slot[64 * i];
        dv[i][0] += slot[64 * (8 + i)];
      }
    }
  }
  if (key >= f.S0) return;
  __bf16* kp = a.dk + (long)b * a.dk_sb + (long)key * a.dk_ss + (long)kvh * a.dk_sh + 32 * j;
  __bf16* vp = a.dv + (long)b * a.dv_sb + (long)key * a.dv_ss + (long)kvh * a.dv_sh + 32 * j;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    store_acc_bf16x8(kp + 8 * p, dk[2 * p][0], dk[2 * p + 1][0], j, a.scale);
    store_acc_bf16x8(vp + 8 * p, dv[2 * p][0], dv[2 * p + 1][0], j, 1.f);
  }
}

// Compute units of the current device (256 without one).
static int compute_units() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 256;
  return n;
}

}  // namespace abkv

extern "C" {

// Workspace bytes of abkv_prefill_masked_attn_bwd: lse * log2(e) and rowsum(dO * O) per (batch, query head, row),
// rows padded to whole 64-row tiles; the dK/dV counts and partial slots (up to 48 MiB, by the device's compute units).
size_t abkv_prefill_masked_bwd_workspace_size(int batch, int seq_len) {
  return abkv::bwd_layout(batch, seq_len, abkv::compute_units()).bytes;
}

int abkv_prefill_masked_attn_bwd(const void* q, long q_stride_b, long q_stride_s, long q_stride_h, const void* k,
                                 long k_stride_b, long k_stride_s, long k_stride_h, const void* v, long v_stride_b,
                                 long v_stride_s, long v_stride_h, const void* out, long out_stride_b,
                                 long out_stride_s, long out_stride_h, const void* dout, long dout_stride_b,
                                 long dout_stride_s, long dout_stride_h, const float* lse, int batch, int block_c,
                                 int codes_k, int num_blocks, int seq_len, const int32_t* prompt_len,
                                 const int32_t* head_quota, int retain_tail, int tail_policy, int pause_xattn,
                                 int pause_passes, int copy_rows, int replay_rows, int replay_exclude, float scale,
                                 void* dq,
                                 long dq_stride_b, long dq_stride_s, long dq_stride_h, void* dk, long dk_stride_b,
                                 long dk_stride_s, long dk_stride_h, void* dv, long dv_stride_b, long dv_stride_s,
                                 long dv_stride_h, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  using namespace abkv;
  if (batch <= 0 || seq_len <= 0) return 0;
  if (q == nullptr || k == nullptr || v == nullptr || out == nullptr || dout == nullptr || lse == nullptr ||
      dq == nullptr || dk == nullptr || dv == nullptr || block_c <= 0 || codes_k < 0 || num_blocks <= 0 ||
      pause_passes <= 0 || copy_rows < 0 || (codes_k == 0 && (pause_passes != 1 || copy_rows)) ||
      replay_rows < 0 || replay_rows > block_c || (replay_rows && (retain_tail || codes_k == 0)) ||
      (replay_exclude && (replay_rows <= 0 || replay_rows >= block_c)) ||
      (long)seq_len != (long)num_blocks * (block_c + (long)pause_passes * codes_k + replay_rows) + copy_rows ||
      retain_tail < 0 || retain_tail > block_c || (retain_tail == block_c && tail_policy != kTailRaw) ||
      tail_policy < kTailStatic || tail_policy > kTailRaw ||
      pause_xattn < kXattnFull || pause_xattn > kXattnNone)
    return (int)hipErrorInvalidValue;
  const BwdLayout lay = bwd_layout(batch, seq_len, compute_units());
  if (workspace == nullptr || workspace_bytes < lay.rows) return (int)hipErrorInvalidValue;
  const bool parts = workspace_bytes >= lay.bytes;          // less: a workgroup per key tile, in tile order
  PrefillBwdArgs a;
  PrefillArgs& f = a.f;
  f.q = static_cast<const __bf16*>(q);
  f.q_sb = q_stride_b; f.q_ss = q_stride_s; f.q_sh = q_stride_h;
  f.k = static_cast<const __bf16*>(k);
  f.k_sb = k_stride_b; f.k_ss = k_stride_s; f.k_sh = k_stride_h;
  f.v = static_cast<const __bf16*>(v);
  f.v_sb = v_stride_b; f.v_ss = v_stride_s; f.v_sh = v_stride_h;
  f.B = batch; f.S0 = seq_len; f.C = block_c; f.K = codes_k; f.N = num_blocks;
  f.prompt_len = prompt_len;
  f.head_quota = head_quota;
  f.scale_log2 = scale * 1.4426950408889634f;
  f.out = nullptr; f.o_sb = f.o_ss = f.o_sh = 0;
  f.lse = nullptr;
  f.tail = retain_tail;
  f.policy = tail_policy;
  f.xattn = pause_xattn;
  f.L = pause_passes;
  f.copy = copy_rows;
  f.R = replay_rows;
  f.rx = replay_exclude != 0;
  f.aligned = (block_c % kBN == 0) && (codes_k % kBN == 0) && pause_xattn == kXattnFull && pause_passes == 1 &&
              copy_rows == 0 && replay_rows == 0 && tail_policy != kTailRaw;
  f.num_q_tiles = (seq_len + kBM - 1) / kBM;
  a.o = static_cast<const __bf16*>(out);
  a.o_sb = out_stride_b; a.o_ss = out_stride_s; a.o_sh = out_stride_h;
  a.dout = static_cast<const __bf16*>(dout);
  a.g_sb = dout_stride_b; a.g_ss = dout_stride_s; a.g_sh = dout_stride_h;
  a.lse = lse;
  a.S0p = f.num_q_tiles * kBM;
  a.lse2 = static_cast<float*>(workspace);
  a.dvec = reinterpret_cast<float*>(static_cast<char*>(workspace) + lay.dvec);
  char* ws = static_cast<char*>(workspace) + (-reinterpret_cast<uintptr_t>(workspace) & 15);
  a.seen = parts ? reinterpret_cast<int*>(ws + lay.seen) : nullptr;
  a.done = reinterpret_cast<int*>(ws + lay.done);
  a.slots = reinterpret_cast<float*>(ws + lay.slots);
  a.slot_cap = parts ? lay.cap : 0;
  a.workers = lay.workers;
  a.count_blocks = parts ? (f.num_q_tiles * batch + 3) / 4 : 0;
  a.scale = scale;
  a.dq = static_cast<__bf16*>(dq);
  a.dq_sb = dq_stride_b; a.dq_ss = dq_stride_s; a.dq_sh = dq_stride_h;
  a.dk = static_cast<__bf16*>(dk);
  a.dk_sb = dk_stride_b; a.dk_ss = dk_stride_s; a.dk_sh = dk_stride_h;
  a.dv = static_cast<__bf16*>(dv);
  a.dv_sb = dv_stride_b; a.dv_ss = dv_stride_s; a.dv_sh = dv_stride_h;
  if (prefill_grid(f.num_q_tiles, batch, 512) == 0) return (int)hipErrorInvalidValue;
  const long rows = (long)batch * kHeadsQ * a.S0p;
  const long gk = ((long)a.slot_cap + (long)f.num_q_tiles * batch) * kHeadsKV;   // at least the items of dkv_item
  // prep: 16 work-items per row and head, and the counting workgroups
  if (rows * 16 + 256L * (a.count_blocks + 1) > 0xFFFFFFFFL || gk * 256 > 0xFFFFFFFFL) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(prefill_bwd_prep_kernel, dim3((unsigned)((rows * 16 + 255) / 256 + a.count_blocks)), dim3(256), 0, stream,
                     a);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return (int)err;
  const unsigned gq = prefill_grid(f.num_q_tiles, batch, 512);
  const bool window = retain_tail > 0 && tail_policy != kTailStatic;
  if (f.aligned && retain_tail == 0)
    hipLaunchKernelGGL((prefill_bwd_dq_kernel<true, false, false>), gq, dim3(512), 0, stream, a);
  else if (f.aligned && !window)
    hipLaunchKernelGGL((prefill_bwd_dq_kernel<true, true, false>), gq, dim3(512), 0, stream, a);
  else if (f.aligned) hipLaunchKernelGGL((prefill_bwd_dq_kernel<true, true, true>), gq, dim3(512), 0, stream, a);
  else hipLaunchKernelGGL((prefill_bwd_dq_kernel<false, false, false>), gq, dim3(512), 0, stream, a);
  err = hipGetLastError();
  if (err != hipSuccess) return (int)err;
  hipLaunchKernelGGL(prefill_bwd_dkv_kernel, dim3((unsigned)gk), dim3(256), 0, stream, a);
  return (int)hipGetLastError();
}

}  // extern "C"
