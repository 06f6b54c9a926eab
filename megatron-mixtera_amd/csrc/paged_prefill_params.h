// Arguments and head mapping shared by the paged varlen prefill kernels (paged_prefill.hip,
// paged_prefill_woven.hip).
#pragma once

#include "mi_common.h"

namespace mi {

struct PrefillParams {
  const uint16_t* q;
  int64_t q_st, q_sh;
  const uint8_t* kc;
  const uint8_t* vc;
  int64_t kv_sc;
  int32_t kv_st, kv_sh;
  int64_t v_sc;          // value cache strides (register-only kernel; equal to the key cache's otherwise)
  int32_t v_st, v_sh;
  const int32_t* bt;
  int64_t bt_stride;
  const int32_t* cu_q;
  const int32_t* lens;
  uint16_t* out;
  int64_t o_st, o_sh;
  uint64_t chunk_magic;  // ceil(2^40 / chunk)
  int32_t T, R, Hq, Hkv, G, g_magic, chunk;  // g_magic = 65536 / G + 1: (n * g_magic) >> 16 == n / G for n <= 64, G <= 16
  int32_t parts;         // workgroups per KV head along the query heads: each takes up to 16 of the G that share it
  int32_t skip_single;  // requests with exactly one query row are handled by the decode kernels
  float scale_log2;
  const float* k_scale;  // fp8 KV only: [n_chunks][Hkv]
  const float* v_scale;
  // Two-phase tile kernel only: the keys of a request cut into gridDim.y ranges, one workgroup each;
  // with more than one range the workgroups write fp32 partials [range][T][Hq][128] and their
  // log-sum-exps [range][T][Hq] (log2 domain) and a merge kernel finishes the rows.
  float* split_o;
  float* split_lse;
  // Queries as the QKV projection left them (one-stream tile kernel only): head norm and rotation happen as they are
  // loaded.  Otherwise q_gst == G * q_sh and the rest is off.
  int64_t q_gst;           // elements between the query heads of two KV heads
  const uint16_t* angles;  // [T][2][head_dim]: cos | sin of every row (see qkv_key_append_kernel), or null
  const uint16_t* q_w;     // RMS norm weight or null
  float eps;
  int32_t norm, interleaved;
};

// The query heads one workgroup serves: with at most 16 query heads per KV head, all G of KV head `hv`; with more,
// `parts` workgroups share a KV head and take 16 query heads each (the last one the rest).
struct HeadSlice {
  int h;        // KV head
  int hq0;      // first query head
  int G;        // query heads (1..16)
  int g_magic;  // 65536 / G + 1
};
static __device__ __forceinline__ HeadSlice head_slice(const PrefillParams& p, int hv) {
  HeadSlice s;
  if (p.parts <= 1) {
    s.h = hv; s.hq0 = hv * p.G; s.G = p.G; s.g_magic = p.g_magic;
  } else {
    s.h = hv / p.parts;
    const int part = hv - s.h * p.parts;
    s.hq0 = s.h * p.G + 16 * part;
    s.G = min(16, p.G - 16 * part);
    s.g_magic = 65536 / s.G + 1;
  }
  return s;
}

// The query block a workgroup of the tile kernels takes.
struct QueryBlock {
  int r;              // request
  int q_begin;        // its first row
  int Lq, Lk;         // its rows and keys
  int q0;             // the block's first row within the request
};

// the largest of the lanes' values (none negative)
static __device__ __forceinline__ int wave_max(int v) {
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));
  return __builtin_amdgcn_readlane(v, 63);
}

constexpr int kOrderedRequests = 128;  // requests whose blocks are handed out longest first (two per lane)
constexpr int kLengthLevels = 16;

// The `rank`-th query block of the batch, blocks of `SBQ` rows; false: there are fewer.  `blocks` is the launch's count
// (an upper bound).  Every wavefront of the workgroup calls this.
//
// The chip takes workgroups in order, so long ones must not come last: in the batch's own order the last ones are the
// first request's, however long its context, and the chip drains while they run.  Requests go by their keys, longest
// first, in 16 levels (within a level by index), and each request's blocks last to first: its shortest end the launch,
// and blocks that run together share their keys in L2.  (Blocks of all requests ranked by their own length balance no
// better and spread the reads: equal prompts 1 % slower than in batch order.)  A lane holds one or two requests; four steps
// of bisection over the levels and a scan find the block.  Steps, against the batch's order: 11 prompts of 33-3 001 tokens,
// head width 64, 149.9 -> 143.1 us; 8 prompts of 2 048 new tokens each over 0-4 096, 1 271 -> 1 273.  With more
// requests than that -- or one, whose blocks are in order as they are -- blocks come last to first: request r's are
// numbered cu_q[r] / SBQ + r onward.
static __device__ __forceinline__ bool find_query_block(const PrefillParams& p, int SBQ, int rank, int blocks,
                                                        QueryBlock* o) {
  const int lane = threadIdx.x & 63;
  if (p.R > 1 && p.R <= kOrderedRequests) {
    const float inv = 1.f / (float)SBQ;
    auto div = [&](int n) {  // n / SBQ for n >= 0: the estimate is at most one off
      int q = (int)((float)n * inv);
      q -= q * SBQ > n ? 1 : 0;
      return q + ((q + 1) * SBQ <= n ? 1 : 0);
    };
    int cq[2], lq[2], lk[2], nb[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int i = lane + 64 * c;
      cq[c] = lq[c] = lk[c] = nb[c] = 0;
      if (i < p.R) {
        cq[c] = p.cu_q[i];
        lq[c] = p.cu_q[i + 1] - cq[c];
        lk[c] = p.lens[i];
        nb[c] = p.skip_single && lq[c] == 1 ? 0 : div(max(lq[c], 0) + SBQ - 1);
      }
    }
    const int top = wave_max(max(nb[0] ? lk[0] : 0, nb[1] ? lk[1] : 0));
    const int step = (top >> 4) + 1;
    static_assert(kLengthLevels == 16, "levels of top / 16 keys");
    // blocks of the lane's request c if it has at least level * step keys
    auto reach = [&](int c, int level) { return lk[c] >= level * step ? nb[c] : 0; };
    auto count = [&](int level) {
      return __builtin_amdgcn_readlane(wave_scan(reach(0, level) + reach(1, level)), 63);
    };
    if (rank >= count(0)) return false;
    int lo = 0, hi = kLengthLevels, above = 0;  // count(lo) > rank >= count(hi) == above
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int mid = (lo + hi) >> 1, n = count(mid);
      if (n > rank) {
        lo = mid;
      } else {
        hi = mid;
        above = n;
      }
    }
    int j = rank - above;  // within the level, request by request
    const int n0 = reach(0, lo) - reach(0, hi), n1 = reach(1, lo) - reach(1, hi);
    const int s0 = wave_scan(n0), s1 = wave_scan(n1), all0 = __builtin_amdgcn_readlane(s0, 63);
    const int c = j < all0 ? 0 : 1;
    if (c) j -= all0;
    const int incl = c ? s1 : s0;
    const int at = __builtin_ctzll(__builtin_amdgcn_ballot_w64(incl > j));
    const int b = __builtin_amdgcn_readlane(incl, at) - 1 - j;  // the request's last block first
    o->r = at + 64 * c;
    o->q_begin = __builtin_amdgcn_readlane(c ? cq[1] : cq[0], at);
    o->Lq = __builtin_amdgcn_readlane(c ? lq[1] : lq[0], at);
    o->Lk = __builtin_amdgcn_readlane(c ? lk[1] : lk[0], at);
    o->q0 = b * SBQ;
    return true;
  }
  // 64 candidates per pass, one per lane (a pass is one trip to memory, and nothing of the workgroup's work can start
  // before its request is known): the last request whose first block is not past this one.  The same pass fetches
  // what is needed of that request.
  const int sb = blocks - 1 - rank;
  int r = 0;
  for (int n = p.R;;) {  // the answer lies in [r, r + n)
    const int stride = (n + 63) >> 6;
    const int idx = r + lane * stride;
    const bool in = lane * stride < n;
    const int cq = in ? p.cu_q[idx] : 0, cq1 = in ? p.cu_q[idx + 1] : 0, len = in ? p.lens[idx] : 0;
    const int c = __builtin_popcountll(__builtin_amdgcn_ballot_w64(in && cq / SBQ + idx <= sb)) - 1;  // >= 0: the first candidate always qualifies
    r += c * stride;
    n = min(stride, n - c * stride);
    if (stride == 1) {
      o->r = r;
      o->q_begin = __builtin_amdgcn_readlane(cq, c);
      o->Lq = __builtin_amdgcn_readlane(cq1, c) - o->q_begin;
      o->Lk = __builtin_amdgcn_readlane(len, c);
      break;
    }
  }
  o->q0 = (sb - (o->q_begin / SBQ + r)) * SBQ;
  return o->q0 < o->Lq && !(p.skip_single && o->Lq == 1);
}

// Query blocks of `SBQ` rows that R requests of T rows in all can have, as find_query_block numbers them: the workgroups a
// launch needs per head.  Not one more: those that find nothing leave at once, but the dispatcher has dealt them out, one
// shader engine after the other, and with every second workgroup an empty one half of the chip stays idle (one request of
// 40 rows over 60 000 keys, 8 heads of 128, 32 ranges: 110 us with one empty block, 65 without).
static inline int prefill_query_blocks(int T, int R, int SBQ) {
  if (R > kOrderedRequests) return T / SBQ + R;
  const int64_t most = ((int64_t)T + (int64_t)R * (SBQ - 1)) / SBQ;  // every request's last block all but empty
  return (int)(most < T ? most : T);
}

// The one-stream ("woven") tile kernel for head_dim 64 and 128 (paged_prefill_woven.hip).  Same grid and request ->
// workgroup map as the two-phase tile kernel: `grid.x` workgroups of `waves` wavefronts (32 rows each; four or, at head_dim
// 128, eight), `grid.y` key ranges (with more than one, `p.split_o` / `p.split_lse` receive the partials).
void launch_prefill_woven(const PrefillParams& p, dim3 grid, int head_dim, bool fp8, bool f16, int waves, hipStream_t stream);

}  // namespace mi
