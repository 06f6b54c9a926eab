// Tail of a decode step: last-token gather, token sampling and the finished-request mask.
//
// What the reference does with torch ops after the forward pass
// (megatron/core/inference/text_generation_controllers/text_generation_controller.py:172-315,
// 519-530 and megatron/core/inference/contexts/dynamic_context.py:890-918):
//   * last_token_logits: rows  cumsum(request_query_lengths) - 1  of the `[T, V]` logits;
//   * sample_from_logits: argmax (top_k == 1), or  logits / temperature -> top-k filter (keep
//     values >= the k-th largest) or top-p filter (sort descending, keep the shortest prefix
//     whose softmax mass exceeds top_p) -> softmax -> one multinomial draw per row;
//   * active_request_mask = (sample != termination_id) & (sequence length + 1 < maximum length).
//
// Here a row is never sorted.  One workgroup of 16 wavefronts owns a row and finds the cut
// value of the filter by selection: a 256-bin histogram over the value range, then four 8-bit
// digit passes over the order-preserving integer image of the floats in the chosen bin (its
// members are listed in LDS; the row is re-read instead when they do not fit).  Probability mass is carried as 64-bit fixed point
// (exp(x - max) rounded to 2^-32), so every sum is an integer sum: the result does not depend on the
// order of the atomic additions and a replay of the same call gives the same token.  The draw
// itself is an inverse-CDF lookup in vocabulary order driven by one caller-supplied uniform
// number per row (three levels: 16 ranges -> 16 sub-ranges -> elements).
#include <type_traits>

#include "mi_common.h"
#include "mi_capi_internal.h"

namespace mi {

struct SampleParams {
  const void* logits; int64_t stride;  // row stride in elements
  int32_t R, V;
  int32_t top_k; float top_p; float inv_temperature;
  const float* uniform;      // [R], unused for top_k == 1
  int32_t vocab_clamp;       // > 0: samples are clamped to [0, vocab_clamp - 1]
  int64_t* samples;          // [R]
  float* cut_out;            // optional [R]: smallest kept (scaled) logit value, -inf = nothing filtered
  const int32_t* kv_off; const int32_t* q_len; const int32_t* out_len;  // optional, [R] each
  int64_t termination_id;
  uint8_t* active_mask;      // optional [R]
};

constexpr int kSampleThreads = 1024;
constexpr int kSampleWaves = kSampleThreads / 64;

// float -> uint32 with the same ordering (and back)
static __device__ __forceinline__ uint32_t order_key(float x) {
  const uint32_t u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
static __device__ __forceinline__ float order_key_value(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// Inclusive prefix sum over the 64 lanes with data-parallel-primitive moves (shifts by 1, 2, 4, 8 inside a row of 16
// lanes, then the last lane of row 0 / 2 broadcast into row 1 / 3 and lane 31 into the upper half): six steps of two
// moves and one 64-bit add, where the shuffle form costs twelve dependent trips through the LDS crossbar.  Lanes
// without a source receive zero.
template <int CTRL, int ROW_MASK>
static __device__ __forceinline__ uint64_t dpp_u64(uint64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, ROW_MASK, 0xF, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, ROW_MASK, 0xF, false);
  return ((uint64_t)hi << 32) | lo;
}
static __device__ __forceinline__ uint64_t wave_scan_incl_u64(uint64_t v, int /*lane*/) {
  v += dpp_u64<0x111, 0xF>(v);  // row_shr:1
  v += dpp_u64<0x112, 0xF>(v);  // row_shr:2
  v += dpp_u64<0x114, 0xF>(v);  // row_shr:4
  v += dpp_u64<0x118, 0xF>(v);  // row_shr:8
  v += dpp_u64<0x142, 0xA>(v);  // row_bcast:15 into rows 1 and 3
  v += dpp_u64<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}
template <int CTRL, int ROW_MASK>
static __device__ __forceinline__ float dpp_f32(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xF, false));
}
static __device__ __forceinline__ float wave_scan_incl_f32(float v) {
  v += dpp_f32<0x111, 0xF>(v);
  v += dpp_f32<0x112, 0xF>(v);
  v += dpp_f32<0x114, 0xF>(v);
  v += dpp_f32<0x118, 0xF>(v);
  v += dpp_f32<0x142, 0xA>(v);
  v += dpp_f32<0x143, 0xC>(v);
  return v;
}
// Sum over the 64 lanes, in every lane: the scan above, then its last lane's value.
static __device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) {
  v = wave_scan_incl_u64(v, 0);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, 63);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), 63);
  return ((uint64_t)hi << 32) | lo;
}

// Largest of the 64 lanes' values, in every lane, by the same moves.
template <int CTRL, int ROW_MASK>
static __device__ __forceinline__ uint32_t dpp_max_u32(uint32_t v) {
  return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xF, false));
}
static __device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  v = dpp_max_u32<0x111, 0xF>(v);
  v = dpp_max_u32<0x112, 0xF>(v);
  v = dpp_max_u32<0x114, 0xF>(v);
  v = dpp_max_u32<0x118, 0xF>(v);
  v = dpp_max_u32<0x142, 0xA>(v);
  v = dpp_max_u32<0x143, 0xC>(v);
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// One row of logits.  DT = element type (0 fp32, 1 bf16, 2 fp16); VEC = elements per 16-byte load (4 fp32,
// 8 of a 16-bit type) when the row is 16-byte aligned, 1 otherwise.
template <int DT, int VEC>
struct RowReader {
  const uint8_t* row; int V; float inv_t; bool scale;
  // the value the filters see: logit * (1 / temperature), rounded to the logits' dtype as the
  // in-place division of the reference rounds it; -0 becomes +0 so that equal values share a key
  __device__ __forceinline__ float finish(float x) const {
    if (scale) {
      x *= inv_t;
      if (DT != 0) x = to_f32<DT == 2>(f32_to_16<DT == 2>(x));
    }
    return x + 0.0f;
  }
  // the same with a -0 left as it is, and fp32 multiplied by one where nothing is scaled
  __device__ __forceinline__ float scaled(float x) const {
    if (DT == 0 || scale) x *= inv_t;
    if (DT != 0 && scale) x = to_f32<DT == 2>(f32_to_16<DT == 2>(x));
    return x;
  }
  __device__ __forceinline__ float at(int i) const {
    return finish(DT != 0 ? to_f32<DT == 2>(reinterpret_cast<const uint16_t*>(row)[i]) : reinterpret_cast<const float*>(row)[i]);
  }
  // elements i0 .. i0+VEC-1 (i0 a multiple of VEC), all inside the row; ZERO = false: a -0 stays one
  template <bool ZERO = true>
  __device__ __forceinline__ void load_full(int i0, float (&x)[VEC]) const {
    if (VEC > 1) {
      const uint4 w = ld16(row + (int64_t)i0 * (DT != 0 ? 2 : 4));
      const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        float v;
        if (DT != 0) v = (j & 1) ? hi_to_f32<DT == 2>(u[(j >> 1) & 3]) : lo_to_f32<DT == 2>(u[(j >> 1) & 3]);
        else v = __uint_as_float(u[j & 3]);
        x[j] = ZERO ? finish(v) : scaled(v);
      }
    } else {
      x[0] = at(i0);
    }
  }
  // the same with slots at or past V set to 0
  __device__ __forceinline__ void load(int i0, float (&x)[VEC]) const {
    if (VEC > 1 && i0 + VEC <= V) {
      const uint4 w = ld16(row + (int64_t)i0 * (DT != 0 ? 2 : 4));
      const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        float v;
        if (DT != 0) v = (j & 1) ? hi_to_f32<DT == 2>(u[(j >> 1) & 3]) : lo_to_f32<DT == 2>(u[(j >> 1) & 3]);
        else v = __uint_as_float(u[j & 3]);
        x[j] = finish(v);
      }
    } else {
#pragma unroll
      for (int j = 0; j < VEC; ++j) x[j] = i0 + j < V ? at(i0 + j) : 0.f;
    }
  }
};

// Calls f(i, x, i < end) for every slot of [begin, end) rounded up to whole strides: `nthreads`
// threads (this one is `t`) take VEC consecutive elements each, U loads in flight.  Every thread
// makes the same number of calls, so f may use wavefront-wide operations.  begin % VEC == 0.
// Whole blocks of U strides run without any bounds test (the flag is the constant true there);
// only the rest of the range pays for guards.
template <int U, int DT, int VEC, typename F>
static __device__ __forceinline__ void sweep(const RowReader<DT, VEC>& rd, int begin, int end, int t, int nthreads, F f) {
  const int stride = nthreads * VEC;
  const int row_end = rd.V - (rd.V % VEC);  // whole 16-byte groups of the row end here
  int base = begin;
  for (; base + U * stride <= min(end, row_end); base += U * stride) {
    float x[U][VEC];
#pragma unroll
    for (int u = 0; u < U; ++u) rd.load_full(base + u * stride + t * VEC, x[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) f(base + u * stride + t * VEC + j, x[u][j], true);
    }
  }
  if (base < end) {  // the rest: fewer than U strides, guarded, loads still issued together
    float x[U][VEC];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i0 = base + u * stride + t * VEC;
      if (i0 < end) {
        rd.load(i0, x[u]);
      } else {
#pragma unroll
        for (int j = 0; j < VEC; ++j) x[u][j] = 0.f;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i0 = base + u * stride + t * VEC;
      if (base + u * stride < end) {  // uniform over the participating threads
#pragma unroll
        for (int j = 0; j < VEC; ++j) f(i0 + j, x[u][j], i0 + j < end);
      }
    }
  }
}

// A thread's next BATCH values of [base, end): U groups of VEC, `nthreads` threads side by side (this one is `t`), all
// loads in flight together; -inf at and past `end`, and zeros of either sign.  base % VEC == 0, and end is a multiple of VEC
// or the row's end.
template <int BATCH, int DT, int VEC>
static __device__ __forceinline__ void load_batch(const RowReader<DT, VEC>& rd, int base, int end, int t, int nthreads,
                                                  float (&x)[BATCH / VEC][VEC]) {
  constexpr int U = BATCH / VEC;
  const int stride = nthreads * VEC;
  const int row_end = rd.V - (rd.V % VEC);  // whole groups of the row end here (there is one)
  if (base + U * stride <= min(end, row_end)) {
#pragma unroll
    for (int u = 0; u < U; ++u) rd.template load_full<false>(base + u * stride + t * VEC, x[u]);
  } else {  // (loads without a branch around them, so that they too are in flight together)
#pragma unroll
    for (int u = 0; u < U; ++u) rd.template load_full<false>(min(base + u * stride + t * VEC, row_end - VEC), x[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i0 = base + u * stride + t * VEC;
#pragma unroll
      for (int j = 0; j < VEC; ++j) x[u][j] = i0 < min(end, row_end) ? x[u][j] : -INFINITY;
    }
    if (VEC > 1 && end > row_end) {  // the row's last values, fewer than a group: one thread's
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (base + u * stride + t * VEC == row_end) {
#pragma unroll
          for (int j = 0; j < VEC - 1; ++j)
            if (row_end + j < end) x[u][j] = rd.at(row_end + j);
        }
    }
  }
}

// exp(x - mx) as fixed point, rounded to the nearest 2^-32: one 32-bit conversion per element
// (sums are carried in 64 bits).  0 for anything that is not a number at or below the maximum.
constexpr float kMassOne = 4294967040.0f;  // largest fp32 below 2^32
static __device__ __forceinline__ float mass_f(float x, float neg_mx_log2e) {
  return __builtin_fmaf(fast_exp2(__builtin_fmaf(x, 1.4426950408889634f, neg_mx_log2e)), kMassOne, 0.5f);
}
// The conversion is the instruction's: truncated, 0 for NaN, and 2^32 - 1 for what does not fit -- a large maximum's
// exponential rounds to more than one -- where C++ leaves it undefined.  (The compiler's own saturating form is five
// instructions, a comparison and a selection cost the walks 3-5 %.)  Inline assembly is not moved out of a branch: where a mass
// may or may not count, it is made first and selected then (200 x 50 304 by one workgroup per row, top-p: 73.2 -> 69.6 us).  Its
// operand comes from a fused multiply-add: a result of the transcendental unit would need a wait that is not inserted here.
static __device__ __forceinline__ uint64_t mass_of(float x, float neg_mx_log2e) {
  uint32_t m = __float_as_uint(mass_f(x, neg_mx_log2e));
  asm("v_cvt_u32_f32 %0, %0" : "+v"(m));
  return m;
}
// The same added to a sum {lo, hi}, in one statement: apart, 32 of them at once spill ten registers (64 x 128 256, top-p: 28.0
// against 30.9 us).
static __device__ __forceinline__ uint32_t add_mass(uint32_t& lo, uint32_t& hi, float x, float neg_mx_log2e) {
  float m = mass_f(x, neg_mx_log2e);
  asm("v_cvt_u32_f32 %2, %2\n\tv_add_co_u32 %0, vcc, %0, %2\n\tv_addc_co_u32 %1, vcc, 0, %1, vcc"
      : "+v"(lo), "+v"(hi), "+v"(m) : : "vcc");
  return __float_as_uint(m);
}

static __device__ __forceinline__ void add_u32(uint32_t& lo, uint32_t& hi, uint32_t m) {
  asm("v_add_co_u32 %0, vcc, %0, %2\n\tv_addc_co_u32 %1, vcc, 0, %1, vcc" : "+v"(lo), "+v"(hi) : "v"(m) : "vcc");
}

// Whether a row with this maximum has a distribution to draw from.  Not where it is not a finite number, and not where it
// is so large (from some 4e8) that the rounding of the product with log2(e) leaves its own mass at nothing: a total of
// zero would have no element to fall on.
static __device__ __forceinline__ bool has_masses(float mx) {
  return fabsf(mx) < INFINITY && mass_of(mx, -mx * 1.4426950408889634f) > 0;
}

// Adds weight() to hist[bin] for the active lanes (weight is only evaluated when some lane of the
// wavefront is active).  When every active lane hits the same bin -- values clustered in one bin
// would otherwise serialise 64 atomics on one address -- the wavefront adds its sum once.
template <typename W>
static __device__ __forceinline__ void hist_add(uint64_t* hist, int bin, bool active, int lane, W weight) {
  const uint64_t m = __builtin_amdgcn_ballot_w64(active);
  if (m == 0) return;
  const uint64_t w = active ? weight() : 0;
  const int first = __builtin_ctzll(m);
  const int b0 = __builtin_amdgcn_readlane(bin, first);
  const uint64_t same = __builtin_amdgcn_ballot_w64(active && bin == b0);
  if (same == m) {
    const uint64_t s = wave_sum_u64(w);
    if (lane == first && s) atomicAdd(reinterpret_cast<unsigned long long*>(&hist[b0]), (unsigned long long)s);
  } else if (active && w) {
    atomicAdd(reinterpret_cast<unsigned long long*>(&hist[bin]), (unsigned long long)w);
  }
}

// Wave 0: first of the 64 N bins b (ascending) whose inclusive running sum, started at `above`, exceeds
// `target`.  Writes {bin or -1, running sum before that bin} to res[0..1].
template <int N = 4>
static __device__ void find_crossing(const uint64_t* hist, uint64_t above, uint64_t target, uint64_t* res, int lane) {
  uint64_t h[N], loc = 0;
#pragma unroll
  for (int j = 0; j < N; ++j) { h[j] = hist[N * lane + j]; loc += h[j]; }
  const uint64_t incl = wave_scan_incl_u64(loc, lane) + above;
  const bool cross = incl > target;
  const uint64_t m = __builtin_amdgcn_ballot_w64(cross);
  if (m == 0) {
    if (lane == 63) { res[0] = (uint64_t)-1; res[1] = incl; }
    return;
  }
  if (lane == __builtin_ctzll(m)) {
    uint64_t run = incl - loc;
    int b = N * lane;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      if (run + h[j] > target) break;
      run += h[j];
      ++b;
    }
    res[0] = (uint64_t)b;
    res[1] = run;
  }
}

static __device__ __forceinline__ void write_sample(const SampleParams& p, int r, int sample, uint32_t cut_key) {
  p.samples[r] = sample;
  // (a cut among NaNs with their sign set, below every number, filters nothing)
  if (p.cut_out) p.cut_out[r] = cut_key > order_key(-INFINITY) ? order_key_value(cut_key) : -INFINITY;
  if (p.active_mask) {
    bool active = (int64_t)sample != p.termination_id;
    if (p.kv_off) active = active && (p.kv_off[r] + p.q_len[r] + 1 < p.out_len[r]);
    p.active_mask[r] = active ? 1 : 0;
  }
}

constexpr int kMemberCap = 4096;  // members of the chosen value bin that fit the LDS list
// Top-k with a small k (the usual 20-100) needs none of the row-wide histogram passes: a threshold is estimated
// from kMemberCap values spread over the row so that a thousand or a few thousand elements lie at or above it, ONE pass
// finds the maximum and lists those candidates, and the exact k-th largest value and the draw are then worked out
// on the list.  Top-p does the same with one more pass for the row's total mass; its cut lies inside the list
// whenever the candidates alone hold more than top_p of that mass (peaked rows: the usual case).  When the estimate
// misses (fewer than k candidates, more than the list holds -- flat rows --, too little mass), the general path
// below runs instead; the result is the same either way.
constexpr int kFastTopK = 768;          // largest k the one-pass form is tried for
constexpr int kFastMinVocab = 16384;    // smallest row it is tried for
// expected candidates: 1 024, or 4 k up to 3 072 (standard deviation ~ target / sqrt(sample rank), i.e. ~10-18 %)
static __device__ __forceinline__ int candidate_target(int top_k) { return max(1024, min(4 * top_k, 3072)); }

template <int DT, int VEC>
__global__ __launch_bounds__(kSampleThreads) void sample_kernel(SampleParams p) {
  __shared__ uint64_t hist[256];
  __shared__ uint64_t res[2];
  __shared__ uint64_t wsum[kSampleWaves];
  __shared__ uint32_t red_key[kSampleWaves];
  __shared__ int32_t red_idx[kSampleWaves];
  __shared__ float red_min[kSampleWaves];
  __shared__ int32_t pick[2];
  __shared__ uint32_t member_count;
  __shared__ uint32_t member_key[kMemberCap];
  __shared__ int32_t member_idx[kMemberCap];    // one-pass top-k only: vocabulary index of a candidate
  __shared__ uint64_t member_mass[kMemberCap];

  const int r = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int V = p.V;
  const bool greedy = p.top_k == 1;
  const RowReader<DT, VEC> rd{reinterpret_cast<const uint8_t*>(p.logits) + (int64_t)r * p.stride * (DT != 0 ? 2 : 4), V,
                                p.inv_temperature, !greedy && p.inv_temperature != 1.0f};
  constexpr int U = VEC == 8 ? 4 : 8;  // 16-byte loads in flight per thread (32 values either way)

  // ---- pass A: maximum (lowest index among equals, NaN counts as largest) and finite minimum ----
  // (a thread meets its elements in rising index order, so "strictly greater" keeps the first)
  uint32_t bk = 0; int bi = 0x7fffffff; float mn = INFINITY;
  const bool filtering = !greedy && (p.top_k > 1 || p.top_p > 0.f);
  // `digit_select`: the key with exactly `target` list members (weights: 1, or the members' masses) above it, by four
  // 8-bit digit passes over member_key[0..n) starting from `above` (the weight already counted above the list).
  // With last_digit > 0 the low digits stay zero: a key at or below the exact one (a threshold that errs on the
  // side of more members).
  auto digit_select = [&](int n, uint64_t target, uint64_t above, bool by_mass, int last_digit) -> uint32_t {
    uint32_t pmask = 0, pval = 0;
    __syncthreads();
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
    for (int d = 3; d >= last_digit; --d) {
      for (int j0 = 0; j0 < n; j0 += kSampleThreads) {
        const int j = j0 + tid;
        const bool in = j < n;
        const uint32_t k = in ? member_key[j] : 0;
        hist_add(hist, 255 - (int)((k >> (8 * d)) & 255u), in && (k & pmask) == pval, lane,
                 [&] { return by_mass ? member_mass[j] : (uint64_t)1; });
      }
      __syncthreads();
      if (wave == 0) {  // the wavefront that reads the bins also clears them for the next digit: two barriers a pass
        find_crossing<4>(hist, above, target, res, lane);
#pragma unroll
        for (int j = 0; j < 4; ++j) hist[4 * lane + j] = 0;
      }
      __syncthreads();
      const uint32_t digit = 255u - (uint32_t)res[0];  // the crossing lies inside the list, so a digit is always found
      above = res[1];
      pmask |= 0xffu << (8 * d);
      pval |= digit << (8 * d);
    }
    return pval;
  };
  const bool one_pass = !greedy && V >= kFastMinVocab &&
                        (p.top_k > 1 ? p.top_k <= kFastTopK : p.top_p > 0.f);  // (top-p: one more pass for the total mass)
  constexpr int kSamplesPerThread = kMemberCap / kSampleThreads;
  uint32_t tau = 0;
  if (one_pass) {
    // threshold: the rank-th largest of kMemberCap sampled values, rank chosen for ~candidate_target(k) candidates
    const int blk = V / kSampleThreads;  // >= 16: thread t samples elements t * blk .. + 3
#pragma unroll
    for (int j = 0; j < kSamplesPerThread; ++j)
      member_key[tid * kSamplesPerThread + j] = order_key(rd.at(tid * blk + j));
    const int rank = min(kMemberCap / 2, (int)(((int64_t)candidate_target(p.top_k) * kMemberCap + V - 1) / V));
    // (the upper 16 bits of the key are enough: sign, exponent and 7 bits of the fraction)
    tau = digit_select(kMemberCap, (uint64_t)(rank - 1), 0, false, 2);
    if (tid == 0) member_count = 0;
    __syncthreads();  // the sample has been read by everyone; the list is reused for the candidates
    // one pass: the maximum (and, for top-p, which falls back to the general path often enough, the finite
    // minimum) and the list of candidates
    auto list_candidate = [&](uint32_t k, int i, bool cand) {
      const uint64_t m = __builtin_amdgcn_ballot_w64(cand);
      if (m == 0) return;
      uint32_t base = 0;
      const int first = __builtin_ctzll(m);
      if (lane == first) base = atomicAdd(&member_count, (uint32_t)__builtin_popcountll(m));
      base = __builtin_amdgcn_readlane(base, first);
      const uint32_t at = base + (uint32_t)__builtin_popcountll(m & (((uint64_t)1 << lane) - 1));
      if (cand && at < (uint32_t)kMemberCap) {
        member_key[at] = k;
        member_idx[at] = i;
      }
    };
    if (p.top_k > 1) {
      sweep<U>(rd, 0, V, tid, kSampleThreads, [&](int i, float x, bool in) {
        const uint32_t k = order_key(x);
        const bool up = in && k > bk;
        bk = up ? k : bk; bi = up ? i : bi;
        list_candidate(k, i, in && k >= tau);
      });
    } else {  // (half the loads in flight: with the minimum the full count no longer fits the registers)
      sweep<U / 2>(rd, 0, V, tid, kSampleThreads, [&](int i, float x, bool in) {
        const uint32_t k = order_key(x);
        const bool up = in && k > bk;
        bk = up ? k : bk; bi = up ? i : bi;
        mn = (in && x > -INFINITY) ? fminf(mn, x) : mn;
        list_candidate(k, i, in && k >= tau);
      });
    }
  } else if (filtering) {
    sweep<U>(rd, 0, V, tid, kSampleThreads, [&](int i, float x, bool in) {
      const uint32_t k = order_key(x);
      const bool up = in && k > bk;
      bk = up ? k : bk; bi = up ? i : bi;
      mn = (in && x > -INFINITY) ? fminf(mn, x) : mn;
    });
  } else {
    sweep<U>(rd, 0, V, tid, kSampleThreads, [&](int i, float x, bool in) {
      const uint32_t k = order_key(x);
      const bool up = in && k > bk;
      bk = up ? k : bk; bi = up ? i : bi;
    });
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    const uint32_t ok = __shfl_xor(bk, m, 64); const int oi = __shfl_xor(bi, m, 64);
    if (ok > bk || (ok == bk && oi < bi)) { bk = ok; bi = oi; }
    mn = fminf(mn, __shfl_xor(mn, m, 64));
  }
  if (lane == 0) { red_key[wave] = bk; red_idx[wave] = bi; red_min[wave] = mn; }
  __syncthreads();
  bk = red_key[0]; bi = red_idx[0]; mn = red_min[0];
#pragma unroll
  for (int w = 1; w < kSampleWaves; ++w) {
    const uint32_t ok = red_key[w]; const int oi = red_idx[w];
    if (ok > bk || (ok == bk && oi < bi)) { bk = ok; bi = oi; }
    mn = fminf(mn, red_min[w]);
  }
  if (bi >= V) bi = 0;  // only when no element compared greater than the start value
  const float mx = order_key_value(bk);
  int sample = bi;
  uint32_t cut_key = 0;  // keep everything

  const bool drawable = !greedy && has_masses(mx);   // (otherwise: the argmax)
  const float neg_mx = -mx * 1.4426950408889634f;
  if (drawable) {
    const bool by_count = p.top_k > 1;
    const bool filtered = by_count || p.top_p > 0.f;
    bool cut_from_list = false;
    int n_candidates = 0;
    if (one_pass) {
      n_candidates = (int)member_count;  // (published by the barrier of the maximum's reduction)
      bool usable = n_candidates <= kMemberCap && (by_count ? n_candidates >= p.top_k : n_candidates > 0);
      uint64_t target = by_count ? (uint64_t)(p.top_k - 1) : 0;
      if (usable && !by_count) {
        // top-p: the row's total mass (one more pass), then the candidates' masses; the cut lies inside the list
        // when those alone exceed top_p of the total
        auto workgroup_sum = [&](uint64_t v) -> uint64_t {
          v = wave_sum_u64(v);
          __syncthreads();
          if (lane == 0) wsum[wave] = v;
          __syncthreads();
          uint64_t t = 0;
#pragma unroll
          for (int w = 0; w < kSampleWaves; ++w) t += wsum[w];
          return t;
        };
        uint64_t c = 0;
        for (int j = tid; j < n_candidates; j += kSampleThreads) {
          const uint64_t m = mass_of(order_key_value(member_key[j]), neg_mx);
          member_mass[j] = m;
          c += m;
        }
        c = workgroup_sum(c);
        // Worth the pass?  The mass below the threshold is many small terms, so the sample estimates it well
        // (unlike the mass above it, which a few elements can hold); a quarter on top of the estimate as margin, so
        // that rows on the edge do not pay for the total-mass pass and then fail.
        // (the sampled values are read again rather than kept in registers through the passes above)
        uint64_t below = 0;
#pragma unroll
        for (int j = 0; j < kSamplesPerThread; ++j) {
          const float x = rd.at(tid * (V / kSampleThreads) + j);
          const uint64_t w = mass_of(x, neg_mx);
          below += order_key(x) < tau ? w : 0;
        }
        const double rest = (double)workgroup_sum(below) * ((double)V / kMemberCap) * 1.25;
        usable = (double)c > (double)p.top_p * ((double)c + rest);
        if (usable) {
          uint64_t z = 0;
          sweep<U>(rd, 0, V, tid, kSampleThreads, [&](int, float x, bool in) {
            const uint64_t w = mass_of(x, neg_mx);
            z += in ? w : 0;
          });
          z = workgroup_sum(z);
          target = (uint64_t)((double)p.top_p * (double)z);
          usable = c > target;
        }
      }
      if (usable) {
        cut_key = digit_select(n_candidates, target, 0, !by_count, 0);
        cut_from_list = true;
      } else if (by_count) {
        // the general path needs the finite minimum, which the one-pass sweep did not track for top-k
        sweep<U>(rd, 0, V, tid, kSampleThreads, [&](int, float x, bool in) {
          mn = (in && x > -INFINITY) ? fminf(mn, x) : mn;
        });
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) mn = fminf(mn, __shfl_xor(mn, m, 64));
        __syncthreads();
        if (lane == 0) red_min[wave] = mn;
        __syncthreads();
        mn = red_min[0];
#pragma unroll
        for (int w = 1; w < kSampleWaves; ++w) mn = fminf(mn, red_min[w]);
      }
    }
    if (filtered && !cut_from_list) {
      // ---- pass B: 256 linear bins over [mx - range, mx], bin 0 = largest values ----
      float range = mx - mn;
      if (!by_count) range = fminf(range, 32.f);  // mass below exp(-32) cannot move a top-p cut
      const float inv_w = range > 0.f ? 256.f / range : 0.f;
      auto lin_bin = [&](float x) {
        const float f = (mx - x) * inv_w;
        return (int)fmaxf(fminf(f, 255.f), 0.f);  // (NaN, of -inf times 0 or with its sign set: the lowest)
      };
      auto weight_of = [&](float x) -> uint64_t { return by_count ? (uint64_t)1 : mass_of(x, neg_mx); };
      if (tid < 256) hist[tid] = 0;
      if (tid == 0) member_count = 0;
      __syncthreads();
      sweep<U>(rd, 0, V, tid, kSampleThreads, [&](int, float x, bool in) {
        hist_add(hist, lin_bin(x), in, lane, [&] { return weight_of(x); });
      });
      __syncthreads();
      uint64_t target;
      if (by_count) {
        target = (uint64_t)(p.top_k - 1);
      } else {
        uint64_t z = 0;
        for (int j = 0; j < 256; ++j) z += hist[j];  // same LDS words for every lane: broadcast reads
        target = (uint64_t)((double)p.top_p * (double)z);
      }
      if (wave == 0) find_crossing<4>(hist, 0, target, res, lane);
      __syncthreads();
      const int lbin = (int)(int64_t)res[0];
      uint64_t above = res[1];
      if (lbin >= 0) {
        // ---- pass C: list the members of the chosen bin in LDS (wavefront-aggregated append) ----
        sweep<U>(rd, 0, V, tid, kSampleThreads, [&](int, float x, bool in) {
          const bool member = in && lin_bin(x) == lbin;
          const uint64_t m = __builtin_amdgcn_ballot_w64(member);
          if (m == 0) return;
          uint32_t base = 0;
          const int first = __builtin_ctzll(m);
          if (lane == first) base = atomicAdd(&member_count, (uint32_t)__builtin_popcountll(m));
          base = __builtin_amdgcn_readlane(base, first);
          const uint32_t at = base + (uint32_t)__builtin_popcountll(m & (((uint64_t)1 << lane) - 1));
          if (member && at < (uint32_t)kMemberCap) {
            member_key[at] = order_key(x);
            member_mass[at] = weight_of(x);
          }
        });
        __syncthreads();
        const int n_members = (int)member_count;
        const bool listed = n_members <= kMemberCap;
        // ---- four 8-bit digit passes over the members (the LDS list, or the row when it overflowed) ----
        uint32_t pmask = 0, pval = 0;
        for (int d = 3; d >= 0; --d) {
          __syncthreads();
          if (tid < 256) hist[tid] = 0;
          __syncthreads();
          if (listed) {
            for (int j0 = 0; j0 < n_members; j0 += kSampleThreads) {
              const int j = j0 + tid;
              const bool in = j < n_members;
              const uint32_t k = in ? member_key[j] : 0;
              hist_add(hist, 255 - (int)((k >> (8 * d)) & 255u), in && (k & pmask) == pval, lane,
                       [&] { return member_mass[j]; });
            }
          } else {
            sweep<U>(rd, 0, V, tid, kSampleThreads, [&](int, float x, bool in) {
              const uint32_t k = order_key(x);
              hist_add(hist, 255 - (int)((k >> (8 * d)) & 255u), in && lin_bin(x) == lbin && (k & pmask) == pval, lane,
                       [&] { return weight_of(x); });
            });
          }
          __syncthreads();
          if (wave == 0) find_crossing<4>(hist, above, target, res, lane);
          __syncthreads();
          // the crossing lies inside the chosen bin, so a digit is always found
          const uint32_t digit = 255u - (uint32_t)res[0];
          above = res[1];
          pmask |= 0xffu << (8 * d);
          pval |= digit << (8 * d);
        }
        cut_key = pval;
      }
    }

    // ---- draw on the candidate list: the kept elements are among the candidates, so when they are few the
    // inverse CDF in vocabulary order is a direct count over the list (each thread owns one kept element and sums
    // the masses of those at or before it) ----
    bool drawn = false;
    if (cut_from_list) {
      __syncthreads();
      if (tid == 0) member_count = 0;
      __syncthreads();
      for (int j0 = 0; j0 < n_candidates; j0 += kSampleThreads) {
        const int j = j0 + tid;
        const bool kept = j < n_candidates && member_key[j] >= cut_key;
        const uint64_t m = __builtin_amdgcn_ballot_w64(kept);
        if (m == 0) continue;
        uint32_t base = 0;
        const int first = __builtin_ctzll(m);
        if (lane == first) base = atomicAdd(&member_count, (uint32_t)__builtin_popcountll(m));
        base = __builtin_amdgcn_readlane(base, first);
        const uint32_t at = base + (uint32_t)__builtin_popcountll(m & (((uint64_t)1 << lane) - 1));
        // (vocabulary index and mass of a kept element in one word: a mass fits 32 bits)
        if (kept) member_mass[at] = ((uint64_t)(uint32_t)member_idx[j] << 32) | mass_of(order_key_value(member_key[j]), neg_mx);
      }
      __syncthreads();
      const int n_kept = (int)member_count;
      if (n_kept <= kSampleThreads) {
        if (wave * 64 < n_kept) {  // only the wavefronts that own a kept element walk the list
          const uint64_t mine = tid < n_kept ? member_mass[tid] : 0;
          const uint32_t my_idx = (uint32_t)(mine >> 32);
          uint64_t total = 0, upto = 0;  // all kept mass; kept mass at vocabulary indices <= mine
          for (int m = 0; m < n_kept; ++m) {
            const uint64_t e = member_mass[m];  // the same word for every lane: a broadcast read
            const uint64_t w = e & 0xffffffffu;
            total += w;
            upto += (uint32_t)(e >> 32) <= my_idx ? w : 0;
          }
          uint64_t want = (uint64_t)((double)p.uniform[r] * (double)total);
          want = want < total ? want : total - 1;
          const uint64_t w_mine = mine & 0xffffffffu;
          if (tid < n_kept && upto > want && upto - w_mine <= want) pick[0] = (int)my_idx;
        }
        drawn = true;
      }
    }
    auto kept_mass = [&](float x) -> uint64_t {
      const uint64_t w = mass_of(x, neg_mx);
      return order_key(x) >= cut_key ? w : 0;
    };
    if (!drawn) {
      const int L1 = ((V + kSampleWaves - 1) / kSampleWaves + 63) & ~63;  // elements per first-level range
      {
        const int a = min(wave * L1, V), b = min(a + L1, V);
        uint64_t s = 0;
        sweep<U>(rd, a, b, lane, 64, [&](int, float x, bool in) { s += in ? kept_mass(x) : 0; });
        s = wave_sum_u64(s);
        if (lane == 0) wsum[wave] = s;
      }
      __syncthreads();
      uint64_t total = 0;
#pragma unroll
      for (int w = 0; w < kSampleWaves; ++w) total += wsum[w];
      // total > 0: the maximum itself is always kept and has the largest mass
      uint64_t want = (uint64_t)((double)p.uniform[r] * (double)total);
      want = want < total ? want : total - 1;
      int w1 = 0;
#pragma unroll
      for (int w = 0; w < kSampleWaves - 1; ++w) {
        const bool pass = w == w1 && want >= wsum[w];
        want -= pass ? wsum[w] : 0;
        w1 += pass ? 1 : 0;
      }
      // (ranges after the last non-empty one hold no mass, so w1 stops inside the vocabulary)
      const int a1 = min(w1 * L1, V), b1 = min(a1 + L1, V);
      const int L2 = (L1 / kSampleWaves + 63) & ~63;  // elements per second-level range
      __syncthreads();
      {
        const int a = min(a1 + wave * L2, b1), b = min(a + L2, b1);
        uint64_t s = 0;
        sweep<1>(rd, a, b, lane, 64, [&](int, float x, bool in) { s += in ? kept_mass(x) : 0; });
        s = wave_sum_u64(s);
        if (lane == 0) wsum[wave] = s;
      }
      __syncthreads();
      int w2 = 0;
#pragma unroll
      for (int w = 0; w < kSampleWaves - 1; ++w) {
        const bool pass = w == w2 && want >= wsum[w];
        want -= pass ? wsum[w] : 0;
        w2 += pass ? 1 : 0;
      }
      const int a2 = min(a1 + w2 * L2, b1), b2 = min(a2 + L2, b1);
      if (wave == 0) {
        // third level: each lane owns a contiguous run of the sub-range
        const int per = L2 / 64;
        const int a = min(a2 + lane * per, b2), b = min(a + per, b2);
        uint64_t s = 0;
        for (int i = a; i < b; ++i) s += kept_mass(rd.at(i));
        const uint64_t incl = wave_scan_incl_u64(s, lane);
        const uint64_t m = __builtin_amdgcn_ballot_w64(incl > want);
        const int owner = m ? __builtin_ctzll(m) : 63;
        if (lane == owner) {
          uint64_t run = incl - s;
          int found = b > a ? b - 1 : bi;
          for (int i = a; i < b; ++i) {
            run += kept_mass(rd.at(i));
            if (run > want) { found = i; break; }
          }
          pick[0] = found;
        }
      }
    }
    __syncthreads();
    sample = pick[0];
    if (p.vocab_clamp > 0) sample = min(max(sample, 0), p.vocab_clamp - 1);
  }

  if (tid == 0) write_sample(p, r, sample, cut_key);
}

// ---- the same over several workgroups per row -------------------------------------------------------------------
// One workgroup per row leaves most of the chip idle while it walks the row up to five times (64 rows: 64 of 256 CUs;
// 64 x 128 256 fp32, top-p 0.9 on flat rows: 105 us against 5 us for one read).  Here a row is cut into parts of one
// workgroup each, and the walk into launches that read the parts once each:
//   sample_first_kernel : a part's maximum (with its index); top-p: the part's mass in bins of 1/64, counted down from the
//                         bin of its maximum on a grid that all parts share; top-k: the part's candidates, listed (the
//                         elements at or above a threshold estimated from 1 024 of them);
//   sample_mass_kernel  : (top-p and plain draws) the exact masses: the part's total, and per run of elements what lies
//                         above the bins that hold the cut; the elements in those bins, listed;
//   sample_pick_kernel  : one workgroup per row: the exact cut among the listed elements, the run of elements the
//                         uniform number falls into, the element.
// Every mass is the integer of the one-workgroup form and every sum that decides is exact, so the tokens are the same
// ones; the estimates only choose what is listed, and the pick checks them.  Where they fail (thousands of equal values,
// more than the list holds) its workgroup walks the row instead of the list.
//
// fp32, 128 256 wide, us per call in a graph, one workgroup per row -> parts (flat rows: N(0, 3); peaked: 32 logits 9-15 above
// N(0, 2)):
//   64 rows: greedy 15 -> 12, plain 37 -> 21, top-k 50 39 -> 31, top-p 0.9 102 -> 28 (flat rows), 54 -> 27 (peaked)
//    1 row : greedy 13 ->  6, plain 34 -> 13, top-k 50 36 -> 18, top-p 0.9  70 -> 21 (flat rows), 50 -> 20 (peaked)
// 64 flat rows, top-p, by trace: 8.4 us for the first walk, 10.3-11 for the second, 8.4-9 for the pick (a chain of loads and
// barriers).  Both walks are vector arithmetic and one burst of loads: what they gained (17.9, 14.5 and 11.7 us) is fewer
// instructions per value.  The first took 38, with bins below a sampled reference, an exponential and a 64-bit addition to
// LDS per value; with the batch in registers its own maximum is the reference, a 32-bit weight within the bin does, and
// bins a quarter as wide leave a third of the values on the lists.  The second claimed its place on the list for one value
// of each lane at a time and held the window's comparison against bins; 1.6 of its time are lists, 1.5 what is kept, 1
// the masses, 3 the bins of the other parts.
constexpr int kBins = 2048;           // of 1/64, from the bin of the largest value down (all that is lower: none)
constexpr float kBinsPerUnit = 64.f;
constexpr int kRuns = kSampleWaves;   // runs of elements per part
constexpr int kMaxParts = 64;
constexpr int kPartSample = 1024;

struct SplitParams {
  SampleParams s;
  int32_t parts, part_len, run_len;    // elements (multiples of 8); a part is kRuns runs
  int32_t list_cap;                    // listed elements per part
  uint32_t* part_key; int32_t* part_idx;  // [R][parts] maximum
  uint32_t* part_tau;                  // [R][parts] top-k: the threshold of the part's candidates; top-p: its first bin's number
  uint32_t* part_listed;               // [R][parts]
  uint32_t* bins;                      // [R][parts][kBins]: sums of exp(x - the bin's upper edge), in units of 1 / bin_one
  float bin_one;                       // (a row of equal values stays below 2^32)
  uint64_t* part_mass;                 // [R][parts] exact total
  uint64_t* run_mass;                  // [R][parts][kRuns] exact mass above the listed bins
  uint2* list;                         // [R][parts][list_cap]: key, vocabulary index
};

template <int DT, int VEC>
static __device__ __forceinline__ RowReader<DT, VEC> row_reader(const SampleParams& p, int r) {
  return RowReader<DT, VEC>{reinterpret_cast<const uint8_t*>(p.logits) + (int64_t)r * p.stride * (DT != 0 ? 2 : 4), p.V,
                            p.inv_temperature, p.top_k != 1 && p.inv_temperature != 1.0f};
}

// The row's maximum (lowest index among equals) from its parts', the same in every lane.
struct RowMax { uint32_t key; int32_t idx; };
static __device__ __forceinline__ RowMax row_max(const SplitParams& p, int r, int lane) {
  RowMax m{0, 0x7fffffff};
  if (lane < p.parts) {
    const int64_t at = (int64_t)r * p.parts + lane;
    m = RowMax{p.part_key[at], p.part_idx[at]};
  }
  const uint32_t key = wave_max_u32(m.key);
  m.idx = (int32_t)~wave_max_u32(m.key == key ? ~(uint32_t)m.idx : 0);  // (the lowest of the indices)
  m.key = key;
  if (m.idx >= p.s.V) m.idx = 0;  // only when no element compared greater than the start value
  return m;
}

// Appends one element per lane with `in` set to a list of `cap` entries; `count` goes on counting past it.
template <typename F>
static __device__ __forceinline__ void list_append(uint32_t* count, uint32_t cap, bool in, int lane, F store) {
  const uint64_t m = __builtin_amdgcn_ballot_w64(in);
  if (m == 0) return;
  uint32_t base = 0;
  const int first = __builtin_ctzll(m);
  if (lane == first) base = atomicAdd(count, (uint32_t)__builtin_popcountll(m));
  base = __builtin_amdgcn_readlane(base, first);
  const uint32_t at = base + (uint32_t)__builtin_popcountll(m & (((uint64_t)1 << lane) - 1));
  if (in && at < cap) store(at);
}

enum { kPickMax = 0, kPickTopK = 1, kPickTopP = 2 };

template <int DT, int VEC, int MODE, int BATCH>
__global__ __launch_bounds__(kSampleThreads) void sample_first_kernel(SplitParams p) {
  __shared__ uint32_t red_key[kSampleWaves];
  __shared__ int32_t red_idx[kSampleWaves];
  __shared__ uint32_t mass[MODE == kPickTopP ? kBins : 1];
  __shared__ uint32_t sampled[MODE == kPickTopK ? kPartSample : 1];
  __shared__ uint64_t hist[MODE == kPickTopK ? 256 : 1];
  __shared__ uint64_t res[2];
  __shared__ uint32_t listed;
  const int part = blockIdx.x, r = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const auto rd = row_reader<DT, VEC>(p.s, r);
  const int a = min(part * p.part_len, p.s.V), b = min(a + p.part_len, p.s.V);
  const int64_t row_part = (int64_t)r * p.parts + part;
  uint32_t tau = 0;
  if (MODE == kPickTopK) {
    // threshold: a rank of the sample that leaves three times this part's share of the top k above it, and twelve
    // of the sample at least (a dozen of it stand for 8-20 of the same spacing in all but a few of 10^5 parts)
    const int len = b - a;
    if (tid < kPartSample / 4) {
      const int at = a + (int)((int64_t)tid * len / (kPartSample / 4));
#pragma unroll
      for (int j = 0; j < 4; ++j) sampled[4 * tid + j] = order_key(rd.at(min(at + j, p.s.V - 1)));
    }
    if (tid < 256) hist[tid] = 0;
    if (tid == 0) listed = 0;
    const int share = (3 * p.s.top_k + p.parts - 1) / p.parts;
    const int rank = min(kPartSample / 2, max(12, (int)(((int64_t)share * kPartSample + len - 1) / max(len, 1))));
    __syncthreads();
    uint32_t pmask = 0;
    uint64_t above = 0;
    for (int d = 3; d >= 2; --d) {  // (the upper 16 bits of the key are enough)
      const uint32_t k = sampled[tid];
      hist_add(hist, 255 - (int)((k >> (8 * d)) & 255u), (k & pmask) == tau, lane, [&] { return (uint64_t)1; });
      __syncthreads();
      if (wave == 0) {
        find_crossing<4>(hist, above, (uint64_t)(rank - 1), res, lane);
#pragma unroll
        for (int j = 0; j < 4; ++j) hist[4 * lane + j] = 0;
      }
      __syncthreads();
      above = res[1];
      pmask |= 0xffu << (8 * d);
      tau |= (255u - (uint32_t)res[0]) << (8 * d);
    }
  }
  uint2* list = p.list + row_part * p.list_cap;
  uint32_t bk = 0; int bi = 0x7fffffff;
  bool indexed = true;
  if (MODE == kPickTopP) {
    // A batch lies in registers while its maximum is found, then goes into bins counted down from the bin of the largest
    // value so far; where that moves up, the bins move with it.
    static_assert(kBins == 2 * kSampleThreads, "two bins per thread");
    float first = -INFINITY;          // number of the first bin: floor(64 x) of the largest value
    mass[tid] = mass[tid + kSampleThreads] = 0;
    for (int base = a; base < b; base += BATCH * kSampleThreads) {
      float x[BATCH / VEC][VEC];
      load_batch<BATCH>(rd, base, b, tid, kSampleThreads, x);
      // as integers, numbers from +0 up are in order, NaN above them; among values below 0 the floats' order counts
      int32_t top_i = INT32_MIN;
      float top_f = -INFINITY;
#pragma unroll
      for (int u = 0; u < BATCH / VEC; ++u)
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
          top_i = max(top_i, __float_as_int(x[u][j]));
          top_f = fmaxf(top_f, x[u][j]);
        }
      bk = max(bk, top_i >= 0 ? (uint32_t)top_i | 0x80000000u : order_key(top_f + 0.f));
      bk = wave_max_u32(bk);
      __syncthreads();   // (the batch before has been read and counted)
      if (lane == 0) red_key[wave] = bk;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < kSampleWaves; ++w) bk = max(bk, red_key[w]);
      const float now = floorf(order_key_value(bk) * kBinsPerUnit);
      if (now > first) {
        if (base > a) {
          const int by = (int)fminf(now - first, (float)kBins), i0 = tid - by, i1 = i0 + kSampleThreads;
          const uint32_t m0 = i0 >= 0 ? mass[i0] : 0, m1 = i1 >= 0 ? mass[i1] : 0;
          __syncthreads();
          mass[tid] = m0;
          mass[tid + kSampleThreads] = m1;
          __syncthreads();
        }
        first = now;
      }
      const float edge = first + 1.f;
#pragma unroll
      for (int u = 0; u < BATCH / VEC; ++u)
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
          // distance from the first bin's upper edge, in bins; exp(-t / 64) by its chord, lowered to within 1.6e-5
          const float f = __builtin_fmaf(x[u][j], -kBinsPerUnit, edge);
          const float w = __builtin_fmaf(__builtin_amdgcn_fractf(f), -0.01550356f * p.bin_one, 0.99998474f * p.bin_one + 0.5f);
          // (a masked value is an infinite distance away, NaN no distance: both fail the comparison)
          if (f < (float)kBins) atomicAdd(&mass[(uint32_t)fmaxf(f, 0.f)], (uint32_t)w);
        }
    }
    // The index matters where there may be nothing to draw from: no finite maximum (that of a part of nothing but -inf and
    // NaN was not found), or one so large that its own mass may round to nothing.
    indexed = !(fabsf(order_key_value(bk)) < 1e6f);
    __syncthreads();
    reinterpret_cast<uint2*>(p.bins + row_part * kBins)[tid] = make_uint2(mass[2 * tid], mass[2 * tid + 1]);
    if (tid == 0) p.part_tau[row_part] = __float_as_uint(first);
    if (!indexed) {
      if (tid == 0) { p.part_key[row_part] = bk; p.part_idx[row_part] = a; p.part_listed[row_part] = 0; }
      return;
    }
    bk = 0;
  }
  sweep<(VEC == 8 ? 4 : 8)>(rd, a, b, tid, kSampleThreads, [&](int i, float x, bool in) {
    const uint32_t k = order_key(x);
    const bool up = in && k > bk;
    bk = up ? k : bk; bi = up ? i : bi;
    if (MODE == kPickTopK)
      list_append(&listed, (uint32_t)p.list_cap, in && k >= tau, lane, [&](uint32_t at) { list[at] = make_uint2(k, (uint32_t)i); });
  });
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    const uint32_t ok = __shfl_xor(bk, m, 64); const int oi = __shfl_xor(bi, m, 64);
    if (ok > bk || (ok == bk && oi < bi)) { bk = ok; bi = oi; }
  }
  if (lane == 0) { red_key[wave] = bk; red_idx[wave] = bi; }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kSampleWaves; ++w) {
      const uint32_t ok = red_key[w]; const int oi = red_idx[w];
      if (ok > bk || (ok == bk && oi < bi)) { bk = ok; bi = oi; }
    }
    p.part_key[row_part] = bk; p.part_idx[row_part] = bi;
    p.part_listed[row_part] = MODE == kPickTopK ? listed : 0;
    if (MODE == kPickTopK) p.part_tau[row_part] = tau;
  }
}

// Exact masses.  top-p lists the values in the bins around the estimated cut; a plain draw lists nothing.
template <int DT, int VEC, int BATCH>
__global__ __launch_bounds__(kSampleThreads) void sample_mass_kernel(SplitParams p) {
  __shared__ float red[kSampleWaves];
  __shared__ int32_t window[2];
  __shared__ uint64_t wsum[kSampleWaves];
  __shared__ uint32_t listed;
  __shared__ uint32_t row_bins[kBins];
  const int part = blockIdx.x, r = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const auto rd = row_reader<DT, VEC>(p.s, r);
  const int pa = part * p.part_len, a = min(pa + wave * p.run_len, p.s.V), b = min(min(a + p.run_len, pa + p.part_len), p.s.V);
  const int64_t row = (int64_t)r * p.parts, row_part = row + part;
  const bool filtered = p.s.top_p > 0.f;
  // (the first batch and the first parts' bins set out before anything is waited for)
  float x[BATCH / VEC][VEC];
  load_batch<BATCH>(rd, a, b, lane, 64, x);
  // (256 bins of one part at a time per wavefront)
  constexpr int kItems = kBins / 256, kFirstItems = 2;
  uint4 first_items[kFirstItems];
  const uint4* const bins_src = reinterpret_cast<const uint4*>(p.bins + row * kBins) + lane;
  const int n_items = filtered ? p.parts * kItems : 0;
  if (filtered) {
#pragma unroll
    for (int n = 0; n < kFirstItems; ++n)
      first_items[n] = bins_src[64 * min(wave + n * kSampleWaves, n_items - 1)];
    row_bins[tid] = row_bins[tid + kSampleThreads] = 0;
  }
  const uint32_t part_key = lane < p.parts ? p.part_key[row + lane] : 0;
  float first = lane < p.parts && filtered ? __uint_as_float(p.part_tau[row + lane]) : -INFINITY;
  const float mx = order_key_value(wave_max_u32(part_key)), neg_mx = -mx * 1.4426950408889634f;
  if (!has_masses(mx)) return;
  if (tid == 0) { window[0] = kBins; window[1] = -1; listed = 0; }
  const float row_first = floorf(mx * kBinsPerUnit);
  const int down = (int)fminf(row_first - first, (float)kBins);   // by how many bins each part's begin below the row's
  uint64_t kept = 0;
  uint32_t all_lo = 0, all_hi = 0;
  auto masses = [&] {
#pragma unroll
    for (int u = 0; u < BATCH / VEC; ++u)
#pragma unroll
      for (int j = 0; j < VEC; ++j) add_mass(all_lo, all_hi, x[u][j], neg_mx);
  };
  masses();
  float over = INFINITY, from = INFINITY;   // kept: above `over`; listed: from `from` to `over`
  if (filtered) {
    // The parts' bins on the row's scale, two per thread; the bin in which the running sum passes top_p of the total, with
    // its neighbours where it passes within `slack` of the edge.  A value's weight is off by up to 1.6e-5 (the chord) and half
    // a unit of 1 / bin_one (rounding) of itself, the share of the total that lies above an edge by a quarter of the range of
    // these: 0.8e-5 + 0.26 / bin_one, 1.6e-5 up to 131 071 values, 4e-5 from 262 144 and 1.3e-4 from 2^20 on.
    auto add_item = [&](int n, uint4 c) {
      const int at = 256 * (n % kItems) + 4 * lane + __builtin_amdgcn_readlane(down, n / kItems);
      const uint32_t v[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (at + j < kBins && v[j]) atomicAdd(&row_bins[at + j], v[j]);
    };
    __syncthreads();   // (the bins are cleared)
#pragma unroll
    for (int n = 0; n < kFirstItems; ++n)
      if (wave + n * kSampleWaves < n_items) add_item(wave + n * kSampleWaves, first_items[n]);
    for (int n0 = wave + kFirstItems * kSampleWaves; n0 < n_items; n0 += 8 * kSampleWaves) {
      uint4 c[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) c[i] = bins_src[64 * min(n0 + i * kSampleWaves, n_items - 1)];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (n0 + i * kSampleWaves < n_items) add_item(n0 + i * kSampleWaves, c[i]);
    }
    __syncthreads();
    const float h0 = (float)row_bins[2 * tid] * fast_exp2((float)(2 * tid) * (-1.4426950408889634f / kBinsPerUnit));
    const float h1 = (float)row_bins[2 * tid + 1] * fast_exp2((float)(2 * tid + 1) * (-1.4426950408889634f / kBinsPerUnit));
    const float h = h0 + h1;
    float incl = wave_scan_incl_f32(h);
    if (lane == 63) red[wave] = incl;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < kSampleWaves; ++w) {
      incl += w < wave ? red[w] : 0.f;
      total += red[w];
    }
    const float want = p.s.top_p * total, slack = fmaxf(1e-4f, 3e-5f + 0.3f / p.bin_one) * total;
    const bool in0 = incl - h - slack <= want && incl - h1 + slack > want && h0 > 0.f;
    const bool in1 = incl - h1 - slack <= want && incl + slack > want && h1 > 0.f;
    if (in0 || in1) {
      atomicMin(&window[0], in0 ? 2 * tid : 2 * tid + 1);
      atomicMax(&window[1], in1 ? 2 * tid + 1 : 2 * tid);
    }
    __syncthreads();
    const int lo = window[0], hi = window[1];
    if (lo <= hi) {   // (nothing found, as where a value is not a number: nothing is listed, and the pick walks the row)
      over = (row_first + 1.f - (float)lo) * (1.f / kBinsPerUnit);
      from = (row_first - (float)hi) * (1.f / kBinsPerUnit);
    }
  } else {
    __syncthreads();
  }
  uint2* list = p.list + row_part * p.list_cap;
  for (int base = a; base < b;) {
    if (filtered) {   // one claim on the list for sixteen values a lane
      constexpr int HALF = BATCH / 2;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        uint64_t in_window[HALF];
        uint32_t found = 0;
#pragma unroll
        for (int n = 0; n < HALF; ++n) {
          const float v = x[(half * HALF + n) / VEC][(half * HALF + n) % VEC];
          uint64_t m = __builtin_amdgcn_ballot_w64(v >= from);
          if (m) {   // (few values are: their mass again is less than holding it)
            const bool is_over = v > over;
            const uint64_t w = mass_of(v, neg_mx);
            kept += is_over ? w : 0;
            m &= ~__builtin_amdgcn_ballot_w64(is_over);
            found += (uint32_t)__builtin_popcountll(m);
          }
          in_window[n] = m;
        }
        if (found == 0) continue;
        uint32_t at = 0;
        if (lane == 0) at = atomicAdd(&listed, found);
        at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
        for (int n = 0; n < HALF; ++n) {
          const uint64_t m = in_window[n];
          if (m == 0) continue;
          const int u = (half * HALF + n) / VEC, j = (half * HALF + n) % VEC;
          const uint32_t mine = at + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
          if (((m >> lane) & 1) && mine < (uint32_t)p.list_cap)
            list[mine] = make_uint2(order_key(x[u][j] + 0.f), (uint32_t)(base + (u * 64 + lane) * VEC + j));
          at += (uint32_t)__builtin_popcountll(m);
        }
      }
    }
    base += BATCH * 64;
    if (base < b) {
      load_batch<BATCH>(rd, base, b, lane, 64, x);
      masses();
    }
  }
  uint64_t all = wave_sum_u64(((uint64_t)all_hi << 32) | all_lo);
  kept = filtered ? wave_sum_u64(kept) : all;
  if (lane == 0) {
    p.run_mass[row_part * kRuns + wave] = kept;
    wsum[wave] = all;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kSampleWaves; ++w) all += wsum[w];
    p.part_mass[row_part] = all;
    p.part_listed[row_part] = listed;
  }
}

// The exact cut of a filter, in LDS: the key with at most `target` of weight above it and more with itself.  `hist` has 512
// cleared words before and after; every thread of the workgroup calls, and every one sees *cut afterwards.
struct CutShared { uint64_t* hist; uint64_t* res; uint32_t* cut; };

// By four 8-bit digits.  each(count) calls count(key, in, weight) for everything that lies below what `before` counts.
template <typename Each>
static __device__ void digit_cut(const CutShared& cs, uint64_t before, uint64_t target, int tid, Each each) {
  const int lane = tid & 63, wave = tid >> 6;
  uint32_t pmask = 0, pval = 0;
  for (int d = 3; d >= 0; --d) {
    each([&](uint32_t k, bool in, auto weight) {
      hist_add(cs.hist, 255 - (int)((k >> (8 * d)) & 255u), in && (k & pmask) == pval, lane, weight);
    });
    __syncthreads();
    if (wave == 0) {  // (the wavefront that reads the bins also clears them for the next digit)
      find_crossing<4>(cs.hist, before, target, cs.res, lane);
#pragma unroll
      for (int j = 0; j < 4; ++j) cs.hist[4 * lane + j] = 0;
    }
    __syncthreads();
    before = cs.res[1];
    pmask |= 0xffu << (8 * d);
    pval |= (255u - (uint32_t)cs.res[0]) << (8 * d);
  }
  if (tid == 0) *cs.cut = pval;
  __syncthreads();
}
template <typename Count>
static __device__ __forceinline__ void count_list(const uint32_t* key, const uint32_t* mass, int n, bool by_count, int tid, Count count) {
  for (int j0 = 0; j0 < n; j0 += kSampleThreads) {
    const int j = j0 + tid;
    count(j < n ? key[j] : 0, j < n, [&]() -> uint64_t { return by_count ? 1u : mass[j]; });
  }
}
// Of up to 256 listed elements, every one against every other: 64 elements a wavefront, the wavefronts of the same elements
// a share of the others each (one wavefront takes 15 ns per other element).
static __device__ __forceinline__ void pair_cut(const CutShared& cs, const uint32_t* key, const uint32_t* mass, int n, bool by_count,
                                                uint64_t above, uint64_t target, int tid) {
  const int lane = tid & 63, wave = tid >> 6;
  const int blocks = n <= 64 ? 1 : n <= 128 ? 2 : 4, shares = kSampleWaves / blocks;
  const int at = 64 * (wave % blocks) + lane, share = wave / blocks;
  const int j1 = (int)((int64_t)n * (share + 1) / shares);
  const uint32_t mine = at < n ? key[at] : 0;
  uint64_t over = 0, equal = 0;
  for (int j = n * share / shares; j < j1; ++j) {   // the same words for every lane: broadcast reads
    const uint32_t k = key[j], w = by_count ? 1u : mass[j];
    over += k > mine ? w : 0;
    equal += k == mine ? w : 0;
  }
  if (at < n) {
    atomicAdd(reinterpret_cast<unsigned long long*>(&cs.hist[at]), (unsigned long long)over);
    atomicAdd(reinterpret_cast<unsigned long long*>(&cs.hist[256 + at]), (unsigned long long)equal);
  }
  __syncthreads();
  if (tid < n && above + cs.hist[tid] <= target && above + cs.hist[tid] + cs.hist[256 + tid] > target) *cs.cut = key[tid];
  __syncthreads();
  if (tid < 512) cs.hist[tid] = 0;   // (for the digits, should the list turn out not to hold the cut)
  __syncthreads();
}

template <int DT, int VEC>
__global__ __launch_bounds__(kSampleThreads) void sample_pick_kernel(SplitParams p) {
  const int r = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  __shared__ uint32_t key[kMemberCap];
  __shared__ uint32_t mass[kMemberCap];     // (a mass fits 32 bits)
  __shared__ uint32_t index[kMemberCap];
  __shared__ uint64_t runs[kMaxParts * kRuns];
  __shared__ uint64_t hist[512];
  __shared__ uint64_t res[2];
  __shared__ uint64_t wsum[3][kSampleWaves];
  __shared__ uint32_t cut;
  __shared__ int32_t pick;
  const bool by_count = p.s.top_k > 1, by_mass = p.s.top_k == 0 && p.s.top_p > 0.f, filtered = by_count || by_mass;
  const int64_t row = (int64_t)r * p.parts;
  const int n_runs = p.parts * kRuns;
  // (everything that does not depend on the maximum is asked for before it is waited for)
  const int c = filtered && lane < p.parts ? (int)p.part_listed[row + lane] : 0;
  uint32_t tau = by_count && lane < p.parts ? p.part_tau[row + lane] : 0;   // top-k: the list holds every element at or above it
  uint64_t z = by_mass && tid < p.parts ? p.part_mass[row + tid] : 0;
  const uint64_t run0 = p.s.top_k == 0 && tid < n_runs ? p.run_mass[row * kRuns + tid] : 0;
  const RowMax m = row_max(p, r, lane);
  const float mx = order_key_value(m.key), neg_mx = -mx * 1.4426950408889634f;
  if (p.s.top_k == 1 || !has_masses(mx)) {
    if (tid == 0) write_sample(p.s, r, m.idx, 0);
    return;
  }
  const auto rd = row_reader<DT, VEC>(p.s, r);
  // ---- the lists of the parts, one after the other: every wavefront copies some of them ----
  int n = 0;
  bool listed = true;
  uint64_t in_list = 0;
  if (filtered) {
    int incl = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(incl, d, 64);
      incl += lane >= d ? v : 0;
      tau = max(tau, (uint32_t)__shfl_xor((int)tau, d, 64));
    }
    n = __builtin_amdgcn_readlane(incl, 63);
    listed = __builtin_amdgcn_ballot_w64(c > p.list_cap) == 0 && n <= kMemberCap;
    for (int g = wave; g < p.parts && listed; g += kSampleWaves) {
      const int mine = __builtin_amdgcn_readlane(c, g), at = __builtin_amdgcn_readlane(incl, g) - mine;
      const uint2* src = p.list + (row + g) * p.list_cap;
      for (int j = lane; j < mine; j += 64) {
        const uint2 e = src[j];
        const uint32_t w = (uint32_t)mass_of(order_key_value(e.x), neg_mx);
        key[at + j] = e.x;
        index[at + j] = e.y;
        mass[at + j] = w;
        in_list += w;
      }
    }
  }
  runs[tid] = run0;   // (n_runs <= the number of threads)
  if (tid < 512) hist[tid] = 0;
  if (tid == 0) { cut = 0; pick = m.idx; }
  uint64_t above = 0, target = (uint64_t)(p.s.top_k - 1);
  bool cuts = by_count;   // (a top-p of the whole mass cuts nothing)
  if (by_mass) {
    z = wave_sum_u64(z);
    above = wave_sum_u64(run0);
    in_list = wave_sum_u64(in_list);
    if (lane == 0) { wsum[0][wave] = z; wsum[1][wave] = above; wsum[2][wave] = in_list; }
    __syncthreads();
    z = above = in_list = 0;
#pragma unroll
    for (int w = 0; w < kSampleWaves; ++w) { z += wsum[0][w]; above += wsum[1][w]; in_list += wsum[2][w]; }
    target = (uint64_t)((double)p.s.top_p * (double)z);
    cuts = z > target;
    listed = listed && (!cuts || (above <= target && above + in_list > target));
  } else {
    listed = listed && (!by_count || n >= p.s.top_k);
    __syncthreads();
  }
  // ---- the smallest kept key ----
  const CutShared cs{hist, res, &cut};
  auto digits = [&](bool from_list) {
    digit_cut(cs, from_list ? above : 0, target, tid, [&](auto count) {
      if (from_list) {
        count_list(key, mass, n, by_count, tid, count);
      } else {
        sweep<4>(rd, 0, p.s.V, tid, kSampleThreads, [&](int, float x, bool in) {
          count(order_key(x), in, [&]() -> uint64_t { return by_count ? 1 : mass_of(x, neg_mx); });
        });
      }
    });
  };
  if (cuts && listed) {
    if (n <= 256) pair_cut(cs, key, mass, n, by_count, above, target, tid);
    else digits(true);
    if (by_count && cut < tau) listed = false;   // (every thread sees the same words)
  }
  if (cuts && !listed) {
    __syncthreads();
    if (tid == 0) cut = 0;
    digits(false);
  }
  const uint32_t cut_key = cuts ? cut : 0;
  // ---- the kept elements that no run has counted yet join theirs ----
  auto join = [&](int i, uint64_t w) {
    const int part = i / p.part_len;
    atomicAdd(reinterpret_cast<unsigned long long*>(&runs[part * kRuns + (i - part * p.part_len) / p.run_len]), (unsigned long long)w);
  };
  if (cuts && listed) {
    for (int j = tid; j < n; j += kSampleThreads)
      if (key[j] >= cut_key) join((int)index[j], mass[j]);
  } else if (filtered) {
    runs[tid] = 0;
    __syncthreads();
    sweep<4>(rd, 0, p.s.V, tid, kSampleThreads, [&](int i, float x, bool in) {
      if (in && order_key(x) >= cut_key) join(i, mass_of(x, neg_mx));
    });
  }
  __syncthreads();
  // ---- the run the uniform number falls into: every thread owns one (there are at most 1 024) ----
  if (tid == 0) res[0] = res[1] = 0;   // (a run of the row, whatever the masses)
  const uint64_t mine = runs[tid];
  uint64_t incl = wave_scan_incl_u64(mine, lane);
  if (lane == 63) wsum[0][wave] = incl;
  __syncthreads();
  uint64_t total = 0;
#pragma unroll
  for (int w = 0; w < kSampleWaves; ++w) {
    incl += w < wave ? wsum[0][w] : 0;
    total += wsum[0][w];
  }
  // total > 0: the maximum itself is always kept and has the largest mass
  uint64_t want = (uint64_t)((double)p.s.uniform[r] * (double)total);
  want = want < total ? want : total - 1;
  if (incl > want && incl - mine <= want) { res[0] = (uint64_t)tid; res[1] = incl - mine; }
  __syncthreads();
  // ---- the element: each thread owns a few neighbours of the run ----
  const int run = (int)res[0];
  want -= res[1];
  const int pa = (run / kRuns) * p.part_len, ra = pa + (run % kRuns) * p.run_len;
  const int rb = min(min(ra + p.run_len, pa + p.part_len), p.s.V);
  const int per = (p.run_len + kSampleThreads - 1) / kSampleThreads;
  auto kept_mass = [&](float x) -> uint64_t {
    const uint64_t w = mass_of(x, neg_mx);
    return order_key(x) >= cut_key ? w : 0;
  };
  const int a = min(ra + tid * per, rb), b = min(a + per, rb);
  uint64_t s = 0;
  for (int i = a; i < b; ++i) s += kept_mass(rd.at(i));
  incl = wave_scan_incl_u64(s, lane);
  if (lane == 63) wsum[1][wave] = incl;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kSampleWaves; ++w) incl += w < wave ? wsum[1][w] : 0;
  if (incl > want && incl - s <= want) {
    uint64_t at = incl - s;
    for (int i = a; i < b; ++i) {
      at += kept_mass(rd.at(i));
      if (at > want) { pick = i; break; }
    }
  }
  __syncthreads();
  if (tid == 0) {
    int sample = pick;
    if (p.s.vocab_clamp > 0) sample = min(max(sample, 0), p.s.vocab_clamp - 1);
    write_sample(p.s, r, sample, cut_key);
  }
}

// ---- a row in the registers of one workgroup ---------------------------------------------------------------------
// elements of a wavefront's run, of `n`
template <int VEC>
static __host__ __device__ __forceinline__ int row_run(int n) { return ((n + kSampleWaves - 1) / kSampleWaves + VEC - 1) & ~(VEC - 1); }

// NG groups of VEC elements a lane; a wavefront holds a run of neighbouring elements, group after group.  Rows start on any
// element (a 16-byte load that is not aligned costs a cache line more now and then); the row's last group, where it is not
// whole, is read as the last VEC elements, of which the lane before holds the first ones.  V >= VEC.
template <int DT, int NG>
struct RowInRegisters {
  static constexpr int VEC = DT != 0 ? 8 : 4;
  uint32_t w[NG][4];   // scaled values, two to a word in a 16-bit type; -inf where the lane has no element
  int at0, last_at;    // the lane's first element; the last group's
  int groups;          // of the wavefront's run: what lies past them is -inf (wave-uniform)

  __device__ __forceinline__ float value(int g, int j) const {
    if (DT != 0) return (j & 1) ? hi_to_f32<DT == 2>(w[g][j >> 1]) : lo_to_f32<DT == 2>(w[g][j >> 1]);
    return __uint_as_float(w[g][j & 3]);
  }
  __device__ __forceinline__ int element(int g, int j) const { return min(at0 + g * 64 * VEC, last_at) + j; }
  // Nothing made of the values lives on from here: conversions of one pass kept for the next spill what they save.
  __device__ __forceinline__ void forget() {
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(w[g][i]));
    asm volatile("" : "+v"(at0));
  }

  __device__ __forceinline__ void load(const SampleParams& p, int r, int wave, int lane) {
    typedef std::conditional_t<DT != 0, uint16_t, uint32_t> element_t;
    constexpr uint32_t kNone = DT == 0 ? 0xff800000u : DT == 1 ? 0xff80ff80u : 0xfc00fc00u;
    const element_t* row = reinterpret_cast<const element_t*>(p.logits) + (int64_t)r * p.stride;
    const int run = row_run<VEC>(p.V);   // (at most NG * 64 * VEC)
    const int end = min((wave + 1) * run, p.V);
    at0 = wave * run + lane * VEC;
    last_at = p.V - VEC;
    groups = __builtin_amdgcn_readfirstlane(max(end - wave * run + 64 * VEC - 1, 0) / (64 * VEC));
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const uint32_t at = (uint32_t)min(at0 + g * 64 * VEC, last_at);
      __builtin_memcpy(w[g], row + at, 16);   // (one load, of the element's alignment)
      __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("" : "+v"(at0));
    if (p.inv_temperature != 1.0f) {     // (rounded to the logits' type, as RowReader::finish)
#pragma unroll
      for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (DT == 0) w[g][i] = __float_as_uint(__uint_as_float(w[g][i]) * p.inv_temperature);
          else w[g][i] = pack2<DT == 2>(lo_to_f32<DT == 2>(w[g][i]) * p.inv_temperature, hi_to_f32<DT == 2>(w[g][i]) * p.inv_temperature);
          if (i == 3) __builtin_amdgcn_sched_barrier(0);
        }
      forget();
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int at = at0 + g * 64 * VEC;
      const int skip = at >= end ? VEC : at - last_at;   // of the lane's group: not its own
      if (__builtin_amdgcn_ballot_w64(skip > 0)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (DT == 0) w[g][i] = skip > i ? kNone : w[g][i];
          else w[g][i] = skip > 2 * i + 1 ? kNone : skip > 2 * i ? (w[g][i] & 0xffff0000u) | (kNone & 0xffffu) : w[g][i];
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    forget();
  }
};

// One workgroup per row, the row read once: maximum, bins around the cut (top-p: the first walk's of the parts; top-k: counts),
// the members of the bins that hold the cut listed in LDS, the exact cut among them, the wavefront and then the element that the
// uniform number falls into.  The masses and every sum that decides are those of the other forms; where the list does not
// hold the cut, four digit passes over the registers find it.
template <int DT, int NG>
__global__ __launch_bounds__(kSampleThreads) void sample_row_kernel(SampleParams p) {
  constexpr int VEC = RowInRegisters<DT, NG>::VEC;
  __shared__ uint32_t bins[kBins + 64];
  __shared__ uint32_t key[kMemberCap];
  __shared__ uint32_t mass[kMemberCap];
  __shared__ uint32_t index[kMemberCap];
  __shared__ uint64_t hist[512];
  __shared__ uint64_t res[2];
  __shared__ uint64_t wsum[2][kSampleWaves];
  __shared__ uint64_t runs[kSampleWaves], kept_runs[kSampleWaves];
  __shared__ uint32_t red[kSampleWaves];
  __shared__ int32_t window[2];
  __shared__ uint32_t listed_n;
  __shared__ uint32_t cut;
  __shared__ int32_t pick;
  const int r = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool by_count = p.top_k > 1, by_mass = p.top_k == 0 && p.top_p > 0.f, filtered = by_count || by_mass;
  const float uniform = p.uniform[r];
  RowInRegisters<DT, NG> row;
  row.load(p, r, wave, lane);
  bins[tid] = bins[tid + kSampleThreads] = 0;
  if (tid < 512) hist[tid] = 0;
  if (tid == 0) { window[0] = kBins; window[1] = -1; listed_n = 0; cut = 0; pick = 0; }

  // ---- the maximum: as integers, numbers from +0 up are in order, NaN above them; below 0 the floats' order counts ----
  int32_t top_i = INT32_MIN;
  float top_f = -INFINITY;
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    if (g >= row.groups) continue;
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const float x = row.value(g, j);
      top_i = max(top_i, __float_as_int(x));
      top_f = fmaxf(top_f, x);
    }
  }
  uint32_t bk = wave_max_u32(top_i >= 0 ? (uint32_t)top_i | 0x80000000u : order_key(top_f + 0.f));
  if (lane == 0) red[wave] = bk;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kSampleWaves; ++w) bk = max(bk, red[w]);
  const float mx = order_key_value(bk), neg_mx = -mx * 1.4426950408889634f;
  const RowReader<DT, 1> rd = row_reader<DT, 1>(p, r);   // (what is rare reads the row again)
  if (!has_masses(mx)) {   // nothing to draw from: the argmax, the lowest index among equals
    uint32_t best = 0, at = 0x7fffffffu;
    sweep<8>(rd, 0, p.V, tid, kSampleThreads, [&](int i, float x, bool in) {
      const uint32_t k = order_key(x);
      const bool up = in && k > best;
      best = up ? k : best;
      at = up ? (uint32_t)i : at;
    });
    const uint32_t wave_best = wave_max_u32(best);
    at = ~wave_max_u32(best == wave_best ? ~at : 0);
    __syncthreads();   // (the maxima have been read)
    if (lane == 0) { red[wave] = wave_best; key[wave] = at; }
    __syncthreads();
    if (tid == 0) {
      best = 0;
      for (int w = 0; w < kSampleWaves; ++w) {
        if (red[w] > best || (red[w] == best && key[w] < at)) { best = red[w]; at = key[w]; }
      }
      write_sample(p, r, at < (uint32_t)p.V ? (int)at : 0, 0);
    }
    return;
  }

  row.forget();
  // ---- the bins, counted down from the maximum's; the bins that hold the cut ----
  float over = INFINITY, from = INFINITY;   // kept: above `over`; listed: from `from` to `over`
  if (filtered) {
    const float row_first = floorf(mx * kBinsPerUnit), edge = row_first + 1.f;
    int bits = 31 - __builtin_clz(p.V);   // V < 2^(bits + 1)
    const float bin_one = (float)(1u << (31 - bits > 16 ? 16 : 31 - bits));
    const uint32_t none = (uint32_t)(kBins + lane);   // (a place of its own for what no bin takes: no branch)
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      if (g >= row.groups) continue;
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        // (the weight of sample_first_kernel)
        const float f = __builtin_fmaf(row.value(g, j), -kBinsPerUnit, edge);
        const float wt = __builtin_fmaf(__builtin_amdgcn_fractf(f), -0.01550356f * bin_one, 0.99998474f * bin_one + 0.5f);
        const bool in = f < (float)kBins;   // (not NaN, nor what is masked)
        atomicAdd(&bins[in ? (uint32_t)fmaxf(in ? f : 0.f, 0.f) : none], by_count ? 1u : (uint32_t)(in ? wt : 0.f));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    const uint32_t c0 = bins[2 * tid], c1 = bins[2 * tid + 1];
    auto count_window = [&](uint32_t n0, uint32_t n1) {   // (bins 2 tid and 2 tid + 1)
      const int h = (int)(n0 + n1);
      int incl = wave_scan(h);
      if (lane == 63) red[wave] = (uint32_t)incl;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < kSampleWaves; ++w) incl += w < wave ? (int)red[w] : 0;
      if (incl >= p.top_k && incl - h < p.top_k) window[0] = window[1] = incl - (int)n1 >= p.top_k ? 2 * tid : 2 * tid + 1;
      __syncthreads();
    };
    if (by_count) {
      count_window(c0, c1);
    } else {   // (the estimate and its slack: see sample_mass_kernel)
      const float h0 = (float)c0 * fast_exp2((float)(2 * tid) * (-1.4426950408889634f / kBinsPerUnit));
      const float h1 = (float)c1 * fast_exp2((float)(2 * tid + 1) * (-1.4426950408889634f / kBinsPerUnit));
      const float h = h0 + h1;
      float incl = wave_scan_incl_f32(h);
      if (lane == 63) red[wave] = __float_as_uint(incl);
      __syncthreads();
      float total = 0.f;
#pragma unroll
      for (int w = 0; w < kSampleWaves; ++w) {
        incl += w < wave ? __uint_as_float(red[w]) : 0.f;
        total += __uint_as_float(red[w]);
      }
      const float want = p.top_p * total, slack = fmaxf(1e-4f, 3e-5f + 0.3f / bin_one) * total;
      const bool in0 = incl - h - slack <= want && incl - h1 + slack > want && h0 > 0.f;
      const bool in1 = incl - h1 - slack <= want && incl + slack > want && h1 > 0.f;
      if (in0 || in1) {
        atomicMin(&window[0], in0 ? 2 * tid : 2 * tid + 1);
        atomicMax(&window[1], in1 ? 2 * tid + 1 : 2 * tid);
      }
      __syncthreads();
    }
    int lo = __builtin_amdgcn_readfirstlane(window[0]), hi = __builtin_amdgcn_readfirstlane(window[1]);
    if (lo <= hi) {
      over = (row_first + 1.f - (float)lo) * (1.f / kBinsPerUnit);
      from = (row_first - (float)hi) * (1.f / kBinsPerUnit);
    } else if (by_count) {
      // The k-th value lies below the bins (32 units: a low temperature spreads the values).  Counted again 16 times as wide, in a
      // walk of the row from memory where the cut's digits would take four (512 x 32 000 bf16, k 50, of them a few such rows:
      // 58.7 us).
      constexpr float kWide = kBinsPerUnit / 16.f;
      bins[2 * tid] = bins[2 * tid + 1] = 0;
      __syncthreads();
      const float wide_first = floorf(mx * kWide);
      sweep<8>(rd, 0, p.V, tid, kSampleThreads, [&](int, float x, bool in) {
        const float f = __builtin_fmaf(x, -kWide, wide_first + 1.f);
        if (in && f < (float)kBins) atomicAdd(&bins[(uint32_t)fmaxf(f, 0.f)], 1u);
      });
      __syncthreads();
      count_window(bins[2 * tid], bins[2 * tid + 1]);
      lo = __builtin_amdgcn_readfirstlane(window[0]);
      if (lo < kBins) {
        over = (wide_first + 1.f - (float)lo) * (1.f / kWide);
        from = (wide_first - (float)lo) * (1.f / kWide);
      }
    }
  }

  // ---- the masses; what lies above the window; its members, listed ----
  uint32_t all_lo = 0, all_hi = 0;   // top-p: of everything; a plain draw keeps all of it
  uint32_t kept_lo = 0, kept_hi = 0, kept_n = 0;
  row.forget();
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    if (g >= row.groups) continue;
    uint32_t m32[VEC];
    if (!by_count) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) m32[j] = add_mass(all_lo, all_hi, row.value(g, j), neg_mx);
    }
    if (!filtered) continue;
    uint64_t in_window[VEC], any = 0;
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const float v = row.value(g, j);
      const bool is_over = v > over;
      const uint64_t above = __builtin_amdgcn_ballot_w64(is_over);
      if (above) {
        if (by_count) kept_n += is_over ? 1u : 0u;
        else add_u32(kept_lo, kept_hi, is_over ? m32[j] : 0u);
      }
      in_window[j] = __builtin_amdgcn_ballot_w64(v >= from) & ~above;
      any |= in_window[j];
    }
    if (any) {
      uint32_t found = 0, at = 0;
#pragma unroll
      for (int j = 0; j < VEC; ++j) found += (uint32_t)__builtin_popcountll(in_window[j]);
      if (lane == 0) at = atomicAdd(&listed_n, found);
      at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const uint64_t m = in_window[j];
        if (m == 0) continue;
        const uint32_t mine = at + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
        if (((m >> lane) & 1) && mine < (uint32_t)kMemberCap) {
          const float v = row.value(g, j);
          key[mine] = order_key(v + 0.f);
          index[mine] = (uint32_t)row.element(g, j);
          mass[mine] = (uint32_t)mass_of(v, neg_mx);
        }
        at += (uint32_t)__builtin_popcountll(m);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  const uint64_t all = wave_sum_u64(((uint64_t)all_hi << 32) | all_lo);
  uint64_t kept = by_mass ? wave_sum_u64(((uint64_t)kept_hi << 32) | kept_lo) : by_count ? wave_sum_u64(kept_n) : all;
  if (lane == 0) { wsum[0][wave] = all; runs[wave] = kept; }
  __syncthreads();
  float cut_value = -INFINITY;
  uint32_t cut_key = 0;
  uint64_t run_mass = 0;   // lane i: kept members of run i that `of_runs` does not count
  const uint64_t* of_runs = runs;
  if (filtered) {
    const uint64_t z = wave_sum_u64(lane < kSampleWaves ? wsum[0][lane & (kSampleWaves - 1)] : 0);
    const uint64_t above = wave_sum_u64(lane < kSampleWaves ? runs[lane & (kSampleWaves - 1)] : 0);
    const uint64_t target = by_count ? (uint64_t)(p.top_k - 1) : (uint64_t)((double)p.top_p * (double)z);
    const bool cuts = by_count || z > target;   // (a top-p of the whole mass cuts nothing)
    const int n = __builtin_amdgcn_readfirstlane((int)listed_n);
    bool listed = n <= kMemberCap, joined = false;
    if (cuts && n <= 16) {
      // few members, one a lane: every wavefront works out the cut and the runs' kept masses by itself, without a barrier
      const bool has = lane < n;
      const uint32_t k = has ? key[lane] : 0, w = !has ? 0 : by_count ? 1u : mass[lane];
      listed = above <= target && above + wave_sum_u64(w) > target;
      if (listed) {
        uint64_t higher = 0, equal = 0;
        for (int j = 0; j < n; ++j) {
          const uint32_t kj = (uint32_t)__builtin_amdgcn_readlane((int)k, j), wj = (uint32_t)__builtin_amdgcn_readlane((int)w, j);
          higher += kj > k ? wj : 0u;
          equal += kj == k ? wj : 0u;
        }
        const uint64_t hit = __builtin_amdgcn_ballot_w64(has && above + higher <= target && above + higher + equal > target);
        cut_key = (uint32_t)__builtin_amdgcn_readlane((int)k, __builtin_ctzll(hit));   // (the list holds it)
        if (by_mass) {
          const int of_run = has && k >= cut_key ? (int)index[lane] / row_run<VEC>(p.V) : -1;
          for (int j = 0; j < n; ++j)
            run_mass += lane == __builtin_amdgcn_readlane(of_run, j) ? (uint32_t)__builtin_amdgcn_readlane((int)w, j) : 0u;
          joined = true;
        }
      }
    } else if (cuts) {
      const CutShared cs{hist, res, &cut};
      if (listed) {   // (does the list hold the cut?)
        uint64_t in_list = (uint64_t)n;
        if (by_mass) {
          in_list = 0;
          for (int j = tid; j < n; j += kSampleThreads) in_list += mass[j];
          in_list = wave_sum_u64(in_list);
          if (lane == 0) wsum[1][wave] = in_list;
          __syncthreads();
          in_list = 0;
#pragma unroll
          for (int w = 0; w < kSampleWaves; ++w) in_list += wsum[1][w];
        }
        listed = above <= target && above + in_list > target;
      }
      if (listed) {
        if (n <= 256) pair_cut(cs, key, mass, n, by_count, above, target, tid);
        else digit_cut(cs, above, target, tid, [&](auto count) { count_list(key, mass, n, by_count, tid, count); });
        cut_key = cut;
      }
    }
    if (cuts && !listed) {
      digit_cut(CutShared{hist, res, &cut}, 0, target, tid, [&](auto count) {
        sweep<8>(rd, 0, p.V, tid, kSampleThreads, [&](int, float x, bool in) {
          count(order_key(x), in, [&]() -> uint64_t { return by_count ? 1 : mass_of(x, neg_mx); });
        });
      });
      cut_key = cut;
    }
    // (a key below -inf's is a negative NaN's, to which every float compares false: such a cut keeps everything)
    if (cut_key > order_key(-INFINITY)) cut_value = order_key_value(cut_key);
    // ---- the kept mass of every wavefront's run ----
    if (!joined) {
      if (by_mass && cuts && listed) {   // the kept members join what lies above the window
        const int run = row_run<VEC>(p.V);
        for (int j = tid; j < n; j += kSampleThreads)
          if (key[j] >= cut_key)
            atomicAdd(reinterpret_cast<unsigned long long*>(&runs[(int)index[j] / run]), (unsigned long long)mass[j]);
      } else {
        kept = 0;
        row.forget();
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          if (g >= row.groups) continue;
#pragma unroll
          for (int j = 0; j < VEC; ++j) {
            const float v = row.value(g, j);
            if (__builtin_amdgcn_ballot_w64(v >= cut_value)) {
              const uint64_t x = mass_of(v, neg_mx);
              kept += v >= cut_value ? x : 0;
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        kept = wave_sum_u64(kept);
        if (lane == 0) kept_runs[wave] = kept;   // (`runs` may still be read)
        of_runs = kept_runs;
      }
      __syncthreads();
    }
  }
  // ---- the wavefront the uniform number falls into (lane i: run i); its group; the lane; the element ----
  if (lane < kSampleWaves) run_mass += of_runs[lane];
  const uint64_t runs_incl = wave_scan_incl_u64(run_mass, lane);
  auto lane_u64 = [](uint64_t v, int at) {
    return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), at) << 32) |
           (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, at);
  };
  const uint64_t total = lane_u64(runs_incl, 63);
  // total > 0: the maximum itself is always kept and has the largest mass
  uint64_t want = (uint64_t)((double)uniform * (double)total);
  want = want < total ? want : total - 1;
  const int owner = __builtin_ctzll(__builtin_amdgcn_ballot_w64(runs_incl > want));
  want -= lane_u64(runs_incl - run_mass, owner);
  row.forget();
  if (wave == owner) {
    bool found = false;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      if (found || g >= row.groups) continue;
      if (filtered) {   // (most of a sharp filter's groups hold nothing)
        uint64_t any = 0;
#pragma unroll
        for (int j = 0; j < VEC; ++j) any |= __builtin_amdgcn_ballot_w64(row.value(g, j) >= cut_value);
        if (!any) continue;
      }
      uint64_t m[VEC], sum = 0;
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const float v = row.value(g, j);
        const uint64_t x = mass_of(v, neg_mx);
        m[j] = v >= cut_value ? x : 0;
        sum += m[j];
      }
      const uint64_t incl = wave_scan_incl_u64(sum, lane), last = lane_u64(incl, 63);
      if (last <= want) {
        want -= last;
        continue;
      }
      if (incl > want && incl - sum <= want) {
        uint64_t at = incl - sum;
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
          if (at <= want && at + m[j] > want) pick = row.element(g, j);
          at += m[j];
        }
      }
      found = true;
    }
  }
  __syncthreads();
  if (tid == 0) {
    int sample = pick;
    if (p.vocab_clamp > 0) sample = min(max(sample, 0), p.vocab_clamp - 1);
    write_sample(p, r, sample, cut_key);
  }
}

struct GatherParams {
  const uint8_t* src; int64_t src_stride_bytes;
  uint8_t* dst; int64_t dst_stride_bytes;
  const int32_t* q_len; int32_t R; int64_t row_bytes; int32_t vec;
};

// dst[r] = src[sum(q_len[0..r]) - 1]; grid = (R, column blocks)
__global__ __launch_bounds__(256) void last_token_gather_kernel(GatherParams p) {
  __shared__ int32_t part[4];
  const int r = blockIdx.x, tid = threadIdx.x;
  int s = 0;
  for (int i = tid; i <= r; i += 256) s += p.q_len[i];
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
  if ((tid & 63) == 0) part[tid >> 6] = s;
  __syncthreads();
  const int64_t row = (int64_t)part[0] + part[1] + part[2] + part[3] - 1;
  if (row < 0) return;
  const uint8_t* src = p.src + row * p.src_stride_bytes;
  uint8_t* dst = p.dst + (int64_t)r * p.dst_stride_bytes;
  const int64_t step = (int64_t)gridDim.y * 256 * p.vec;
  for (int64_t o = ((int64_t)blockIdx.y * 256 + tid) * p.vec; o < p.row_bytes; o += step) {
    if (p.vec == 16) st16(dst + o, ld16(src + o));
    else if (p.vec == 4) *reinterpret_cast<uint32_t*>(dst + o) = *reinterpret_cast<const uint32_t*>(src + o);
    else *reinterpret_cast<uint16_t*>(dst + o) = *reinterpret_cast<const uint16_t*>(src + o);
  }
}

struct LogProbParams {
  const void* logits; int64_t stride; int32_t T, V;
  const int64_t* token_ids; float* out;
};

constexpr int kLogProbThreads = 512;

// out[t] = log_softmax(logits[t])[token_ids[t]] in fp32: one pass over the row with a running
// (maximum, sum of exp(x - maximum)) pair per thread, merged over the workgroup.  One workgroup per row.
template <int DT, int VEC>
__global__ __launch_bounds__(kLogProbThreads) void selected_log_probs_kernel(LogProbParams p) {
  __shared__ float red_m[kLogProbThreads / 64], red_s[kLogProbThreads / 64];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  RowReader<DT, VEC> rd;
  rd.row = reinterpret_cast<const uint8_t*>(p.logits) + (int64_t)t * p.stride * (DT != 0 ? 2 : 4);
  rd.V = p.V; rd.inv_t = 1.f; rd.scale = false;
  constexpr float kLog2e = 1.4426950408889634f;
  // a finite start keeps exp(-inf - m) = 0 for masked (-inf) logits
  float m = -3.0e38f, sum = 0.f;
  // Whole batches of U 16-byte groups per thread: the batch maximum first (one three-way maximum per
  // two elements), a rescale only when it raises the running maximum (rare after a thread's first
  // batches), then one fused multiply-add, one exp2 and one add per element.
  constexpr int U = 4;
  const int stride = kLogProbThreads * VEC;
  const int row_end = p.V - (p.V % VEC);
  int base = 0;
  if (VEC > 1) {
    for (; base + U * stride <= row_end; base += U * stride) {
      float x[U * VEC];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint4 w = ld16(rd.row + (int64_t)(base + u * stride + tid * VEC) * (DT != 0 ? 2 : 4));
        const uint32_t q[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int j = 0; j < VEC; ++j)
          x[u * VEC + j] = DT != 0 ? ((j & 1) ? hi_to_f32<DT == 2>(q[(j >> 1) & 3]) : lo_to_f32<DT == 2>(q[(j >> 1) & 3]))
                                : __uint_as_float(q[j & 3]);
      }
      float bm = x[0];
#pragma unroll
      for (int j = 1; j + 1 < U * VEC; j += 2) bm = fmaxf(fmaxf(bm, x[j]), x[j + 1]);
      bm = fmaxf(bm, x[U * VEC - 1]);
      if (bm > m) {
        sum *= fast_exp2((m - bm) * kLog2e);
        m = bm;
      }
      const float nm = -m * kLog2e;
      float part = 0.f;
#pragma unroll
      for (int j = 0; j < U * VEC; ++j) part += fast_exp2(__builtin_fmaf(x[j], kLog2e, nm));
      sum += part;
    }
  }
  sweep<U>(rd, base, p.V, tid, kLogProbThreads, [&](int, float x, bool valid) {
    if (valid) {
      if (x > m) {
        sum *= fast_exp2((m - x) * kLog2e);
        m = x;
      }
      sum += fast_exp2((x - m) * kLog2e);
    }
  });
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    const float m2 = __shfl_xor(m, d, 64), s2 = __shfl_xor(sum, d, 64);
    const float mm = fmaxf(m, m2);
    sum = sum * fast_exp2((m - mm) * kLog2e) + s2 * fast_exp2((m2 - mm) * kLog2e);
    m = mm;
  }
  if (lane == 0) { red_m[wave] = m; red_s[wave] = sum; }
  __syncthreads();
  if (tid == 0) {
    float mm = red_m[0];
#pragma unroll
    for (int w = 1; w < kLogProbThreads / 64; ++w) mm = fmaxf(mm, red_m[w]);
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < kLogProbThreads / 64; ++w) total += red_s[w] * fast_exp2((red_m[w] - mm) * kLog2e);
    const int64_t id = p.token_ids[t];
    float r = __builtin_nanf("");
    if (id >= 0 && id < p.V) r = (rd.at((int)id) - mm) - __logf(total);
    p.out[t] = r;
  }
}

}  // namespace mi

using namespace mi;

extern "C" int mi_last_token_gather(const void* src, int64_t src_stride_row, void* dst, int64_t dst_stride_row,
                                    const int32_t* request_query_lengths, int32_t R, int32_t row_elems,
                                    int32_t elem_bytes, void* stream) {
  if (R == 0 || row_elems == 0) return MI_OK;
  if (!src || !dst || !request_query_lengths) return mi_fail(MI_ERR_NULL, "mi_last_token_gather: null pointer argument");
  if (R < 0 || row_elems < 0 || (elem_bytes != 2 && elem_bytes != 4))
    return mi_fail(MI_ERR_SHAPE, "mi_last_token_gather: need R, row_elems >= 0 and 2- or 4-byte elements");
  if (src_stride_row < row_elems || dst_stride_row < row_elems)
    return mi_fail(MI_ERR_SHAPE, "mi_last_token_gather: row strides are shorter than a row");
  GatherParams p;
  p.src = (const uint8_t*)src; p.src_stride_bytes = src_stride_row * elem_bytes;
  p.dst = (uint8_t*)dst; p.dst_stride_bytes = dst_stride_row * elem_bytes;
  p.q_len = request_query_lengths; p.R = R; p.row_bytes = (int64_t)row_elems * elem_bytes;
  const bool wide = !(((uintptr_t)src | (uintptr_t)dst | (uintptr_t)p.src_stride_bytes | (uintptr_t)p.dst_stride_bytes |
                       (uintptr_t)p.row_bytes) & 15);
  p.vec = wide ? 16 : elem_bytes;
  const int64_t per_block = 256 * (int64_t)p.vec;
  int ny = (int)((p.row_bytes + per_block - 1) / per_block);
  ny = ny < 1 ? 1 : (ny > 64 ? 64 : ny);
  hipLaunchKernelGGL(last_token_gather_kernel, dim3(R, ny), dim3(256), 0, (hipStream_t)stream, p);
  return mi_check_launch("mi_last_token_gather");
}

// Parts a row is cut into: as many workgroups as the chip takes at once (one per CU: a second round costs more than
// larger parts, 83 x 50 304 top-p in 4 parts 45 us, in 3 33 with the walks of then, 24 now), parts of at least 4 096 elements.
static int sample_parts(int R, int V) {
  int parts = 256 / R;
  if (parts > V / 4096) parts = V / 4096;
  return parts < 1 ? 1 : (parts > kMaxParts ? kMaxParts : parts);
}
// Whether the rows are done in parts, for some type of logits at least.  The further launches cost 3-6 us, so the walks they shorten
// have to be long enough.  Draws from rows that fit the registers of a workgroup go there, workspace or not, but where row_groups
// says otherwise; the lines here leave those rows out.  fp32 in a graph, us, one workgroup per row that walks it / parts:
//   greedy, one walk to shorten: 64 x 151 936 16.9 / 12.0, 64 x 32 768 below the line 6.2 / 7.5;
//   plain draws, two: 64 x 128 256 37 / 21;
//   top-k, whose pick grows with its lists: 64 x 128 256 39.1 / 31.1, and does not gain from two: 128 x 100 352 35.2 / 37.7;
//   top-p, three: 64 x 128 256 101.8 / 28.1.
// More than 128 rows have one part each, and are done this way for the walks alone: a top-p row that does not fit the registers
// of a workgroup.  fp32 / bf16: 256 x 128 256 119 / 115 -> 67 / 60, 512 x 151 936 255 / 253 -> 139 / 124; peaked rows 512 x
// 128 256 130 / 122 -> 115 / 95.  That takes 40 KB of scratch a row, at most 40 MB: more rows are walked.
constexpr int kManyRows = 1024;
constexpr int kRowInRegisters = 32768;     // widest row whose filter does not gain from parts
constexpr int kWidestInRegisters = 65536;
static bool sample_in_parts(int R, int V, int top_k, float top_p) {
  const bool by_mass = top_k == 0 && top_p > 0.f;
  if (R > 128) return by_mass && R <= kManyRows && V > kWidestInRegisters;
  if (V < kFastMinVocab || top_k > kFastTopK) return false;
  if (top_k == 1) return V >= 1600 * (R > 50 ? R : 50);
  if (top_k > 1) return R <= 85 && V > kRowInRegisters;
  if (!by_mass) return V > kWidestInRegisters || (R <= 16 && V > 57344);
  if (V <= kRowInRegisters) return false;
  return R > 85 ? V >= 65536 : V >= 49152 || R <= 64;
}

static int64_t align256(int64_t n) { return (n + 255) & ~(int64_t)255; }
static int64_t sample_layout(SplitParams* p, uint8_t* base, int R, int V, int top_k, float top_p) {
  const int parts = sample_parts(R, V);
  int run = (V + parts * kRuns - 1) / (parts * kRuns);
  run = (run + 7) & ~7;
  int64_t at = 0;
  auto take = [&](int64_t bytes) { uint8_t* q = base + at; at += align256(bytes); return q; };
  const int64_t n = (int64_t)R * parts;
  const bool draws = top_k != 1, by_count = top_k > 1, by_mass = draws && !by_count && top_p > 0.f;
  p->parts = parts; p->run_len = run; p->part_len = run * kRuns;
  p->list_cap = kMemberCap;   // (one part's list may hold all that the pick takes)
  if (parts > 4) p->list_cap = kMemberCap / 4;
  p->part_key = (uint32_t*)take(4 * n); p->part_idx = (int32_t*)take(4 * n);
  p->part_tau = (uint32_t*)take(4 * n); p->part_listed = (uint32_t*)take(4 * n);
  p->bins = (uint32_t*)take(by_mass ? n * kBins * 4 : 0);
  int bits = 0;
  while (bits < 30 && (V >> bits) > 1) ++bits;   // V < 2^(bits + 1)
  p->bin_one = (float)(1u << (31 - bits > 16 ? 16 : 31 - bits));
  p->part_mass = (uint64_t*)take(draws && !by_count ? n * 8 : 0);
  p->run_mass = (uint64_t*)take(draws && !by_count ? n * kRuns * 8 : 0);
  p->list = (uint2*)take(by_count || by_mass ? n * p->list_cap * 8 : 0);
  return at;
}

// Whether draws from rows of V elements take the registers of one workgroup, and how many groups of 16 bytes a lane: 0 = no.
// Up to 65 536 elements fit without spilling.  A plain draw is faster than any other form, but for a few of the widest fp32 rows,
// which parts scale by the temperature.  A filter's bins and lists are work that parts share: above 32 768 elements parts, where
// the rows are few enough for them, are level or better.  Without parts the one other form walks the row several times; only
// top-k up to kFastTopK, which it reads once, stays there above 32 768: over fp32, and over a 16-bit type where more than 256
// rows, which it takes two to a CU, are not the widest.  In a graph, us, the other form -> this one, fp32 / bf16, N(0, 3):
//   plain: 16 x 32 000 15.1 / 17.0 -> 7.4 / 9.1, 256 x 32 000 17.4 / 17.9 -> 9.6 / 9.8, 1 x 65 536 12.1 / 12.6 -> 10.7 / 11.0 (fp32 with a
//          temperature 12.8, here 13.7; 1 x 50 257 13.0 -> 11.0), 256 x 65 536 30.7 / 23.5 -> 20.6 / 12.3;
//   top-k 50: 16 x 32 000 16.8 / 17.0 -> 13.0 / 15.5, 128 x 32 000 24.0 / 24.3 -> 13.5 / 16.1; 16 x 65 536 17.3 / 17.7, here 21.8 /
//          20.6; bf16 512 x 32 769 34.1, here 38.1, 512 x 50 257 44.1 -> 43.5, 1 024 x 50 257 76.3, here 83.0,
//          1 024 x 65 536 118 -> 85; k 1 500, bf16: 512 x 50 257 70 -> 51;
//   top-p 0.9: 16 x 32 000 19.4 / 20.2 -> 16.0 / 18.8, 256 x 32 000 51.4 / 50.0 -> 17.9 / 19.7, 256 x 65 536 82 / 74 -> 33 / 26; 16 x
//          65 536 22.6 / 23.5, here 24.0 / 25.5; peaked rows 1 x 32 000 18.1 / 18.6 -> 13.4 / 15.3; but top-p 0.999: 7 x 32 000 22.3 / 23.2, here 23.4 / 25.6.
template <int DT>
static int row_groups(const SampleParams& s, bool in_parts) {
  constexpr int VEC = DT != 0 ? 8 : 4;
  if (s.top_k == 1 || s.V < VEC || s.V > kWidestInRegisters) return 0;
  if (s.top_k > 1) {
    const int widest_walked = s.top_k > kFastTopK || s.R <= 256 ? 0 : s.R <= 512 ? 49152 : 57344;
    if (s.V > kRowInRegisters && (in_parts || DT == 0 || s.V < widest_walked)) return 0;
  } else if (in_parts) {
    if (s.top_p > 0.f ? s.V > kRowInRegisters : DT == 0 && s.inv_temperature != 1.0f) return 0;
  }
  return (row_run<VEC>(s.V) + 64 * VEC - 1) / (64 * VEC);
}

template <int DT, int VEC>
static void launch_sample(const SampleParams& s, SplitParams* split, hipStream_t st) {
  const int groups = row_groups<DT>(s, split != nullptr);
  if (groups > 8) {   // (fp32 only)
    hipLaunchKernelGGL((sample_row_kernel<DT, DT == 0 ? 16 : 8>), dim3(s.R), dim3(kSampleThreads), 0, st, s);
    return;
  }
  if (groups > 0) {
    hipLaunchKernelGGL((sample_row_kernel<DT, 8>), dim3(s.R), dim3(kSampleThreads), 0, st, s);
    return;
  }
  if (!split) {
    hipLaunchKernelGGL((sample_kernel<DT, VEC>), dim3(s.R), dim3(kSampleThreads), 0, st, s);
    return;
  }
  const dim3 grid(split->parts, s.R), block(kSampleThreads);
  // Values a thread holds at a time: short runs (many parts per row) have few, and what is loaded past their end is worked
  // on all the same (2 x 138 767 bf16, top-p: 27.0 us with 32, 20.9 with 8).
  // Rows off 16 bytes load value by value: 32 of them spill.
  constexpr int kLarge = VEC == 1 ? 16 : 32, kSmall = 8;
  const bool small = split->run_len <= 64 * kSmall;
#define MI_PARTS_LAUNCH(K_, ...)                                                          \
  do {                                                                                    \
    if (small) hipLaunchKernelGGL((K_<__VA_ARGS__, kSmall>), grid, block, 0, st, *split); \
    else hipLaunchKernelGGL((K_<__VA_ARGS__, kLarge>), grid, block, 0, st, *split);       \
  } while (0)
  if (s.top_k > 1) hipLaunchKernelGGL((sample_first_kernel<DT, VEC, kPickTopK, kSmall>), grid, block, 0, st, *split);
  else if (s.top_k == 0 && s.top_p > 0.f) MI_PARTS_LAUNCH(sample_first_kernel, DT, VEC, kPickTopP);
  else hipLaunchKernelGGL((sample_first_kernel<DT, VEC, kPickMax, kSmall>), grid, block, 0, st, *split);
  if (s.top_k == 0) MI_PARTS_LAUNCH(sample_mass_kernel, DT, VEC);
#undef MI_PARTS_LAUNCH
  hipLaunchKernelGGL((sample_pick_kernel<DT, VEC>), dim3(s.R), block, 0, st, *split);
}

extern "C" int64_t mi_sample_workspace_bytes(int32_t R, int32_t vocab, int32_t top_k, float top_p) {
  SplitParams p;
  return R > 0 && vocab > 0 && sample_in_parts(R, vocab, top_k, top_p) ? sample_layout(&p, nullptr, R, vocab, top_k, top_p) : 0;
}

extern "C" int mi_sample_from_logits_ws(const void* logits, int64_t stride_row, int32_t logits_dtype, int32_t R,
                                        int32_t vocab, int32_t top_k, float top_p, float temperature,
                                        const float* uniform, int32_t vocab_clamp, int64_t* samples,
                                        float* cut_values, const int32_t* request_kv_length_offsets,
                                        const int32_t* request_query_lengths, const int32_t* request_output_lengths,
                                        int64_t termination_id, uint8_t* active_request_mask, void* workspace,
                                        int64_t workspace_bytes, void* stream) {
  if (R == 0) return MI_OK;
  if (!logits || !samples) return mi_fail(MI_ERR_NULL, "mi_sample_from_logits: null pointer argument");
  if (R < 0 || vocab <= 0 || stride_row < vocab)
    return mi_fail(MI_ERR_SHAPE, "mi_sample_from_logits: need R >= 0, vocab > 0 and a row stride of at least vocab");
  if (logits_dtype < 0 || logits_dtype > 2)
    return mi_fail(MI_ERR_UNSUPPORTED, "mi_sample_from_logits: logits must be fp32 (0), bf16 (1) or fp16 (2)");
  if (top_k < 0 || !(top_p >= 0.f && top_p <= 1.f))
    return mi_fail(MI_ERR_SHAPE, "mi_sample_from_logits: need top_k >= 0 and top_p in [0, 1]");
  if (top_k > 0 && top_p > 0.f)
    return mi_fail(MI_ERR_SHAPE, "mi_sample_from_logits: cannot have top-p and top-k both greater than zero");
  if (top_k > vocab) return mi_fail(MI_ERR_SHAPE, "mi_sample_from_logits: top-k is larger than logit size");
  if (top_k != 1 && !(temperature > 0.f))
    return mi_fail(MI_ERR_SHAPE, "mi_sample_from_logits: temperature must be positive");
  if (top_k != 1 && !uniform)
    return mi_fail(MI_ERR_NULL, "mi_sample_from_logits: sampling needs one uniform number per row");
  const bool any_len = request_kv_length_offsets || request_query_lengths || request_output_lengths;
  if (any_len && !(request_kv_length_offsets && request_query_lengths && request_output_lengths))
    return mi_fail(MI_ERR_NULL, "mi_sample_from_logits: the three request length rows go together");
  if (any_len && !active_request_mask)
    return mi_fail(MI_ERR_NULL, "mi_sample_from_logits: request lengths were given without a mask to write");
  SampleParams p;
  p.logits = logits; p.stride = stride_row; p.R = R; p.V = vocab;
  p.top_k = top_k; p.top_p = top_p; p.inv_temperature = top_k == 1 ? 1.0f : 1.0f / temperature;
  p.uniform = uniform; p.vocab_clamp = vocab_clamp; p.samples = samples; p.cut_out = cut_values;
  p.kv_off = request_kv_length_offsets; p.q_len = request_query_lengths; p.out_len = request_output_lengths;
  p.termination_id = termination_id; p.active_mask = active_request_mask;
  const int esize = logits_dtype != 0 ? 2 : 4;
  const bool wide = !(((uintptr_t)logits | (uintptr_t)(stride_row * esize)) & 15);  // 16-byte loads
  SplitParams split, *in_parts = nullptr;
  // (more than 128 rows do without a workspace that does not serve: for those none is asked for at every size)
  const bool optional = R > 128 && (((uintptr_t)workspace & 255) || sample_layout(&split, nullptr, R, vocab, top_k, top_p) > workspace_bytes);
  if (workspace && !optional && sample_in_parts(R, vocab, top_k, top_p)) {
    if ((uintptr_t)workspace & 255) return mi_fail(MI_ERR_ALIGN, "mi_sample_from_logits_ws: the workspace must be 256-byte aligned");
    if (sample_layout(&split, (uint8_t*)workspace, R, vocab, top_k, top_p) > workspace_bytes)
      return mi_fail(MI_ERR_WORKSPACE, "mi_sample_from_logits_ws: workspace smaller than mi_sample_workspace_bytes()");
    split.s = p;
    in_parts = &split;
  }
  hipStream_t st = (hipStream_t)stream;
  if (logits_dtype == 2) {
    if (wide) launch_sample<2, 8>(p, in_parts, st);
    else launch_sample<2, 1>(p, in_parts, st);
  } else if (logits_dtype == 1) {
    if (wide) launch_sample<1, 8>(p, in_parts, st);
    else launch_sample<1, 1>(p, in_parts, st);
  } else {
    if (wide) launch_sample<0, 4>(p, in_parts, st);
    else launch_sample<0, 1>(p, in_parts, st);
  }
  return mi_check_launch("mi_sample_from_logits");
}

extern "C" int mi_sample_from_logits(const void* logits, int64_t stride_row, int32_t logits_dtype, int32_t R,
                                     int32_t vocab, int32_t top_k, float top_p, float temperature,
                                     const float* uniform, int32_t vocab_clamp, int64_t* samples,
                                     float* cut_values, const int32_t* request_kv_length_offsets,
                                     const int32_t* request_query_lengths, const int32_t* request_output_lengths,
                                     int64_t termination_id, uint8_t* active_request_mask, void* stream) {
  return mi_sample_from_logits_ws(logits, stride_row, logits_dtype, R, vocab, top_k, top_p, temperature, uniform, vocab_clamp,
                                  samples, cut_values, request_kv_length_offsets, request_query_lengths,
                                  request_output_lengths, termination_id, active_request_mask, nullptr, 0, stream);
}

extern "C" int mi_selected_log_probs(const void* logits, int64_t stride_row, int32_t logits_dtype, int32_t T,
                                     int32_t vocab, const int64_t* token_ids, float* log_probs, void* stream) {
  if (T == 0) return MI_OK;
  if (!logits || !token_ids || !log_probs) return mi_fail(MI_ERR_NULL, "mi_selected_log_probs: null pointer argument");
  if (T < 0 || vocab <= 0 || stride_row < vocab)
    return mi_fail(MI_ERR_SHAPE, "mi_selected_log_probs: need T >= 0, vocab > 0 and a row stride of at least vocab");
  if (logits_dtype < 0 || logits_dtype > 2)
    return mi_fail(MI_ERR_UNSUPPORTED, "mi_selected_log_probs: logits must be fp32 (0), bf16 (1) or fp16 (2)");
  LogProbParams p;
  p.logits = logits; p.stride = stride_row; p.T = T; p.V = vocab; p.token_ids = token_ids; p.out = log_probs;
  const int esize = logits_dtype != 0 ? 2 : 4;
  const bool wide = !(((uintptr_t)logits | (uintptr_t)(stride_row * esize)) & 15);  // 16-byte loads
  const dim3 grid(T), block(kLogProbThreads);
  hipStream_t st = (hipStream_t)stream;
  if (logits_dtype == 2) {
    if (wide) hipLaunchKernelGGL((selected_log_probs_kernel<2, 8>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((selected_log_probs_kernel<2, 1>), grid, block, 0, st, p);
  } else if (logits_dtype == 1) {
    if (wide) hipLaunchKernelGGL((selected_log_probs_kernel<1, 8>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((selected_log_probs_kernel<1, 1>), grid, block, 0, st, p);
  } else {
    if (wide) hipLaunchKernelGGL((selected_log_probs_kernel<0, 4>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((selected_log_probs_kernel<0, 1>), grid, block, 0, st, p);
  }
  return mi_check_launch("mi_selected_log_probs");
}
