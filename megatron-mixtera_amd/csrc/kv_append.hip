// KV-append into the chunked ("paged") KV cache.
//
// Two addressing modes:
//  * mi_kv_append: the slot of every token is given by the reference's per-token
//    rows `token_to_chunk_idx` / `token_to_local_position_within_kv_chunk`
//    (int64), i.e. memory_buffer[0|1, layer, chunk_idx, local] = key|value
//    (megatron/core/inference/contexts/dynamic_context.py:511-545).
//  * mi_kv_append_decode: one new token per request; the slot is derived on the
//    GPU from the block table and the kv length that already counts the new
//    token: pos = len-1, chunk = block_table[r][pos / C], local = pos % C.
//    Rows with len <= 0 (batch padding) write nothing.
// Both are pure copies: the cache holds the source bits unchanged.
//
// fp8 variants quantise on the way in (OCP e4m3fn, round to nearest even,
// saturating at +-448) with one fp32 scale per (chunk, KV head).
#include "mi_common.h"
#include "mi_capi_internal.h"

namespace mi {

struct AppendParams {
  const uint8_t* key;
  const uint8_t* value;
  int64_t src_stride;  // bytes between tokens in key / value
  uint8_t* kc;
  uint8_t* vc;
  int64_t chunk_bytes;  // bytes between chunks
  int64_t tok_bytes;    // bytes between tokens inside a chunk
  const int64_t* tok_chunk;
  const int64_t* tok_local;
  const int32_t* bt;
  int64_t bt_stride;
  const int32_t* lens;
  int32_t chunk, row_bytes, T;
};

// grid = (T, 2): blockIdx.y selects key / value.  VEC = bytes moved per thread step.
template <int VEC, bool DECODE>
__global__ __launch_bounds__(256) void kv_append_kernel(AppendParams p) {
  const int t = blockIdx.x;
  int64_t c, l;
  if (DECODE) {
    const int len = p.lens[t];
    if (len <= 0) return;
    const int pos = len - 1;
    const int ci = pos / p.chunk;
    c = p.bt[(int64_t)t * p.bt_stride + ci];
    l = pos - ci * p.chunk;
  } else {
    c = p.tok_chunk[t];
    l = p.tok_local[t];
  }
  const uint8_t* src = (blockIdx.y ? p.value : p.key) + (int64_t)t * p.src_stride;
  uint8_t* dst = (blockIdx.y ? p.vc : p.kc) + c * p.chunk_bytes + l * p.tok_bytes;
  for (int i = threadIdx.x * VEC; i < p.row_bytes; i += 256 * VEC) {
    if (VEC == 16) st16(dst + i, ld16(src + i));
    else if (VEC == 4) *reinterpret_cast<uint32_t*>(dst + i) = *reinterpret_cast<const uint32_t*>(src + i);
    else if (VEC == 2) *reinterpret_cast<uint16_t*>(dst + i) = *reinterpret_cast<const uint16_t*>(src + i);
    else dst[i] = src[i];
  }
}

struct QuantParams {
  const uint16_t* src;   // rows in the 16-bit type the kernel is instantiated for
  int64_t src_stride;    // elements between tokens (bulk: between chunk tokens)
  int64_t src_chunk;     // bulk: elements between chunks
  uint8_t* dst;          // fp8 cache
  int64_t chunk_bytes, tok_bytes;
  float* scale;          // [n_chunks][Hkv]
  const int32_t* bt;
  int64_t bt_stride;
  const int32_t* lens;
  int32_t chunk, Hkv, d;
  float headroom;
};

// One workgroup (256 threads) per (chunk, KV head): amax over the whole
// chunk-head tile, scale = amax / 448, then quantise.  Used to fill an fp8 cache
// from bf16 chunks (prefill-style writes and benchmark set-up).
template <bool F16>
__global__ __launch_bounds__(256) void quantize_chunks_fp8_kernel(QuantParams p) {
  const int c = blockIdx.x, h = blockIdx.y;
  const uint16_t* src = p.src + (int64_t)c * p.src_chunk + (int64_t)h * p.d;
  const int n = p.chunk * p.d;
  float amax = 0.f;
  for (int i = threadIdx.x; i < n; i += 256) {
    const int tok = i / p.d, e = i - tok * p.d;
    amax = fmaxf(amax, fabsf(to_f32<F16>(src[(int64_t)tok * p.src_stride + e])));
  }
  __shared__ float red[256];
  red[threadIdx.x] = amax;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  amax = red[0];
  const float scale = amax > 0.f ? amax / 448.f : 1.f;
  if (threadIdx.x == 0) p.scale[(int64_t)c * p.Hkv + h] = scale;
  uint8_t* dst = p.dst + (int64_t)c * p.chunk_bytes + (int64_t)h * p.d;
  for (int i = threadIdx.x; i < n; i += 256) {
    const int tok = i / p.d, e = i - tok * p.d;
    const float v = to_f32<F16>(src[(int64_t)tok * p.src_stride + e]) / scale;
    dst[(int64_t)tok * p.tok_bytes + e] = (uint8_t)f32_to_e4m3_sat(v);
  }
}

// One workgroup per (request, KV head): quantise the newly generated token.
// A token that opens a chunk (local position 0) fixes that chunk-head's scale to
// headroom * amax(token) / 448; later tokens reuse the stored scale and saturate.
template <bool F16>
__global__ __launch_bounds__(64) void kv_append_decode_fp8_kernel(QuantParams p) {
  const int r = blockIdx.x, h = blockIdx.y;
  const int len = p.lens[r];
  if (len <= 0) return;
  const int pos = len - 1;
  const int ci = pos / p.chunk;
  const int64_t c = p.bt[(int64_t)r * p.bt_stride + ci];
  const int l = pos - ci * p.chunk;
  const uint16_t* src = p.src + (int64_t)r * p.src_stride + (int64_t)h * p.d;
  float scale;
  if (l == 0) {
    float amax = 0.f;
    for (int e = threadIdx.x; e < p.d; e += 64) amax = fmaxf(amax, fabsf(to_f32<F16>(src[e])));
    for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
    scale = amax > 0.f ? p.headroom * amax / 448.f : 1.f;
    if (threadIdx.x == 0) p.scale[c * p.Hkv + h] = scale;
  } else {
    scale = p.scale[c * p.Hkv + h];
  }
  uint8_t* dst = p.dst + c * p.chunk_bytes + (int64_t)l * p.tok_bytes + (int64_t)h * p.d;
  for (int e = threadIdx.x; e < p.d; e += 64) dst[e] = (uint8_t)f32_to_e4m3_sat(to_f32<F16>(src[e]) / scale);
}

// ---- fp8 append of many tokens per request (prefill / mixed steps) ----------------------------
// Slots come from the per-token rows.  Tokens of one chunk are neighbours in the token dimension
// with rising local positions (that is how the context lays requests out), so the tokens a call
// writes into a chunk form one run.  A run that starts at local position 0 opens the chunk and fixes
// the scale of each of its heads: amax over the whole run / 448, times `headroom` unless the run
// fills the chunk (later tokens of a partly filled chunk reuse the scale and saturate).  A run that
// starts further in reuses the stored scale.
struct AppendFp8Params {
  const uint16_t* src[2];          // key, value rows (16-bit)
  int64_t src_st[2], src_sh[2];    // elements between tokens / heads
  uint8_t* dst[2];                 // fp8 caches
  int64_t chunk_bytes, tok_bytes;
  float* scale[2];                 // [n_chunks][Hkv] each
  const int64_t* tok_chunk;
  const int64_t* tok_local;
  int32_t T, chunk, Hkv, d, slice;
  float headroom;
};

// Byte of clamp(v / scale): the quotient by the scale's correctly rounded reciprocal and one residual step.  The bytes
// are those of the division: a quotient that lies on a boundary between two bytes (5 significant bits) comes out as
// that boundary, because the residual is exact and its product with the reciprocal is off by 2^-24 of it, and no other
// quotient of a 16-bit value and a 24-bit scale is near enough to a boundary to be rounded across it.  (That needs
// residuals above the underflow limit: scales outside 2^+-60 take the division.)  5 instructions instead of 12 or so.
struct Fp8Scale {
  float scale, inv, lim;
  bool fast;
};
static __device__ __forceinline__ Fp8Scale fp8_scale(float scale) {
  Fp8Scale q;
  q.scale = scale;
  q.inv = 1.f / scale;
  q.lim = 448.f * scale;
  q.fast = scale > 0x1p-60f && scale < 0x1p60f;
  return q;
}
static __device__ __forceinline__ float fp8_quotient(float v, const Fp8Scale& q) {
  const float c = __builtin_amdgcn_fmed3f(v, -q.lim, q.lim);  // (NaN: the lower limit, as in the saturating conversion)
  const float q1 = c * q.inv;
  return __builtin_fmaf(-__builtin_fmaf(q1, q.scale, -c), q.inv, q1);  // (the residual's sign this way round: -0 stays -0)
}
template <bool F16, bool FAST>
static __device__ __forceinline__ uint2 fp8_bytes8(uint4 w, const Fp8Scale& q) {
  const uint32_t u[4] = {w.x, w.y, w.z, w.w};
  uint32_t out[2] = {0u, 0u};
  if (FAST) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      int r = __builtin_amdgcn_cvt_pk_fp8_f32(fp8_quotient(lo_to_f32<F16>(u[2 * j]), q), fp8_quotient(hi_to_f32<F16>(u[2 * j]), q), 0, false);
      r = __builtin_amdgcn_cvt_pk_fp8_f32(fp8_quotient(lo_to_f32<F16>(u[2 * j + 1]), q), fp8_quotient(hi_to_f32<F16>(u[2 * j + 1]), q), r, true);
      out[j] = (uint32_t)r;
    }
  } else {
#pragma unroll 1
    for (int j = 0; j < 4; ++j) {
      const uint32_t x = j == 0 ? w.x : j == 1 ? w.y : j == 2 ? w.z : w.w;
      const uint32_t lo = f32_to_e4m3_sat(lo_to_f32<F16>(x) / q.scale), hi = f32_to_e4m3_sat(hi_to_f32<F16>(x) / q.scale);
      const uint32_t b = (lo | (hi << 8)) << (16 * (j & 1));
      if (j < 2) out[0] |= b; else out[1] |= b;
    }
  }
  return make_uint2(out[0], out[1]);
}
// Largest magnitude of eight values, as bit patterns (whose order is that of the magnitudes): two packed 16-bit maxima
// per instruction.  A NaN is above every number here, so a result above infinity asks for `amax8`, which skips NaNs.
typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));
static __device__ __forceinline__ u16x2_t amax_bits8(uint4 w, u16x2_t m) {
  const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2_t, u[j] & 0x7fff7fffu));
  return m;
}
template <bool F16>
static __device__ __forceinline__ float amax8(uint4 w, float m) {
  const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) m = fmaxf(m, fmaxf(fabsf(lo_to_f32<F16>(u[j])), fabsf(hi_to_f32<F16>(u[j]))));
  return m;
}

// grid = (ceil(T / slice), Hkv, 2): a workgroup takes the runs that START among `slice` <= kFp8Slice tokens -- one head of the
// key (z = 0) or value (z = 1) rows of each -- and quantises them whole: the run's values stay in registers between
// the maximum that gives the scale and the conversion, so they are read once and there is no second launch.
// Bound by memory for long prompts (3 bytes per value) and by the chain of loads (slots -> run -> values) for short
// ones.  13 900 tokens x 8 heads of 128, key and value, kernel time by trace: 27 us as a prompt step runs it, 23 with the
// rows in the last-level cache (scales in a launch of their own, then the rows: 65 us); 1 000 tokens and 24 padded rows:
// 12 us (57: each padded row was a run that a workgroup walked on its own).
//   A run of one token, and a token that continues a chunk opened by an earlier call, need no more than a row: those
//   of the slice are taken together, the threads spread over rows x pieces.
//   A longer run is walked by the whole workgroup: the first kFp8Keep pieces (16 bytes each) of every thread -- a
//   256-token chunk's head of 128 -- stay in registers, what a larger chunk has beyond them is read again.
// WIDE: rows of whole 16-byte pieces, 16-byte aligned, whose number divides the threads (the bytes 8-byte aligned, a
// chunk's rows within 32-bit offsets); anything else goes element by element.
constexpr int kFp8Slice = 128, kFp8Keep = 8, kFp8Threads = 512;
template <bool F16, bool WIDE>
__global__ __launch_bounds__(kFp8Threads, 4) void kv_append_fp8_kernel(AppendFp8Params p) {
  const int t0 = blockIdx.x * p.slice, h = blockIdx.y, kv = blockIdx.z;
  const int tid = threadIdx.x;
  __shared__ int long_s[kFp8Slice], row_s[kFp8Slice];   // tokens that open a longer run; tokens taken row by row
  __shared__ int64_t chunk_s[kFp8Slice], local_s[kFp8Slice];
  __shared__ int n_long_s, n_row_s;
  __shared__ int count_s[2], end_s[2];
  __shared__ float red[kFp8Threads / 64];
  // maximum over the workgroup (its two barriers also separate uses of `red`)
  auto block_max = [&](float m) {
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    __syncthreads();
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    for (int w = 0; w < kFp8Threads / 64; ++w) m = fmaxf(m, red[w]);
    return m;
  };
  if (tid == 0) n_long_s = n_row_s = count_s[0] = end_s[0] = count_s[1] = end_s[1] = 0;
  __syncthreads();
  if (tid < p.slice && t0 + tid < p.T) {
    const int t = t0 + tid;
    const int64_t c = p.tok_chunk[t], l = p.tok_local[t];
    chunk_s[tid] = c;
    local_s[tid] = l;
    // the token that would have opened this one's run, and whether a run of two or more starts there
    const int64_t o = t - l;
    const bool opened = o >= 0 && o + 1 < p.T && p.tok_chunk[o] == c && p.tok_local[o] == 0 && p.tok_chunk[o + 1] == c &&
                        p.tok_local[o + 1] == 1 && l < p.chunk;
    if (!opened) row_s[atomicAdd(&n_row_s, 1)] = tid;
    else if (l == 0) long_s[atomicAdd(&n_long_s, 1)] = tid;
  }
  __syncthreads();
  const int n_long = n_long_s, n_row = n_row_s;
  constexpr int EPP = WIDE ? 8 : 1;    // elements per piece
  const int per_row = p.d / EPP;       // pieces per head row
  const int64_t st = p.src_st[kv];
  const uint16_t* const src_h = p.src[kv] + (int64_t)h * p.src_sh[kv];
  uint8_t* const dst_h = p.dst[kv] + (int64_t)h * p.d;

  // ---- rows: one wavefront lane group per row where the pieces of a row fill whole groups, else a row per thread group
  if (n_row > 0) {
    const int group = WIDE && per_row <= 64 ? per_row : kFp8Threads;  // threads per row
    const int sub = tid % group;
    for (int k = tid / group; k < n_row; k += kFp8Threads / group) {   // (uniform over the threads of a group)
      const int i = row_s[k], t = t0 + i;
      const int64_t c = chunk_s[i];
      const uint16_t* src = src_h + (int64_t)t * st;
      uint8_t* dst = dst_h + c * p.chunk_bytes + local_s[i] * p.tok_bytes;
      float* scale_at = p.scale[kv] + c * p.Hkv + h;
      if (WIDE && group < kFp8Threads) {
        const uint4 w = ld16(src + 8 * sub);
        float scale;
        if (local_s[i] == 0) {  // the token opens its chunk
          float m = amax8<F16>(w, 0.f);
          for (int o = group >> 1; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
          const float hr = p.chunk == 1 ? 1.f : p.headroom;
          scale = m > 0.f ? hr * m / 448.f : 1.f;
          if (sub == 0) *scale_at = scale;
        } else {
          scale = *scale_at;
        }
        const Fp8Scale q = fp8_scale(scale);
        uint2 bytes;
        if (q.fast) bytes = fp8_bytes8<F16, true>(w, q); else bytes = fp8_bytes8<F16, false>(w, q);
        st8(dst + 8 * sub, bytes);
      } else {
        float scale;
        if (local_s[i] == 0) {
          float m = 0.f;
          for (int e = tid; e < p.d; e += kFp8Threads) m = fmaxf(m, fabsf(to_f32<F16>(src[e])));
          m = block_max(m);
          const float hr = p.chunk == 1 ? 1.f : p.headroom;
          scale = m > 0.f ? hr * m / 448.f : 1.f;
          if (tid == 0) *scale_at = scale;
        } else {
          scale = *scale_at;
        }
        for (int e = tid; e < p.d; e += kFp8Threads) dst[e] = (uint8_t)f32_to_e4m3_sat(to_f32<F16>(src[e]) / scale);
      }
    }
  }

  // ---- longer runs -------------------------------------------------------------------------------------------------
  for (int k = 0; k < n_long; ++k) {
    const int i0 = __builtin_amdgcn_readfirstlane(long_s[k]), t = t0 + i0;
    const int64_t c = ((int64_t)__builtin_amdgcn_readfirstlane((int)(chunk_s[i0] >> 32)) << 32) |
                      (uint32_t)__builtin_amdgcn_readfirstlane((int)chunk_s[i0]);
    auto in_run = [&](int i) { return t + i < p.T && p.tok_chunk[t + i] == c && p.tok_local[t + i] == i; };
    // the run's tokens: their number and the last one's position (equal, unless the caller's rows have gaps)
    int cnt = 0, end = 0;
    for (int i = tid; i < p.chunk; i += kFp8Threads)
      if (in_run(i)) { ++cnt; end = i + 1; }
    for (int o = 32; o > 0; o >>= 1) {
      cnt += __shfl_xor(cnt, o, 64);
      end = max(end, __shfl_xor(end, o, 64));
    }
    if ((tid & 63) == 0) {
      atomicAdd(&count_s[k & 1], cnt);
      atomicMax(&end_s[k & 1], end);
    }
    __syncthreads();
    const int n = __builtin_amdgcn_readfirstlane(count_s[k & 1]), n_end = __builtin_amdgcn_readfirstlane(end_s[k & 1]);
    if (tid == 0) count_s[(k + 1) & 1] = end_s[(k + 1) & 1] = 0;  // (everyone has left the other pair: a barrier lies between)
    const bool gaps = n != n_end;
    const uint16_t* src = src_h + (int64_t)t * st;
    uint8_t* dst = dst_h + c * p.chunk_bytes;
    if (WIDE) {
      // a thread keeps its piece of the row and takes every rstep-th row; rows past the last repeat it
      const int rstep = kFp8Threads / per_row, row0 = tid / per_row, e = 8 * (tid - row0 * per_row);
      const int kept = gaps ? 0 : min(n_end, rstep * kFp8Keep);   // rows that stay in registers
      const uint32_t off0 = 2u * (uint32_t)(row0 * (int)st + e), off_step = 2u * (uint32_t)(rstep * (int)st),
                     off_lim = 2u * (uint32_t)((kept - 1) * (int)st + e);
      uint4 keep[kFp8Keep];
      u16x2_t mb = {0, 0};
      if (kept > 0) {
#pragma unroll
        for (int j = 0; j < kFp8Keep; ++j)
          keep[j] = ld16(reinterpret_cast<const uint8_t*>(src) + min(off0 + (uint32_t)j * off_step, off_lim));
#pragma unroll
        for (int j = 0; j < kFp8Keep; ++j) mb = amax_bits8(keep[j], mb);
      }
      for (int row = kept + row0; row < n_end; row += rstep)
        if (!gaps || in_run(row)) mb = amax_bits8(ld16(src + (int64_t)row * st + e), mb);
      float amax = block_max((float)max(mb.x, mb.y));   // (exact: the patterns are below 2^16)
      if (amax > (F16 ? 0x7c00 : 0x7f80)) {             // some value is NaN: the maximum of the others
        float m = 0.f;
        for (int row = row0; row < n_end; row += rstep)
          if (!gaps || in_run(row)) m = amax8<F16>(ld16(src + (int64_t)row * st + e), m);
        amax = block_max(m);
      } else {
        amax = lo_to_f32<F16>((uint32_t)amax);
      }
      const float scale = amax > 0.f ? (n == p.chunk ? 1.f : p.headroom) * amax / 448.f : 1.f;
      if (tid == 0) p.scale[kv][c * p.Hkv + h] = scale;
      const Fp8Scale q = fp8_scale(scale);
      if (q.fast) {
        const uint32_t tokb = (uint32_t)p.tok_bytes;
#pragma unroll
        for (int j = 0; j < kFp8Keep; ++j)
          if (row0 + rstep * j < kept) st8(dst + (uint32_t)(row0 + rstep * j) * tokb + e, fp8_bytes8<F16, true>(keep[j], q));
        for (int row = kept + row0; row < n_end; row += rstep)
          if (!gaps || in_run(row)) st8(dst + (int64_t)row * p.tok_bytes + e, fp8_bytes8<F16, true>(ld16(src + (int64_t)row * st + e), q));
      } else {
        for (int row = row0; row < n_end; row += rstep)
          if (!gaps || in_run(row)) st8(dst + (int64_t)row * p.tok_bytes + e, fp8_bytes8<F16, false>(ld16(src + (int64_t)row * st + e), q));
      }
    } else {
      const int pieces = n_end * per_row;
      float amax = 0.f;
      for (int idx = tid; idx < pieces; idx += kFp8Threads) {
        const int row = idx / per_row;
        if (!(gaps && !in_run(row))) amax = fmaxf(amax, fabsf(to_f32<F16>(src[(int64_t)row * st + (idx - row * per_row)])));
      }
      amax = block_max(amax);
      const float scale = amax > 0.f ? (n == p.chunk ? 1.f : p.headroom) * amax / 448.f : 1.f;
      if (tid == 0) p.scale[kv][c * p.Hkv + h] = scale;
      for (int idx = tid; idx < pieces; idx += kFp8Threads) {
        const int row = idx / per_row, e = idx - row * per_row;
        if (!(gaps && !in_run(row)))
          dst[(int64_t)row * p.tok_bytes + e] = (uint8_t)f32_to_e4m3_sat(to_f32<F16>(src[(int64_t)row * st + e]) / scale);
      }
    }
    __syncthreads();
  }
}

// n_tensors = 2: key and value; 1: the key alone (a cache with one row per token, e.g. MLA latents)
template <bool DECODE>
static int launch_append(AppendParams& p, hipStream_t st, int n_tensors = 2) {
  const uintptr_t bits = (uintptr_t)p.key | (uintptr_t)p.value | (uintptr_t)p.kc | (uintptr_t)p.vc |
                         (uintptr_t)p.src_stride | (uintptr_t)p.chunk_bytes | (uintptr_t)p.tok_bytes |
                         (uintptr_t)p.row_bytes;
  dim3 grid(p.T, n_tensors), block(256);
  if (!(bits & 15)) hipLaunchKernelGGL((kv_append_kernel<16, DECODE>), grid, block, 0, st, p);
  else if (!(bits & 3)) hipLaunchKernelGGL((kv_append_kernel<4, DECODE>), grid, block, 0, st, p);
  else if (!(bits & 1)) hipLaunchKernelGGL((kv_append_kernel<2, DECODE>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((kv_append_kernel<1, DECODE>), grid, block, 0, st, p);
  return MI_OK;
}

}  // namespace mi

using namespace mi;

extern "C" int mi_kv_append(const void* key, const void* value, int64_t src_stride_tok,
                            void* k_cache, void* v_cache, int64_t kv_stride_chunk,
                            int64_t kv_stride_tok, const int64_t* token_to_chunk_idx,
                            const int64_t* token_to_local_pos, int32_t T, int32_t row_elems,
                            int32_t elem_bytes, void* stream) {
  if (T == 0) return MI_OK;
  if (!key || !k_cache || !token_to_chunk_idx || !token_to_local_pos || (value == nullptr) != (v_cache == nullptr))
    return mi_fail(MI_ERR_NULL, "mi_kv_append: null pointer argument (value and v_cache go together)");
  if (T < 0 || row_elems <= 0 || elem_bytes <= 0 || src_stride_tok < row_elems || kv_stride_tok < row_elems)
    return mi_fail(MI_ERR_SHAPE, "mi_kv_append: bad sizes or strides");
  AppendParams p = {};
  p.key = (const uint8_t*)key; p.value = (const uint8_t*)value;
  p.src_stride = src_stride_tok * elem_bytes;
  p.kc = (uint8_t*)k_cache; p.vc = (uint8_t*)v_cache;
  p.chunk_bytes = kv_stride_chunk * elem_bytes; p.tok_bytes = kv_stride_tok * elem_bytes;
  p.tok_chunk = token_to_chunk_idx; p.tok_local = token_to_local_pos;
  p.row_bytes = row_elems * elem_bytes; p.T = T; p.chunk = 1;
  launch_append<false>(p, (hipStream_t)stream, value ? 2 : 1);
  return mi_check_launch("mi_kv_append");
}

extern "C" int mi_kv_append_decode(const void* key, const void* value, int64_t src_stride_tok,
                                   void* k_cache, void* v_cache, int64_t kv_stride_chunk,
                                   int64_t kv_stride_tok, const int32_t* block_table,
                                   int64_t bt_stride, const int32_t* kv_lens, int32_t R,
                                   int32_t chunk_tokens, int32_t row_elems, int32_t elem_bytes,
                                   void* stream) {
  if (R == 0) return MI_OK;
  if (!key || !value || !k_cache || !v_cache || !block_table || !kv_lens)
    return mi_fail(MI_ERR_NULL, "mi_kv_append_decode: null pointer argument");
  if (R < 0 || row_elems <= 0 || elem_bytes <= 0 || chunk_tokens <= 0 || src_stride_tok < row_elems ||
      kv_stride_tok < row_elems)
    return mi_fail(MI_ERR_SHAPE, "mi_kv_append_decode: bad sizes or strides");
  AppendParams p = {};
  p.key = (const uint8_t*)key; p.value = (const uint8_t*)value;
  p.src_stride = src_stride_tok * elem_bytes;
  p.kc = (uint8_t*)k_cache; p.vc = (uint8_t*)v_cache;
  p.chunk_bytes = kv_stride_chunk * elem_bytes; p.tok_bytes = kv_stride_tok * elem_bytes;
  p.bt = block_table; p.bt_stride = bt_stride; p.lens = kv_lens;
  p.row_bytes = row_elems * elem_bytes; p.T = R; p.chunk = chunk_tokens;
  launch_append<true>(p, (hipStream_t)stream);
  return mi_check_launch("mi_kv_append_decode");
}

extern "C" int mi_kv_quantize_chunks_fp8(const void* src, int64_t src_stride_chunk,
                                         int64_t src_stride_tok, void* dst_fp8,
                                         int64_t dst_stride_chunk, int64_t dst_stride_tok,
                                         float* scales, int32_t n_chunks, int32_t chunk_tokens,
                                         int32_t Hkv, int32_t head_dim, int32_t dtype, void* stream) {
  if (n_chunks == 0) return MI_OK;
  if (dtype != MI_DTYPE_BF16 && dtype != MI_DTYPE_FP16)
    return mi_fail(MI_ERR_UNSUPPORTED, "mi_kv_quantize_chunks_fp8: dtype must be MI_DTYPE_BF16 or MI_DTYPE_FP16");
  if (!src || !dst_fp8 || !scales) return mi_fail(MI_ERR_NULL, "mi_kv_quantize_chunks_fp8: null pointer argument");
  if (n_chunks < 0 || chunk_tokens <= 0 || Hkv <= 0 || head_dim <= 0 || Hkv > 65535)
    return mi_fail(MI_ERR_SHAPE, "mi_kv_quantize_chunks_fp8: bad sizes");
  QuantParams p = {};
  p.src = (const uint16_t*)src; p.src_chunk = src_stride_chunk; p.src_stride = src_stride_tok;
  p.dst = (uint8_t*)dst_fp8; p.chunk_bytes = dst_stride_chunk; p.tok_bytes = dst_stride_tok;
  p.scale = scales; p.chunk = chunk_tokens; p.Hkv = Hkv; p.d = head_dim; p.headroom = 1.f;
  if (dtype == MI_DTYPE_FP16) hipLaunchKernelGGL(quantize_chunks_fp8_kernel<true>, dim3(n_chunks, Hkv), dim3(256), 0, (hipStream_t)stream, p);
  else hipLaunchKernelGGL(quantize_chunks_fp8_kernel<false>, dim3(n_chunks, Hkv), dim3(256), 0, (hipStream_t)stream, p);
  return mi_check_launch("mi_kv_quantize_chunks_fp8");
}

extern "C" int mi_kv_append_decode_fp8(const void* key, const void* value,
                                       int64_t src_stride_tok, void* k_cache_fp8, void* v_cache_fp8,
                                       int64_t kv_stride_chunk, int64_t kv_stride_tok,
                                       float* k_scales, float* v_scales, const int32_t* block_table,
                                       int64_t bt_stride, const int32_t* kv_lens, int32_t R,
                                       int32_t chunk_tokens, int32_t Hkv, int32_t head_dim,
                                       float headroom, int32_t dtype, void* stream) {
  if (R == 0) return MI_OK;
  if (dtype != MI_DTYPE_BF16 && dtype != MI_DTYPE_FP16)
    return mi_fail(MI_ERR_UNSUPPORTED, "mi_kv_append_decode_fp8: dtype must be MI_DTYPE_BF16 or MI_DTYPE_FP16");
  if (!key || !value || !k_cache_fp8 || !v_cache_fp8 || !k_scales || !v_scales || !block_table || !kv_lens)
    return mi_fail(MI_ERR_NULL, "mi_kv_append_decode_fp8: null pointer argument");
  if (R < 0 || chunk_tokens <= 0 || Hkv <= 0 || head_dim <= 0 || Hkv > 65535 || !(headroom > 0.f))
    return mi_fail(MI_ERR_SHAPE, "mi_kv_append_decode_fp8: bad sizes");
  QuantParams p = {};
  p.src_stride = src_stride_tok; p.chunk_bytes = kv_stride_chunk; p.tok_bytes = kv_stride_tok;
  p.bt = block_table; p.bt_stride = bt_stride; p.lens = kv_lens;
  p.chunk = chunk_tokens; p.Hkv = Hkv; p.d = head_dim; p.headroom = headroom;
  const auto kernel = dtype == MI_DTYPE_FP16 ? kv_append_decode_fp8_kernel<true> : kv_append_decode_fp8_kernel<false>;
  p.src = (const uint16_t*)key; p.dst = (uint8_t*)k_cache_fp8; p.scale = k_scales;
  hipLaunchKernelGGL(kernel, dim3(R, Hkv), dim3(64), 0, (hipStream_t)stream, p);
  p.src = (const uint16_t*)value; p.dst = (uint8_t*)v_cache_fp8; p.scale = v_scales;
  hipLaunchKernelGGL(kernel, dim3(R, Hkv), dim3(64), 0, (hipStream_t)stream, p);
  return mi_check_launch("mi_kv_append_decode_fp8");
}

extern "C" int mi_kv_append_fp8_strided(const void* key, int64_t k_stride_tok, int64_t k_stride_head, const void* value,
                                        int64_t v_stride_tok, int64_t v_stride_head, void* k_cache_fp8,
                                        void* v_cache_fp8, int64_t kv_stride_chunk, int64_t kv_stride_tok,
                                        float* k_scales, float* v_scales, const int64_t* token_to_chunk_idx,
                                        const int64_t* token_to_local_pos, int32_t T, int32_t chunk_tokens, int32_t Hkv,
                                        int32_t head_dim, float headroom, int32_t dtype, void* stream) {
  if (T == 0) return MI_OK;
  if (dtype != MI_DTYPE_BF16 && dtype != MI_DTYPE_FP16)
    return mi_fail(MI_ERR_UNSUPPORTED, "mi_kv_append_fp8: dtype must be MI_DTYPE_BF16 or MI_DTYPE_FP16");
  if (!key || !value || !k_cache_fp8 || !v_cache_fp8 || !k_scales || !v_scales || !token_to_chunk_idx ||
      !token_to_local_pos)
    return mi_fail(MI_ERR_NULL, "mi_kv_append_fp8: null pointer argument");
  // (a head stride below the head's width is taken for one head only: it is never used)
  const auto rows_ok = [&](int64_t st, int64_t sh) {
    return Hkv == 1 ? st >= head_dim : sh >= head_dim && st >= (int64_t)(Hkv - 1) * sh + head_dim;
  };
  if (T < 0 || chunk_tokens <= 0 || Hkv <= 0 || head_dim <= 0 || Hkv > 65535 || !(headroom > 0.f) ||
      !rows_ok(k_stride_tok, k_stride_head) || !rows_ok(v_stride_tok, v_stride_head) ||
      kv_stride_tok < (int64_t)Hkv * head_dim)
    return mi_fail(MI_ERR_SHAPE, "mi_kv_append_fp8: bad sizes or strides");
  AppendFp8Params p = {};
  p.src[0] = (const uint16_t*)key; p.src_st[0] = k_stride_tok; p.src_sh[0] = k_stride_head;
  p.src[1] = (const uint16_t*)value; p.src_st[1] = v_stride_tok; p.src_sh[1] = v_stride_head;
  p.dst[0] = (uint8_t*)k_cache_fp8; p.dst[1] = (uint8_t*)v_cache_fp8;
  p.chunk_bytes = kv_stride_chunk; p.tok_bytes = kv_stride_tok;
  p.scale[0] = k_scales; p.scale[1] = v_scales;
  p.tok_chunk = token_to_chunk_idx; p.tok_local = token_to_local_pos;
  p.T = T; p.chunk = chunk_tokens; p.Hkv = Hkv; p.d = head_dim; p.headroom = headroom;
  const bool wide = head_dim % 8 == 0 && kFp8Threads % (head_dim / 8) == 0 &&
                    chunk_tokens * k_stride_tok < (int64_t)1 << 30 && chunk_tokens * v_stride_tok < (int64_t)1 << 30 &&
                    chunk_tokens * kv_stride_tok < (int64_t)1 << 31 && !((head_dim | k_stride_tok | k_stride_head | v_stride_tok | v_stride_head) & 7) &&
                    !(((uintptr_t)key | (uintptr_t)value) & 15) &&
                    !(((uintptr_t)k_cache_fp8 | (uintptr_t)v_cache_fp8 | (uintptr_t)kv_stride_chunk | (uintptr_t)kv_stride_tok) & 7);
  const bool f16 = dtype == MI_DTYPE_FP16;
  // Tokens per workgroup: a workgroup without a run start is all latency (13 900 tokens in slices of 32: 43 us), one
  // with several walks them in turn (256: 28 us, 128: 27) -- 128 while that leaves the chip two workgroups per CU.
  const int64_t want = (int64_t)T * Hkv * 2 / 512;
  p.slice = want >= 128 ? 128 : want >= 64 ? 64 : 32;
  const dim3 grid((T + p.slice - 1) / p.slice, Hkv, 2), block(kFp8Threads);
  hipStream_t st = (hipStream_t)stream;
  if (wide && f16) hipLaunchKernelGGL((kv_append_fp8_kernel<true, true>), grid, block, 0, st, p);
  else if (wide) hipLaunchKernelGGL((kv_append_fp8_kernel<false, true>), grid, block, 0, st, p);
  else if (f16) hipLaunchKernelGGL((kv_append_fp8_kernel<true, false>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((kv_append_fp8_kernel<false, false>), grid, block, 0, st, p);
  return mi_check_launch("mi_kv_append_fp8");
}

extern "C" int mi_kv_append_fp8(const void* key, const void* value, int64_t src_stride_tok,
                                void* k_cache_fp8, void* v_cache_fp8, int64_t kv_stride_chunk,
                                int64_t kv_stride_tok, float* k_scales, float* v_scales,
                                const int64_t* token_to_chunk_idx, const int64_t* token_to_local_pos,
                                int32_t T, int32_t chunk_tokens, int32_t Hkv, int32_t head_dim,
                                float headroom, int32_t dtype, void* stream) {
  return mi_kv_append_fp8_strided(key, src_stride_tok, head_dim, value, src_stride_tok, head_dim, k_cache_fp8,
                                  v_cache_fp8, kv_stride_chunk, kv_stride_tok, k_scales, v_scales, token_to_chunk_idx,
                                  token_to_local_pos, T, chunk_tokens, Hkv, head_dim, headroom, dtype, stream);
}
