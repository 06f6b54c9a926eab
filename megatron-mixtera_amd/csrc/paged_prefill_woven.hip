// Paged varlen causal attention tiles for chunked prefill on gfx950: one instruction stream per wavefront.
//
// Serves the same call as the two-phase tile kernel of paged_prefill.hip -- flash_attn_varlen_func(..., causal=True,
// block_table=...) from Attention.flash_decode_and_prefill (megatron/core/transformer/attention.py:546-557) -- for
// head_dim 64 and 128 over a 16-bit or fp8 cache whose chunk size is a multiple of 64.
//
// A workgroup of 8 wavefronts (two per SIMD, 256 registers each) takes 256 consecutive (query token, head-in-group)
// rows of one (request, KV head), 32 rows per wavefront, and walks the keys in staged tiles of 64.  Workgroups of 4
// wavefronts share a CU by twos (74 KB of LDS each) and cover each other's start and end where walks are short
// (prefill_woven_waves).  At head_dim 64 the accumulators are half as many and the exponentials per product twice: there
// workgroups of 4 wavefronts, three per CU (168 registers, 41 KB of LDS each), put a third wavefront on every SIMD to fill
// the vector pipe (11 ragged prompts of 164-2 911 tokens, fp16: 148 us, the two-phase kernel 170).  Over an fp8 cache a
// call of no more than three workgroups per CU, where the third wavefront would come for a moment only, takes a build for
// two per CU and with more fragments ahead (bf16, 32/8 heads: two prompts of 1 100 tokens 48.0 -> 46.7 us, of 1 500 57 -> 54.5, one
// of 2 600 67.3 -> 64.5, of 1 000 level; but one of 4 000, 1 000 workgroups, 112 -> 120).  There are no
// matrix / vector phases and no per-phase barriers: every wavefront runs the whole tile pipeline in ONE stream, cut
// into 32-key steps and software-pipelined so that three independent chains are always open --
//     products    S^T(step s+1) = K Q^T          and  O^T += V^T P^T(step s-1)     (matrix cores)
//     vector ALU  P(step s) = exp2(S(step s) * scale - reference)  and the mask of S(step s+1)
//     LDS         the fragments of the products, one or three fragments ahead
// -- and the source orders them product pair / fragment read / a few vector instructions, pinned by scheduling
// barriers.  Whatever one wavefront of a SIMD cannot issue (a product waiting for the matrix core, a wait for LDS),
// the SIMD's other wavefront fills with its own stream; nothing but the one barrier per tile keeps them in step.
//
// Staging: a 64-key tile goes straight from memory into LDS (buffer loads with the LDS destination: no staging
// registers, no LDS stores), as 18 instructions of 64 lanes x 16 bytes over a line of 64 rows x 18 pieces (288-byte
// row pitch, the last two pieces of a row are padding).  The loads go through a buffer descriptor that covers the
// tile's rows up to the request's last key: rows beyond it arrive as zeros (their probabilities are masked to zero,
// and zero times a stale value must not be NaN).  Key and value tiles are double-buffered (values are multiplied one tile
// after their keys: the second half of a value tile is loaded one barrier after the first, when the half it replaces has
// been read); loads are issued right after the tile's barrier and are waited for at the next one.
//
// An fp8 cache (e4m3 bytes, one scale per chunk and KV head; a tile lies in one chunk) is staged through registers, a
// tile ahead: 8-byte loads set out after one barrier and are stored, converted, before the next.  Key bytes are
// converted exactly (four instructions per eight; e4m3 is a subset of both 16-bit types) and their scale multiplies the
// softmax scale of the tile instead.  Value bytes are converted as cheaply, times the power of two of their scale; the rest of
// the scale (value_factor) goes into the exponent of the tile's probabilities and out of their sum, which is kept per tile (values
// multiplied by their scale and rounded took 48 more vector instructions per tile; 2 x 8 000 tokens 1 081 -> 1 066 us).  At
// head_dim 64, half the values for as many probabilities and no registers for it, values are multiplied and rounded (the factor
// there: 12 prompts of 1 000 tokens 145 -> 148 us, two of 175-2 806 109 -> 111).  After a barrier the next keys set out before the
// second half of the values is converted (three prompts of 4 000, width 128, 617 -> 607).
//
// Softmax: exponentials are taken against a per-row reference that moves only when a probability leaves a window (a
// factor of 2^31 with bf16 operands, 2^8 with fp16); the row sums come out of the matrix cores (an all-ones A fragment).
// No maximum is taken beside the products: the step's finished probabilities are looked at two to a word (5 instructions for
// 16 scores a lane, where the maximum of the scores took 10), and where one has left the window the scores, still in
// registers, give the new reference, the accumulators and sums are rescaled and the step's probabilities made again.  (Steps,
// the maximum of every score -> this: 11 ragged prompts of width 64 147.0 -> 144.4 us, 6 prompts over an fp8 cache 456 -> 446, 8 x 2 048
// new tokens beside decoding requests 1 307 -> 1 280, 509 new tokens over 61 234 877 -> 854.)
#include <type_traits>

#include "mi_common.h"
#include "mi_capi_internal.h"
#include "paged_prefill_params.h"

namespace mi {

constexpr int kWvTile = 64;                      // keys per staged tile
// Fragment registers: fragment n lives in slot n % ring and is requested ring - 1 fragments ahead of its products.  Width 64 over
// an fp8 cache at three workgroups per CU: two fragments less are the registers that it lacks, and the SIMD's other two wavefronts
// cover the wait (with four it spilled nine; 12 prompts of 1 000 tokens 146 -> 136 us, 11 of 33-3 001 176 -> 167, 3 x 6 000 601 -> 568;
// over a 16-bit cache, which spills nothing, level).
template <int HD, bool FP8, int PER_SIMD> constexpr int wv_ring() { return FP8 && HD == 64 && PER_SIMD == 3 ? 2 : 4; }
// LDS bytes per staged row: the row and 32 bytes of padding (288 or 160: conflict-free fragment reads)
template <int HD> constexpr int wv_pitch() { return 2 * HD + 32; }
// A row's reference is moved where a probability leaves the window, to where the row's largest one is 2^-headroom: with bf16
// operands, whose exponents reach far below, 2^-30 under the 2 that the check looks for (one bit of a word); with fp16 1
// under 2^8.
template <bool F16> constexpr float kWvHeadroom = F16 ? 0.f : 30.f;
constexpr float kNoReference = 3e38f;   // any score leaves the window; a masked one (-inf) stays a probability of zero
// piece u of a tile's line -> its row, by multiplication
template <int HD> constexpr unsigned wv_magic() { return 65536u / (wv_pitch<HD>() / 16) + 1; }
template <int HD> constexpr bool wv_piece_division_ok() {
  for (unsigned u = 0; u < (unsigned)(kWvTile * wv_pitch<HD>() / 16); ++u)
    if (((u * wv_magic<HD>()) >> 16) != u / (wv_pitch<HD>() / 16)) return false;
  return true;
}
static_assert(wv_piece_division_ok<128>() && wv_piece_division_ok<64>(), "piece -> (row, column)");

template <int HD, bool FP8, bool SPLIT, bool F16, int WAVES, int PER_SIMD>
__global__ __launch_bounds__(64 * WAVES, PER_SIMD) void paged_prefill_woven_kernel(PrefillParams p) {
  constexpr int KS = HD / 32, DV = HD / 16, NQ = 2, THREADS = 64 * WAVES;
  constexpr bool FACTOR = FP8 && HD == 128;   // the value scales' mantissas go into the probabilities (see above)
  constexpr int PITCH = wv_pitch<HD>(), PIECES = PITCH / 16, LOADS = kWvTile * PIECES / 64, BUF = LOADS * 1024;
  constexpr int NKF = 2 * KS, NVF = DV;  // key and value fragments of a 32-key slot
  constexpr int ESZ = FP8 ? 1 : 2;       // bytes per cache element
  static_assert(HD == 128 || HD == 64, "head widths");
  static_assert(wv_ring<HD, FP8, PER_SIMD>() - 1 <= NKF && (NKF + NVF) % wv_ring<HD, FP8, PER_SIMD>() == 0, "next slot's key fragments are requested after the tile's barrier");
  // Key tile t lives in Ks[t & 1], value tile t in Vs[t & 1], whose halves are filled one barrier apart (see `iteration`).
  constexpr int HALF = BUF / 2;  // 32 rows of a tile
  __shared__ __attribute__((aligned(16))) uint8_t Ks[2][BUF];
  __shared__ __attribute__((aligned(16))) uint8_t Vs[2][BUF];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m16 = lane & 15, g = lane >> 4;
  const int HV = p.Hkv * p.parts;  // workgroups along the heads
  const HeadSlice hs = head_slice(p, blockIdx.x % HV);
  const int h = hs.h, G = hs.G, g_magic = hs.g_magic, hq0 = hs.hq0;
  const int rank = blockIdx.x / HV;
  const int BQ = ((16 * NQ) * p.g_magic) >> 16;  // query tokens per wavefront (the widest head slice's count)
  const int SBQ = WAVES * BQ;

  // rows beyond the last request (token padding of the batch) are defined as zeros
  if (rank == 0 && (!SPLIT || blockIdx.y == 0)) {
    const int tq = p.cu_q[p.R];
    const int per_row = G * HD;
    for (int64_t i = (int64_t)tid * 8; i < (int64_t)(p.T - tq) * per_row; i += THREADS * 8) {
      const int row = (int)(i / per_row), e = (int)(i - (int64_t)row * per_row);
      st16(p.out + (int64_t)(tq + row) * p.o_st + (int64_t)(hq0 + e / HD) * p.o_sh + (e % HD), make_uint4(0, 0, 0, 0));
    }
  }

  QueryBlock qb;
  if (!find_query_block(p, SBQ, rank, (int)(gridDim.x / HV), &qb)) return;  // workgroup-uniform
  const int r = qb.r, q_begin = qb.q_begin, Lq = qb.Lq, Lk = qb.Lk, q0_wg = qb.q0;
  const int shift = Lk - Lq;
  const int last = Lk - 1;
  const int kend_wg = min(Lk, shift + min(q0_wg + SBQ, Lq));
  const int ntl_all = (kend_wg + kWvTile - 1) / kWvTile;  // staged tiles the rows of this workgroup can see
  const int n_split = SPLIT ? (int)gridDim.y : 1, split = SPLIT ? (int)blockIdx.y : 0;
  // (workgroup-uniform values the tile loop's bookkeeping is built from: held in scalar registers)
  const int tb = __builtin_amdgcn_readfirstlane(SPLIT ? (int)((int64_t)ntl_all * split / n_split) : 0);
  const int te = __builtin_amdgcn_readfirstlane(SPLIT ? (int)((int64_t)ntl_all * (split + 1) / n_split) : ntl_all);
  const int ntl = te - tb;  // this workgroup walks tiles [tb, te)

  const int q0 = q0_wg + wave * BQ;
  const int nq = max(0, min(BQ, Lq - q0));
  const int full_until = shift + q0;  // keys up to here are visible to every valid row of the wavefront

  uint4 qf[NQ][KS];
  int qpos[NQ];
#pragma unroll
  for (int nt = 0; nt < NQ; ++nt) {
    const int n = 16 * nt + m16;
    const int qi = (n * g_magic) >> 16, u = n - qi * G;  // n / G, n % G
    const bool valid = qi < nq;
    qpos[nt] = valid ? shift + q0 + qi : last;
    const uint16_t* qrow = p.q + (int64_t)(q_begin + q0 + qi) * p.q_st + (int64_t)h * p.q_gst + (int64_t)(hq0 - h * p.G + u) * p.q_sh;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk)
      qf[nt][kk] = valid ? ld16(qrow + 32 * kk + 8 * g) : make_uint4(0, 0, 0, 0);
  }
  // Queries straight from the QKV projection: head norm and rotation in registers, with the roundings of the separate
  // launch.  A row's values lie in four lanes (g), the partner of a half-split pair KS / 2 fragments away in the same
  // lane.  What that needs is requested here, together with the queries; the arithmetic (some 900 instructions, three
  // microseconds of a workgroup's tens) runs while the first tiles are on their way.
  const bool raw = p.norm != MI_NORM_NONE || p.angles;
  uint4 cw[NQ][KS], sw[NQ][KS], qw[KS];
  if (raw) {
#pragma unroll
    for (int kk = 0; kk < KS; ++kk)
      qw[kk] = p.norm == MI_NORM_RMS && p.q_w ? ld16(p.q_w + 32 * kk + 8 * g)
                                              : make_uint4(ones2<F16>(), ones2<F16>(), ones2<F16>(), ones2<F16>());
    if (p.angles) {
#pragma unroll
      for (int nt = 0; nt < NQ; ++nt) {
        const int qi = ((16 * nt + m16) * g_magic) >> 16;
        const uint16_t* cs = p.angles + (int64_t)(qi < nq ? q_begin + q0 + qi : q_begin) * (2 * HD) + 8 * g;
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
          cw[nt][kk] = ld16(cs + 32 * kk);
          sw[nt][kk] = ld16(cs + HD + 32 * kk);
        }
      }
    }
  }
  auto norm_and_rotate = [&] {
#pragma unroll
    for (int nt = 0; nt < NQ; ++nt) {
      const bool valid = (((16 * nt + m16) * g_magic) >> 16) < nq;
      uint32_t y[KS][4];   // the row's values, two to a word
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) {
        y[kk][0] = qf[nt][kk].x; y[kk][1] = qf[nt][kk].y; y[kk][2] = qf[nt][kk].z; y[kk][3] = qf[nt][kk].w;
      }
      if (p.norm != MI_NORM_NONE) {
        float ss = 0.f;
#pragma unroll
        for (int kk = 0; kk < KS; ++kk)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float lo = lo_to_f32<F16>(y[kk][i]), hi = hi_to_f32<F16>(y[kk][i]);
            ss += lo * lo;
            ss += hi * hi;
          }
        ss += xor16(ss);
        ss += xor32(ss);
        const float rstd = rsqrtf(ss * (1.f / HD) + p.eps);
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
          const uint32_t w4[4] = {qw[kk].x, qw[kk].y, qw[kk].z, qw[kk].w};
#pragma unroll
          for (int i = 0; i < 4; ++i)
            y[kk][i] = pack2<F16>(lo_to_f32<F16>(y[kk][i]) * rstd * lo_to_f32<F16>(w4[i]),
                                  hi_to_f32<F16>(y[kk][i]) * rstd * hi_to_f32<F16>(w4[i]));
        }
      }
      // (fp16 in packed arithmetic, which rounds as the conversions of the 32-bit form do: a product of two fp16 is exact in
      // fp32, and a sum rounded to fp32 rounds on to fp16 as the exact one would; 3 instructions for two values, not 12)
      auto rotated_pair = [](uint32_t x, uint32_t partner, uint32_t c, uint32_t sn) -> uint32_t {
        if constexpr (F16) {
#pragma clang fp contract(off)
          const f16x2_t a = __builtin_bit_cast(f16x2_t, x) * __builtin_bit_cast(f16x2_t, c);
          const f16x2_t b = __builtin_bit_cast(f16x2_t, partner) * __builtin_bit_cast(f16x2_t, sn);
          return __builtin_bit_cast(uint32_t, a + b);
        } else {
          const uint32_t a = pack2<F16>(lo_to_f32<F16>(x) * lo_to_f32<F16>(c), hi_to_f32<F16>(x) * hi_to_f32<F16>(c));
          const uint32_t b = pack2<F16>(lo_to_f32<F16>(partner) * lo_to_f32<F16>(sn), hi_to_f32<F16>(partner) * hi_to_f32<F16>(sn));
          return pack2<F16>(lo_to_f32<F16>(a) + lo_to_f32<F16>(b), hi_to_f32<F16>(a) + hi_to_f32<F16>(b));
        }
      };
      auto rotated = [&](auto Ic) {
        constexpr bool INTERLEAVED = decltype(Ic)::value;
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
          const uint32_t c4[4] = {cw[nt][kk].x, cw[nt][kk].y, cw[nt][kk].z, cw[nt][kk].w};
          const uint32_t s4[4] = {sw[nt][kk].x, sw[nt][kk].y, sw[nt][kk].z, sw[nt][kk].w};
          uint32_t o4[4];
#pragma unroll
          for (int i = 0; i < 4; ++i)
            o4[i] = rotated_pair(y[kk][i], INTERLEAVED ? __builtin_amdgcn_alignbit(y[kk][i], y[kk][i], 16) : y[kk ^ (KS / 2)][i],
                                 c4[i], s4[i]);
          qf[nt][kk] = valid ? make_uint4(o4[0], o4[1], o4[2], o4[3]) : make_uint4(0, 0, 0, 0);
        }
      };
      if (!p.angles) {
#pragma unroll
        for (int kk = 0; kk < KS; ++kk)
          qf[nt][kk] = valid ? make_uint4(y[kk][0], y[kk][1], y[kk][2], y[kk][3]) : make_uint4(0, 0, 0, 0);
      } else if (p.interleaved) {
        rotated(std::true_type{});
      } else {
        rotated(std::false_type{});
      }
    }
  };

  float neg_run[NQ];  // the reference: a probability is 2^(score * scale + neg_run); kNoReference until a row has one
  f32x4_t acc[NQ][DV], accl[NQ];
  float row_sum[NQ];  // FACTOR only
#pragma unroll
  for (int nt = 0; nt < NQ; ++nt) {
    neg_run[nt] = kNoReference;
    row_sum[nt] = 0.f;
    accl[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < DV; ++e) acc[nt][e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  if (ntl > 0) {
#define MI_SB() __builtin_amdgcn_sched_barrier(0)
    auto uniform64 = [](uint64_t x) {
      return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(x >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((int)x);
    };
    // (48-bit addresses: what a descriptor's second word holds above them are its stride and swizzle fields)
    const uint64_t kbase = uniform64((uint64_t)(uintptr_t)(p.kc + (int64_t)h * p.kv_sh * ESZ)) & 0xffffffffffffull;
    const uint64_t vbase = uniform64((uint64_t)(uintptr_t)(p.vc + (int64_t)h * p.kv_sh * ESZ)) & 0xffffffffffffull;
    const int last_key = __builtin_amdgcn_readfirstlane(last);
    const int64_t chunk_bytes = p.kv_sc * ESZ;
    const int tok_bytes = p.kv_st * ESZ;
    const int tiles_per_chunk = p.chunk / kWvTile;
    const int tile_bytes = kWvTile * tok_bytes;
    const int32_t* bt_row = p.bt + (int64_t)r * p.bt_stride;
    const uint32_t ks_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)&Ks[0][0];
    const uint32_t vs_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)&Vs[0][0];

    // ---- 16-bit cache: this wavefront's direct loads of an iteration: a key tile's line, then the first half of a value
    // tile's and the second half of the value tile's before it -------------------------------------------------------
    // Load k of the 2 LOADS belongs to wavefront k % WAVES; with 36 loads over 8 wavefronts the fifth load of wavefronts 4-7
    // repeats their fourth, so that every wavefront issues as many.  Where load i of a wavefront is of one kind for some
    // wavefronts and of the next for the others, the wavefront's number decides.
    static_assert(LOADS % 2 == 0, "half a tile is whole loads");
    constexpr int NL = (2 * LOADS + WAVES - 1) / WAVES;
    auto load_number = [&](int i, int w) { return w + WAVES * i < 2 * LOADS ? w + WAVES * i : w + WAVES * i - WAVES; };
    // wavefronts (from 0) whose load i lies below `end`: all, none, or some
    auto below = [&](int i, int end) {
      if (load_number(i, WAVES - 1) < end && load_number(i, 0) < end) return true;
      if (WAVES * i >= end + (WAVES * i + WAVES > 2 * LOADS ? WAVES : 0)) return false;
      return load_number(i, wave) < end;
    };
    uint32_t ld_off[NL];  // per lane: where its piece of the load comes from, relative to the tile's first row
    uint32_t ld_dst[NL];  // scalar: LDS offset of the load's 1 KiB inside its tile buffer
    if constexpr (!FP8) {
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const int k = load_number(i, wave);
        const bool is_key = k < LOADS;
        const int kp = is_key ? k : k - LOADS;
        ld_dst[i] = (uint32_t)__builtin_amdgcn_readfirstlane(1024 * kp);
        const uint32_t u = 64u * (uint32_t)kp + (uint32_t)lane;
        const uint32_t prow = (u * wv_magic<HD>()) >> 16, pcol = u - (uint32_t)PIECES * prow;
        ld_off[i] = prow * (uint32_t)tok_bytes + 16u * min(pcol, (uint32_t)(PIECES - 3));
      }
    }
    // ---- fp8 cache: a thread fetches 8 bytes (8 elements) of NP8 rows of a tile into registers, one tile ahead, and
    // stores them converted.  Keys are converted exactly (e4m3 is a subset of both 16-bit types) and their scale goes
    // into the softmax scale of their tile; values are multiplied by their scale and rounded.
    constexpr int PPR8 = HD / 8, RPP8 = THREADS / PPR8, NP8 = kWvTile / RPP8;
    static_assert(NP8 * RPP8 == kWvTile && NP8 <= NKF && NP8 <= NVF, "one row per fragment position");
    uint2 kraw[NP8], vraw[NP8];
    const uint32_t f_row0 = (uint32_t)(tid / PPR8) * (uint32_t)tok_bytes + 8u * (uint32_t)(tid % PPR8),
                   f_step = (uint32_t)RPP8 * (uint32_t)tok_bytes;
    const int f_lds = (tid / PPR8) * PITCH + 16 * (tid % PPR8);
    // (through a descriptor of the tile's rows, as the direct loads: rows past the request's last key arrive as zeros)
    auto fetch_fp8 = [&](uint64_t base, int64_t off, uint32_t nrec, uint2 (&reg)[NP8]) {
      const auto rs = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(base + (uint64_t)off), 0, (int)nrec, 0x00020000);
#pragma unroll
      for (int i = 0; i < NP8; ++i)
        reg[i] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rs, (int)(f_row0 + (uint32_t)i * f_step), 0, 0));
    };
    auto store_k_fp8 = [&](uint8_t* buf, int i) {
      const uint2 lo = fp8x4_to_16x4<F16>(kraw[i].x), hi = fp8x4_to_16x4<F16>(kraw[i].y);
      *reinterpret_cast<uint4*>(buf + f_lds + i * RPP8 * PITCH) = make_uint4(lo.x, lo.y, hi.x, hi.y);
    };
    // A value scale as sign, power of two and what is left, its factor, which goes into its tile's probabilities (the exponent) and
    // out of their sum: from 1 to 2, or, where bytes times the power of two round in fp16 (subnormal numbers, below 2^-15), from
    // 1/2 to 1, so that this error is no larger than that of value times scale.  A scale of zero counts as 2^-126; NaN and
    // infinite ones are in the factor, and so in all results over the tile.
    auto scale_bits = [](float vscale) { return max(__float_as_uint(vscale) & 0x7fffffffu, 0x00800000u); };
    auto factor_below_one = [](uint32_t bits) { return F16 && bits < (uint32_t)(127 - 15) << 23; };
    auto value_factor = [&](float vscale) {
      const uint32_t bits = scale_bits(vscale);
      if (bits >= 0x7f800000u) return __uint_as_float(0x7fc00000u);
      return __uint_as_float((bits & 0x007fffffu) | (factor_below_one(bits) ? 0x3f000000u : 0x3f800000u));
    };
    auto value_pow2 = [&](float vscale) {
      const uint32_t bits = scale_bits(vscale);
      return __uint_as_float((bits & 0x7f800000u) + (factor_below_one(bits) ? 0x00800000u : 0u));
    };
    // the sign goes to the fetched bytes, in a branch of its own: as an operation of every store it takes 1.6 % of prompts (six of
    // 129-4 097 tokens 433.6 -> 440.6 us)
    auto negate_values_fp8 = [&](int32_t sign) {
      if (__builtin_expect(sign >= 0, 1)) return;
#pragma unroll
      for (int i = 0; i < NP8; ++i) vraw[i] = make_uint2(vraw[i].x ^ 0x80808080u, vraw[i].y ^ 0x80808080u);
    };
    auto store_v_fp8 = [&](uint8_t* buf, int i, float vscale) {   // (FACTOR: their scale's value_pow2)
      if constexpr (!FACTOR) {
        const f32x2_t a = fp8x2_lo_to_f32(vraw[i].x), b = fp8x2_hi_to_f32(vraw[i].x);
        const f32x2_t c = fp8x2_lo_to_f32(vraw[i].y), d = fp8x2_hi_to_f32(vraw[i].y);
        *reinterpret_cast<uint4*>(buf + f_lds + i * RPP8 * PITCH) =
            make_uint4(pack2<F16>(a.x * vscale, a.y * vscale), pack2<F16>(b.x * vscale, b.y * vscale),
                       pack2<F16>(c.x * vscale, c.y * vscale), pack2<F16>(d.x * vscale, d.y * vscale));
        return;
      }
      const uint2 lo = fp8x4_to_16x4<F16>(vraw[i].x, vscale), hi = fp8x4_to_16x4<F16>(vraw[i].y, vscale);
      *reinterpret_cast<uint4*>(buf + f_lds + i * RPP8 * PITCH) = make_uint4(lo.x, lo.y, hi.x, hi.y);
    };
    // descriptor of a tile: its rows up to the request's last key (reads beyond return zeros)
    auto tile_rsrc = [&](uint64_t base, int64_t off, uint32_t nrec) {
      const uint64_t a = base + (uint64_t)off;
      u32x4_t rs;
      rs.x = (uint32_t)a;
      rs.y = (uint32_t)(a >> 32);
      rs.z = nrec;
      rs.w = 0x00020000u;
      return rs;
    };
    auto issue_load = [&](int i, const u32x4_t& rs_k, const u32x4_t& rs_v0, const u32x4_t& rs_v1, uint32_t kdst, uint32_t v0dst,
                          uint32_t v1dst) {
      const bool is_key = below(i, LOADS), first_half = below(i, LOADS + LOADS / 2);
      const u32x4_t rs = is_key ? rs_k : first_half ? rs_v0 : rs_v1;
      const uint32_t m0 = (is_key ? kdst : first_half ? v0dst : v1dst) + ld_dst[i];
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(m0), "v"(ld_off[i]), "s"(rs)
                   : "memory", "m0");
    };
    // the tile cursor: all members wave-uniform; it sticks to the workgroup's last tile
    struct Cursor { int tile, ci, tin; };
    auto cursor_at = [&](int t) {
      Cursor c;
      c.tile = __builtin_amdgcn_readfirstlane(min(t, te - 1));
      c.ci = __builtin_amdgcn_readfirstlane(c.tile / tiles_per_chunk);
      c.tin = c.tile - c.ci * tiles_per_chunk;
      return c;
    };
    auto cursor_next = [&](Cursor& c) {
      const bool adv = c.tile + 1 < te;
      const bool wrap = adv && (c.tin + 1 == tiles_per_chunk);
      c.tile += adv ? 1 : 0;
      c.tin = wrap ? 0 : c.tin + (adv ? 1 : 0);
      c.ci += wrap ? 1 : 0;
    };
    auto tile_off = [&](const Cursor& c, int pc) { return (int64_t)pc * chunk_bytes + (int64_t)c.tin * tile_bytes; };
    auto tile_nrec = [&](const Cursor& c) { return (uint32_t)(min(last_key - c.tile * kWvTile, kWvTile - 1) + 1) * (uint32_t)tok_bytes; };
    // block-table entries by scalar loads the compiler does not see (a vector load in the tile loop would make it
    // wait on the vector-memory counter, i.e. for the direct loads in flight)
    auto bt_request = [&](int ci) {
      const int byte_off = 4 * ci;
      int pc;
      asm volatile("s_load_dword %0, %1, %2" : "=s"(pc) : "s"(bt_row), "s"(byte_off) : "memory");
      return pc;
    };
    auto bt_arrived = [&](int& pc) { asm volatile("s_waitcnt lgkmcnt(0)" : "+s"(pc)::"memory"); };
    // fp8: a tile's block-table entry, then its two scales, by vector loads (one address for all lanes) that the
    // compiler tracks with the other loads into registers: a value in flight across the loop's edge may be copied there
    int vzero = 0;
    asm volatile("" : "+v"(vzero));
    int pc_v = 0;
    float ks_v = 1.f, vs_v = 1.f;
    auto scales_request = [&](int pc) {
      ks_v = p.k_scale[(int64_t)pc * p.Hkv + h + vzero];
      vs_v = p.v_scale[(int64_t)pc * p.Hkv + h + vzero];
    };
    auto uniform_float = [](float x) { return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x))); };

    // 16-bit: one scale for all scores.  fp8: a tile's own (kept off zero: zero times the -inf of a masked score would be NaN).
    auto tile_scale = [&](float ks) { return FP8 ? fmaxf(ks * p.scale_log2, 1.17549435e-38f) : p.scale_log2; };
    float scale_prev = p.scale_log2, scale_cur = p.scale_log2, scale_next = p.scale_log2, vscale = 1.f;
    float factor_prev = 1.f, factor_cur = 1.f;   // fp8: value_factor of the tiles whose scales are scale_prev and scale_cur
    float factor_next = 1.f;                     // (and of the tile of `vscale`, whose sign is `vsign`'s)
    int32_t vsign = 0;
    auto values_scale = [&](float vs) {          // uniform; vscale: what store_v_fp8 takes
      vscale = FACTOR ? value_pow2(vs) : vs;
      if constexpr (FACTOR) {
        vsign = __float_as_int(vs);
        factor_next = value_factor(vs);
      }
    };
    const uint4 ones = make_uint4(ones2<F16>(), ones2<F16>(), ones2<F16>(), ones2<F16>());
    const f32x4_t zero4 = {0.f, 0.f, 0.f, 0.f};
    // per-lane starts of the fragment reads inside a tile buffer
    const uint8_t* const k_lane = &Ks[0][0] + m16 * PITCH + 16 * g;
    const uint8_t* const v_lane = &Vs[0][0] + (4 * g + (m16 >> 2)) * PITCH + 8 * (m16 & 3);

    // S[x]: scores of the even (x = 0) / odd (x = 1) 32-key steps, P[x]: their probabilities as the B operand
    f32x4_t S[2][NQ][2];
    uint4 P[2][NQ];
    constexpr int RING = wv_ring<HD, FP8, PER_SIMD>(), AHEAD = RING - 1;
    uint4 fr[RING];  // fragments in flight: fragment n of the stream lives in fr[n % RING]
#pragma unroll
    for (int nt = 0; nt < NQ; ++nt) {
      P[0][nt] = P[1][nt] = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
      for (int u = 0; u < 2; ++u) S[0][nt][u] = S[1][nt][u] = f32x4_t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    }

    auto read_k = [&](const uint8_t* ka, int half, int f) {  // key fragment f of a half tile: sub-tile f & 1, columns 32 (f >> 1)
      return *reinterpret_cast<const uint4*>(ka + (32 * half + 16 * (f & 1)) * PITCH + 64 * (f >> 1));
    };
    auto read_v = [&](const uint8_t* va, int half, int e) {  // transposed value fragment: 32 keys x output columns 16 e
      const uint2 a = lds_ld8_tr(va + 32 * half * PITCH + 32 * e), b = lds_ld8_tr(va + (32 * half + 16) * PITCH + 32 * e);
      return make_uint4(a.x, a.y, b.x, b.y);
    };
    // probabilities of two scores (chunk c of a step's 8 per lane): rows nt = c >> 2, sub-tile (c >> 1) & 1, pair c & 1
    auto exp_chunk = [&](const f32x4_t (&Sx)[NQ][2], uint4 (&Px)[NQ], int c, float scale, const float (&neg)[NQ]) {
      const int nt = c >> 2, u = (c >> 1) & 1, q2 = 2 * (c & 1);
      const float p0 = fast_exp2(__builtin_fmaf(Sx[nt][u][q2], scale, neg[nt]));
      const float p1 = fast_exp2(__builtin_fmaf(Sx[nt][u][q2 + 1], scale, neg[nt]));
      const uint32_t w = pack2<F16>(p0, p1);
      const int d = 2 * u + (c & 1);
      if (d == 0) Px[nt].x = w; else if (d == 1) Px[nt].y = w; else if (d == 2) Px[nt].z = w; else Px[nt].w = w;
    };
    // whether one of a step's probabilities has left the window
    auto leaves_window = [&](const uint4 (&Px)[NQ]) -> bool {
      if constexpr (F16) {   // 2^8 or more (or NaN): in both halves at once
        uint32_t t;
        asm("v_pk_maximum3_f16 %0, %1, %2, %3" : "=v"(t) : "v"(Px[0].x), "v"(Px[0].y), "v"(Px[0].z));
        asm("v_pk_maximum3_f16 %0, %0, %1, %2" : "+v"(t) : "v"(Px[0].w), "v"(Px[1].x));
        asm("v_pk_maximum3_f16 %0, %0, %1, %2" : "+v"(t) : "v"(Px[1].y), "v"(Px[1].z));
        asm("v_pk_maximum3_f16 %0, %0, %1, %1" : "+v"(t) : "v"(Px[1].w));
        asm("v_pk_add_u16 %0, %0, %1" : "+v"(t) : "v"(0x24002400u));   // (0x5c00, 256.0, becomes the sign)
        return (t & 0x80008000u) != 0;
      } else {               // 2 or more: the exponent's highest bit
        const uint32_t t = ((Px[0].x | Px[0].y | Px[0].z) | (Px[0].w | Px[1].x | Px[1].y)) | (Px[1].z | Px[1].w);
        return (t & 0x40004000u) != 0;
      }
    };
    // The reference of some row has to move (rare): it goes to the row's largest score of the step, what was summed against the old
    // one is rescaled, and the step's probabilities are made again.
    auto move_reference = [&](const f32x4_t (&Sx)[NQ][2], uint4 (&Px)[NQ], float scale, float factor) {
      float shifted[NQ];
#pragma unroll
      for (int nt = 0; nt < NQ; ++nt) {
        float tm = -INFINITY;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) tm = fmaxf(tm, Sx[nt][u][i]);
        const float neg = fminf(neg_run[nt], __builtin_fmaf(-rowgroup_max(tm), scale, -kWvHeadroom<F16>));
        const float alpha = fast_exp2(neg - neg_run[nt]);
        neg_run[nt] = neg;
        if (__builtin_amdgcn_ballot_w64(alpha != 1.f)) {
#pragma unroll
          for (int e = 0; e < DV; ++e) {
            acc[nt][e][0] *= alpha; acc[nt][e][1] *= alpha; acc[nt][e][2] *= alpha; acc[nt][e][3] *= alpha;
          }
          accl[nt][0] *= alpha; accl[nt][1] *= alpha; accl[nt][2] *= alpha; accl[nt][3] *= alpha;
          if (FACTOR) row_sum[nt] *= alpha;
        }
        shifted[nt] = FACTOR ? neg + fast_log2(factor) : neg;
      }
#pragma unroll
      for (int c = 0; c < 8; ++c) exp_chunk(Sx, Px, c, scale, shifted);
    };

    // ---- one 32-key slot.  H: the half of the key tile whose scores are multiplied (into S[H]); the vector ALU turns
    // S[1-H] into P[1-H]; the value product takes P[H] and half H of the value tile before.  ka / va: this lane's
    // fragment starts in the key tile's and the value tile's buffers, ka_next in the next key tile's.  key0: position
    // of the first key of S[H] (MASK only).  at_barrier (H == 1): runs between the two groups of products, and requests the
    // first value fragments behind its barrier.
    auto slot = [&](auto Hc, auto Mc, const uint8_t* ka, const uint8_t* ka_next, const uint8_t* va, int key0,
                    auto&& at_barrier, auto&& under_scores, auto&& under_values) {
      constexpr int H = decltype(Hc)::value;
      constexpr bool MASK = decltype(Mc)::value;
      f32x4_t (&Sn)[NQ][2] = S[H];
      const f32x4_t (&Sx)[NQ][2] = S[1 - H];
      uint4 (&Px)[NQ] = P[1 - H];
      const uint4 (&Pv)[NQ] = P[H];
      const float scale = FP8 ? (H == 0 ? scale_prev : scale_cur) : p.scale_log2;  // of the scores in Sx
      const float factor = FACTOR ? (H == 0 ? factor_prev : factor_cur) : 1.f;
      float neg[NQ];
#pragma unroll
      for (int nt = 0; nt < NQ; ++nt) neg[nt] = FACTOR ? neg_run[nt] + fast_log2(factor) : neg_run[nt];
      // fragment n of the slot's stream: NKF key fragments, NVF value fragments, then the next slot's first keys
      auto request = [&](int n) {
        if (n < NKF) fr[n % RING] = read_k(ka, H, n);
        else if (n < NKF + NVF) fr[n % RING] = read_v(va, H, n - NKF);
        else fr[n % RING] = H == 0 ? read_k(ka, 1, n - NKF - NVF) : read_k(ka_next, 0, n - NKF - NVF);
      };
      // The probabilities of S[1-H], two scores ("chunk") at a time in three stages -- scale and subtract, exponential,
      // pack -- one stage of three different chunks per position, so that no instruction waits for the one before it:
      // position n holds stage one of chunk n, stage two of chunk n - 1, stage three of chunk n - 2.
      float xs[8][2], ps[8][2];
      auto exp_stages = [&](int n) {
        if (n >= 2 && n < 10) {
          const int c = n - 2, nt = c >> 2, d = 2 * ((c >> 1) & 1) + (c & 1);
          const uint32_t w = pack2<F16>(ps[c][0], ps[c][1]);
          if (d == 0) Px[nt].x = w; else if (d == 1) Px[nt].y = w; else if (d == 2) Px[nt].z = w; else Px[nt].w = w;
        }
        if (n >= 1 && n < 9) {
          ps[n - 1][0] = fast_exp2(xs[n - 1][0]);
          ps[n - 1][1] = fast_exp2(xs[n - 1][1]);
        }
        if (n < 8) {
          const int nt = n >> 2, u = (n >> 1) & 1, q2 = 2 * (n & 1);
          xs[n][0] = __builtin_fmaf(Sx[nt][u][q2], scale, neg[nt]);
          xs[n][1] = __builtin_fmaf(Sx[nt][u][q2 + 1], scale, neg[nt]);
        }
      };
      // scores: sub-tiles alternate, so a product meets its accumulator again four products later
      constexpr int EPP = 8 / NKF;  // positions of the probabilities' stages per key fragment: 1, or 2 at head width 64
#pragma unroll
      for (int n = 0; n < NKF; ++n) {
        if (H == 0 || n + AHEAD < NKF) request(n + AHEAD);   // (the second half of a value tile: behind the barrier)
        MI_SB();
        const int u = n & 1, kk = n >> 1;
        Sn[0][u] = mfma_16x16x32<F16>(fr[n % RING], qf[0][kk], kk ? Sn[0][u] : zero4);
        Sn[1][u] = mfma_16x16x32<F16>(fr[n % RING], qf[1][kk], kk ? Sn[1][u] : zero4);
        MI_SB();
#pragma unroll
        for (int i = 0; i < EPP; ++i) exp_stages(EPP * n + i);
        under_scores(n);
        MI_SB();
      }
      if constexpr (H == 1) {
        at_barrier([&] {
#pragma unroll
          for (int n = 0; n < AHEAD; ++n) request(NKF + n);
          MI_SB();
        });
      }
      // the mask of the scores just multiplied, rows nt
      auto mask_step = [&](int nt) {
        if (!MASK) return;
        const int dpos = qpos[nt] - (key0 + 4 * g);
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i2 = 0; i2 < 4; ++i2)
            if (16 * u + i2 > dpos) Sn[nt][u][i2] = -INFINITY;
      };
      // values; beside them the last probabilities, then the mask of the scores just multiplied
#pragma unroll
      for (int e = 0; e < NVF; ++e) {
        const int n = NKF + e;
        request(n + AHEAD);
        MI_SB();
        acc[0][e] = mfma_16x16x32<F16>(fr[n % RING], Pv[0], acc[0][e]);
        acc[1][e] = mfma_16x16x32<F16>(fr[n % RING], Pv[1], acc[1][e]);
        MI_SB();
        if (HD == 128) {
          if (e < 2) exp_stages(8 + e);
          if (e == 3 || e == 5) mask_step((e - 3) / 2);
        } else {
          if (e == 0) { exp_stages(8); exp_stages(9); }
          if (e == 1 || e == 2) mask_step(e - 1);
        }
        under_values(e);
        MI_SB();
      }
      // (fp8: the sums of one value tile, whose factor comes out of them in end_of_sums)
      accl[0] = mfma_16x16x32<F16>(ones, Pv[0], FACTOR && H == 0 ? zero4 : accl[0]);
      accl[1] = mfma_16x16x32<F16>(ones, Pv[1], FACTOR && H == 0 ? zero4 : accl[1]);
      MI_SB();
      if (__builtin_amdgcn_ballot_w64(leaves_window(Px))) move_reference(Sx, Px, scale, factor);
      MI_SB();
    };

    // ---- prologue: clear the buffer of the value tile "before the first" (its probabilities are zeros, and zero times
    // a stale value must not be NaN; every other buffer is filled whole before it is read), start the first tiles ----
    for (int i = tid * 16; i < BUF; i += THREADS * 16) *reinterpret_cast<uint4*>(&Vs[1][0] + i) = make_uint4(0u, 0u, 0u, 0u);
    Cursor cur = cursor_at(tb + 2);
    int64_t off_first[2];   // tiles tb and tb + 1, started here
    uint32_t nrec_first[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const Cursor c = cursor_at(tb + i);
      const int pc = __builtin_amdgcn_readfirstlane(bt_row[c.ci]);
      off_first[i] = tile_off(c, pc);
      nrec_first[i] = tile_nrec(c);
      if constexpr (FP8) {
        scales_request(pc);
        if (i == 0) {
          scale_prev = scale_cur = tile_scale(uniform_float(ks_v));
          values_scale(uniform_float(vs_v));
          factor_prev = factor_cur = factor_next;
        }
      }
    }
    int pc_next = 0;
    if constexpr (FP8) pc_v = bt_row[cur.ci + vzero];
    else pc_next = __builtin_amdgcn_readfirstlane(bt_row[cur.ci]);
    // (the query fragments count as used here: the compiler then waits for their loads now and not in the tile
    // loop, where a wait on the vector-memory counter would wait for the direct loads in flight as well)
#pragma unroll
    for (int nt = 0; nt < NQ; ++nt)
#pragma unroll
      for (int kk = 0; kk < KS; ++kk)
        asm volatile("" ::"v"(qf[nt][kk].x), "v"(qf[nt][kk].y), "v"(qf[nt][kk].z), "v"(qf[nt][kk].w));
    if (raw) {
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) {
        asm volatile("" ::"v"(qw[kk].x), "v"(qw[kk].y), "v"(qw[kk].z), "v"(qw[kk].w));
#pragma unroll
        for (int nt = 0; nt < NQ; ++nt) {
          asm volatile("" ::"v"(cw[nt][kk].x), "v"(cw[nt][kk].y), "v"(cw[nt][kk].z), "v"(cw[nt][kk].w));
          asm volatile("" ::"v"(sw[nt][kk].x), "v"(sw[nt][kk].y), "v"(sw[nt][kk].z), "v"(sw[nt][kk].w));
        }
      }
    }
    __syncthreads();
    int64_t off_prev, off_prev2 = off_first[0];   // of tiles j+1 and j
    uint32_t nrec_prev, nrec_prev2 = nrec_first[0];
    if constexpr (FP8) {
      fetch_fp8(kbase, off_first[0], nrec_first[0], kraw);
      MI_SB();
      if (raw) norm_and_rotate();
      MI_SB();
#pragma unroll
      for (int i = 0; i < NP8; ++i) store_k_fp8(&Ks[0][0], i);
      fetch_fp8(kbase, off_first[1], nrec_first[1], kraw);  // stored by iteration 0
      fetch_fp8(vbase, off_first[0], nrec_first[0], vraw);
      off_prev = off_first[1];
      nrec_prev = nrec_first[1];
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    } else {
      const u32x4_t rk0 = tile_rsrc(kbase, off_first[0], nrec_first[0]);
#pragma unroll
      for (int i = 0; i < NL; ++i)
        if (below(i, LOADS)) issue_load(i, rk0, rk0, rk0, ks_lds, ks_lds, ks_lds);  // key tile 0 -> Ks[0]
      // key tile 1 -> Ks[1], value tile 0 -> Vs[0], whole
      const u32x4_t rk1 = tile_rsrc(kbase, off_first[1], nrec_first[1]), rv0 = tile_rsrc(vbase, off_first[0], nrec_first[0]);
#pragma unroll
      for (int i = 0; i < NL; ++i) issue_load(i, rk1, rv0, rv0, ks_lds + BUF, vs_lds, vs_lds);
      off_prev = off_first[1];
      nrec_prev = nrec_first[1];
    }
    if constexpr (!FP8) {
      MI_SB();
      if (raw) norm_and_rotate();
      MI_SB();
    }
    // key tile 0 has landed (this wavefront's share): only the loads issued after it may still be on their way
    if constexpr (!FP8) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NL) : "memory");
    }
    __builtin_amdgcn_s_barrier();
    MI_SB();

    const int t_mask = max(0, (full_until + 1) >> 6);              // first tile with a masked score for this wavefront
    const int jm = min(max(t_mask - tb, 0), ntl);                  // iterations [0, jm) need no mask
    int j = 0;
    int even = 0;   // BUF where j is odd
#pragma unroll
    for (int n = 0; n < AHEAD; ++n) fr[n] = read_k(k_lane, 0, n);

    auto end_of_sums = [&](float factor) {
      const float inv = __builtin_amdgcn_rcpf(factor);
#pragma unroll
      for (int nt = 0; nt < NQ; ++nt) row_sum[nt] = __builtin_fmaf(accl[nt][0], inv, row_sum[nt]);
    };
    // Iteration j: scores of key tile j, values of tile j-1.  After its barrier, which follows the last score, every wavefront
    // has left key tile j, the first half of value tile j-1 and the second half of value tile j-2: key tile j+2 and value
    // tiles j+1 (first half) and j (second half) take their places, under the products that follow, for the next barrier.
    auto iteration = [&](auto Mc) {
      const uint8_t* ka = k_lane + even;
      const uint8_t* ka_next = k_lane + (BUF - even);
      const uint8_t* va = v_lane + (BUF - even);
      const int key0 = (tb + j) * kWvTile;
      u32x4_t rs_k, rs_v0, rs_v1;
      const uint32_t kdst = ks_lds + (uint32_t)even, v0dst = vs_lds + (uint32_t)(BUF - even), v1dst = vs_lds + (uint32_t)even;
      // fp8: key tile j+1 and the first half of value tile j, fetched since the last barrier, go into LDS before this one
      uint8_t* const kst = &Ks[0][0] + (BUF - even);
      uint8_t* const vst = &Vs[0][0] + even;
      slot(std::integral_constant<int, 0>{}, Mc, ka, ka_next, va, key0, [](auto) {}, [](int) {},
           [&](int e) {
             if constexpr (FP8) {
               if (e >= NVF - NP8) store_k_fp8(kst, e - (NVF - NP8));
             }
           });
      if constexpr (FACTOR) negate_values_fp8(vsign);
      slot(std::integral_constant<int, 1>{}, Mc, ka, ka_next, va, key0 + 32,
           [&](auto first_values) {
             // this wavefront's share of key tile j+1 and of the value tiles has landed
             if constexpr (FP8) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
             else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
             __builtin_amdgcn_s_barrier();
             first_values();
             if constexpr (FP8) pc_next = __builtin_amdgcn_readfirstlane(pc_v);
             else bt_arrived(pc_next);
             const int64_t off = tile_off(cur, pc_next);
             const uint32_t nrec = tile_nrec(cur);
             if constexpr (FP8) {
               scale_next = tile_scale(uniform_float(ks_v));  // (of tile j+1)
               const float vscale_last = vscale;
               values_scale(uniform_float(vs_v));
               scales_request(pc_next);
               fetch_fp8(kbase, off, nrec, kraw);
#pragma unroll
               for (int i = NP8 / 2; i < NP8; ++i) store_v_fp8(vst, i, vscale_last);
               fetch_fp8(vbase, off_prev, nrec_prev, vraw);
             } else {
               rs_k = tile_rsrc(kbase, off, nrec);
               rs_v0 = tile_rsrc(vbase, off_prev, nrec_prev);
               rs_v1 = tile_rsrc(vbase, off_prev2, nrec_prev2);
             }
             off_prev2 = off_prev;
             nrec_prev2 = nrec_prev;
             off_prev = off;
             nrec_prev = nrec;
             cursor_next(cur);
             if constexpr (FP8) pc_v = bt_row[cur.ci + vzero];
             else pc_next = bt_request(cur.ci);
           },
           [&](int n) {
             if constexpr (FP8) {
               if (n < NP8 / 2) store_v_fp8(vst, n, vscale);
             }
           },
           [&](int e) {
             if constexpr (!FP8) {
#pragma unroll
               for (int i = e; i < NL; i += NVF) issue_load(i, rs_k, rs_v0, rs_v1, kdst, v0dst, v1dst);
             }
           });
      if constexpr (FP8) {
        if (FACTOR) end_of_sums(factor_prev);   // (the values of tile j-1)
        scale_prev = scale_cur;
        scale_cur = scale_next;
        factor_prev = factor_cur;
        factor_cur = factor_next;
      }
      ++j;
      even = BUF - even;
    };
    for (; j < jm;) iteration(std::false_type{});
    for (; j < ntl;) iteration(std::true_type{});

    // ---- drain: the last two steps' values (tile ntl - 1), the second half when it has landed; S[1] is masked already ----
    {
      const uint8_t* va = v_lane + (BUF - even);
      if (FACTOR) accl[0] = accl[1] = zero4;
      auto values = [&](int half, const uint4 (&Pv)[NQ]) {
#pragma unroll
        for (int e = 0; e < DV; ++e) {
          const uint4 a = read_v(va, half, e);
          acc[0][e] = mfma_16x16x32<F16>(a, Pv[0], acc[0][e]);
          acc[1][e] = mfma_16x16x32<F16>(a, Pv[1], acc[1][e]);
        }
        accl[0] = mfma_16x16x32<F16>(ones, Pv[0], accl[0]);
        accl[1] = mfma_16x16x32<F16>(ones, Pv[1], accl[1]);
      };
      values(0, P[0]);
      float neg_last[NQ];
#pragma unroll
      for (int nt = 0; nt < NQ; ++nt) neg_last[nt] = FACTOR ? neg_run[nt] + fast_log2(factor_prev) : neg_run[nt];
#pragma unroll
      for (int c = 0; c < 8; ++c) exp_chunk(S[1], P[1], c, FP8 ? scale_prev : p.scale_log2, neg_last);
      if (__builtin_amdgcn_ballot_w64(leaves_window(P[1]))) move_reference(S[1], P[1], FP8 ? scale_prev : p.scale_log2, factor_prev);
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      values(1, P[1]);
      if (FACTOR) end_of_sums(factor_prev);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no direct load may still be on its way into this workgroup's LDS
#undef MI_SB
  }

  // ---- epilogue: acc[nt][e][i] is output element d = 16e + 4g + i of row (nt, m16) --------------
#pragma unroll
  for (int nt = 0; nt < NQ; ++nt) {
    const float l_tot = FACTOR ? row_sum[nt] : accl[nt][0];
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    const int n = 16 * nt + m16;
    const int qi = (n * g_magic) >> 16, u = n - qi * G;  // n / G, n % G
    if (qi < nq) {
      if (!SPLIT) {
        uint16_t* o = p.out + (int64_t)(q_begin + q0 + qi) * p.o_st + (int64_t)(hq0 + u) * p.o_sh + 4 * g;
#pragma unroll
        for (int e = 0; e < DV; ++e)
          st8(o + 16 * e, make_uint2(pack2<F16>(acc[nt][e][0] * inv, acc[nt][e][1] * inv),
                                     pack2<F16>(acc[nt][e][2] * inv, acc[nt][e][3] * inv)));
      } else {  // a range without visible keys leaves zeros and -inf
        const int64_t prow = ((int64_t)split * p.T + (q_begin + q0 + qi)) * p.Hq + (hq0 + u);
        float* o = p.split_o + prow * HD + 4 * g;
#pragma unroll
        for (int e = 0; e < DV; ++e)
          *reinterpret_cast<float4*>(o + 16 * e) =
              make_float4(acc[nt][e][0] * inv, acc[nt][e][1] * inv, acc[nt][e][2] * inv, acc[nt][e][3] * inv);
        if (g == 0) p.split_lse[prow] = l_tot > 0.f ? fast_log2(l_tot) - neg_run[nt] : -INFINITY;
      }
    }
  }
}


void launch_prefill_woven(const PrefillParams& p, dim3 grid, int head_dim, bool fp8, bool f16, int waves, hipStream_t st) {
  const bool split = grid.y > 1;
#define MI_WV_LAUNCH(HD_, FP8_, W_, PS_)                                                                                 \
  do {                                                                                                              \
    const dim3 block(64 * W_);                                                                                      \
    if (split && f16) hipLaunchKernelGGL((paged_prefill_woven_kernel<HD_, FP8_, true, true, W_, PS_>), grid, block, 0, st, p); \
    else if (split) hipLaunchKernelGGL((paged_prefill_woven_kernel<HD_, FP8_, true, false, W_, PS_>), grid, block, 0, st, p); \
    else if (f16) hipLaunchKernelGGL((paged_prefill_woven_kernel<HD_, FP8_, false, true, W_, PS_>), grid, block, 0, st, p); \
    else hipLaunchKernelGGL((paged_prefill_woven_kernel<HD_, FP8_, false, false, W_, PS_>), grid, block, 0, st, p);      \
  } while (0)
  if (head_dim == 64 && fp8 && (int64_t)grid.x * grid.y <= 3 * device_cu_count()) MI_WV_LAUNCH(64, true, 4, 2);
  else if (head_dim == 64 && fp8) MI_WV_LAUNCH(64, true, 4, 3);
  else if (head_dim == 64) MI_WV_LAUNCH(64, false, 4, 3);
  else if (fp8 && waves == 4) MI_WV_LAUNCH(128, true, 4, 2);
  else if (fp8) MI_WV_LAUNCH(128, true, 8, 2);
  else if (waves == 4) MI_WV_LAUNCH(128, false, 4, 2);
  else MI_WV_LAUNCH(128, false, 8, 2);
#undef MI_WV_LAUNCH
}

}  // namespace mi
