// The two projections either side of the attention path, at decode size:  y[T, N] = x[T, K] . W[N, K]^T (+ bias).
//
// Replaces, for steps of at most 256 tokens,
//   mixed_qkv, _ = self.linear_qkv(hidden_states)        (megatron/core/transformer/attention.py:985-992; N = (Hq + 2 Hkv) d)
//   output, bias = self.linear_proj(core_attn_out)       (attention.py:829-845; skip_bias_add: the bias is returned, not added)
// as ColumnParallelLinear / RowParallelLinear compute them at tensor-parallel size 1
// (megatron/core/tensor_parallel/layers.py:946-1010,1225-1290): 16-bit inputs, fp32 accumulation, 16-bit result.
// With a few dozen rows of x the weight matrix is the traffic -- 50 MB for 4096 -> 6144 -- and each of its bytes is
// used once: the kernel is a stream of W from HBM with the products riding along.
//
// Work split: K is cut into slices of at most 512 columns, and the result is the slices' fp32 sums added in slice order,
// part by part -- fixed by (T, N, K) alone, so a call is reproducible bit for bit.  A workgroup takes
// 8 RH rows of W and all of K (or one of up to three parts) for a block of at most 64 tokens, one wavefront per slice:
// each piece of W and of x that a workgroup needs enters the CU exactly once, straight into the registers of the wavefront that multiplies it -- no
// staging shared between wavefronts, no barrier before or between the products, and a ring of loads that stays full
// from the first instruction on.  The slices' sums meet in LDS at the end: one kernel and no partial sums in memory, but
// for calls whose row blocks alone would not fill the chip (linear_plan).
//
// 64 tokens, weights from HBM (GPU time per call, graph replay; before: 128 rows of one slice per workgroup, x staged
// in LDS, partial sums in memory and a second kernel to add them):
//   4096 -> 6144   23.9 -> 19.9 us,  1 token 16.1 -> 12.8,  256 tokens 65 -> 45
//   4096 -> 4096   22.0 -> 16.4 us,  1 token 14.5 -> 10.0,  256 tokens 46 -> 25
//   2048 -> 1280   11.4 ->  6.6 us,  1 token  7.3 ->  4.9,  256 tokens 18 ->  9
// The matrix alone streams in 10.3 us (4096 -> 6144); beside it the CU's miss queue carries x (32 tokens: 4 KB per 6 KB of
// a 48-row tile of W), at 52-60 KB/us: 168 MB into the CUs by counter, each request 680 clocks on its way.
#include "mi_common.h"
#include "mi_capi_internal.h"

namespace mi {

constexpr int kLinTok = 64;      // tokens per workgroup, at most (and in the slice rule)
constexpr int kLinStep = 64;     // columns a wavefront multiplies per step: whole 128-byte lines of 8 rows
constexpr int kLinSlice = 512;   // columns per slice, at most
constexpr int kLinRows = 128;    // (only in the slice rule)
constexpr int kLinParts = 3;     // parts of K with workgroups of their own, at most
constexpr int kLinLds = 160 * 1024;

struct LinearParams {
  const uint16_t* x; int64_t x_st;
  const uint16_t* w; int64_t w_st;
  const uint16_t* bias;
  uint16_t* out; int64_t o_st;
  int32_t T, N, K, kslice, S, waves;  // S slices of kslice columns (a multiple of 32), `waves` of them at a time
  int32_t per_part;                   // slices of a part (S: the only one); part z of the grid takes z per_part onward
  float* part;                        // with several parts their sums, [part][T][N]; else null
};

// RH = 8-row half tiles of W, XH = 8-token half tiles of x, P = steps in flight, NW = wavefronts at most (8: 256 registers
// each, 12: 168, 16: 128).
//
// The products want lane (m16, g) to hold columns 8 g .. + 7 (of 32) of row m16 of W, and the same of token m16 of x.
// Loads in that order are slow wherever they hit: neighbouring lanes ask for different rows, and the vector memory
// pipe takes them at 17 bytes per clock and CU (measured on 512 KB in L2 read by every CU; 54-60 when eight
// neighbouring lanes ask for one 128-byte line).  So lane l loads 16-byte piece l & 7 of row l >> 3, eight rows per
// instruction, and the wavefront turns its own piece of LDS -- written as loaded, read in the products' order, both
// without bank conflicts by the exclusive-or of piece and row.  A wavefront's LDS operations execute in order and no
// other wavefront touches its piece, so there is no barrier and no wait between the two.
template <bool F16, int RH, int XH, int P, int NW>
__global__ __launch_bounds__(64 * NW) void linear_decode_kernel(LinearParams p) {
  constexpr int TT = (XH + 1) / 2, RT = (RH + 1) / 2;
  constexpr int kTurn = (2 * RT + 2 * TT) * 1024;   // bytes of a wavefront's piece of LDS: one step of W and of x
  constexpr int kTile = 1024;                       // a 16 x 16 tile of sums: 16 bytes per lane
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (8 * RH);
  const int t0 = blockIdx.y * (8 * XH);
  const int nt = min(8 * XH, p.T - t0);

  const int lo = lane >> 3, col = 8 * (lane & 7);
  uint8_t* const turn_put = lds + wave * kTurn + lo * 128 + (((lane & 7) ^ lo) << 4);
  const uint8_t* const turn_get = lds + wave * kTurn + m16 * 128;
  const int piece0 = (g ^ (m16 & 7)) << 4, piece1 = ((4 + g) ^ (m16 & 7)) << 4;   // columns 0-31 / 32-63 of the step
  // Rows beyond the last of W repeat its last eight or sixteen, tokens beyond the last repeat it: their results are not stored.
  const uint32_t w_lane = (uint32_t)(lo * p.w_st + col);
  uint32_t x_lane[XH];
#pragma unroll
  for (int i = 0; i < XH; ++i) x_lane[i] = (uint32_t)(min(8 * i + lo, nt - 1) * p.x_st + col);
  const uint16_t* xbase = p.x + (int64_t)t0 * p.x_st;
  auto w_at = [&](int i, int k) {
    const int row = RH % 2 ? min(n0 + 8 * i, p.N - 8) : min(n0 + 16 * (i >> 1), p.N - 16) + 8 * (i & 1);
    return p.w + (int64_t)row * p.w_st + k + w_lane;
  };
  auto x_at = [&](int i, int k) { return xbase + k + x_lane[i]; };

  struct Stage { uint4 w[RH]; uint4 x[XH]; };
  Stage st[P];
  int k0 = 0, k1 = 0, ka = 0;   // columns of the slice at hand; where its first whole step of 64 starts
  auto load = [&](Stage& s, int step) {
    const int k = ka + step * kLinStep;
    if (k + kLinStep <= p.K) {
#pragma unroll
      for (int i = 0; i < RH; ++i) s.w[i] = ld16_stream(w_at(i, k));
#pragma unroll
      for (int i = 0; i < XH; ++i) s.x[i] = ld16(x_at(i, k));
    } else {  // the last 32 columns of a K that is no multiple of 64: zeros beyond them
      const bool live = k + col < p.K;
#pragma unroll
      for (int i = 0; i < RH; ++i) s.w[i] = live ? ld16_stream(w_at(i, k)) : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
      for (int i = 0; i < XH; ++i) s.x[i] = live ? ld16(x_at(i, k)) : make_uint4(0u, 0u, 0u, 0u);
    }
  };
  f32x4_t acc[RT * TT];
  auto multiply = [&](Stage& s, int step) {
    // (a slice of an odd number of 32 columns shares its first or last 64 with its neighbour: each multiplies its half)
    const bool first = ka + step * kLinStep >= k0, second = ka + step * kLinStep + 32 < k1;
#pragma unroll
    for (int i = 0; i < RH; ++i) *reinterpret_cast<uint4*>(turn_put + i * 1024) = s.w[i];
#pragma unroll
    for (int i = 0; i < XH; ++i) *reinterpret_cast<uint4*>(turn_put + (2 * RT + i) * 1024) = s.x[i];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    uint4 wa[RT], wb[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      wa[i] = *reinterpret_cast<const uint4*>(turn_get + i * 2048 + piece0);
      wb[i] = *reinterpret_cast<const uint4*>(turn_get + i * 2048 + piece1);
    }
#pragma unroll
    for (int j = 0; j < TT; ++j) {   // (an odd XH or RH leaves its last half tile as it was: values that are not stored)
      const uint4 xa = *reinterpret_cast<const uint4*>(turn_get + (RT + j) * 2048 + piece0);
      const uint4 xb = *reinterpret_cast<const uint4*>(turn_get + (RT + j) * 2048 + piece1);
      if (first) {
#pragma unroll
        for (int i = 0; i < RT; ++i) acc[i * TT + j] = mfma_16x16x32<F16>(wa[i], xa, acc[i * TT + j]);
      }
      if (second) {
#pragma unroll
        for (int i = 0; i < RT; ++i) acc[i * TT + j] = mfma_16x16x32<F16>(wb[i], xb, acc[i * TT + j]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  auto tile_at = [&](int slot, int tile) { return reinterpret_cast<f32x4_t*>(lds + (slot * RT * TT + tile) * kTile + 16 * lane); };
  static_assert(RT * TT * kTile <= kTurn, "the sums of a wavefront lie over its piece");
  const int base = blockIdx.z * p.per_part, mine = min(p.per_part, p.S - base);
  auto before = [&](int tile) { return reinterpret_cast<f32x4_t*>(lds + p.waves * kTurn + tile * kTile + 16 * lane); };
  for (int s0 = 0; s0 < mine; s0 += p.waves) {   // (one round unless there are more than 16 slices)
    if (s0 > 0) __syncthreads();                 // the sums have been read
    const int slice = base + s0 + wave;
    k0 = slice * p.kslice;
    k1 = s0 + wave < mine ? min(k0 + p.kslice, p.K) : k0;
    ka = k0 & ~(kLinStep - 1);
    const int steps = k1 > k0 ? (k1 - ka + kLinStep - 1) / kLinStep : 0;
#pragma unroll
    for (int i = 0; i < RT * TT; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < P; ++u)
      if (u < steps) load(st[u], u);
    for (int s = 0; s < steps; s += P) {
#pragma unroll
      for (int u = 0; u < P; ++u) {
        if (s + u < steps) {
          multiply(st[u], s + u);
          if (s + u + P < steps) load(st[u], s + u + P);
        }
      }
    }
    // ---- acc[i * TT + j][e] = y[token 16 j + m16][row n0 + 16 i + 4 g + e] of this slice ----
    __syncthreads();  // (everyone has read its last step)
#pragma unroll
    for (int i = 0; i < RT * TT; ++i) *tile_at(wave, i) = acc[i];
    __syncthreads();
    const int live = min(p.waves, mine - s0);
    const bool last = s0 + p.waves >= mine;
    for (int tile = wave; tile < RT * TT; tile += p.waves) {
      f32x4_t sum = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (s0 > 0) sum = *before(tile);
      for (int w = 0; w < live; ++w) {
        const f32x4_t v = *tile_at(w, tile);
        sum[0] += v[0]; sum[1] += v[1]; sum[2] += v[2]; sum[3] += v[3];
      }
      if (!last) {
        *before(tile) = sum;
        continue;
      }
      const int n = n0 + 16 * (tile / TT) + 4 * g, t = 16 * (tile % TT) + m16;
      if (n >= (RH % 2 ? min(n0 + 8 * RH, p.N) : p.N) || t >= nt) continue;
      if (p.part) {
        *reinterpret_cast<f32x4_t*>(p.part + ((int64_t)blockIdx.z * p.T + t0 + t) * p.N + n) = sum;
        continue;
      }
      if (p.bias) {
        const uint2 bw = ld8(p.bias + n);
        sum[0] += lo_to_f32<F16>(bw.x); sum[1] += hi_to_f32<F16>(bw.x); sum[2] += lo_to_f32<F16>(bw.y); sum[3] += hi_to_f32<F16>(bw.y);
      }
      st8(p.out + (int64_t)(t0 + t) * p.o_st + n, make_uint2(pack2<F16>(sum[0], sum[1]), pack2<F16>(sum[2], sum[3])));
    }
  }
}

// The parts' sums added in order, with the bias: a thread takes four values, and its four results lie `quad` values past
// those of the thread before (8, with p.out the workspace: over the first part's sums that it has read).
template <bool F16>
__global__ __launch_bounds__(256) void linear_parts_kernel(LinearParams p, int parts, int quad) {
  const int quads = p.N / 4, i = blockIdx.x * 256 + threadIdx.x;
  if (i >= p.T * quads) return;
  const int t = i / quads, n = 4 * (i - t * quads);
  const float* from = p.part + (int64_t)t * p.N + n;
  f32x4_t sum = *reinterpret_cast<const f32x4_t*>(from);
  for (int z = 1; z < parts; ++z) {
    const f32x4_t v = *reinterpret_cast<const f32x4_t*>(from + (int64_t)z * p.T * p.N);
    sum[0] += v[0]; sum[1] += v[1]; sum[2] += v[2]; sum[3] += v[3];
  }
  if (p.bias) {
    const uint2 bw = ld8(p.bias + n);
    sum[0] += lo_to_f32<F16>(bw.x); sum[1] += hi_to_f32<F16>(bw.x); sum[2] += lo_to_f32<F16>(bw.y); sum[3] += hi_to_f32<F16>(bw.y);
  }
  st8(p.out + t * p.o_st + (i - t * quads) * quad, make_uint2(pack2<F16>(sum[0], sum[1]), pack2<F16>(sum[2], sum[3])));
}

// `out` over one of the inputs: workgroups store their rows while others still load, so the results go to the workspace
// (four of them every `quad` values) and this launch puts them in place.
__global__ __launch_bounds__(256) void linear_place_kernel(const uint16_t* from, int quad, uint16_t* out, int64_t o_st, int T, int N) {
  const int quads = N / 4, i = blockIdx.x * 256 + threadIdx.x;   // (T N / 4 fits: T <= 256)
  if (i >= T * quads) return;
  const int t = i / quads, n = 4 * (i - t * quads);
  st8(out + t * o_st + n, ld8(from + (int64_t)i * quad));
}

}  // namespace mi

using namespace mi;

// Whether `rows_a` rows of `width_a` values every `st_a` and the same of b share memory.  Columns of one buffer's rows
// (equal strides) that lie side by side do not; other layouts are taken by their first and last value.
static bool linear_overlap(const void* a, int64_t rows_a, int64_t width_a, int64_t st_a, const void* b, int64_t rows_b,
                           int64_t width_b, int64_t st_b) {
  const intptr_t a0 = (intptr_t)a / 2, b0 = (intptr_t)b / 2;
  if (a0 + (rows_a - 1) * st_a + width_a <= b0 || b0 + (rows_b - 1) * st_b + width_b <= a0) return false;
  if (st_a != st_b || rows_a == 1 || rows_b == 1) return true;
  const intptr_t at = ((b0 - a0) % st_a + st_a) % st_a;   // b's first column, counted from a's
  return at < width_a || at + width_b > st_a;
}

// The slices of K, and with them the order of summation: at least one per 512 columns, more where 128-row blocks of W
// times 64-token blocks are few (a slice keeps at least 128 columns), a multiple of 32 columns each.
static void linear_slices(int T, int N, int K, int* n_slices, int* kslice) {
  const int row_blocks = (N + kLinRows - 1) / kLinRows, tok_blocks = (T + kLinTok - 1) / kLinTok;
  int s = (K + kLinSlice - 1) / kLinSlice;
  const int want = (384 + row_blocks * tok_blocks - 1) / (row_blocks * tok_blocks);
  if (want > s) s = want;
  if (s > K / 128) s = K / 128 > 0 ? K / 128 : 1;
  int len = ((K + s - 1) / s + 31) & ~31;
  if (len > kLinSlice) len = kLinSlice;
  *kslice = len;
  *n_slices = (K + len - 1) / len;
}

// LDS of a workgroup: a step of every wavefront (at the end its sums, over it) and, where the slices come in rounds, the
// sums of the rounds before.
static int linear_lds(int rt, int half_tiles, int waves, int slices) {
  const int tt = (half_tiles + 1) / 2;
  return (waves * (2 * rt + 2 * tt) + (slices > waves ? rt * tt : 0)) * 1024;
}

// (the instances there are: eight wavefronts have the registers for four row tiles, sixteen for one or two; 24 rows for few
// tokens)
static bool linear_instance(int rh, int xh, int waves, int slices) {
  const int most = waves > 12 ? (xh <= 2 ? 4 : 2) : waves > 8 || xh <= 2 ? 4 : xh <= 4 ? 6 : 8;
  return rh <= most && (rh != 3 || xh <= 4) && linear_lds((rh + 1) / 2, xh, waves, slices) <= kLinLds;
}
// How a call is spread: tokens per workgroup (8 half_tiles), rows (8 row_halves), slices at a time (waves), and the parts
// that the slices are cut into, with workgroups of their own and a second launch that adds their sums.
struct LinearPlan {
  int half_tiles, row_halves, waves, parts;
};
// The plan with the least estimated time.  A workgroup fills a CU (its registers or its LDS), so the launch runs in rounds
// of 256 workgroups; a round costs 4.6 us, 3 us more for every further round of slices, and the bytes it brings into a CU,
// whose miss queue carries 52 KB/us of W (from HBM) or 60 KB/us of x (from L2); several parts cost 5 us and their sums
// written and read.  Fitted to ten shapes from 1280 x 2048 to 10240 x 2048 at 1 .. 256 tokens: within 16 % of the fastest
// plan everywhere, within 4 % for most.  More rows per workgroup read x less often, fewer fill the chip.  Where W has
// fewer row blocks than the chip has CUs, or a few more, smaller token blocks (W once more for each, from the last-level
// cache) or parts fill it; 64 tokens, against 64 in a workgroup and one part:
//   2048 x 8192 28.3 -> 19.1 us,  5120 x 8192 34.7 -> 26.3,  1280 x 5120 22.6 -> 12.7,  2048 x 4096 15.4 -> 12.5
// With few tokens 32 rows leave a quarter of the CUs without any (6144 rows: 192 workgroups) and 16 need a second round:
// 24 fill the chip.  Without them -> with them (weights from HBM):  6144 x 4096, 16 tokens 12.9 -> 12.1 us, 24 tokens 15.1 ->
// 13.8 (1 to 8 tokens 12.1-12.5 either way);  5120 x 5120, one token 14.5 -> 13.1, 16 tokens 15.7 -> 14.1;  10240 x 5120, one
// token 26.3 -> 23.5;  5120 x 8192, one token 18.7 -> 17.3.
// Where a few more rows than the chip takes at once would need a second round, a workgroup with room for more tokens than
// there are has 48 or 64 rows, and one round does: 10240 x 2048, one token 16.4 -> 12.3 us;  8448 x 4096 19.6 -> 16.0;
// 10240 x 4096, 16 tokens 20.5 -> 18.3;  16384 x 4096, 24 tokens 32.2 -> 28.3.  (Not with up to four wavefronts, two such
// workgroups share a CU: 16384 x 2048, one token 14.3 -> 16.7.)
static LinearPlan linear_plan(int T, int N, int K, int slices) {
  LinearPlan best{};
  float least = 0.f;
  int undivided = 0;  // workgroups of the best plan of one part
  const int row_halves = N / 8;
  for (int z = 1; z <= kLinParts; ++z) {
    const int per = (slices + z - 1) / z, fewest = (per + 15) / 16;
    // (as many parts as have slices; none where the chip is filled more than twice as it is: 10240 x 8192, 256 tokens,
    // two parts 153 us against 149)
    if ((z - 1) * per >= slices || undivided > 512) break;
    const float column = (float)K * 2.f / (float)z, merge = z > 1 ? 5.f + (float)z * (float)T * (float)N * (8.f / 4.5e6f) : 0.f;
    int covered = 0;
    for (const int xh : {1, 2, 4, 6, 8}) {
      const int blocks = (T + 8 * xh - 1) / (8 * xh) * z;
      const bool beyond = covered >= T;  // (the last one held all tokens)
      if (beyond && z > 1) break;
      covered = 8 * xh;
      for (int rounds = fewest; rounds <= fewest + 2; ++rounds) {
        const int w = (per + rounds - 1) / rounds;
        for (const int rh : {2, 3, 4, 6, 8}) {
          if (!linear_instance(rh, xh, w, per)) continue;
          const int groups = (row_halves + rh - 1) / rh * blocks;
          if (beyond && (w <= 4 || groups > 256)) continue;
          float us = merge + (float)((groups + 255) >> 8) *
                                       (4.6f + 3.f * (float)(rounds - 1) + column * ((float)rh * (8.f / 52e3f) + (float)xh * (8.f / 60e3f)));
          if (rh == 3) us *= 1.06f;   // (for less than that it is not the faster)
          if (beyond) us *= 1.1f;     // (nor this)
          if (best.waves == 0 || us < least) {
            least = us;
            if (z == 1) undivided = groups;
            best = LinearPlan{xh, rh, w, z};
          }
        }
        if (w <= 8) break;  // (fewer at a time have no instance more)
      }
    }
  }
  return best;
}

int mi::linear_rows_per_workgroup(int T, int N, int K) {
  if (T <= 0 || T > 256) return 0;
  int slices, len;
  linear_slices(T, N, K, &slices, &len);
  const LinearPlan plan = linear_plan(T, N, K, slices);
  const int rows = 8 * plan.row_halves, across = (N + rows - 1) / rows;
  return plan.parts == 1 && (T <= 8 * plan.half_tiles || across % 8 == 0) ? rows : 0;
}

template <bool F16, int RH, int XH, int P, int NW>
static void launch_linear(const LinearParams& p, hipStream_t st) {
  const dim3 grid((p.N + 8 * RH - 1) / (8 * RH), (p.T + 8 * XH - 1) / (8 * XH), (p.S + p.per_part - 1) / p.per_part);
  hipLaunchKernelGGL((linear_decode_kernel<F16, RH, XH, P, NW>), grid, dim3(64 * p.waves), linear_lds((RH + 1) / 2, XH, p.waves, p.per_part), st, p);
}
// (steps in flight: what fits the registers without spilling)
template <bool F16>
static void launch_linear(const LinearParams& p, const LinearPlan& plan, hipStream_t st) {
  const int rh = plan.row_halves, xh = plan.half_tiles;
#define LIN(RH, XH, P, NW) launch_linear<F16, RH, XH, P, NW>(p, st)
  if (p.waves <= 8) {
    switch (10 * xh + rh) {
      case 12: LIN(2, 1, 8, 8); break;
      case 13: LIN(3, 1, 7, 8); break;
      case 14: LIN(4, 1, 6, 8); break;
      case 22: LIN(2, 2, 6, 8); break;
      case 23: LIN(3, 2, 5, 8); break;
      case 24: LIN(4, 2, 4, 8); break;
      case 42: LIN(2, 4, 6, 8); break;
      case 43: LIN(3, 4, 4, 8); break;
      case 44: LIN(4, 4, 4, 8); break;
      case 46: LIN(6, 4, 3, 8); break;
      case 62: LIN(2, 6, 5, 8); break;
      case 64: LIN(4, 6, 4, 8); break;
      case 66: LIN(6, 6, 2, 8); break;
      case 68: LIN(8, 6, 2, 8); break;
      case 82: LIN(2, 8, 4, 8); break;
      case 84: LIN(4, 8, 3, 8); break;
      case 86: LIN(6, 8, 2, 8); break;
      default: LIN(8, 8, 1, 8); break;
    }
  } else if (p.waves <= 12) {
    switch (10 * xh + rh) {
      case 12: LIN(2, 1, 6, 12); break;
      case 13: LIN(3, 1, 5, 12); break;
      case 14: LIN(4, 1, 4, 12); break;
      case 22: LIN(2, 2, 5, 12); break;
      case 23: LIN(3, 2, 4, 12); break;
      case 24: LIN(4, 2, 3, 12); break;
      case 42: LIN(2, 4, 4, 12); break;
      case 43: LIN(3, 4, 3, 12); break;
      case 44: LIN(4, 4, 2, 12); break;
      case 62: LIN(2, 6, 3, 12); break;
      case 64: LIN(4, 6, 1, 12); break;
      case 82: LIN(2, 8, 2, 12); break;
      default: LIN(4, 8, 1, 12); break;
    }
  } else {
    switch (10 * xh + rh) {
      case 12: LIN(2, 1, 6, 16); break;
      case 13: LIN(3, 1, 4, 16); break;
      case 14: LIN(4, 1, 3, 16); break;
      case 22: LIN(2, 2, 4, 16); break;
      case 23: LIN(3, 2, 3, 16); break;
      case 24: LIN(4, 2, 2, 16); break;
      case 42: LIN(2, 4, 2, 16); break;
      case 62: LIN(2, 6, 1, 16); break;
      default: LIN(2, 8, 1, 16); break;
    }
  }
#undef LIN
}

// Room for the sums of as many parts as a plan can have, or for the results where `out` lies over an input.  A K of 256
// and more asks for it on every call, so that a caller who sizes none is told at the first.
static int64_t linear_workspace(int T, int N, int slices) {
  return ((int64_t)T * N * 4 * (slices < kLinParts ? slices : kLinParts) + 255) & ~(int64_t)255;
}

extern "C" int64_t mi_linear_decode_workspace_bytes(int32_t T, int32_t N, int32_t K) {
  if (T <= 0 || N <= 0 || K <= 0) return 0;
  int slices, len;
  linear_slices(T, N, K, &slices, &len);
  return linear_workspace(T, N, slices);
}

extern "C" int mi_linear_decode(const void* x, int64_t x_stride_tok, const void* weight, int64_t w_stride_row,
                                const void* bias, void* out, int64_t out_stride_tok, void* workspace,
                                int64_t workspace_bytes, int32_t T, int32_t N, int32_t K, int32_t dtype, void* stream) {
  if (T == 0) return MI_OK;
  if (dtype != MI_DTYPE_BF16 && dtype != MI_DTYPE_FP16)
    return mi_fail(MI_ERR_UNSUPPORTED, "mi_linear_decode: dtype must be MI_DTYPE_BF16 or MI_DTYPE_FP16");
  if (!x || !weight || !out) return mi_fail(MI_ERR_NULL, "mi_linear_decode: null pointer argument");
  if (T < 0 || T > 256) return mi_fail(MI_ERR_SHAPE, "mi_linear_decode: 1..256 tokens per call (decode-sized steps)");
  if (N <= 0 || K <= 0 || N % 16 || K % 32)
    return mi_fail(MI_ERR_SHAPE, "mi_linear_decode: N must be a multiple of 16 and K a multiple of 32");
  if (((uintptr_t)x | (uintptr_t)weight | (uintptr_t)out) & 15 || ((uintptr_t)bias & 7))
    return mi_fail(MI_ERR_ALIGN, "mi_linear_decode: x / weight / out must be 16-byte aligned, bias 8-byte aligned");
  if ((x_stride_tok | w_stride_row) % 8 || out_stride_tok % 4 || x_stride_tok < K || w_stride_row < K || out_stride_tok < N)
    return mi_fail(MI_ERR_ALIGN, "mi_linear_decode: strides must cover a row and keep rows 16-byte (out: 8-byte) aligned");
  LinearParams p;
  p.x = (const uint16_t*)x; p.x_st = x_stride_tok; p.w = (const uint16_t*)weight; p.w_st = w_stride_row;
  p.bias = (const uint16_t*)bias; p.out = (uint16_t*)out; p.o_st = out_stride_tok;
  p.T = T; p.N = N; p.K = K;
  linear_slices(T, N, K, &p.S, &p.kslice);
  const LinearPlan plan = linear_plan(T, N, K, p.S);
  // (with several parts only the second launch stores, and reads nothing but the bias)
  const bool staged = (bias && linear_overlap(out, T, N, out_stride_tok, bias, 1, N, N)) ||
                      (plan.parts == 1 && (linear_overlap(out, T, N, out_stride_tok, x, T, K, x_stride_tok) ||
                                           linear_overlap(out, T, N, out_stride_tok, weight, N, K, w_stride_row)));
  if (staged || plan.parts > 1 || K >= 256) {
    if (!workspace || workspace_bytes < linear_workspace(T, N, p.S))
      return mi_fail(MI_ERR_WORKSPACE, "mi_linear_decode: workspace smaller than mi_linear_decode_workspace_bytes()");
    if ((uintptr_t)workspace & 15) return mi_fail(MI_ERR_ALIGN, "mi_linear_decode: the workspace must be 16-byte aligned");
  }
  p.waves = plan.waves;
  p.per_part = (p.S + plan.parts - 1) / plan.parts;
  p.part = plan.parts > 1 ? (float*)workspace : nullptr;
  const int quad = staged && plan.parts > 1 ? 8 : 4;
  if (staged) {
    p.out = (uint16_t*)workspace;
    p.o_st = N / 4 * quad;
  }
  hipStream_t st = (hipStream_t)stream;
  hipEvent_t ev_a, ev_b;
  const bool timed = mi_profile_next(&ev_a, &ev_b);
  if (timed) (void)hipEventRecord(ev_a, st);
  if (dtype == MI_DTYPE_FP16) launch_linear<true>(p, plan, st);
  else launch_linear<false>(p, plan, st);
  if (timed) (void)hipEventRecord(ev_b, st);
  const dim3 after((T * (N / 4) + 255) / 256);
  if (plan.parts > 1) {
    if (dtype == MI_DTYPE_FP16) hipLaunchKernelGGL(linear_parts_kernel<true>, after, dim3(256), 0, st, p, plan.parts, quad);
    else hipLaunchKernelGGL(linear_parts_kernel<false>, after, dim3(256), 0, st, p, plan.parts, quad);
  }
  if (staged)
    hipLaunchKernelGGL(linear_place_kernel, after, dim3(256), 0, st, p.out, quad, (uint16_t*)out, out_stride_tok, T, N);
  return mi_check_launch("mi_linear_decode");
}

extern "C" int mi_linear_qkv_decode_step(const void* hidden_states, int64_t x_stride_tok, const void* qkv_weight,
                                         int64_t w_stride_row, const void* qkv_bias, void* mixed_qkv,
                                         int64_t out_stride_tok, void* workspace, int64_t workspace_bytes, int32_t T,
                                         int32_t hidden_size, int32_t Hq, int32_t Hkv, int32_t head_dim, int32_t dtype,
                                         void* stream) {
  if (Hq <= 0 || Hkv <= 0 || head_dim <= 0 || Hq % Hkv)
    return mi_fail(MI_ERR_SHAPE, "mi_linear_qkv_decode_step: need Hq a positive multiple of Hkv");
  return mi_linear_decode(hidden_states, x_stride_tok, qkv_weight, w_stride_row, qkv_bias, mixed_qkv, out_stride_tok,
                          workspace, workspace_bytes, T, (Hq + 2 * Hkv) * head_dim, hidden_size, dtype, stream);
}

extern "C" int mi_attention_out_linear_proj(const void* core_attn_out, int64_t x_stride_tok, const void* proj_weight,
                                            int64_t w_stride_row, void* output, int64_t out_stride_tok, void* workspace,
                                            int64_t workspace_bytes, int32_t T, int32_t hidden_size, int32_t Hq,
                                            int32_t head_dim, int32_t dtype, void* stream) {
  if (Hq <= 0 || head_dim <= 0) return mi_fail(MI_ERR_SHAPE, "mi_attention_out_linear_proj: need Hq, head_dim > 0");
  return mi_linear_decode(core_attn_out, x_stride_tok, proj_weight, w_stride_row, nullptr, output, out_stride_tok,
                          workspace, workspace_bytes, T, hidden_size, Hq * head_dim, dtype, stream);
}
