// Gated delta rule (delta.hip) over long runs, blocks of 16 tokens, two at a time.  With G_t the product of the block's
// decays up to token t, per key channel, a block is
//
//   A[t, s] = beta_t sum_c k_t k_s G_t / G_s (s < t),   P[t, s] = sum_c q_t k_s G_t / G_s (s <= t)
//   (1 + A) [V0 | W] = beta [V | G k],   U = V0 - W S,   O = (G q) S + P U
//   S <- G_15 S + sum_s (G_15 / G_s) k_s u_s^T
//
// delta_prepare computes everything without S for all pairs of blocks at once and leaves it in the order of the matrix
// operands.  delta_blocks walks a head's pairs with S in registers.  All fp32; projections in bfloat16.
#include "blocks.h"

namespace {

constexpr int kMaxTaps = 8;

struct RunArgs {
  zp_delta d;
  float* ws;
  int row0;      // first token row of the first segment
  Pieces pieces;
  // PROJECTED: the decays' and the gates' pre-activations are products made here, of `rank` columns of a.in from low_at on, the
  // first a_rank of them for the decays, with rows (heads * (dk + dv), rank) as [rows / 16][columns / 32][64 lanes][8]
  const uint16_t* low_weights;
  int low_at, rank, a_rank;
};
constexpr int kLowSteps = 4, kLowRank = 256;   // of 32 columns for either product; columns in all

// Two blocks after one another are one step of the chain, which splits the state once for both and meets once (a block at a
// time, 160 heads 3.2 us for 16 tokens, now 2.4): with D the decays of a whole block and S the state before both,
//
//   U0 = V0 - W0 S,   U1 = V1 - W1 D0 S - (W1 K0^T) U0,   S <- D1 D0 S + D1 K0^T U0 + K1^T U1
//   O0 = Q0 S + P0 U0,   O1 = Q1 D0 S + (Q1 K0^T) U0 + P1 U1      (Q: G q, K: keys with the decays behind them)
//
// A pair in memory, whole KBs: tiles of [64 lanes][4] of -W0, Q0, -W1 D0, Q1 D0 (16 columns each, left operands) and, by 16
// rows, of D1 K0 and K1; V0 and V1 as result tiles; planes of P0, P1, -W1 K0^T, Q1 K0^T; D0 D1; the gates' pre-activations
// as result tiles in bfloat16.
__host__ __device__ inline constexpr int small_floats(int dk) { return 4 * kPairFloats + dk; }
__host__ __device__ inline constexpr int pair_floats(int dk, int dv) {
  return (2 * kBlock * (3 * dk + dv) + small_floats(dk) + kBlock * dv + 255) / 256 * 256;
}
__host__ __device__ inline constexpr int gates_at(int dk, int dv) { return 2 * kBlock * (3 * dk + dv) + small_floats(dk); }
__device__ __forceinline__ int64_t pair_slot(int row0, const Segment& sg, int seg, int b) { return (sg.row - row0) / (2 * kBlock) + seg + b; }

// A pair of blocks: 256 threads each, and the products of the second with the first.  Bound by vector issue (four fifths of its
// time).  Ratios of decays are running products of the decays behind a token, A and P sums in fp32.  As products of G k and G q with
// k / G on the matrix cores they take less of it (8 prompts of 2048 tokens, 32 heads 899 us in all, now 945; one of 110, 16 heads 39.0 and
// 40.4), but quotients carry the roundings of what both have in common: where channels forget 3 bits a token, the state was 2.7e-7 of its
// norm off 64 bits, now 1.1e-7.
constexpr int kPrepareLd = 132;                // floats of a row: reads across tokens meet no conflicts, offsets are constants
constexpr int kPrepareHalf = kBlock * 4 * kPrepareLd + 6 * kBlock * kBlock + kBlock + 128;
// A lane of 16, one of each row, gets its left neighbour's times its own decay; the first keeps its own.  Eight side by side, as a
// lane that is moved has to be written two instructions before.
__device__ __forceinline__ void to_next_token(float (&x)[8], const float (&g)[8]) {
#ifdef __HIP_DEVICE_COMPILE__
#define ZP_MOVED(i, by) "v_mul_f32_dpp %" #i ", %" #i ", %" #by " row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
  asm("s_nop 1\n\t" ZP_MOVED(0, 8) ZP_MOVED(1, 9) ZP_MOVED(2, 10) ZP_MOVED(3, 11) ZP_MOVED(4, 12) ZP_MOVED(5, 13) ZP_MOVED(6, 14) ZP_MOVED(7, 15)
      : "+&v"(x[0]), "+&v"(x[1]), "+&v"(x[2]), "+&v"(x[3]), "+&v"(x[4]), "+&v"(x[5]), "+&v"(x[6]), "+&v"(x[7])
      : "v"(g[0]), "v"(g[1]), "v"(g[2]), "v"(g[3]), "v"(g[4]), "v"(g[5]), "v"(g[6]), "v"(g[7]));
#undef ZP_MOVED
#endif
}
// The left neighbour's of 16, the first's one.
__device__ __forceinline__ float before_or_one(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0x3f800000, __builtin_bit_cast(int, x), 0x111, 0xf, 0xf, false));
}
// Sums over the wave's four groups of 16 lanes; group g has that of x[g].
__device__ __forceinline__ float sums_of_groups(const float (&x)[4]) {
  auto bits = [](float v) { return __builtin_bit_cast(uint32_t, v); };
  auto value = [](uint32_t v) { return __builtin_bit_cast(float, v); };
  const auto a = __builtin_amdgcn_permlane16_swap(bits(x[0]), bits(x[1]), false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(bits(x[2]), bits(x[3]), false, false);
  const auto c = __builtin_amdgcn_permlane32_swap(bits(value(a[0]) + value(a[1])), bits(value(b[0]) + value(b[1])), false, false);
  return value(c[0]) + value(c[1]);
}
template <int TAPS, bool PROJECTED>
__global__ __launch_bounds__(512, 4) void delta_prepare_kernel(RunArgs ra) {
  extern __shared__ __align__(16) float lds[];
  const zp_delta& a = ra.d;
  constexpr int ld = kPrepareLd;
  const int dk = a.dk, dv = a.dv, taps = a.taps;
  const Segment sg = segment_of(a.seg, blockIdx.z);
  const int half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), t0 = (2 * blockIdx.x + half) * kBlock;
  if ((int)blockIdx.x * 2 * kBlock >= sg.count || sg.row < ra.row0) return;
  const int cnt = max(min(kBlock, sg.count - t0), 0);          // of the second block: maybe none
  const int h = blockIdx.y, hk = h / (a.heads / a.kv_heads);
  float* const qs = lds + half * kPrepareHalf;                 // [16][ld], later G q
  float* const ks = qs + kBlock * ld;          // later G k, then -W
  float* const gs = ks + kBlock * ld;          // decays, later keys with those behind them
  float* const vs = gs + kBlock * ld;
  float* const As = vs + kBlock * ld;          // [16][16]
  float* const Ps = As + kBlock * kBlock;      // [16][16]; both over parts of them, [3][2][64][4]
  float* const beta = As + 6 * kBlock * kBlock;
  float* const decays = beta + kBlock;         // [dk] of the whole block
  float* const other_decays = decays + (half ? -kPrepareHalf : kPrepareHalf);
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cw = 2 * dk + dv;
  const char* const tail = (const char*)a.conv_state + ((int64_t)sg.slot * a.heads + h) * (taps - 1) * cw * 2;
  const int channels = 2 * a.kv_heads * dk + a.heads * dv;
  auto place = [&](int c) -> int {
    return c < dk ? hk * dk + c : (c < 2 * dk ? a.kv_heads * dk + hk * dk + c - dk : 2 * a.kv_heads * dk + h * dv + c - 2 * dk);
  };
  const int tiles = dk / 16, wave8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, g4 = lane >> 4;
  float* const to = ra.ws + (pair_slot(ra.row0, sg, blockIdx.z, blockIdx.x) * a.heads + h) * pair_floats(dk, dv);
  // ---- requests first: the decays' pre-activations (two pieces a thread at most), the step sizes'; or what they are products of
  const int piece_bits = 31 - __builtin_clz(dk / 4);           // pieces of four channels: 8, 16 or 32 a row
  f32x4 z[2], zb[2];
  u32x4 low[2], wa[kLowSteps], wg[kLowSteps];
  const int g_step = ra.a_rank >> 5;                           // the gates' first step; they share it with the decays where that ends inside
  if constexpr (PROJECTED) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {                              // rows of up to 32 pieces of 16 bytes
      const int i = tid + u * 256, t = min(t0 + (i >> 5), sg.count - 1), c = (i & 31) * 8;
      low[u] = u32x4{0u, 0u, 0u, 0u};
      if (c < ra.rank) low[u] = *(const u32x4*)((const uint16_t*)a.in + (int64_t)(sg.row + t) * a.in_stride + ra.low_at + c);
    }
    const int steps = (ra.rank + 31) >> 5;
    auto weights = [&](int tile, int step, bool there) {
      u32x4 v = {0u, 0u, 0u, 0u};
      if (there && step < steps) v = *(const u32x4*)(ra.low_weights + ((int64_t)tile * steps + step) * 512 + lane * 8);
      return v;
    };
#pragma unroll
    for (int i = 0; i < kLowSteps; ++i) {
      wa[i] = weights(h * tiles + wave8, i, wave8 < tiles && i * 32 < ra.a_rank);
      wg[i] = weights(a.heads * tiles + h * (dv / 16) + wave8, g_step + i, wave8 < dv / 16);
    }
  } else {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int i = tid + u * 256, t = min(t0 + (i >> piece_bits), sg.count - 1), c = (i & ((1 << piece_bits) - 1)) * 4;
      z[u] = load4<BF16>(a.low, (int64_t)(sg.row + t) * a.low_stride + h * dk + c);
      zb[u] = *(const f32x4*)(a.dt_bias + h * dk + c);
    }
    if (wave8 < dv / 16)
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int first = (2 * blockIdx.x + k) * kBlock;
        const BlockRows rows(a.low, sg.row + first, min(max(sg.count - first, 0), kBlock), a.low_stride);
        uint32_t v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = rows.ld((4 * g4 + r) * (int)a.low_stride * 2 + (a.g_at + h * dv + wave8 * 16 + l16) * 2, 0);
        *(uint2*)(to + gates_at(dk, dv) + ((k * (dv / 16) + wave8) * 64 + lane) * 2) = uint2{v[0] | v[1] << 16, v[2] | v[3] << 16};
      }
  }
  const float b_in = tid < cnt ? Elem<BF16>::ld(a.in, (int64_t)(sg.row + t0 + tid) * a.in_stride + a.b_at + h) : 0.f;
  const float rate = expf(a.a_log[h]) * 1.44269504088896f;      // in bits
  // ---- convolutions: a thread's two channels, the block's 16 tokens from a sliding window.  Rows behind the run's end read
  // as zero, and those before its beginning too, unless they come from the history.
  const int row_bytes = (int)a.in_stride * 2;
  const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const char*)a.in + (int64_t)(sg.row + t0) * row_bytes), 0, cnt * row_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t before = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const char*)a.in + (int64_t)(sg.row + t0 - (TAPS - 1)) * row_bytes), 0, t0 > 0 && cnt > 0 ? (TAPS - 1) * row_bytes : 0, 0x00020000);
  // at most 384 channels, which leave a wave of each half without work: not those on one SIMD
  const int c = 2 * ((tid + 64 * (blockIdx.x + 2 * half)) & 255);
  uint32_t x[kBlock + TAPS - 1];               // two channels' bf16
  float f[2][TAPS];                            // f[.][j]: j tokens back
  if (c < cw) {
    const int at = place(c);
#pragma unroll
    for (int i = 0; i < kBlock + TAPS - 1; ++i)
      x[i] = (uint32_t)(i < TAPS - 1 ? __builtin_amdgcn_raw_buffer_load_b32(before, at * 2, i * row_bytes, 0)
                                     : __builtin_amdgcn_raw_buffer_load_b32(rows, at * 2, (i - (TAPS - 1)) * row_bytes, 0));
#pragma unroll
    for (int j = 0; j < TAPS; ++j)
#pragma unroll
      for (int e = 0; e < 2; ++e) f[e][j] = a.filters[(int64_t)max(taps - 1 - j, 0) * channels + at + e];
#pragma unroll
    for (int j = 1; j < TAPS; ++j)
#pragma unroll
      for (int e = 0; e < 2; ++e) f[e][j] = j < taps ? f[e][j] : 0.f;
    if (t0 == 0 && sg.start > 0) {
#pragma unroll
      for (int i = 0; i < TAPS - 1; ++i)
        if (i >= TAPS - taps) x[i] = *(const uint32_t*)(tail + ((int64_t)(taps - TAPS + i) * cw + c) * 2);
    }
  }
  if constexpr (PROJECTED) {
#pragma unroll
    for (int u = 0; u < 2; ++u) *(u32x4*)((char*)qs + ((tid + u * 256) >> 5) * ld * 4 + (tid & 31) * 16) = low[u];
    __syncthreads();
    // A wave 16 channels of decays and 16 of gates, of both blocks.  The library's product of rows that are half zeros takes as
    // long as this does in all for many tokens and a launch more (8 prompts of 2048 tokens, 32 heads 19 us of 936, 2 of about 1250
    // 21 of 261, one of 110, 16 heads 3.6 of 42.3); weights row by row, which touch twice as many lines, cost 27 of the first.
    const f32x4 bias = wave8 < tiles ? *(const f32x4*)(a.dt_bias + h * dk + wave8 * 16 + g4 * 4) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const char* const rows = (const char*)(lds + k * kPrepareHalf) + l16 * ld * 4 + g4 * 16;
      f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = x;
#pragma unroll
      for (int i = 0; i < kLowSteps; ++i) {
        x = mfma_bf16(wa[i], *(const u32x4*)(rows + i * 64), x);
        y = mfma_bf16(*(const u32x4*)(rows + (g_step + i) * 64), wg[i], y);
      }
      if (wave8 < dv / 16)
        *(uint2*)(to + gates_at(dk, dv) + ((k * (dv / 16) + wave8) * 64 + lane) * 2) = uint2{pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3])};
      if (wave8 < tiles) {
        const uint32_t lo = pack_bf16(x[0], x[1]), hi = pack_bf16(x[2], x[3]);     // as rows `low` would hold them
        x = f32x4{__uint_as_float(lo << 16), __uint_as_float(lo & 0xffff0000u), __uint_as_float(hi << 16), __uint_as_float(hi & 0xffff0000u)} + bias;
        const bool there = (2 * (int)blockIdx.x + k) * kBlock + l16 < sg.count;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = there ? __builtin_amdgcn_exp2f(-rate * fast_softplus(x[e])) : 1.f;
        *(f32x4*)(lds + k * kPrepareHalf + 2 * kBlock * ld + l16 * ld + wave8 * 16 + g4 * 4) = x;
      }
    }
    __syncthreads();                           // the rows are used up
  }
  if (c < cw) {
    float* const dst = c < dk ? qs + c : (c < 2 * dk ? ks + c - dk : vs + c - 2 * dk);
    if (cnt > 0)
#pragma unroll
    for (int t = 0; t < kBlock; ++t) {
      float2 y = {0.f, 0.f};
#pragma unroll
      for (int j = 0; j < TAPS; ++j) {
        const uint32_t v = x[t + TAPS - 1 - j];
        y.x = fmaf(f[0][j], __uint_as_float(v << 16), y.x);
        y.y = fmaf(f[1][j], __uint_as_float(v & 0xffff0000u), y.y);
      }
      y.x *= fast_sigmoid(y.x);
      y.y *= fast_sigmoid(y.y);
      *(float2*)(dst + t * ld) = y;
      if (t % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    for (int t = cnt; t < kBlock; ++t) *(float2*)(dst + t * ld) = float2{0.f, 0.f};
  }
  if constexpr (!PROJECTED)
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int i = tid + u * 256, t = i >> piece_bits, c = (i & ((1 << piece_bits) - 1)) * 4;
    if (t < kBlock) {
      f32x4 g;
#pragma unroll
      for (int e = 0; e < 4; ++e) g[e] = t < cnt ? __builtin_amdgcn_exp2f(-rate * fast_softplus(z[u][e] + zb[u][e])) : 1.f;
      *(f32x4*)(gs + t * ld + c) = g;
    }
  }
  if (tid < kBlock) beta[tid] = tid < cnt ? fast_sigmoid(b_in) : 0.f;
  __syncthreads();
  // ---- unit vectors: a wave its four tokens, 16 lanes each
  {
    const int t = wave * 4 + (lane >> 4), pieces = dk / 4;
    f32x4 q[2], k[2], q2 = {0.f, 0.f, 0.f, 0.f}, k2 = q2;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int pc = min(l16 + 16 * p, pieces - 1);
      q[p] = *(const f32x4*)(qs + t * ld + pc * 4);
      k[p] = *(const f32x4*)(ks + t * ld + pc * 4);
      if (l16 + 16 * p < pieces) {
        q2 += q[p] * q[p];
        k2 += k[p] * k[p];
      }
    }
    const float rq = a.q_scale / sqrtf(row16_sum(q2[0] + q2[1] + q2[2] + q2[3]) + 1e-6f);
    const float rk = 1.f / sqrtf(row16_sum(k2[0] + k2[1] + k2[2] + k2[3]) + 1e-6f);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int pc = l16 + 16 * p;
      if (pc < pieces) {
        *(f32x4*)(qs + t * ld + pc * 4) = q[p] * rq;
        *(f32x4*)(ks + t * ld + pc * 4) = k[p] * rk;
      }
    }
  }
  __syncthreads();
  // ---- A and P: a wave 32 channels (of fewer than 128, some of the distances too), a lane one token's of them.  Keys go down the tokens, from lane to lane, and decay on the way:
  // after d moves a lane has k_s with the decays behind s, s = t - d, for A[t, s] and P[t, s], and the last lane what the state gets of
  // k_s.  One comes in before the first token, and once it has reached a lane, that has the decays up to it.
  const int waves = dk / 32, mine = wave & (waves - 1), from = wave & -waves, row_at = (lane & 15) * ld + mine * 32 + (lane >> 4) * 4;
  float* const oU = to + 6 * kBlock * dk + half * kBlock * dv;
  float* const oSmall = to + 6 * kBlock * dk + 2 * kBlock * dv;
  auto put_small = [&](int i, const f32x4& v) {
    const Planes x(v);
    *(u32x4*)(oSmall + i * kPairFloats + lane * 4) = u32x4{x.hi.x, x.hi.y, x.mid.x, x.mid.y};
    *(uint2*)(oSmall + i * kPairFloats + 256 + lane * 2) = x.lo;
  };
  auto split = [](const f32x4 (&v)[2], u32x4 (&o)[3]) {
    const Planes x(v[0]), y(v[1]);
    o[0] = u32x4{x.hi.x, x.hi.y, y.hi.x, y.hi.y};
    o[1] = u32x4{x.mid.x, x.mid.y, y.mid.x, y.mid.y};
    o[2] = u32x4{x.lo.x, x.lo.y, y.lo.x, y.lo.y};
  };
  auto products = [](const u32x4 (&l)[3], const u32x4 (&r)[2][3], f32x4 (&y)[2]) {      // the smallest first
    y[0] = y[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 2; i >= 0; --i)
#pragma unroll
      for (int j = 2 - i; j >= 0; --j)
#pragma unroll
        for (int u = 0; u < 2; ++u) y[u] = mfma_bf16(l[i], r[u][j], y[u]);
  };
  f32x4 y[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};       // A and P, distances 4 u + lane / 16 in element u
  if (cnt == 0) {                              // a second block without tokens leaves the SIMDs to the first (beside zeros for keys and queries)
    if (waves < 4) __syncthreads();
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      *(f32x4*)(gs + row_at + 16 * p) = f32x4{0.f, 0.f, 0.f, 0.f};
      if ((lane & 15) == 15) *(f32x4*)(decays + mine * 32 + 16 * p + (lane >> 4) * 4) = f32x4{1.f, 1.f, 1.f, 1.f};
    }
  } else {
    float k[8], q[8], g[8], x[8];              // of this lane's own elements, all three, which nobody else reads
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const f32x4 kp = *(const f32x4*)(ks + row_at + 16 * p), qp = *(const f32x4*)(qs + row_at + 16 * p), gp = *(const f32x4*)(gs + row_at + 16 * p);
#pragma unroll
      for (int e = 0; e < 4; ++e) k[4 * p + e] = kp[e], q[4 * p + e] = qp[e], g[4 * p + e] = gp[e], x[4 * p + e] = kp[e];
    }
    if (waves < 4) __syncthreads();            // others read them too
    auto put = [](float* at, const float (&v)[8]) {
      *(f32x4*)at = f32x4{v[0], v[1], v[2], v[3]};
      *(f32x4*)(at + 16) = f32x4{v[4], v[5], v[6], v[7]};
    };
#pragma unroll
    for (int u = 0; u < 4; ++u) {              // those before its first only move, and behind its last nothing does
      if (u >= from + waves) continue;
      float sa[4], sp[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = 4 * u + j;
        if (d == 1)
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i] = before_or_one(x[i]) * g[i];
        if (d > 1) to_next_token(x, g);
        if (u < from) continue;
        if ((lane & 15) == 15) put(gs + row_at - d * ld, x);
        sa[j] = sp[j] = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if (d > 0) sa[j] += x[i] * k[i];
          sp[j] += x[i] * q[i];
        }
      }
      if (u < from) continue;
      y[0][u] = sums_of_groups(sa);
      y[1][u] = sums_of_groups(sp);
    }
    if (from + waves == 4) {
      to_next_token(x, g);                     // the decays up to the lane's token
      if ((lane & 15) == 15) put(decays + mine * 32 + (lane >> 4) * 4, x);
#pragma unroll
      for (int i = 0; i < 8; ++i) k[i] *= x[i], q[i] *= x[i];
      put(ks + row_at, k);
      put(qs + row_at, q);
    }
  }
  if (wave > 0)
#pragma unroll
    for (int u = 0; u < 2; ++u) *(f32x4*)(As + (((wave - 1) * 2 + u) * 64 + lane) * 4) = y[u];
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int j = 1; j < 4; ++j)
#pragma unroll
      for (int u = 0; u < 2; ++u) y[u] += *(const f32x4*)(As + (((j - 1) * 2 + u) * 64 + lane) * 4);
    asm volatile("" ::: "memory");             // the parts are read before rows of A and P lie there
    const int t = lane & 15, g4 = lane >> 4;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (const int d = 4 * u + g4; d <= t) {  // A's with itself is not read
        As[t * kBlock + t - d] = y[0][u] * beta[t];
        Ps[t * kBlock + t - d] = y[1][u];
      }
    asm volatile("" ::: "memory");
    f32x4 P = *(const f32x4*)(Ps + t * kBlock + 4 * g4);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (4 * g4 + r > t) P[r] = 0.f;
    put_small(half, P);
  }
  __syncthreads();
  // ---- columns: forward substitution.  A thread reads and writes its own column only.
  float w[kBlock];
  auto substitute = [&](int t, float b) {      // w_t = b - sum_{s < t} A[t, s] w_s
    float x[4] = {b, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < t; s += 4) {
      const f32x4 A = *(const f32x4*)(As + t * kBlock + s);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (s + i < t) x[i] = fmaf(-A[i], w[s + i], x[i]);
    }
    w[t] = (x[0] + x[1]) + (x[2] + x[3]);
    if (t % 2 == 1) __builtin_amdgcn_sched_barrier(0);
  };
  if (tid < dk + dv) {                         // at most 256
    const bool key = tid < dk;
    const int c = key ? tid : tid - dk;
    const float* const column = (key ? ks : vs) + c;
    if (cnt > 0) {
#pragma unroll
      for (int t = 0; t < kBlock; ++t) substitute(t, beta[t] * column[t * ld]);
    } else {
#pragma unroll
      for (int t = 0; t < kBlock; ++t) w[t] = 0.f;
    }
    if (key) {
      const float D = other_decays[c], by = half ? 1.f : D;
      if (!half) oSmall[4 * kPairFloats + c] = decays[c] * D;
      float* const oK = to + (4 * tiles + 2 * (c >> 4) + half) * 256 + (c & 15) * 4;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 x;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          x[r] = gs[(4 * g + r) * ld + c] * by;
          ks[(4 * g + r) * ld + c] = -w[4 * g + r];
        }
        *(f32x4*)(oK + g * 64) = x;
      }
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *(f32x4*)(oU + ((c >> 4) * 64 + g * 16 + (c & 15)) * 4) = f32x4{w[4 * g], w[4 * g + 1], w[4 * g + 2], w[4 * g + 3]};
    }
  }
  __syncthreads();
  // ---- -W and G q, as left operands hold them; the second block's with the first one's keys, transposed like these
  float* const part = lds + kPrepareHalf + 3 * kBlock * ld;    // over the second block's values: [dk / 32][2][64][4]
  if (wave < waves) {
    f32x4 W[2], Q[2], K[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      W[p] = *(const f32x4*)(ks + row_at + 16 * p);
      Q[p] = *(const f32x4*)(qs + row_at + 16 * p);
      K[p] = *(const f32x4*)(lds + 2 * kBlock * ld + row_at + 16 * p);
      const f32x4 D = *(const f32x4*)(other_decays + wave * 32 + 16 * p + (lane >> 4) * 4);
      float* const o = to + (2 * half * tiles + 2 * wave + p) * 256 + lane * 4;
      *(f32x4*)o = half ? W[p] * D : W[p];
      *(f32x4*)(o + tiles * 256) = half ? Q[p] * D : Q[p];
    }
    if (half) {
      u32x4 left[3], rows2[2][3];
      split(K, left);
      split(W, rows2[0]);
      split(Q, rows2[1]);
      products(left, rows2, y);
#pragma unroll
      for (int u = 0; u < 2; ++u) *(f32x4*)(part + ((wave * 2 + u) * 64 + lane) * 4) = y[u];
    }
  }
  __syncthreads();
  if (half && wave < 2) {
    f32x4 x = *(const f32x4*)(part + (wave * 64 + lane) * 4);
    for (int j = 1; j < waves; ++j) x += *(const f32x4*)(part + ((j * 2 + wave) * 64 + lane) * 4);
    put_small(2 + wave, x);
  }
}

// ------------------------------------------------------------------ runs in pieces, of heads with as many keys as values
// A piece keeps M S of a state S before it, M the product of its blocks' (diag(G_15) - keys^T W).  Its columns walk through
// the piece as those of a state do, from one on, with nothing of the values.  A piece's state: its sums, or the state before
// it, then M as a left operand, [rows / 16][columns / 16][64 lanes][4].
__host__ __device__ inline constexpr int piece_floats(int dk) { return 2 * dk * dk; }

// From sums to the states before the pieces, in place; a wave 16 columns, a workgroup half of them, which splits all of M: 4.3 us
// a piece.  With all columns in one workgroup the products and reads of eight waves take 5.7; with a quarter, the splitting by two
// waves 5.0 (a prompt of 700 tokens, 16 heads, in six pieces 34.2, 25.9 and 30.1 us; the whole scan 106 -> 98).
template <int KT, int NW>
__global__ __launch_bounds__(64 * NW, 1) void delta_states_kernel(RunArgs ra) {
  extern __shared__ __align__(16) float planes[];              // [rows / 16][pairs of columns / 16][3][64 lanes][4]
  constexpr int dk = 16 * KT, J = KT / 2, kParts = KT / NW;
  const zp_delta& a = ra.d;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int unit = blockIdx.x / kParts, h = unit % a.heads, seg = unit / a.heads, mine = blockIdx.x % kParts * NW + wave;
  const Segment whole = segment_of(a.seg, seg);
  if (whole.count <= 0 || whole.row < ra.row0) return;
  f32x4 S[KT][1], x[kParts][KT], add[KT];
  load_state<KT, 1>(S, a.state + ((int64_t)whole.slot * a.heads + h) * ((int64_t)dk * dk), dk, mine * 16, whole.start == 0);
  const int tokens = ra.pieces.blocks * kBlock, count = (whole.count + tokens - 1) / tokens;
  const int64_t stride = (int64_t)a.heads * piece_floats(dk);
  float* const at = ra.pieces.states + Piece(ra.pieces, ra.row0, whole, seg, 0).slot * stride + (int64_t)h * piece_floats(dk) + lane * 4;
  auto load = [&](int c) {                                     // this wave's share of M's columns, for all waves
#pragma unroll
    for (int u = 0; u < kParts; ++u)
#pragma unroll
      for (int t = 0; t < KT; ++t) x[u][t] = *(const f32x4*)(at + c * stride + dk * dk + (t * KT + wave + u * NW) * 256);
  };
  auto meet = [] {                                             // LDS alone: what comes from memory and goes there stays on its way
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto load_sums = [&](int c, int t) { add[t] = *(const f32x4*)(at + c * stride + (mine * KT + t) * 256); };
  if (count > 1) {
    load(0);
#pragma unroll
    for (int t = 0; t < KT; ++t) load_sums(0, t);
  }
#pragma unroll 1
  for (int c = 0; c < count; ++c) {
    const bool more = c + 1 < count;                           // the last piece has no sums
    u32x4 sp[3][J];
    meet();                                                    // the planes before these are used up
    if (more) {
#pragma unroll
      for (int u = 0; u < kParts; ++u)
#pragma unroll
        for (int t = 0; t < KT; ++t) {
          const Planes p(x[u][t]);
          const int column = wave + u * NW;
          float* const to = planes + (t * J + (column >> 1)) * 768 + lane * 4 + (column & 1) * 2;
          *(uint2*)to = p.hi;
          *(uint2*)(to + 256) = p.mid;
          *(uint2*)(to + 512) = p.lo;
        }
      load(min(c + 1, count - 2));
    }
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      *(f32x4*)(at + c * stride + (mine * KT + kt) * 256) = S[kt][0];
      const Planes p(S[kt][0]);
      const int e = (kt & 1) * 2;
      sp[0][kt >> 1][e] = p.hi.x, sp[0][kt >> 1][e + 1] = p.hi.y;
      sp[1][kt >> 1][e] = p.mid.x, sp[1][kt >> 1][e + 1] = p.mid.y;
      sp[2][kt >> 1][e] = p.lo.x, sp[2][kt >> 1][e + 1] = p.lo.y;
    }
    meet();
    if (!more) break;
#pragma unroll
    for (int t = 0; t < KT; t += 2) {                          // two rows of tiles: each product waits for the one before
      f32x4 y[2] = {add[t], add[t + 1]};
      load_sums(min(c + 1, count - 2), t);
      load_sums(min(c + 1, count - 2), t + 1);
#pragma unroll
      for (int i = 2; i >= 0; --i)                             // the smallest products first
#pragma unroll
        for (int k = 2 - i; k >= 0; --k)
#pragma unroll
          for (int j = 0; j < J; ++j)
#pragma unroll
            for (int u = 0; u < 2; ++u)
              y[u] = mfma_bf16(*(const u32x4*)(planes + (((t + u) * J + j) * 3 + i) * 256 + lane * 4), sp[k][j], y[u]);
      S[t][0] = y[0];
      S[t + 1][0] = y[1];
    }
  }
}

// A head's pairs of blocks, one after the other, a wave 16 columns of the state.  On the fp32 matrix cores the products would be
// the bound, so operands are split into three bf16 planes: the products that count take a quarter of that, beside the vector
// units.  The state is split where it is updated; what comes from memory passes through registers, asked for a pair ahead, and
// is split into LDS by all waves together under the products with the state; rows are normed and stored in the next pair.
// What bounds it: of 11 300 cycles a pair and SIMD the products take 5100, vector issue 6200 beside them, LDS 4300, and the
// younger of its two waves the rest.  8 prompts of 2048 tokens, 32 heads of 128 x 128, with the kernel above: 1017 -> 945 us, 5 of
// 1640 to 2037 717 -> 621, one 261 -> 217; 7 of 625 to 1499 with 16 heads 417 -> 357; error of the state against 64 bits, where channels
// forget 0.01, 1 and 3 bits a token, 3.9e-7 -> 3.7e-7, 1.7e-7 -> 1.4e-7 and 1.3e-7 -> 1.1e-7 of its norm.  All products are six of the planes;
// with eight in the update of the state, 3.694e-7 instead of 3.695e-7, 1.437e-7 and 1.142e-7, and 1 to 2 % longer.
// SUMS: no state comes in and no rows go out; every second workgroup takes what the piece keeps, where values are none.
template <int KT, int NW> struct PairStage {
  static constexpr int kTiles = 6 * KT, kPlanes = kTiles * 384, kSmall = small_floats(16 * KT);      // floats in LDS
  static constexpr int kMine = (kTiles + NW - 1) / NW, kRing = kMine <= 6 ? kMine : kMine % 6 == 0 ? 6 : kMine % 4 == 0 ? 4 : 3;      // a wave's tiles; asked for ahead
  static constexpr int kPieces = (kSmall / 4 + 64 * NW - 1) / (64 * NW);     // a thread's 16 bytes of the small ones
  static constexpr int kBytes = (2 * kPlanes + 2 * kSmall + 4 * NW * kBlock) * 4;
  static_assert(kMine % kRing == 0, "places of the ring are constants");
};
template <int KT, int NW, bool SUMS>
__global__ __launch_bounds__(64 * NW, 2) void delta_blocks_kernel(RunArgs ra) {
  extern __shared__ __align__(16) float lds[];
  typedef PairStage<KT, NW> Stage;
  const zp_delta& a = ra.d;
  constexpr int dk = 16 * KT, dv = 16 * NW, size = pair_floats(dk, dv), J = KT / 2;
  constexpr int kMine = Stage::kMine, kRing = Stage::kRing, kPlanes = Stage::kPlanes, kSmall = Stage::kSmall, kPieces = Stage::kPieces;
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  float* const planes = lds;                   // [2][pairs of tiles][3][64 lanes][4]
  float* const small = planes + 2 * kPlanes;   // [2][kSmall]
  float* const red = small + 2 * kSmall;       // [2][2][NW * 16]
  const bool keeps = SUMS && blockIdx.x & 1;
  const int id = SUMS ? blockIdx.x >> 1 : blockIdx.x, most = ra.pieces.most - SUMS, unit = id / most, h = unit % a.heads, seg = unit / a.heads;
  const Segment whole = segment_of(a.seg, seg);
  if (whole.count <= 0 || whole.row < ra.row0) return;
  const Piece piece(ra.pieces, ra.row0, whole, seg, id % most);
  const Segment& sg = piece.sg;
  if (SUMS ? piece.last : sg.count <= 0) return;
  const int64_t item = (int64_t)sg.slot * a.heads + h;
  float* const state = a.state + item * ((int64_t)dk * dv);
  float* const between = ra.pieces.states + (piece.slot * a.heads + h) * piece_floats(dk);
  const int col0 = wave * 16;
  f32x4 S[KT][1];
  if constexpr (SUMS) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[kt][0][r] = keeps && 16 * kt + 4 * g + r == col0 + l16 ? 1.f : 0.f;
  } else if (ra.pieces.blocks) {
    load_piece_state(S, between, wave);
  } else {
    load_state<KT, 1>(S, state, dv, col0, sg.start == 0);
  }
  const float nrm = a.norm[h * dv + col0 + l16] * a.out_scale;
  const float* const base = ra.ws + (pair_slot(ra.row0, sg, seg, 0) * a.heads + h) * size;
  const int64_t stride = (int64_t)a.heads * size;
  const int pairs = (sg.count + 2 * kBlock - 1) / (2 * kBlock);
  auto at_pair = [&](int b) { return base + min(b, pairs - 1) * stride; };     // behind the last: it again, and nobody looks
  // A wave's tile u of a pair: on its way through registers, then its planes in LDS.  The last may come twice.
  auto tile_index = [&](int u) { return min(wave + u * NW, Stage::kTiles - 1); };
  f32x4 raw[kRing], rest[kPieces], values[2];
  auto ask = [&](int b, int u) { raw[u % kRing] = *(const f32x4*)(at_pair(b) + tile_index(u) * 256 + lane * 4); };
  auto put = [&](int b, int u) {
    const int i = tile_index(u);
    float* const to = planes + (b & 1) * kPlanes + (i >> 1) * 768 + (i & 1) * 2 + lane * 4;
    const Planes p(raw[u % kRing]);
    *(uint2*)to = p.hi;
    *(uint2*)(to + 256) = p.mid;
    *(uint2*)(to + 512) = p.lo;
  };
  auto next_tile = [&](int b, int u) {         // put tile u of pair b, ask for the one kRing further
    put(b, u);
    if (u + kRing < kMine) ask(b, u + kRing);
    else ask(b + 1, u + kRing - kMine);
  };
  auto ask_values = [&](int b) {
#pragma unroll
    for (int i = 0; i < 2; ++i) values[i] = *(const f32x4*)(at_pair(b) + 6 * kBlock * dk + i * kBlock * dv + wave * 256 + lane * 4);
  };
  auto ask_rest = [&](int b) {
    const float* const p = at_pair(b) + 2 * kBlock * (3 * dk + dv);
#pragma unroll
    for (int u = 0; u < kPieces; ++u) rest[u] = *(const f32x4*)(p + min(tid + u * 64 * NW, kSmall / 4 - 1) * 4);
  };
  auto put_rest = [&](int b) {
#pragma unroll
    for (int u = 0; u < kPieces; ++u) *(f32x4*)(small + (b & 1) * kSmall + min(tid + u * 64 * NW, kSmall / 4 - 1) * 4) = rest[u];
  };
  f32x4 done[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  uint2 gate[2] = {{0, 0}, {0, 0}};
  const float inv_v = 1.f / (float)a.vdim;
  const int out_at = (4 * g * (int)a.out_stride + h * dv + col0 + l16) * 2;
  auto rows_of = [&](int b) { return b < 0 ? 0 : min(2 * kBlock, sg.count - b * 2 * kBlock); };
  auto finish = [&](int b, int r, const f32x4& ss) {               // row 16 (r / 4) + 4 g + r % 4 of pair b; none of pair -1
    const BlockRows out(a.out, sg.row + b * 2 * kBlock, rows_of(b), a.out_stride);
    const float rs = __builtin_amdgcn_rsqf(ss[r & 3] * inv_v + a.eps);
    const uint32_t two = r & 2 ? gate[r / 4].y : gate[r / 4].x;
    out.st(out_at + (r / 4 * kBlock + (r & 3)) * (int)a.out_stride * 2, 0,
           done[r / 4][r & 3] * rs * nrm * fast_sigmoid(__uint_as_float(r & 1 ? two & 0xffff0000u : two << 16)));
  };
  u32x4 sp[3][J];                              // the state's planes, pairs of tiles
  auto split_state = [&](int kt) {
    const Planes x(S[kt][0]);
    const int at = (kt & 1) * 2;
    sp[0][kt >> 1][at] = x.hi.x, sp[0][kt >> 1][at + 1] = x.hi.y;
    sp[1][kt >> 1][at] = x.mid.x, sp[1][kt >> 1][at + 1] = x.mid.y;
    sp[2][kt >> 1][at] = x.lo.x, sp[2][kt >> 1][at + 1] = x.lo.y;
  };
  auto meet = [] {                             // LDS alone: what comes from memory and goes there stays on its way
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
#pragma unroll
  for (int u = 0; u < kRing; ++u) ask(0, u);
  ask_rest(0);
  ask_values(0);
#pragma unroll
  for (int kt = 0; kt < (J > 1 ? KT - 2 : KT); ++kt) split_state(kt);      // the last two beside the first products
#pragma unroll
  for (int u = 0; u < kMine; ++u) next_tile(0, u);
  put_rest(0);
  ask_rest(1);
#pragma unroll 1
  for (int b = 0; b < pairs; ++b) {
    meet();
    const float* const mine = small + (b & 1) * kSmall;
    const float* const pl = planes + (b & 1) * kPlanes + lane * 4;
    u32x4 W[2][3], Q[2][3];
    auto operands = [&](int n) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        W[n & 1][i] = *(const u32x4*)(pl + ((n / J * 2 * J + n % J) * 3 + i) * 256);
        if constexpr (!SUMS) Q[n & 1][i] = *(const u32x4*)(pl + (((n / J * 2 + 1) * J + n % J) * 3 + i) * 256);
      }
    };
    operands(0);
    f32x4 U[2] = {values[0], values[1]}, O[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    if (keeps) U[0] = U[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    ask_values(b + 1);
    f32x4 ss;
    uint2 next[2];
    if constexpr (!SUMS)
#pragma unroll
      for (int i = 0; i < 2; ++i) next[i] = *(const uint2*)(at_pair(b) + gates_at(dk, dv) + ((i * NW + wave) * 64 + lane) * 2);
    __builtin_amdgcn_sched_barrier(0);
    u32x4 left[2], up[3], u0[4], K[2][2][3];   // up: planes of U0 and U1, one contraction of 32
    uint2 left_lo[2];
    f32x4 dec[2][2];
    auto small_operands = [&](int i, int k) {
      left[0] = *(const u32x4*)(mine + i * kPairFloats + lane * 4);
      left_lo[0] = *(const uint2*)(mine + i * kPairFloats + 256 + lane * 2);
      left[1] = *(const u32x4*)(mine + k * kPairFloats + lane * 4);
      left_lo[1] = *(const uint2*)(mine + k * kPairFloats + 256 + lane * 2);
    };
    auto keys = [&](int j) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int k = 0; k < 3; ++k) K[j & 1][i][k] = *(const u32x4*)(pl + ((4 * J + 2 * j + i) * 3 + k) * 256);
        dec[j & 1][i] = *(const f32x4*)(mine + 4 * kPairFloats + 16 * (2 * j + i) + 4 * g);
      }
    };
    // What follows from U0: its planes, the second block's U and O.  Within the second half where that is long enough.
    auto split_first = [&] {
      const PlanePairs u(U[0]);
      u0[0] = u.hh, u0[1] = u.mm, u0[2] = u.ll, u0[3] = u.hm;
      up[0][0] = u.hh[0], up[0][1] = u.hh[1], up[1][0] = u.mm[0], up[1][1] = u.mm[1], up[2][0] = u.ll[0], up[2][1] = u.ll[1];
    };
    auto cross = [&] {
      const PlanePairs u(u0);
      if constexpr (SUMS) u.add(left[0], left_lo[0], U[1]);
      else u.add(left, left_lo, U[1], O[1]);
    };
    constexpr bool kLate = J < 4;
#pragma unroll
    for (int n = 0; n < 2 * J; ++n) {          // beside: the pair before is finished, the next one's planes are made
      const int half = n / J;
      if (n + 1 < 2 * J) operands(n + 1);
      else keys(0);
      if constexpr (!SUMS)
        if (n % J == 0) ss = block_squares_total<NW>(red + (((b - 1) & 1) * 2 + half) * NW * kBlock);
      if (!kLate && n == J + 1) small_operands(2, 3);
#pragma unroll
      for (int i = 2; i >= 0; --i)             // the smallest products first
#pragma unroll
        for (int k = 2 - i; k >= 0; --k) {
          U[half] = mfma_bf16(W[n & 1][i], sp[k][n % J], U[half]);
          if constexpr (!SUMS) O[half] = mfma_bf16(Q[n & 1][i], sp[k][n % J], O[half]);
        }
      if (J > 1 && n == 0) {
        split_state(KT - 2);
        split_state(KT - 1);
      }
      if constexpr (!SUMS)
#pragma unroll
        for (int r = n * 8 / (2 * J); r < (n + 1) * 8 / (2 * J); ++r) finish(b - 1, r, ss);
#pragma unroll
      for (int u = n * kMine / (2 * J); u < (n + 1) * kMine / (2 * J); ++u) next_tile(b + 1, u);
      if (!kLate && n == J) split_first();
      if (!kLate && n == J + 2) cross();
      spread_over_products<SUMS ? 6 : 12, 4>();
    }
    if constexpr (kLate) {
      small_operands(2, 3);
      split_first();
      cross();
    }
    put_rest(b + 1);
    ask_rest(b + 2);
    if constexpr (!SUMS) {
#pragma unroll
      for (int i = 0; i < 2; ++i) gate[i] = next[i];
      small_operands(0, 1);
    }
    S[0][0] *= dec[0][0];
    S[1][0] *= dec[0][1];
    const PlanePairs u1(U[1]);
    up[0][2] = u1.hh[0], up[0][3] = u1.hh[1], up[1][2] = u1.mm[0], up[1][3] = u1.mm[1], up[2][2] = u1.ll[0], up[2][3] = u1.ll[1];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < J; ++j) {              // beside: two tiles before are split, the next two decay, rows are squared
      if (j + 1 < J) {
        keys(j + 1);
        S[2 * j + 2][0] *= dec[(j + 1) & 1][0];
        S[2 * j + 3][0] *= dec[(j + 1) & 1][1];
      }
      if constexpr (!SUMS)
        if (j == 0) {
          PlanePairs(u0).add(left[0], left_lo[0], O[0]);
          u1.add(left[1], left_lo[1], O[1]);
        }
#pragma unroll
      for (int i = 2; i >= 0; --i)
#pragma unroll
        for (int k = 2 - i; k >= 0; --k)
#pragma unroll
          for (int t = 0; t < 2; ++t) S[2 * j + t][0] = mfma_bf16(K[j & 1][t][i], up[k], S[2 * j + t][0]);
      if (j > 0) {
        split_state(2 * j - 2);
        split_state(2 * j - 1);
      }
      if constexpr (!SUMS)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          if (j == min(i + 1, J - 1)) {
            f32x4 o[1] = {O[i]};
            block_squares<1>(o, red + ((b & 1) * 2 + i) * NW * kBlock, wave);
            done[i] = O[i];
          }
      spread_over_products<12, 4>();
    }
    if constexpr (J == 1) {
      split_state(KT - 2);
      split_state(KT - 1);
    }
  }
  meet();
  if constexpr (SUMS) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      if (keeps) {
        float* const to = between + dk * dk + ((kt * KT + wave) * 64 + (l16 >> 2) * 16 + 4 * g) * 4 + (l16 & 3);
#pragma unroll
        for (int r = 0; r < 4; ++r) to[r * 4] = S[kt][0][r];
      } else {
        *(f32x4*)(between + ((wave * KT + kt) * 64 + lane) * 4) = S[kt][0];
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const f32x4 ss = block_squares_total<NW>(red + (((pairs - 1) & 1) * 2 + i) * NW * kBlock);
#pragma unroll
    for (int r = 0; r < 4; ++r) finish(pairs - 1, 4 * i + r, ss);
  }
  if (!piece.last) return;
  store_state<KT, 1>(S, state, dv, col0);
  // the last inputs of the head's convolutions (runs are longer than a filter)
  const int taps = a.taps, cw = 2 * dk + dv, hk = h / (a.heads / a.kv_heads);
  char* const tail = (char*)a.conv_state + item * (taps - 1) * cw * 2;
  for (int i = tid; i < (taps - 1) * cw; i += blockDim.x) {
    const int e = i / cw, c = i - e * cw;
    const int at = c < dk ? hk * dk + c : (c < 2 * dk ? a.kv_heads * dk + hk * dk + c - dk : 2 * a.kv_heads * dk + h * dv + c - 2 * dk);
    Elem<BF16>::st(tail, i, Elem<BF16>::ld(a.in, (int64_t)(whole.row + max(whole.count - (taps - 1) + e, 0)) * a.in_stride + at));
  }
}

template <typename F> int launch_kernel(F* kernel, int64_t groups, int threads, int smem, const RunArgs& ra, hipStream_t st) {
  if (smem > 60 * 1024 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, smem) != hipSuccess) {
    zp_set_error("delta_runs: cannot reserve %d bytes of LDS", smem);
    return ZP_EHIP;
  }
  hipLaunchKernelGGL(kernel, dim3((unsigned)groups), dim3(threads), smem, st, ra);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}
template <int KT, int NW> int launch_blocks(const RunArgs& ra, hipStream_t st) {
  constexpr int smem = PairStage<KT, NW>::kBytes;
  const int64_t units = (int64_t)ra.d.seg.n * ra.d.heads;
  if constexpr (KT == NW)
    if (ra.pieces.blocks) {
      int rc = launch_kernel(delta_blocks_kernel<KT, NW, true>, units * (ra.pieces.most - 1) * 2, 64 * NW, smem, ra, st);
      if (rc == ZP_OK) rc = launch_kernel(delta_states_kernel<KT, KT / 2>, units * 2, 32 * KT, KT * KT / 2 * 3072, ra, st);
      if (rc != ZP_OK) return rc;
    }
  return launch_kernel(delta_blocks_kernel<KT, NW, false>, units * ra.pieces.most, 64 * NW, smem, ra, st);
}
template <int KT> int launch_blocks(const RunArgs& ra, hipStream_t st) {
  switch (ra.d.dv / 32) {
    case 1: return launch_blocks<KT, 2>(ra, st);
    case 2: return launch_blocks<KT, 4>(ra, st);
    case 3: return launch_blocks<KT, 6>(ra, st);
    default: return launch_blocks<KT, 8>(ra, st);
  }
}

template <int TAPS, bool PROJECTED> int launch_prepare(const RunArgs& ra, int longest, hipStream_t st) {
  const zp_delta& a = ra.d;
  const size_t smem = sizeof(float) * 2 * kPrepareHalf;
  if (smem > 60 * 1024 && hipFuncSetAttribute((const void*)delta_prepare_kernel<TAPS, PROJECTED>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                              (int)smem) != hipSuccess) {
    zp_set_error("delta_runs: cannot reserve %zu bytes of LDS", smem);
    return ZP_EHIP;
  }
  hipLaunchKernelGGL((delta_prepare_kernel<TAPS, PROJECTED>), dim3((unsigned)((longest + 2 * kBlock - 1) / (2 * kBlock)), (unsigned)a.heads, (unsigned)a.seg.n),
                     dim3(512), smem, st, ra);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}

int launch_runs(const RunArgs& ra, int longest, hipStream_t st) {
  const zp_delta& a = ra.d;
  const int rc = ra.low_weights ? (a.taps <= 4 ? launch_prepare<4, true>(ra, longest, st) : launch_prepare<kMaxTaps, true>(ra, longest, st))
                                : (a.taps <= 4 ? launch_prepare<4, false>(ra, longest, st) : launch_prepare<kMaxTaps, false>(ra, longest, st));
  if (rc != ZP_OK) return rc;
  switch (a.dk) {
    case 32: return launch_blocks<2>(ra, st);
    case 64: return launch_blocks<4>(ra, st);
    default: return launch_blocks<8>(ra, st);
  }
}

}  // namespace

static int64_t pairs_bytes(int64_t rows, int64_t segments, int64_t heads, int dk, int dv) {
  return (rows / (2 * kBlock) + segments) * heads * pair_floats(dk, dv) * 4;
}

// A piece as dear as when its states took 5.7 us: with 18, shorter pieces of 500 and 700 tokens, 16 heads, take 93 and 101 us instead
// of 86 and 98, what begins and ends them being paid more often.
constexpr PieceCost kCost = {2, 8, 72, 24};

// With room for the states between pieces of few heads' runs, whatever the longest run.
extern "C" int64_t zp_delta_runs_workspace(int32_t rows, int32_t segments, int32_t heads, int32_t dk, int32_t dv) {
  if (rows < 0 || segments < 0 || heads <= 0 || dk <= 0 || dv <= 0) return -1;
  return pairs_bytes(rows, segments, heads, dk, dv) +
         (dk == dv && dk <= 128 ? most_states(rows, segments, heads, kCost) * piece_floats(dk) * 4 : 0);
}

static int delta_runs(const zp_delta* args, const void* low_weights, int low_at, int a_rank, int rank, int first_row, int longest,
                      void* workspace, int64_t workspace_bytes, int dtype, void* stream) {
  ZP_REQUIRE(args, "delta_runs: null arguments");
  const zp_delta& a = *args;
  ZP_REQUIRE(a.seg.n >= 0 && a.heads > 0 && a.kv_heads > 0 && a.heads % a.kv_heads == 0 && a.vdim > 0 && a.vdim <= a.dv &&
                 a.seg.num_slots > 0 && a.out_stride >= (int64_t)a.heads * a.dv && first_row >= 0 && longest >= 0 &&
                 first_row <= a.seg.num_rows, "delta_runs: bad dims");
  if (dtype != ZP_BF16 || (a.dk != 32 && a.dk != 64 && a.dk != 128) || a.dv % 32 || a.dv > 128 || a.taps < 1 || a.taps > kMaxTaps || a.heads > 65535 ||
      a.seg.n > 65535 || a.in_stride % 8 || a.out_stride >= (1 << 24) || (!low_weights && (a.low_stride % 8 || a.low_stride >= (1 << 24)))) {
    zp_set_error("delta_runs: bfloat16, head sizes %d (32, 64, 128) and %d (a multiple of 32, <= 128), %d taps (1 .. %d) unsupported",
                 a.dk, a.dv, a.taps, kMaxTaps);
    return ZP_EUNSUPPORTED;
  }
  if (a.seg.n == 0 || longest == 0) return ZP_OK;
  ZP_REQUIRE(a.in && (a.low || low_weights) && a.filters && a.a_log && a.dt_bias && a.norm && a.state && (a.conv_state || a.taps == 1) && a.out &&
                 a.seg.rows && a.seg.counts && a.seg.slots && a.seg.starts && aligned16(a.state) && aligned16(a.in) && (low_weights ? aligned16(low_weights) : aligned16(a.low)) &&
                 aligned16(a.dt_bias) && aligned16(workspace),
             "delta_runs: null or unaligned pointer");
  const int64_t rows = a.seg.num_rows - first_row, whole = pairs_bytes(rows, a.seg.n, a.heads, a.dk, a.dv);
  ZP_REQUIRE(workspace && workspace_bytes >= whole, "delta_runs: workspace too small");
  RunArgs ra = {a, (float*)workspace, first_row, {}, (const uint16_t*)low_weights, low_at, rank, a_rank};
  if (a.dk == a.dv) ra.pieces = pieces_of(rows, a.seg.n, a.heads, longest, kCost, 2, (workspace_bytes - whole) / 4 / piece_floats(a.dk));
  ra.pieces.states = (float*)workspace + whole / 4;
  ra.d.seg.max_count = longest;               // no segment has more blocks than were prepared
  return launch_runs(ra, longest, (hipStream_t)stream);
}

extern "C" int zp_delta_runs(const zp_delta* args, int32_t first_row, int32_t longest, void* workspace,
                             int64_t workspace_bytes, int32_t dtype, void* stream) {
  return delta_runs(args, nullptr, 0, 0, 0, first_row, longest, workspace, workspace_bytes, dtype, stream);
}

extern "C" int zp_delta_runs_projected(const zp_delta* args, const void* low_weights, int32_t low_at, int32_t a_rank, int32_t rank,
                                       int32_t first_row, int32_t longest, void* workspace, int64_t workspace_bytes, int32_t dtype,
                                       void* stream) {
  ZP_REQUIRE(args && low_weights && low_at >= 0 && a_rank >= 0 && rank >= a_rank && low_at + (int64_t)rank <= args->in_stride,
             "delta_runs: bad low-rank products");
  if (low_at % 8 || rank % 8 || rank > kLowRank || (a_rank + 31) / 32 > kLowSteps || (rank + 31) / 32 - a_rank / 32 > kLowSteps) {
    zp_set_error("delta_runs: low-rank products of %d and %d columns from column %d on unsupported (multiples of 8, up to 128)", a_rank,
                 rank - a_rank, low_at);
    return ZP_EUNSUPPORTED;
  }
  return delta_runs(args, low_weights, low_at, a_rank, rank, first_row, longest, workspace, workspace_bytes, dtype, stream);
}
