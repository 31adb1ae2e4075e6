// Gated delta rule (delta.hip) over long runs, 16 tokens at a time.  With G_t the product of the block's
// decays up to token t, per key channel, a block is
//
//   A[t, s] = beta_t sum_c k_t k_s G_t / G_s (s < t),   P[t, s] = sum_c q_t k_s G_t / G_s (s <= t)
//   (1 + A) [U0 | W] = beta [V | G k],   U = U0 - W S,   O = (G q) S + P U
//   S <- G_15 S + sum_s (G_15 / G_s) k_s u_s^T
//
// delta_prepare computes everything without S for all blocks at once and leaves it in the order of the
// matrix operands; ratios of decays are running products of the decays themselves, so nothing is divided
// and nothing overflows.  delta_blocks walks a head's blocks with S in registers.  All fp32; projections in
// bfloat16.
#include "blocks.h"

namespace {

constexpr int kMaxTaps = 8;

struct RunArgs {
  zp_delta d;
  float* ws;
  int row0;      // first token row of the first segment
  Pieces pieces;
};

// [-W | G q] and the keys as left operands, U0 as a result tile, P's planes, the block's decays; whole KBs
__host__ __device__ inline constexpr int block_floats(int dk, int dv) {
  return (kBlock * (3 * dk + dv) + kPairFloats + dk + 255) / 256 * 256;
}

template <int TAPS>
__global__ __launch_bounds__(256, 4) void delta_prepare_kernel(RunArgs ra) {
  extern __shared__ __align__(16) float lds[];
  const zp_delta& a = ra.d;
  constexpr int ld = 132;                      // every row: reads across tokens meet no conflicts, offsets are constants
  const int dk = a.dk, dv = a.dv, taps = a.taps;
  const Segment sg = segment_of(a.seg, blockIdx.z);
  const int t0 = blockIdx.x * kBlock;
  if (t0 >= sg.count || sg.row < ra.row0) return;
  const int cnt = min(kBlock, sg.count - t0);
  const int h = blockIdx.y, hk = h / (a.heads / a.kv_heads);
  float* const qs = lds;                       // [16][ld], later G q
  float* const ks = qs + kBlock * ld;
  float* const gs = ks + kBlock * ld;          // decays, later -W
  float* const vs = gs + kBlock * ld;
  float* const As = vs + kBlock * ld;          // [16][16]
  float* const Ps = As + kBlock * kBlock;      // [16][16]
  float* const beta = Ps + kBlock * kBlock;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int cw = 2 * dk + dv;
  const char* const tail = (const char*)a.conv_state + ((int64_t)sg.slot * a.heads + h) * (taps - 1) * cw * 2;
  const int channels = 2 * a.kv_heads * dk + a.heads * dv;
  auto place = [&](int c) -> int {
    return c < dk ? hk * dk + c : (c < 2 * dk ? a.kv_heads * dk + hk * dk + c - dk : 2 * a.kv_heads * dk + h * dv + c - 2 * dk);
  };
  // ---- requests first: the decays' pre-activations (two pieces a thread at most), the step sizes'
  const int piece_bits = 31 - __builtin_clz(dk / 4);           // pieces of four channels: 8, 16 or 32 a row
  f32x4 z[2], zb[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int i = tid + u * 256, t = min(i >> piece_bits, cnt - 1), c = (i & ((1 << piece_bits) - 1)) * 4;
    z[u] = load4<BF16>(a.low, (int64_t)(sg.row + t0 + t) * a.low_stride + h * dk + c);
    zb[u] = *(const f32x4*)(a.dt_bias + h * dk + c);
  }
  const float b_in = tid < cnt ? Elem<BF16>::ld(a.in, (int64_t)(sg.row + t0 + tid) * a.in_stride + a.b_at + h) : 0.f;
  const float rate = __expf(a.a_log[h]);
  // ---- convolutions: a thread's two channels, the block's 16 tokens from a sliding window.  Rows behind the run's end read
  // as zero, and those before its beginning too, unless they come from the history.
  const int row_bytes = (int)a.in_stride * 2;
  const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const char*)a.in + (int64_t)(sg.row + t0) * row_bytes), 0, cnt * row_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t before = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const char*)a.in + (int64_t)(sg.row + t0 - (TAPS - 1)) * row_bytes), 0, t0 > 0 ? (TAPS - 1) * row_bytes : 0, 0x00020000);
  if (const int c = 2 * tid; c < cw) {         // at most 384 channels
    const int at = place(c);
    uint32_t x[kBlock + TAPS - 1];             // two channels' bf16
#pragma unroll
    for (int i = 0; i < kBlock + TAPS - 1; ++i)
      x[i] = (uint32_t)(i < TAPS - 1 ? __builtin_amdgcn_raw_buffer_load_b32(before, at * 2, i * row_bytes, 0)
                                     : __builtin_amdgcn_raw_buffer_load_b32(rows, at * 2, (i - (TAPS - 1)) * row_bytes, 0));
    float f[2][TAPS];
#pragma unroll
    for (int j = 0; j < TAPS; ++j)                            // f[.][j]: j tokens back
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
    float* const dst = c < dk ? qs + c : (c < 2 * dk ? ks + c - dk : vs + c - 2 * dk);
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
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int i = tid + u * 256, t = i >> piece_bits, c = (i & ((1 << piece_bits) - 1)) * 4;
    if (t < kBlock) {
      f32x4 g;
#pragma unroll
      for (int e = 0; e < 4; ++e) g[e] = t < cnt ? __expf(-rate * fast_softplus(z[u][e] + zb[u][e])) : 1.f;
      *(f32x4*)(gs + t * ld + c) = g;
    }
  }
  if (tid < kBlock) beta[tid] = tid < cnt ? fast_sigmoid(b_in) : 0.f;
  if (tid < 2 * kBlock * kBlock / 4) *(f32x4*)(As + tid * 4) = f32x4{0.f, 0.f, 0.f, 0.f};       // and Ps behind it
  __syncthreads();
  // ---- unit vectors: a wave its four tokens, 16 lanes each
  {
    const int t = wave * 4 + (lane >> 4), l16 = lane & 15, pieces = dk / 4;
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
  // ---- A and P: 16 lanes walk k_s down the tokens from s on, in pieces of four channels.  A wave takes four
  // neighbours, so that it starts at the first of them; which four changes with the block, as the waves' shares differ (all
  // tokens for every s: 1135 us for 8 prompts of 2048 tokens, 32 heads, with the kernel below, now 1100).
  {
    const int first = 4 * ((wave + blockIdx.x) & 3), l16 = lane & 15, s = first + (lane >> 4), pieces = dk / 4;
    int at[2];
    f32x4 kk[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int pc = l16 + 16 * p;
      at[p] = min(pc, pieces - 1) * 4;
      kk[p] = *(const f32x4*)(ks + s * ld + at[p]);
      if (pc >= pieces) kk[p] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // Two tokens at a time, four sums over 16 lanes: lanes 8 .. 15 keep those of P, of each eight the upper half the second
    // token's (eleven additions and choices instead of sixteen additions, one store instead of four).
    const bool is_p = l16 & 8, second = l16 & 4;
    float* const to = (is_p ? Ps : As) + s;
    auto tokens = [&](int t, bool all) {       // all: they lie behind the four
      float sa[2], sp[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        f32x4 pa = {0.f, 0.f, 0.f, 0.f}, pp = pa;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const f32x4 gt = *(const f32x4*)(gs + (t + u) * ld + at[p]);
#pragma unroll
          for (int e = 0; e < 4; ++e) kk[p][e] *= all || t + u > s ? gt[e] : 1.f;
          pa += kk[p] * *(const f32x4*)(ks + (t + u) * ld + at[p]);
          pp += kk[p] * *(const f32x4*)(qs + (t + u) * ld + at[p]);
        }
        sa[u] = (pa[0] + pa[1]) + (pa[2] + pa[3]);
        sp[u] = (pp[0] + pp[1]) + (pp[2] + pp[3]);
        sa[u] += dpp_row_ror<8>(sa[u]);
        sp[u] += dpp_row_ror<8>(sp[u]);
        sa[u] = is_p ? sp[u] : sa[u];
        sa[u] += half_row_mirror(sa[u]);
      }
      const float x = quad_sum(second ? sa[1] : sa[0]);
      const int mine = t + second;
      const float by = is_p ? 1.f : beta[mine];
      if (all || (is_p ? mine >= s : mine > s)) to[mine * kBlock] = x * by;
    };
#pragma unroll
    for (int u = 0; u < 4; u += 2) tokens(first + u, false);
#pragma unroll 1
    for (int t = first + 4; t < kBlock; t += 2) tokens(t, true);
  }
  __syncthreads();
  // ---- columns: forward substitution, and the block's decays.  A thread reads and writes its own column only.
  const int64_t base = (block_slot(ra.row0, sg, blockIdx.z, blockIdx.x) * a.heads + h) * block_floats(dk, dv);
  float* const oWQ = ra.ws + base;             // [2][dk / 16][64 lanes][4]
  float* const oK = oWQ + 2 * kBlock * dk;     // [dk / 16][64][4]
  float* const oU = oK + kBlock * dk;          // [dv / 16][64][4]
  float* const oP = oU + kBlock * dv;          // [64][hi 4, mid 4], [64][lo 4]
  float* const oG = oP + kPairFloats;          // [dk]
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
  for (int c = tid; c < dk; c += 256) {
    float G = 1.f;
#pragma unroll
    for (int t = 0; t < kBlock; ++t) {
      G *= gs[t * ld + c];
      qs[t * ld + c] *= G;
      substitute(t, beta[t] * ks[t * ld + c] * G);
    }
    oG[c] = G;
    asm volatile("" ::: "memory");            // keys and decays are read again rather than kept
    float R = 1.f;
#pragma unroll
    for (int g = 3; g >= 0; --g) {
      f32x4 x;
#pragma unroll
      for (int r = 3; r >= 0; --r) {
        const int t = 4 * g + r;
        x[r] = ks[t * ld + c] * R;
        R *= gs[t * ld + c];
        gs[t * ld + c] = -w[t];
      }
      *(f32x4*)(oK + ((c >> 4) * 64 + g * 16 + (c & 15)) * 4) = x;
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  for (int v = (tid + 256 - dk) % 256; v < dv; v += 256) {      // on the threads the keys leave free, as far as they go
#pragma unroll
    for (int t = 0; t < kBlock; ++t) substitute(t, beta[t] * vs[t * ld + v]);
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *(f32x4*)(oU + ((v >> 4) * 64 + g * 16 + (v & 15)) * 4) = f32x4{w[4 * g], w[4 * g + 1], w[4 * g + 2], w[4 * g + 3]};
  }
  if (tid < 64) {
    const Planes x(*(const f32x4*)(Ps + (tid & 15) * kBlock + (tid >> 4) * 4));
    *(u32x4*)(oP + tid * 4) = u32x4{x.hi.x, x.hi.y, x.mid.x, x.mid.y};
    *(uint2*)(oP + 256 + tid * 2) = x.lo;
  }
  __syncthreads();
  for (int i = tid; i < 2 * kBlock * dk / 4; i += 256) {       // lane (g, row) of tile kt: columns 16 kt + 4 g ..
    const int tile = i >> 6, l = i & 63, kt = tile & (dk / 16 - 1);
    *(f32x4*)(oWQ + i * 4) = *(const f32x4*)((tile < dk / 16 ? gs : qs) + (l & 15) * ld + kt * 16 + (l >> 4) * 4);
  }
}

// ------------------------------------------------------------------ runs in pieces, of heads with as many keys as values
// A piece keeps M S of a state S before it, M the product of its blocks' (diag(G_15) - keys^T W).  Its columns walk through
// the piece as those of a state do, from one on, with nothing of the values.  A piece's state: its sums, or the state before
// it, then M as a left operand, [rows / 16][columns / 16][64 lanes][4].
__host__ __device__ inline constexpr int piece_floats(int dk) { return 2 * dk * dk; }

// From sums to the states before the pieces, in place; a wave 16 columns.  The products are those of the blocks, M split by
// all waves together while the piece before is worked on: 2.4 us a piece.
template <int KT>
__global__ __launch_bounds__(64 * KT, 2) void delta_states_kernel(RunArgs ra) {
  extern __shared__ __align__(16) float planes[];              // [rows / 16][pairs of columns / 16][3][64 lanes][4]
  constexpr int dk = 16 * KT, J = KT / 2;
  const zp_delta& a = ra.d;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = blockIdx.x % a.heads, seg = blockIdx.x / a.heads;
  const Segment whole = segment_of(a.seg, seg);
  if (whole.count <= 0 || whole.row < ra.row0) return;
  f32x4 S[KT][1], x[KT], add[KT];
  load_state<KT, 1>(S, a.state + ((int64_t)whole.slot * a.heads + h) * ((int64_t)dk * dk), dk, wave * 16, whole.start == 0);
  const int tokens = ra.pieces.blocks * kBlock, count = (whole.count + tokens - 1) / tokens;
  const int64_t stride = (int64_t)a.heads * piece_floats(dk);
  float* const at = ra.pieces.states + Piece(ra.pieces, ra.row0, whole, seg, 0).slot * stride + (int64_t)h * piece_floats(dk) + lane * 4;
  auto load = [&](int c) {                                     // this wave's columns of M, for all waves
#pragma unroll
    for (int t = 0; t < KT; ++t) x[t] = *(const f32x4*)(at + c * stride + dk * dk + (t * KT + wave) * 256);
  };
  auto meet = [] {                                             // LDS alone: what comes from memory and goes there stays on its way
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto load_sums = [&](int c, int t) { add[t] = *(const f32x4*)(at + c * stride + (wave * KT + t) * 256); };
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
      for (int t = 0; t < KT; ++t) {
        const Planes p(x[t]);
        float* const to = planes + (t * J + (wave >> 1)) * 768 + lane * 4 + (wave & 1) * 2;
        *(uint2*)to = p.hi;
        *(uint2*)(to + 256) = p.mid;
        *(uint2*)(to + 512) = p.lo;
      }
      load(min(c + 1, count - 2));
    }
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      *(f32x4*)(at + c * stride + (wave * KT + kt) * 256) = S[kt][0];
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

// A head's blocks, one after the other, a wave 16 columns of the state.  On the fp32 matrix cores the products would be the
// bound (208 of 32 cycles a block on each SIMD, which keep its vector units idle as well), so operands are split into
// three bf16 planes: the products that count take a quarter of that, beside the vector units.  The state is split
// where it is updated, what comes from memory by all waves together, a block ahead and under the products with the state;
// rows are normed and stored behind the next meeting of the waves, which the norm needs too.  What bounds it now is a wave's
// chain of work: two per SIMD are all there are (twice the columns per wave, one per SIMD: 2 to 12 % more time in all).
// 8 prompts of 2048 tokens, 32 heads of 128 x 128, with the kernel above: 1161 -> 1106 us, one of them 566 -> 491; error of the
// state against 64 bits 4.0e-7 -> 3.6e-7 of its size.
// SUMS: no state comes in and no rows go out; every second workgroup takes what the piece keeps, where values are none.
template <int KT, int NW, bool SUMS>
__global__ __launch_bounds__(64 * NW, 2) void delta_blocks_kernel(RunArgs ra) {
  extern __shared__ __align__(16) float lds[];
  const zp_delta& a = ra.d;
  constexpr int dk = 16 * KT, dv = 16 * NW, size = block_floats(dk, dv), J = KT / 2;
  constexpr int kSplit = 3 * kBlock * dk, kRest = size - kSplit;      // floats of a block: operands to be split, the others
  constexpr int kP = kBlock * dv, kG = kP + kPairFloats;              // in the rest, behind U0
  constexpr int kPlanes = 3 * KT * 384, kMine = ((SUMS ? 2 : 3) * KT + NW - 1) / NW;    // floats of a block's planes; tiles of a wave
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  float* const split = lds;                    // [2][kSplit]
  float* const rest = split + 2 * kSplit;      // [3][kRest]
  float* const planes = rest + 3 * kRest;      // [2][kPlanes]
  float* const red = planes + 2 * kPlanes;     // [2][NW * 16]
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
  const float* const base = ra.ws + (block_slot(ra.row0, sg, seg, 0) * a.heads + h) * size;
  const int64_t stride = (int64_t)a.heads * size;
  const int blocks = (sg.count + kBlock - 1) / kBlock;
  auto tile_at = [](int i) { return SUMS && i >= KT ? i + KT : i; };      // without those of G q
  auto request = [&](int b) {                  // a block behind the last: nothing is read
    const StageLoads from(base + b * stride, b < blocks ? size * 4 : 0);
    constexpr int kKBs = size / 256 - (SUMS ? KT : 0);
#pragma unroll
    for (int u = 0; u < (kKBs + NW - 1) / NW; ++u) {
      const int i = tile_at(min(wave + u * NW, kKBs - 1));         // the last may come twice
      float* const to = i < kSplit / 256 ? split + (b & 1) * kSplit + i * 256 : rest + b % 3 * kRest + (i * 256 - kSplit);
      from.ld(to, lane * 16, i * 1024);
    }
  };
  // Planes of a block's tiles: for pairs of those of -W and of G q [3][64 lanes][two tiles' 4], for those of keys
  // [64][hi 4, mid 4], [64][lo 4].  A wave's tile u; the last may be made twice.
  auto tile_of = [&](int b, int u) {
    return *(const f32x4*)(split + (b & 1) * kSplit + tile_at(min(wave + u * NW, (SUMS ? 2 : 3) * KT - 1)) * 256 + lane * 4);
  };
  auto put_planes = [&](int b, int u, const f32x4& x) {
    const int i = tile_at(min(wave + u * NW, (SUMS ? 2 : 3) * KT - 1));
    const int key = i >= 2 * KT;               // multiplied, not branched on: the products beside stay in one stretch
    float* const to = planes + (b & 1) * kPlanes + (i >> 1) * 768 + (i & 1) * (2 + 382 * key) + lane * 4;
    const Planes p(x);
    *(uint2*)to = p.hi;
    *(uint2*)(to + 256 - 254 * key) = p.mid;
    *(uint2*)(to + 512 - (256 + lane * 2) * key) = p.lo;
  };
  f32x4 done = {0.f, 0.f, 0.f, 0.f};
  uint16_t gate[4] = {0, 0, 0, 0};
  const float inv_v = 1.f / (float)a.vdim;
  const int out_at = (4 * g * (int)a.out_stride + h * dv + col0 + l16) * 2;
  const int low_at = (4 * g * (int)a.low_stride + a.g_at + h * dv + col0 + l16) * 2;
  auto finish = [&](int b, int r, const f32x4& ss) {               // row r of block b, whose squares are ss; none of block -1
    const int cnt = b < 0 ? 0 : min(kBlock, sg.count - b * kBlock);
    const BlockRows out(a.out, sg.row + b * kBlock, cnt, a.out_stride);
    const float rs = __builtin_amdgcn_rsqf(ss[r] * inv_v + a.eps);
    out.st(out_at + r * (int)a.out_stride * 2, 0, done[r] * rs * nrm * fast_sigmoid(bf16_bits_to_float(gate[r])));
  };
  u32x4 sp[3][J];                              // the state's planes, pairs of tiles
  auto split_state = [&](int kt) {
    const Planes x(S[kt][0]);
    const int at = (kt & 1) * 2;
    sp[0][kt >> 1][at] = x.hi.x, sp[0][kt >> 1][at + 1] = x.hi.y;
    sp[1][kt >> 1][at] = x.mid.x, sp[1][kt >> 1][at + 1] = x.mid.y;
    sp[2][kt >> 1][at] = x.lo.x, sp[2][kt >> 1][at + 1] = x.lo.y;
  };
  request(0);
  __builtin_amdgcn_s_waitcnt(0);               // the state is there: the loop's first use of it must not wait in every pass
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) split_state(kt);
  wait_and_meet();
  request(1);
#pragma unroll
  for (int u = 0; u < kMine; ++u) put_planes(0, u, tile_of(0, u));
#pragma unroll 1
  for (int b = 0; b < blocks; ++b) {
    wait_and_meet();
    const float* const mine = rest + b % 3 * kRest;
    const float* const pl = planes + (b & 1) * kPlanes + lane * 4;
    u32x4 W[2][3], Q[2][3];
    auto operands = [&](int j) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        W[j & 1][i] = *(const u32x4*)(pl + (j * 3 + i) * 256);
        if constexpr (!SUMS) Q[j & 1][i] = *(const u32x4*)(pl + ((J + j) * 3 + i) * 256);
      }
    };
    operands(0);
    f32x4 U = *(const f32x4*)(mine + wave * 256 + lane * 4), O = {0.f, 0.f, 0.f, 0.f};
    if (keeps) U = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 tile = tile_of(b + 1, 0), ss;
    if constexpr (!SUMS) ss = block_squares_total<NW>(red + ((b - 1) & 1) * NW * kBlock);
    request(b + 2);
    const int cnt = min(kBlock, sg.count - b * kBlock);
    const BlockRows low(a.low, sg.row + b * kBlock, cnt, a.low_stride);
    uint16_t next[4];
    if constexpr (!SUMS)
#pragma unroll
    for (int r = 0; r < 4; ++r) next[r] = low.ld(low_at + r * (int)a.low_stride * 2, 0);
    __builtin_amdgcn_sched_barrier(0);
    u32x4 K[2][2];
    uint2 Kl[2][2];
    f32x4 dec[2][2];
    auto keys = [&](int j) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float* const at = planes + (b & 1) * kPlanes + (2 * KT + 2 * j + i) * 384;
        K[j & 1][i] = *(const u32x4*)(at + lane * 4);
        Kl[j & 1][i] = *(const uint2*)(at + 256 + lane * 2);
        dec[j & 1][i] = *(const f32x4*)(mine + kG + 16 * (2 * j + i) + 4 * g);
      }
    };
#pragma unroll
    for (int j = 0; j < J; ++j) {              // beside: the block before is finished, the next one's planes are made
      if (j + 1 < J) operands(j + 1);
      else keys(0);
#pragma unroll
      for (int i = 2; i >= 0; --i)             // the smallest products first
#pragma unroll
        for (int k = 2 - i; k >= 0; --k) {
          U = mfma_bf16(W[j & 1][i], sp[k][j], U);
          if constexpr (!SUMS) O = mfma_bf16(Q[j & 1][i], sp[k][j], O);
        }
      if constexpr (!SUMS)
#pragma unroll
        for (int r = j * 4 / J; r < (j + 1) * 4 / J; ++r) finish(b - 1, r, ss);
#pragma unroll
      for (int u = j * kMine / J; u < (j + 1) * kMine / J; ++u) {
        put_planes(b + 1, u, tile);
        if (u + 1 < kMine) tile = tile_of(b + 1, u + 1);
      }
      spread_over_products<SUMS ? 6 : 12, 4>();
    }
    u32x4 P;
    uint2 Pl;
    if constexpr (!SUMS) {
#pragma unroll
      for (int r = 0; r < 4; ++r) gate[r] = next[r];
      P = *(const u32x4*)(mine + kP + lane * 4);
      Pl = *(const uint2*)(mine + kP + 256 + lane * 2);
    }
    const PlanePairs u(U);
    __builtin_amdgcn_sched_barrier(0);
    S[0][0] *= dec[0][0];
    S[1][0] *= dec[0][1];
#pragma unroll
    for (int j = 0; j < J; ++j) {              // beside: two tiles before are split, the next two decay
      if (j + 1 < J) {
        keys(j + 1);
        S[2 * j + 2][0] *= dec[(j + 1) & 1][0];
        S[2 * j + 3][0] *= dec[(j + 1) & 1][1];
      }
      u.add(K[j & 1], Kl[j & 1], S[2 * j][0], S[2 * j + 1][0]);
      if (j > 0) {
        split_state(2 * j - 2);
        split_state(2 * j - 1);
      }
      spread_over_products<8, 5>();
    }
    if constexpr (!SUMS) u.add(P, Pl, O);
    split_state(KT - 2);
    split_state(KT - 1);
#pragma unroll
    for (int i = 0; i < 3; ++i)                // here, not behind the squares
#pragma unroll
      for (int j = 0; j < J; ++j) settle(sp[i][j]);
    if constexpr (!SUMS) {
      f32x4 o[1] = {O};
      block_squares<1>(o, red + (b & 1) * NW * kBlock, wave);
      done = O;
    }
  }
  wait_and_meet();
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
  const f32x4 ss = block_squares_total<NW>(red + ((blocks - 1) & 1) * NW * kBlock);
#pragma unroll
  for (int r = 0; r < 4; ++r) finish(blocks - 1, r, ss);
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
  constexpr int kSplit = 3 * kBlock * 16 * KT;
  constexpr int smem = (3 * block_floats(16 * KT, 16 * NW) - kSplit + 2 * 3 * KT * 384 + 2 * NW * kBlock) * 4;
  const int64_t units = (int64_t)ra.d.seg.n * ra.d.heads;
  if constexpr (KT == NW)
    if (ra.pieces.blocks) {
      int rc = launch_kernel(delta_blocks_kernel<KT, NW, true>, units * (ra.pieces.most - 1) * 2, 64 * NW, smem, ra, st);
      if (rc == ZP_OK) rc = launch_kernel(delta_states_kernel<KT>, units, 64 * KT, KT * KT / 2 * 3072, ra, st);
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

template <int TAPS> int launch_prepare(const RunArgs& ra, int longest, hipStream_t st) {
  const zp_delta& a = ra.d;
  const size_t smem = sizeof(float) * (kBlock * 4 * 132 + 2 * kBlock * kBlock + kBlock);
  if (smem > 60 * 1024 && hipFuncSetAttribute((const void*)delta_prepare_kernel<TAPS>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                              (int)smem) != hipSuccess) {
    zp_set_error("delta_runs: cannot reserve %zu bytes of LDS", smem);
    return ZP_EHIP;
  }
  hipLaunchKernelGGL((delta_prepare_kernel<TAPS>), dim3((unsigned)((longest + kBlock - 1) / kBlock), (unsigned)a.heads, (unsigned)a.seg.n),
                     dim3(256), smem, st, ra);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}

int launch_runs(const RunArgs& ra, int longest, hipStream_t st) {
  const zp_delta& a = ra.d;
  const int rc = a.taps <= 4 ? launch_prepare<4>(ra, longest, st) : launch_prepare<kMaxTaps>(ra, longest, st);
  if (rc != ZP_OK) return rc;
  switch (a.dk) {
    case 32: return launch_blocks<2>(ra, st);
    case 64: return launch_blocks<4>(ra, st);
    default: return launch_blocks<8>(ra, st);
  }
}

}  // namespace

static int64_t blocks_bytes(int64_t rows, int64_t segments, int64_t heads, int dk, int dv) {
  return (rows / kBlock + segments) * heads * block_floats(dk, dv) * 4;
}

constexpr PieceCost kCost = {2, 8, 60, 10};

// With room for the states between pieces of few heads' runs, whatever the longest run.
extern "C" int64_t zp_delta_runs_workspace(int32_t rows, int32_t segments, int32_t heads, int32_t dk, int32_t dv) {
  if (rows < 0 || segments < 0 || heads <= 0 || dk <= 0 || dv <= 0) return -1;
  return blocks_bytes(rows, segments, heads, dk, dv) +
         (dk == dv && dk <= 128 ? most_states(rows, segments, heads, kCost) * piece_floats(dk) * 4 : 0);
}

extern "C" int zp_delta_runs(const zp_delta* args, int32_t first_row, int32_t longest, void* workspace,
                             int64_t workspace_bytes, int32_t dtype, void* stream) {
  ZP_REQUIRE(args, "delta_runs: null arguments");
  const zp_delta& a = *args;
  ZP_REQUIRE(a.seg.n >= 0 && a.heads > 0 && a.kv_heads > 0 && a.heads % a.kv_heads == 0 && a.vdim > 0 && a.vdim <= a.dv &&
                 a.seg.num_slots > 0 && a.out_stride >= (int64_t)a.heads * a.dv && first_row >= 0 && longest >= 0 &&
                 first_row <= a.seg.num_rows, "delta_runs: bad dims");
  if (dtype != ZP_BF16 || (a.dk != 32 && a.dk != 64 && a.dk != 128) || a.dv % 32 || a.dv > 128 || a.taps < 1 || a.taps > kMaxTaps || a.heads > 65535 ||
      a.seg.n > 65535 || a.in_stride % 8 || a.low_stride % 8 || a.out_stride >= (1 << 24) || a.low_stride >= (1 << 24)) {
    zp_set_error("delta_runs: bfloat16, head sizes %d (32, 64, 128) and %d (a multiple of 32, <= 128), %d taps (1 .. %d) unsupported",
                 a.dk, a.dv, a.taps, kMaxTaps);
    return ZP_EUNSUPPORTED;
  }
  if (a.seg.n == 0 || longest == 0) return ZP_OK;
  ZP_REQUIRE(a.in && a.low && a.filters && a.a_log && a.dt_bias && a.norm && a.state && (a.conv_state || a.taps == 1) && a.out &&
                 a.seg.rows && a.seg.counts && a.seg.slots && a.seg.starts && aligned16(a.state) && aligned16(a.in) && aligned16(a.low) &&
                 aligned16(a.dt_bias) && aligned16(workspace),
             "delta_runs: null or unaligned pointer");
  const int64_t rows = a.seg.num_rows - first_row, whole = blocks_bytes(rows, a.seg.n, a.heads, a.dk, a.dv);
  ZP_REQUIRE(workspace && workspace_bytes >= whole, "delta_runs: workspace too small");
  RunArgs ra = {a, (float*)workspace, first_row, {}};
  if (a.dk == a.dv) ra.pieces = pieces_of(rows, a.seg.n, a.heads, longest, kCost, (workspace_bytes - whole) / 4 / piece_floats(a.dk));
  ra.pieces.states = (float*)workspace + whole / 4;
  ra.d.seg.max_count = longest;               // no segment has more blocks than were prepared
  return launch_runs(ra, longest, (hipStream_t)stream);
}
