// Linear attention with decay (linear.hip) over long runs, 16 tokens at a time.  With G_t the product of the
// block's decays up to token t, per key channel, a block is
//
//   P[t, s] = sum_c q_t k_s G_t / G_s (s <= t),   O = (G q) S + P V,   S <- G_15 S + sum_s (G_15 / G_s) k_s v_s^T
//
// linear_prepare turns q and k, takes the decays, and computes everything without S for all blocks at once, in
// the order of the matrix operands; ratios of decays are running products of the decays themselves, so nothing
// is divided and nothing overflows.  linear_blocks walks a head's blocks with S in registers.  All fp32;
// projections in bfloat16.
#include "blocks.h"
#include "linear.h"
#include <type_traits>

namespace {

struct RunArgs {
  zp_linear d;
  float* ws;
  int row0;      // first token row of the first segment
  Pieces pieces;
};

// G q and the keys as left operands, P's planes, the block's decays; whole KBs
__host__ __device__ inline constexpr int block_floats(int dk) {
  return (2 * kBlock * dk + kPairFloats + dk + 255) / 256 * 256;
}

__global__ __launch_bounds__(256, 4) void linear_prepare_kernel(RunArgs ra) {
  const zp_linear& a = ra.d;
  constexpr int ld = 132;                      // every row: reads across tokens meet no conflicts, offsets are constants
  __shared__ __align__(16) float qs[kBlock * ld], ks[kBlock * ld], gs[kBlock * ld], Ps[kBlock * kBlock];
  const int dk = a.dk, half = a.rot / 2;
  const Segment sg = segment_of(a.seg, blockIdx.z);
  const int t0 = blockIdx.x * kBlock;
  if (t0 >= sg.count || sg.row < ra.row0) return;
  const int cnt = min(kBlock, sg.count - t0);
  const int h = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float fixed = a.low ? 1.f : a.decay[h];
#pragma unroll
  for (int u = 0; u < 2; ++u) {                // dk <= 128: two pieces a thread at most
    const int i = tid + u * 256, t = i / (dk / 4), c = (i - t * (dk / 4)) * 4;
    if (t >= kBlock) continue;
    f32x4 q = {0.f, 0.f, 0.f, 0.f}, k = q, g = {1.f, 1.f, 1.f, 1.f};
    if (t < cnt) {
      const int64_t row = sg.row + t0 + t;
      q = load4<BF16>(a.in, row * a.in_stride + a.q_at + h * dk + c) * a.q_scale;
      k = load4<BF16>(a.in, row * a.in_stride + a.k_at + h * dk + c) * a.k_scale;
      g *= fixed;
      if (a.low) {
        const f32x4 z = load4<BF16>(a.low, row * a.low_stride + h * dk + c) + *(const f32x4*)(a.decay + h * dk + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) g[e] = __expf(-a.inv_tau * fast_softplus(-z[e]));
      }
    }
    *(f32x4*)(qs + t * ld + c) = q;
    *(f32x4*)(ks + t * ld + c) = k;
    *(f32x4*)(gs + t * ld + c) = g;
  }
  if (tid < kBlock * kBlock / 4) *(f32x4*)(Ps + tid * 4) = f32x4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();
  if (half > 0) {                              // uniform
    for (int i = tid; i < cnt * half; i += 256) {
      const int t = i / half, c = i - t * half;
      const float2 r = rotary_turn(sg.start + t0 + t, a.freqs[c]);
      float* const q = qs + t * ld + c;
      float* const k = ks + t * ld + c;
      turn_pair(q[0], q[half], r.x, r.y);
      turn_pair(k[0], k[half], r.x, r.y);
    }
    __syncthreads();
  }
  // ---- P: 16 lanes walk k_s down the tokens from s on, in pieces of four channels.  A wave takes four neighbours, so that it
  // starts at the first of them; which four changes with the block, as the waves' shares differ (all tokens for every s: 8
  // prompts of 2048 tokens, 32 heads, with the kernels below 618 us, now 601)
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
    auto token = [&](int t, bool all) {        // all: it lies behind the four
      f32x4 pp = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const f32x4 gt = *(const f32x4*)(gs + t * ld + at[p]);
#pragma unroll
        for (int e = 0; e < 4; ++e) kk[p][e] *= all || t > s ? gt[e] : 1.f;
        pp += kk[p] * *(const f32x4*)(qs + t * ld + at[p]);
      }
      const float sp = row16_sum((pp[0] + pp[1]) + (pp[2] + pp[3]));
      if (all || t >= s) Ps[t * kBlock + s] = sp;              // all 16 lanes, the same value
    };
#pragma unroll
    for (int u = 0; u < 4; ++u) token(first + u, false);
#pragma unroll 2
    for (int t = first + 4; t < kBlock; ++t) token(t, true);
  }
  __syncthreads();
  // ---- columns: a thread reads and writes its own only
  float* const oQ = ra.ws + (block_slot(ra.row0, sg, blockIdx.z, blockIdx.x) * a.heads + h) * block_floats(dk);
  float* const oK = oQ + kBlock * dk;          // [dk / 16][64 lanes][4], as oQ
  float* const oP = oK + kBlock * dk;          // [64][hi 4, mid 4], [64][lo 4]
  float* const oG = oP + kPairFloats;          // [dk]
  if (tid < dk) {                              // G q
    const int c = tid;
    float G = 1.f;
#pragma unroll
    for (int t = 0; t < kBlock; ++t) {
      G *= gs[t * ld + c];
      qs[t * ld + c] *= G;
    }
    oG[c] = G;
  }
  if (tid >= 256 - dk) {                       // keys, on the threads the queries leave free as far as they go
    const int c = tid - (256 - dk);
    float R = 1.f;
#pragma unroll
    for (int g = 3; g >= 0; --g) {
      f32x4 x;
#pragma unroll
      for (int r = 3; r >= 0; --r) {
        const int t = 4 * g + r;
        x[r] = ks[t * ld + c] * R;
        R *= gs[t * ld + c];
      }
      *(f32x4*)(oK + ((c >> 4) * 64 + g * 16 + (c & 15)) * 4) = x;
    }
  }
  __syncthreads();
  if (tid < 64) {
    const Planes x(*(const f32x4*)(Ps + (tid & 15) * kBlock + (tid >> 4) * 4));
    *(u32x4*)(oP + tid * 4) = u32x4{x.hi.x, x.hi.y, x.mid.x, x.mid.y};
    *(uint2*)(oP + 256 + tid * 2) = x.lo;
  }
  for (int i = tid; i < kBlock * dk / 4; i += 256) {           // lane (g, row) of tile kt: columns 16 kt + 4 g ..
    const int l = i & 63, kt = i >> 6;
    *(f32x4*)(oQ + i * 4) = *(const f32x4*)(qs + (l & 15) * ld + kt * 16 + (l >> 4) * 4);
  }
}

// ------------------------------------------------------------------ runs in pieces
// A piece's state: its sums, or the state before it, then its decays.
__host__ __device__ inline constexpr int piece_floats(int dk, int dv) { return dk * dv + dk; }

// What a piece adds to the state and its decays; pieces behind which there is another, whose blocks are whole.  A wave 16
// rows of the state, so that every key is split once; value rows of four blocks come into LDS while four are worked on.
template <int KT, int NW>
__global__ __launch_bounds__(64 * KT) void linear_sums_kernel(RunArgs ra) {
  constexpr int kAhead = 4, dk = 16 * KT, dv = 16 * NW, size = block_floats(dk), kRows = kBlock * dv;
  __shared__ __align__(16) uint16_t rows[2][kAhead * kRows];
  const zp_linear& a = ra.d;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int kt = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = blockIdx.x % (ra.pieces.most - 1), unit = blockIdx.x / (ra.pieces.most - 1), h = unit % a.heads, seg = unit / a.heads;
  const Segment whole = segment_of(a.seg, seg);
  if (whole.count <= 0 || whole.row < ra.row0) return;
  const Piece piece(ra.pieces, ra.row0, whole, seg, c);
  if (piece.last) return;
  const Segment& sg = piece.sg;
  const int blocks = ra.pieces.blocks;
  const int64_t stride = (int64_t)a.heads * size;
  const float* const base = ra.ws + (block_slot(ra.row0, sg, seg, 0) * a.heads + h) * size;
  const float* const keys = base + kBlock * dk + (kt * 64 + lane) * 4;
  const float* const decays = base + 2 * kBlock * dk + kPairFloats + 16 * kt + 4 * g;
  f32x4 k[2][kAhead], dec[2][kAhead];
  auto request = [&](int b0, int to) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int b = min(b0 + i, blocks - 1);                   // the last may come again
      k[to][i] = *(const f32x4*)(keys + b * stride);
      dec[to][i] = *(const f32x4*)(decays + b * stride);
    }
    for (int u = kt; u < kAhead * NW / 2; u += KT) {
      const int i = u / (NW / 2), part = u % (NW / 2), b = min(b0 + i, blocks - 1), s = part * 64 + lane, row = s / (dv / 8);
      const StageLoads from((const char*)a.in + (int64_t)(sg.row + b * kBlock) * a.in_stride * 2, kBlock * a.in_stride * 2);
      from.ld(rows[to] + i * kRows + part * 512, row * (int)a.in_stride * 2 + (s - row * (dv / 8)) * 16, (a.v_at + h * dv) * 2);
    }
  };
  f32x4 S[NW], D = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
  for (int nc = 0; nc < NW; ++nc) S[nc] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto work = [&](int b0, int at) {
    wait_and_meet();
    if (b0 + kAhead < blocks) request(b0 + kAhead, at ^ 1);
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      if (b0 + i >= blocks) break;
      const Planes x(k[at][i]);
      const uint16_t* const from = rows[at] + i * kRows + (4 * g + (l16 >> 2)) * dv + (l16 & 3) * 4;
      D *= dec[at][i];
#pragma unroll
      for (int nc = 0; nc < NW; ++nc) {
        const uint2 v = read_transposed(from + nc * 16);
        S[nc] *= dec[at][i];
        S[nc] = mfma_bf16(u32x4{x.lo.x, x.lo.y, 0u, 0u}, u32x4{v.x, v.y, v.x, v.y}, S[nc]);
        S[nc] = mfma_bf16(u32x4{x.hi.x, x.hi.y, x.mid.x, x.mid.y}, u32x4{v.x, v.y, v.x, v.y}, S[nc]);
      }
    }
  };
  request(0, 0);
#pragma unroll 1
  for (int b0 = 0; b0 < blocks; b0 += 2 * kAhead) {
    work(b0, 0);
    if (b0 + kAhead < blocks) work(b0 + kAhead, 1);
  }
  float* const to = ra.pieces.states + (piece.slot * a.heads + h) * piece_floats(dk, dv);
#pragma unroll
  for (int nc = 0; nc < NW; ++nc) *(f32x4*)(to + ((nc * KT + kt) * 64 + lane) * 4) = S[nc];
  if (l16 == 0) *(f32x4*)(to + dk * dv + 16 * kt + 4 * g) = D;
}

// From sums to the states before the pieces, in place; a thread four rows of a column.
template <int KT, int NW>
__global__ __launch_bounds__(256) void linear_states_kernel(RunArgs ra) {
  constexpr int dk = 16 * KT, dv = 16 * NW, kAhead = 4;
  const zp_linear& a = ra.d;
  const int h = blockIdx.x % a.heads, seg = blockIdx.x / a.heads, f = blockIdx.y * 256 + threadIdx.x;
  const Segment whole = segment_of(a.seg, seg);
  if (whole.count <= 0 || whole.row < ra.row0) return;
  const int lane = f & 63, kt = (f >> 6) % KT, nc = (f >> 6) / KT, row = 16 * kt + 4 * (lane >> 4);
  const float* const state = a.state + ((int64_t)whole.slot * a.heads + h) * ((int64_t)dk * dv) + row * dv + nc * 16 + (lane & 15);
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  if (whole.start != 0)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[r] = state[r * dv];
  const int tokens = ra.pieces.blocks * kBlock, count = (whole.count + tokens - 1) / tokens;
  const int64_t stride = (int64_t)a.heads * piece_floats(dk, dv);
  float* const at = ra.pieces.states + Piece(ra.pieces, ra.row0, whole, seg, 0).slot * stride + (int64_t)h * piece_floats(dk, dv);
  for (int c0 = 0; c0 < count; c0 += kAhead) {
    f32x4 x[kAhead], D[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int c = min(c0 + i, max(count - 2, 0));            // the last piece has no sums
      x[i] = *(const f32x4*)(at + c * stride + f * 4);
      D[i] = *(const f32x4*)(at + c * stride + dk * dv + row);
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
      if (c0 + i < count) {
        *(f32x4*)(at + (c0 + i) * stride + f * 4) = S;
        S = S * D[i] + x[i];
      }
  }
}

// A head's blocks, one after the other, a wave 16 columns of the state.  Operands in fp32 enter the bf16 matrix cores in three
// planes each, as in delta_blocks: the state is split where it is updated, what comes from memory by all waves together,
// a block ahead; value rows are bf16 as they come.  Rows are normed and stored behind the next meeting of the
// waves, which the norm needs too.  8 prompts of 2048 tokens, 32 heads of 128 x 128, with the kernel above: 677 -> 647 us,
// 16 heads 422 -> 358; error of the state against 64 bits 2.0e-7 -> 1.8e-7 of its size.
template <int KT, int NW>
__global__ __launch_bounds__(64 * NW, 2) void linear_blocks_kernel(RunArgs ra) {
  extern __shared__ __align__(16) float lds[];
  const zp_linear& a = ra.d;
  constexpr int dk = 16 * KT, dv = 16 * NW, size = block_floats(dk), J = KT / 2;
  constexpr int kSplit = 2 * kBlock * dk, kV = size - kSplit, kRest = kV + kBlock * dv / 2;   // floats to be split; the others
  constexpr int kG = kPairFloats;                                     // in the others, behind P; then from kV on the value rows
  constexpr int kPlanes = 2 * KT * 384, kMine = (2 * KT + NW - 1) / NW;      // floats of a block's planes; tiles of a wave
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  float* const split = lds;                    // [2][kSplit]
  float* const rest = split + 2 * kSplit;      // [3][kRest]
  float* const planes = rest + 3 * kRest;      // [2][kPlanes]
  float* const red = planes + 2 * kPlanes;     // [2][NW * 16]
  const int unit = blockIdx.x / ra.pieces.most, h = unit % a.heads, seg = unit / a.heads;
  const Segment whole = segment_of(a.seg, seg);
  if (whole.count <= 0 || whole.row < ra.row0) return;
  const Piece piece(ra.pieces, ra.row0, whole, seg, blockIdx.x % ra.pieces.most);
  const Segment& sg = piece.sg;
  if (sg.count <= 0) return;
  float* const state = a.state + ((int64_t)sg.slot * a.heads + h) * ((int64_t)dk * dv);
  const int col0 = wave * 16;
  f32x4 S[KT][1];
  if (ra.pieces.blocks) load_piece_state(S, ra.pieces.states + (piece.slot * a.heads + h) * piece_floats(dk, dv), wave);
  else load_state<KT, 1>(S, state, dv, col0, sg.start == 0);
  const float nrm = a.norm[h * dv + col0 + l16];
  const float* const base = ra.ws + (block_slot(ra.row0, sg, seg, 0) * a.heads + h) * size;
  const int64_t stride = (int64_t)a.heads * size;
  const int blocks = (sg.count + kBlock - 1) / kBlock;
  auto request = [&](int b) {                  // a block behind the last: nothing is read
    const int cnt = b < blocks ? min(kBlock, sg.count - b * kBlock) : 0;
    const StageLoads from(base + b * stride, cnt > 0 ? size * 4 : 0);
#pragma unroll
    for (int u = 0; u < (size / 256 + NW - 1) / NW; ++u) {
      const int i = min(wave + u * NW, size / 256 - 1);            // the last may come twice
      float* const to = i < kSplit / 256 ? split + (b & 1) * kSplit + i * 256 : rest + b % 3 * kRest + (i * 256 - kSplit);
      from.ld(to, lane * 16, i * 1024);
    }
    const StageLoads rows((const char*)a.in + (int64_t)(sg.row + b * kBlock) * a.in_stride * 2, cnt * a.in_stride * 2);
    const int w = wave % (NW / 2), s = w * 64 + lane, row = s / (dv / 8), pc = s - row * (dv / 8);       // each comes twice
    rows.ld(rest + b % 3 * kRest + kV + w * 256, max(min(row, cnt - 1), 0) * (int)a.in_stride * 2 + pc * 16, (a.v_at + h * dv) * 2);
  };
  // Planes of a block's tiles: for pairs of those of G q [3][64 lanes][two tiles' 4], for those of keys [64][hi 4, mid 4],
  // [64][lo 4].  A wave's tile u; the last may be made twice.
  auto tile_of = [&](int b, int u) {
    return *(const f32x4*)(split + (b & 1) * kSplit + min(wave + u * NW, 2 * KT - 1) * 256 + lane * 4);
  };
  auto put_planes = [&](int b, int u, const f32x4& x) {
    const int i = min(wave + u * NW, 2 * KT - 1);
    const int key = i >= KT;                   // multiplied, not branched on: the products beside stay in one stretch
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
  const int gate_at = (4 * g * (int)a.in_stride + a.g_at + h * dv + col0 + l16) * 2;
  auto finish = [&](int b, int r, const f32x4& ss) {               // row r of block b, whose squares are ss; none of block -1
    const int cnt = b < 0 ? 0 : min(kBlock, sg.count - b * kBlock);
    const BlockRows out(a.out, sg.row + b * kBlock, cnt, a.out_stride);
    const float rs = __builtin_amdgcn_rsqf(ss[r] * inv_v + a.eps), z = bf16_bits_to_float(gate[r]);
    out.st(out_at + r * (int)a.out_stride * 2, 0, done[r] * rs * nrm * z * fast_sigmoid(z));
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
    const float* const pl = planes + (b & 1) * kPlanes;
    u32x4 Q[2][3], K[2][2];
    uint2 Kl[2][2];
    f32x4 dec[2][2];
    auto operands = [&](int j) {
#pragma unroll
      for (int i = 0; i < 3; ++i) Q[j & 1][i] = *(const u32x4*)(pl + (j * 3 + i) * 256 + lane * 4);
    };
    auto keys = [&](int j) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float* const at = pl + (KT + 2 * j + i) * kPairFloats;
        K[j & 1][i] = *(const u32x4*)(at + lane * 4);
        Kl[j & 1][i] = *(const uint2*)(at + 256 + lane * 2);
        dec[j & 1][i] = *(const f32x4*)(mine + kG + 16 * (2 * j + i) + 4 * g);
      }
    };
    operands(0);
    keys(0);
    f32x4 tile = tile_of(b + 1, 0);
    const f32x4 ss = block_squares_total<NW>(red + ((b - 1) & 1) * NW * kBlock);
    const uint2 v4 = read_transposed((const uint16_t*)(mine + kV) + (4 * g + (l16 >> 2)) * dv + col0 + (l16 & 3) * 4);
    const u32x4 v = {v4.x, v4.y, v4.x, v4.y};
    const u32x4 P = *(const u32x4*)(mine + lane * 4);
    const uint2 Pl = *(const uint2*)(mine + 256 + lane * 2);
    request(b + 2);
    const BlockRows gp(a.in, sg.row + b * kBlock, min(kBlock, sg.count - b * kBlock), a.in_stride);
    uint16_t next[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) next[r] = gp.ld(gate_at + r * (int)a.in_stride * 2, 0);
    __builtin_amdgcn_sched_barrier(0);
    f32x4 O[1] = {mfma_bf16(u32x4{Pl.x, Pl.y, 0u, 0u}, v, f32x4{0.f, 0.f, 0.f, 0.f})};
    O[0] = mfma_bf16(P, v, O[0]);
#pragma unroll
    for (int j = 0; j < J; ++j) {              // beside: the block before is finished, the next one's planes are made
      if (j + 1 < J) {
        operands(j + 1);
        keys(j + 1);
      }
#pragma unroll
      for (int i = 2; i >= 0; --i)             // the smallest products first
#pragma unroll
        for (int k = 2 - i; k >= 0; --k) O[0] = mfma_bf16(Q[j & 1][i], sp[k][j], O[0]);
#pragma unroll
      for (int i = 0; i < 2; ++i) {            // the state's tiles are behind their products
        f32x4& s = S[2 * j + i][0];
        s *= dec[j & 1][i];
        s = mfma_bf16(u32x4{Kl[j & 1][i].x, Kl[j & 1][i].y, 0u, 0u}, v, s);
        s = mfma_bf16(K[j & 1][i], v, s);
      }
#pragma unroll
      for (int r = j * 4 / J; r < (j + 1) * 4 / J; ++r) finish(b - 1, r, ss);
#pragma unroll
      for (int u = j * kMine / J; u < (j + 1) * kMine / J; ++u) {
        put_planes(b + 1, u, tile);
        if (u + 1 < kMine) tile = tile_of(b + 1, u + 1);
      }
      if (j > 0) {
        split_state(2 * j - 2);
        split_state(2 * j - 1);
      }
      spread_over_products<10, 6>();
    }
    split_state(KT - 2);
    split_state(KT - 1);
#pragma unroll
    for (int i = 0; i < 3; ++i)                // here, not behind the squares
#pragma unroll
      for (int j = 0; j < J; ++j) settle(sp[i][j]);
#pragma unroll
    for (int r = 0; r < 4; ++r) gate[r] = next[r];
    block_squares<1>(O, red + (b & 1) * NW * kBlock, wave);
    done = O[0];
  }
  wait_and_meet();
  const f32x4 ss = block_squares_total<NW>(red + ((blocks - 1) & 1) * NW * kBlock);
#pragma unroll
  for (int r = 0; r < 4; ++r) finish(blocks - 1, r, ss);
  if (piece.last) store_state<KT, 1>(S, state, dv, col0);
}

template <int KT, int NW> int launch_blocks(const RunArgs& ra, hipStream_t st) {
  constexpr int kSplit = 2 * kBlock * 16 * KT;
  constexpr int smem = (3 * (block_floats(16 * KT) + kBlock * 8 * NW) - kSplit + 2 * 2 * KT * 384 + 2 * NW * kBlock) * 4;
  if (smem > 60 * 1024 && hipFuncSetAttribute((const void*)linear_blocks_kernel<KT, NW>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                              smem) != hipSuccess) {
    zp_set_error("linear_runs: cannot reserve %d bytes of LDS", smem);
    return ZP_EHIP;
  }
  const int64_t units = (int64_t)ra.d.seg.n * ra.d.heads;
  if (ra.pieces.blocks) {
    hipLaunchKernelGGL((linear_sums_kernel<KT, NW>), dim3((unsigned)(units * (ra.pieces.most - 1))), dim3(64 * KT), 0, st, ra);
    ZP_LAUNCH_CHECK();
    hipLaunchKernelGGL((linear_states_kernel<KT, NW>), dim3((unsigned)units, KT * NW / 4), dim3(256), 0, st, ra);
    ZP_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL((linear_blocks_kernel<KT, NW>), dim3((unsigned)(units * ra.pieces.most)), dim3(64 * NW), smem, st, ra);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}
template <int KT> int launch_blocks(const RunArgs& ra, hipStream_t st) {
  switch (ra.d.dv / 32) {
    case 1: return launch_blocks<KT, 2>(ra, st);
    case 2: return launch_blocks<KT, 4>(ra, st);
    case 3: return launch_blocks<KT, 6>(ra, st);
    default: return launch_blocks<KT, 8>(ra, st);
  }
}

}  // namespace

static int64_t blocks_bytes(int64_t rows, int64_t segments, int64_t heads, int dk) {
  return (rows / kBlock + segments) * heads * block_floats(dk) * 4;
}

constexpr PieceCost kCost = {1, 3, 75, 0};

// With room for the states between pieces of few heads' runs, whatever the values' size and the longest run.
extern "C" int64_t zp_linear_runs_workspace(int32_t rows, int32_t segments, int32_t heads, int32_t dk) {
  if (rows < 0 || segments < 0 || heads <= 0 || dk <= 0) return -1;
  return blocks_bytes(rows, segments, heads, dk) + (dk <= 128 ? most_states(rows, segments, heads, kCost) * piece_floats(dk, 128) * 4 : 0);
}

extern "C" int zp_linear_runs(const zp_linear* args, int32_t first_row, int32_t longest, void* workspace,
                              int64_t workspace_bytes, int32_t dtype, void* stream) {
  ZP_REQUIRE(args, "linear_runs: null arguments");
  const zp_linear& a = *args;
  ZP_REQUIRE(linear_dims_fit(a) && first_row >= 0 && longest >= 0 && first_row <= a.seg.num_rows, "linear_runs: bad dims");
  if (dtype != ZP_BF16 || (a.dk != 32 && a.dk != 64 && a.dk != 128) || a.dv % 32 || a.dv > 128 || a.heads > 65535 ||
      a.seg.n > 65535 || a.in_stride % 8 || a.q_at % 8 || a.k_at % 8 || a.v_at % 8 || a.low_stride % 8 ||
      a.in_stride >= (1 << 24) || a.out_stride >= (1 << 24)) {
    zp_set_error("linear_runs: bfloat16, head sizes %d (32, 64, 128) and %d (a multiple of 32, <= 128) unsupported", a.dk, a.dv);
    return ZP_EUNSUPPORTED;
  }
  if (a.seg.n == 0 || longest == 0) return ZP_OK;
  ZP_REQUIRE(a.in && a.decay && (a.rot == 0 || a.freqs) && a.norm && a.state && a.out && a.seg.rows && a.seg.counts &&
                 a.seg.slots && a.seg.starts && aligned16(a.in) && aligned16(a.low) && (!a.low || aligned16(a.decay)) &&
                 aligned16(a.state) && aligned16(workspace), "linear_runs: null or unaligned pointer");
  const int64_t rows = a.seg.num_rows - first_row, whole = blocks_bytes(rows, a.seg.n, a.heads, a.dk);
  ZP_REQUIRE(workspace && workspace_bytes >= whole, "linear_runs: workspace too small");
  RunArgs ra = {a, (float*)workspace, first_row, {}};
  ra.pieces = pieces_of(rows, a.seg.n, a.heads, longest, kCost, 1, (workspace_bytes - whole) / 4 / piece_floats(a.dk, a.dv));
  ra.pieces.states = (float*)workspace + whole / 4;
  ra.d.seg.max_count = longest;               // no segment has more blocks than were prepared
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(linear_prepare_kernel, dim3((unsigned)((longest + kBlock - 1) / kBlock), (unsigned)a.heads, (unsigned)a.seg.n),
                     dim3(256), 0, st, ra);
  ZP_LAUNCH_CHECK();
  switch (a.dk) {
    case 32: return launch_blocks<2>(ra, st);
    case 64: return launch_blocks<4>(ra, st);
    default: return launch_blocks<8>(ra, st);
  }
}
