// Matrix memory with exponential gates (mlstm.hip) over long runs, 16 tokens at a time.  With F_t the sum of
// the block's log forget gates up to token t, x_s = i_s - F_s and m the running maximum,
//
//   D[t, s] = e^{F_t + x_s - m_t} q_t . k_s (s <= t),  a_t = e^{F_t + m_0 - m_t}
//   O = a (Q S) + D V,   n . q_t = a_t (n . q_t) + sum_s D[t, s]
//   S <- e^{F_15 + m_0 - m_15} S + sum_s e^{F_15 + x_s - m_15} k_s v_s^T,  n likewise with k alone
//
//   mlstm_gates     gates and the running maximum
//   mlstm_prepare   D and the block's factors, for all blocks at once
//   mlstm_blocks    a head's blocks one after the other, S in registers
//
// All fp32, on the bf16 matrix cores: the products q . k are exact products of the projections, added up in fp32, and S, D
// and the rows that are written are split into three bf16 planes each.  Projections in bfloat16.
#include "blocks.h"
#include <type_traits>

namespace {

struct RunArgs {
  zp_mlstm d;
  float* aux;    // per block and head: kAux floats
  float4* scal;  // per token row from row0 on and head: F, x, m, m before the block
  int row0;
  Pieces pieces;
};
// D's planes as a left operand, then a, write factors, e^{-m}, row sums of D (16 each), the keep factor
constexpr int kAux = 512, kInter = kPairFloats, kWrite = kInter + 16, kFloor = kWrite + 16, kSum = kFloor + 16, kKeep = kSum + 16;

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// lane i <- lane i - N of its row of 16, or `edge`
template <int N> __device__ __forceinline__ float row_shr(float v, float edge) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, edge), __builtin_bit_cast(int, v), 0x110 + N,
                                                               0xf, 0xf, false));
}

// A workgroup per head and run, a wave 64 tokens of every stretch: sums and maxima of blocks side by side, then one wave takes the
// maximum from block to block.  As many waves as the longest run keeps busy, up to 16.  (One wave for all, 64 tokens at a
// time: 14.2 us for 970 tokens of 16 heads, now 7.4; three runs of 844 to 2043 21.2, now 9.7.  With 16 waves for any run 40 runs of
// 17 tokens, 64 heads of 64, took 57.9 us with the kernels behind; with one wave each 45.3.)
constexpr int kGateWaves = 16;
__global__ __launch_bounds__(64 * kGateWaves) void mlstm_gates_kernel(RunArgs ra) {
  __shared__ float ends[2][64], before[65];                    // of 64 blocks: F and the maximum of x at the last token; m before it
  const zp_mlstm& a = ra.d;
  const int tid = threadIdx.x, lane = tid & 63, block = tid >> 4, h = blockIdx.x % a.heads;
  const Segment sg = segment_of(a.seg, blockIdx.x / a.heads);
  if (sg.count <= 0 || sg.row < ra.row0) return;
  float* const mstate = a.state + ((int64_t)sg.slot * a.heads + h) * ((int64_t)a.dk * a.dv + a.dk + 4) + (int64_t)a.dk * a.dv + a.dk;
  float m = sg.start == 0 ? 0.f : *mstate;
  const float icap = 1.f / a.cap, ib = a.i_bias[h], fb = a.f_bias[h];
  float zi = 0.f, zf = 0.f;
  auto fetch = [&](int t0) {
    const int64_t src = (int64_t)(sg.row + min(t0 + tid, sg.count - 1)) * a.gate_stride + h;
    zi = a.gates[src];
    zf = a.gates[src + a.heads];
  };
  fetch(0);
  const int stretch = blockDim.x;
  for (int t0 = 0; t0 < sg.count; t0 += stretch) {
    const int cnt = min(stretch, sg.count - t0);
    const float gi = a.cap * tanhf((zi + ib) * icap), x = a.cap * tanhf((zf + fb) * icap);
    const float gf = fminf(x, 0.f) - log1pf(expf(-fabsf(x)));
    if (t0 + stretch < sg.count) fetch(t0 + stretch);
    // sums and maxima inside each block of 16 lanes: m_t = F_t + max(m before the block, max_{s <= t} x_s)
    float F = tid < cnt ? gf : 0.f;
    F += row_shr<1>(F, 0.f);
    F += row_shr<2>(F, 0.f);
    F += row_shr<4>(F, 0.f);
    F += row_shr<8>(F, 0.f);
    const float xs = tid < cnt ? gi - F : -INFINITY;
    float top = xs;
    top = fmaxf(top, row_shr<1>(top, -INFINITY));
    top = fmaxf(top, row_shr<2>(top, -INFINITY));
    top = fmaxf(top, row_shr<4>(top, -INFINITY));
    top = fmaxf(top, row_shr<8>(top, -INFINITY));
    if ((lane & 15) == 15) {
      ends[0][block] = F;
      ends[1][block] = top;
    }
    __syncthreads();
    if (tid < 64) {
      const bool there = lane * kBlock < stretch;
      const float Fe = there ? ends[0][lane] : 0.f, te = there ? ends[1][lane] : -INFINITY;
      float mine = m;
#pragma unroll 1
      for (int b0 = 0; b0 * kBlock < cnt; b0 += 8)             // blocks behind the end change nothing
#pragma unroll
        for (int b = b0; b < b0 + 8; ++b) {
          if (lane == b) mine = m;
          m = lane_value(Fe, b) + fmaxf(m, lane_value(te, b));
        }
      before[lane] = mine;
      if (lane == 0) before[64] = m;
    }
    __syncthreads();
    const float m0 = before[block];
    m = before[64];
    const float mine_m = F + fmaxf(m0, top);
    if (tid < cnt)
      ra.scal[(int64_t)(sg.row + t0 + tid - ra.row0) * a.heads + h] = make_float4(F, xs, mine_m, m0);
  }
  if (tid == 0) *mstate = m;
}

// A wave per (block, head).
template <int KT>
__global__ __launch_bounds__(256) void mlstm_prepare_kernel(RunArgs ra) {
  const zp_mlstm& a = ra.d;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4, h = blockIdx.y * 4 + (threadIdx.x >> 6);
  const Segment sg = segment_of(a.seg, blockIdx.z);
  const int t0 = blockIdx.x * kBlock;
  if (t0 >= sg.count || sg.row < ra.row0 || h >= a.heads) return;
  const int cnt = min(kBlock, sg.count - t0);
  const int64_t mine = sg.row + t0 + min(l16, cnt - 1);
  const float4 sc = ra.scal[(mine - ra.row0) * a.heads + h];
  const uint16_t* const in = (const uint16_t*)a.in + mine * a.in_stride + h * (16 * KT) + g * 8;
  f32x4 P = {0.f, 0.f, 0.f, 0.f};              // rows s = 4 g + r, column t = l16
#pragma unroll
  for (int ks = 0; ks < KT / 2; ++ks)
    P = mfma_bf16(*(const u32x4*)(in + a.k_at + ks * 32), *(const u32x4*)(in + a.q_at + ks * 32), P);
  float sum = 0.f;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int s = 4 * g + r;
    const float xs = __shfl(sc.y, s);
    P[r] = s <= l16 && s < cnt && l16 < cnt ? P[r] * expf(sc.x + xs - sc.z) : 0.f;
    sum += P[r];
  }
  sum += lane_xor16(sum);
  sum += lane_xor32(sum);
  const float F_end = lane_value(sc.x, cnt - 1), m_end = lane_value(sc.z, cnt - 1);
  float* const aux = ra.aux + (block_slot(ra.row0, sg, blockIdx.z, blockIdx.x) * a.heads + h) * kAux;
  const Planes planes(P);
  *(u32x4*)(aux + lane * 4) = u32x4{planes.hi.x, planes.hi.y, planes.mid.x, planes.mid.y};
  *(uint2*)(aux + 256 + lane * 2) = planes.lo;
  if (g == 0) {
    aux[kInter + l16] = expf(sc.x + sc.w - sc.z);
    aux[kWrite + l16] = l16 < cnt ? expf(F_end + sc.y - m_end) : 0.f;
    aux[kFloor + l16] = expf(-sc.z);
    aux[kSum + l16] = sum;
    if (l16 == 0) aux[kKeep] = expf(F_end + sc.w - m_end);
  }
}

// ------------------------------------------------------------------ runs in pieces
// A piece's state: its sums, or the state before it; the same of the normaliser; the factor that keeps what was before.
__host__ __device__ inline constexpr int piece_floats(int dk, int dv) { return dk * dv + dk + 4; }

// What a piece adds to the state and the normaliser; pieces behind which there is another, whose blocks are whole.  A wave 16
// rows of the state, so that every key is weighted and split once; key and value rows of four blocks come into LDS while
// four are worked on.
template <int KT, int NW>
__global__ __launch_bounds__(64 * KT) void mlstm_sums_kernel(RunArgs ra) {
  constexpr int kAhead = 4, dk = 16 * KT, dv = 16 * NW, kKeys = kBlock * dk, kRows = kBlock * dv;
  __shared__ __align__(16) uint16_t krows[2][kAhead * kKeys], vrows[2][kAhead * kRows];
  const zp_mlstm& a = ra.d;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int kt = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = blockIdx.x % (ra.pieces.most - 1), unit = blockIdx.x / (ra.pieces.most - 1), h = unit % a.heads, seg = unit / a.heads;
  const Segment whole = segment_of(a.seg, seg);
  if (whole.count <= 0 || whole.row < ra.row0) return;
  const Piece piece(ra.pieces, ra.row0, whole, seg, c);
  if (piece.last) return;
  const Segment& sg = piece.sg;
  const int blocks = ra.pieces.blocks;
  const float* const aux = ra.aux + (block_slot(ra.row0, sg, seg, 0) * a.heads + h) * kAux;
  const int64_t stride = (int64_t)a.heads * kAux;
  f32x4 wr[2][kAhead];
  float keep[2][kAhead];
  // rows of `cols` columns from column `at` on
  auto stage = [&](auto cols_, uint16_t* to, int b, int part, int at) {
    constexpr int cols = cols_.value;
    const int s = part * 64 + lane, row = s / (cols / 8);
    const StageLoads from((const char*)a.in + (int64_t)(sg.row + b * kBlock) * a.in_stride * 2, kBlock * a.in_stride * 2);
    from.ld(to + part * 512, row * (int)a.in_stride * 2 + (s - row * (cols / 8)) * 16, at * 2);
  };
  auto request = [&](int b0, int to) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int b = min(b0 + i, blocks - 1);                   // the last may come again
      wr[to][i] = *(const f32x4*)(aux + b * stride + kWrite + 4 * g);
      keep[to][i] = aux[b * stride + kKeep];
    }
    for (int u = kt; u < kAhead * KT / 2; u += KT)
      stage(std::integral_constant<int, dk>(), krows[to] + u / (KT / 2) * kKeys, min(b0 + u / (KT / 2), blocks - 1), u % (KT / 2), a.k_at + h * dk);
    for (int u = kt; u < kAhead * NW / 2; u += KT)
      stage(std::integral_constant<int, dv>(), vrows[to] + u / (NW / 2) * kRows, min(b0 + u / (NW / 2), blocks - 1), u % (NW / 2), a.v_at + h * dv);
  };
  f32x4 S[NW];
  float n = 0.f, kept = 1.f;
#pragma unroll
  for (int nc = 0; nc < NW; ++nc) S[nc] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto work = [&](int b0, int at) {
    wait_and_meet();
    if (b0 + kAhead < blocks) request(b0 + kAhead, at ^ 1);
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      if (b0 + i >= blocks) break;
      const float f = keep[at][i];
      const int row = 4 * g + (l16 >> 2);
      const f32x4 k = read_columns((const char*)(krows[at] + i * kKeys + row * dk + 16 * kt + (l16 & 3) * 4)) * wr[at][i];
      const uint16_t* const from = vrows[at] + i * kRows + row * dv + (l16 & 3) * 4;
      const Planes x(k);
      n = fmaf(n, f, (k[0] + k[1]) + (k[2] + k[3]));
      kept *= f;
#pragma unroll
      for (int nc = 0; nc < NW; ++nc) {
        const uint2 v = read_transposed(from + nc * 16);
        S[nc] *= f;
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
  n += lane_xor16(n);
  n += lane_xor32(n);
  float* const to = ra.pieces.states + (piece.slot * a.heads + h) * piece_floats(dk, dv);
#pragma unroll
  for (int nc = 0; nc < NW; ++nc) *(f32x4*)(to + ((nc * KT + kt) * 64 + lane) * 4) = S[nc];
  if (g == 0) to[dk * dv + 16 * kt + l16] = n;
  if (threadIdx.x == 0) to[dk * dv + dk] = kept;
}

// From sums to the states before the pieces, in place; a thread four rows of a column, or a row of the normaliser.
template <int KT, int NW>
__global__ __launch_bounds__(256) void mlstm_states_kernel(RunArgs ra) {
  constexpr int dk = 16 * KT, dv = 16 * NW, kAhead = 4;
  const zp_mlstm& a = ra.d;
  const int h = blockIdx.x % a.heads, seg = blockIdx.x / a.heads, f = blockIdx.y * 256 + threadIdx.x;
  const Segment whole = segment_of(a.seg, seg);
  if (whole.count <= 0 || whole.row < ra.row0) return;
  const int lane = f & 63, kt = (f >> 6) % KT, nc = (f >> 6) / KT;
  const float* const state = a.state + ((int64_t)whole.slot * a.heads + h) * ((int64_t)dk * dv + dk + 4);
  const bool fresh = whole.start == 0, norm = f < dk;
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  float n = 0.f;
  if (!fresh) {
#pragma unroll
    for (int r = 0; r < 4; ++r) S[r] = state[(16 * kt + 4 * (lane >> 4) + r) * dv + nc * 16 + (lane & 15)];
    if (norm) n = state[dk * dv + f];
  }
  const int tokens = ra.pieces.blocks * kBlock, count = (whole.count + tokens - 1) / tokens;
  const int64_t stride = (int64_t)a.heads * piece_floats(dk, dv);
  float* const at = ra.pieces.states + Piece(ra.pieces, ra.row0, whole, seg, 0).slot * stride + (int64_t)h * piece_floats(dk, dv);
  for (int c0 = 0; c0 < count; c0 += kAhead) {
    f32x4 x[kAhead];
    float y[kAhead], kept[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int c = min(c0 + i, max(count - 2, 0));            // the last piece has no sums
      x[i] = *(const f32x4*)(at + c * stride + f * 4);
      y[i] = norm ? at[c * stride + dk * dv + f] : 0.f;
      kept[i] = at[c * stride + dk * dv + dk];
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
      if (c0 + i < count) {
        *(f32x4*)(at + (c0 + i) * stride + f * 4) = S;
        if (norm) at[(c0 + i) * stride + dk * dv + f] = n;
        S = S * kept[i] + x[i];
        n = fmaf(n, kept[i], y[i]);
      }
  }
}

// A wave owns 16 columns of the state, which is split into planes where it is updated (8 prompts of 2048 tokens, 16 heads
// of 128 x 128, with the kernels above: 595 us with products on the fp32 matrix cores, 440; error of the state against 64
// bits 3.1e-7 -> 2.9e-7 of its size).  What bounds it is a wave's chain of work from meeting to meeting: the normaliser is
// with the waves that are ahead (407), the rows of the block before are finished under the products (402).
// LDS of a stage: Q and K rows, their 16-byte pieces xor-ed with the row so that neither operand order meets bank
// conflicts; V rows; the block's factors.  The next stage comes in while this one is worked on.
template <int KT, int NW>
__global__ __launch_bounds__(64 * NW, 2) void mlstm_blocks_kernel(RunArgs ra) {
  extern __shared__ __align__(16) char lds_raw[];
  const zp_mlstm& a = ra.d;
  constexpr int dk = 16 * KT, dv = 16 * NW, PR = dk / 8, J = KT / 2;      // PR: pieces per row of Q and K
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int unit = blockIdx.x / ra.pieces.most, h = unit % a.heads, seg = unit / a.heads;
  const Segment whole = segment_of(a.seg, seg);
  if (whole.count <= 0 || whole.row < ra.row0) return;
  const Piece piece(ra.pieces, ra.row0, whole, seg, blockIdx.x % ra.pieces.most);
  const Segment& sg = piece.sg;
  if (sg.count <= 0) return;
  constexpr int v_bytes = kBlock * dv * 2, stage = 2 * kBlock * dk * 2 + v_bytes + kAux * 4;
  float (*const red)[NW * kBlock] = (float (*)[NW * kBlock])(lds_raw + 2 * stage);
  float (*const den)[kBlock] = (float (*)[kBlock])(red + 2);
  float (*const nl)[dk] = (float (*)[dk])(den + 2);
  float* const state = a.state + ((int64_t)sg.slot * a.heads + h) * ((int64_t)dk * dv + dk + 4);
  float* const nstate = state + (int64_t)dk * dv;
  const bool fresh = sg.start == 0;
  const int col0 = wave * 16;
  f32x4 S[KT][1];
  if (ra.pieces.blocks) {
    const float* const from = ra.pieces.states + (piece.slot * a.heads + h) * piece_floats(dk, dv);
    load_piece_state(S, from, wave);
    for (int c = tid; c < dk; c += blockDim.x) nl[0][c] = from[dk * dv + c];
  } else {
    load_state<KT, 1>(S, state, dv, col0, fresh);
    for (int c = tid; c < dk; c += blockDim.x) nl[0][c] = fresh ? 0.f : nstate[c];
  }
  const float nrm = a.norm[h * dv + col0 + l16] * a.out_scale;
  const int blocks = (sg.count + kBlock - 1) / kBlock;
  const float* const aux0 = ra.aux + (block_slot(ra.row0, sg, seg, 0) * a.heads + h) * kAux;
  constexpr int kQK = KT / 2;                  // KBs of Q, and of K
  // a share of `kbs` KBs; the last may come twice
  auto share = [&](auto kbs, auto ld) {
#pragma unroll
    for (int u = 0; u < (kbs.value + NW - 1) / NW; ++u) ld(min(wave + u * NW, kbs.value - 1));
  };
  auto request = [&](int b) {                  // of a block behind the last nothing is read
    char* const st = lds_raw + (b & 1) * stage;
    const int cnt = b < blocks ? min(kBlock, sg.count - b * kBlock) : 0;
    const StageLoads rows((const char*)a.in + (int64_t)(sg.row + b * kBlock) * a.in_stride * 2, cnt * a.in_stride * 2);
    const StageLoads aux(aux0 + (int64_t)b * a.heads * kAux, cnt > 0 ? kAux * 4 : 0);
    share(std::integral_constant<int, kQK>(), [&](int i) {
      const int s = i * 64 + lane, row = s / PR, pc = (s % PR) ^ (row & (PR - 1));
      const int at = max(min(row, cnt - 1), 0) * (int)a.in_stride * 2 + pc * 16;
      rows.ld(st + i * 1024, at, (a.q_at + h * dk) * 2);
      rows.ld(st + (kQK + i) * 1024, at, (a.k_at + h * dk) * 2);
    });
    share(std::integral_constant<int, NW / 2>(), [&](int i) {
      const int s = i * 64 + lane, row = s / (dv / 8), pc = s - row * (dv / 8);
      rows.ld(st + (2 * kQK + i) * 1024, max(min(row, cnt - 1), 0) * (int)a.in_stride * 2 + pc * 16, (a.v_at + h * dv) * 2);
    });
    share(std::integral_constant<int, 2>(), [&](int i) { aux.ld(st + (2 * kQK + NW / 2 + i) * 1024, lane * 16, i * 1024); });
  };
  f32x4 done = {0.f, 0.f, 0.f, 0.f};
  uint16_t gate[4] = {0, 0, 0, 0};
  const float inv_v = 1.f / (float)a.vdim;
  const int out_at = (4 * g * (int)a.out_stride + h * dv + col0 + l16) * 2;
  const int gate_at = (4 * g * (int)a.in_stride + a.g_at + h * dv + col0 + l16) * 2;
  auto finish = [&](int b) {                   // rows of block b, whose squares and denominators are in LDS; none of block -1
    const f32x4 ss = block_squares_total<NW>(red[b & 1]);
    const f32x4 dn = *(const f32x4*)(den[b & 1] + 4 * g);
    const int cnt = b < 0 ? 0 : min(kBlock, sg.count - b * kBlock);
    const BlockRows out(a.out, sg.row + b * kBlock, cnt, a.out_stride);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float f = a.q_scale * __builtin_amdgcn_rcpf(dn[r]), rs = f * __builtin_amdgcn_rsqf(ss[r] * f * f * inv_v + a.eps);
      out.st(out_at + r * (int)a.out_stride * 2, 0, done[r] * rs * nrm * fast_sigmoid(bf16_bits_to_float(gate[r])));
    }
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
#pragma unroll 1
  for (int b = 0; b < blocks; ++b) {
    wait_and_meet();
    request(b + 1);
    const int cnt = min(kBlock, sg.count - b * kBlock);
    const BlockRows gp(a.in, sg.row + b * kBlock, cnt, a.in_stride);
    uint16_t next[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) next[r] = gp.ld(gate_at + r * (int)a.in_stride * 2, 0);
    const char* const st = lds_raw + (b & 1) * stage;
    const char* const ks = st + kBlock * dk * 2;
    const uint16_t* const vs = (const uint16_t*)(ks + kBlock * dk * 2);
    const float* const aux = (const float*)((const char*)vs + v_bytes);
    // ---- read-outs
    f32x4 O[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
    const char* const qrow = st + l16 * dk * 2 + (g & 1) * 8;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const uint2 q0 = *(const uint2*)(qrow + ((4 * j + (g >> 1)) ^ (l16 & (PR - 1))) * 16);
      const uint2 q1 = *(const uint2*)(qrow + ((4 * j + 2 + (g >> 1)) ^ (l16 & (PR - 1))) * 16);
#pragma unroll
      for (int k = 2; k >= 0; --k) O[0] = mfma_bf16(u32x4{q0.x, q0.y, q1.x, q1.y}, sp[k][j], O[0]);      // the smallest first
    }
    const u32x4 P = *(const u32x4*)(aux + lane * 4);
    const uint2 Pl = *(const uint2*)(aux + 256 + lane * 2);
    const f32x4 inter = *(const f32x4*)(aux + kInter + 4 * g), wr = *(const f32x4*)(aux + kWrite + 4 * g);
    const float keep = aux[kKeep];
    const uint2 v4 = read_transposed(vs + (4 * g + (l16 >> 2)) * dv + col0 + (l16 & 3) * 4);
    O[0] *= inter;
    O[0] = mfma_bf16(u32x4{Pl.x, Pl.y, 0u, 0u}, u32x4{v4.x, v4.y, v4.x, v4.y}, O[0]);
    O[0] = mfma_bf16(P, u32x4{v4.x, v4.y, v4.x, v4.y}, O[0]);
    // ---- the state behind the block
    const f32x4 v = {__uint_as_float(v4.x << 16), __uint_as_float(v4.x & 0xffff0000u), __uint_as_float(v4.y << 16), __uint_as_float(v4.y & 0xffff0000u)};
    const Planes vw(v * wr);
    const int kr = 4 * g + (l16 >> 2), kz = ((l16 & 3) >> 1) ^ (kr & (PR - 1));
    const char* const krow = ks + kr * dk * 2 + (l16 & 1) * 8;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      const uint2 k4 = read_transposed((const uint16_t*)(krow + ((2 * kt) ^ kz) * 16));
      S[kt][0] *= keep;
      S[kt][0] = mfma_bf16(u32x4{k4.x, k4.y, 0u, 0u}, u32x4{vw.lo.x, vw.lo.y, 0u, 0u}, S[kt][0]);
      S[kt][0] = mfma_bf16(u32x4{k4.x, k4.y, k4.x, k4.y}, u32x4{vw.hi.x, vw.hi.y, vw.mid.x, vw.mid.y}, S[kt][0]);
    }
    finish(b - 1);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) split_state(kt);
#pragma unroll
    for (int i = 0; i < 3; ++i)                // here, not behind the squares
#pragma unroll
      for (int j = 0; j < J; ++j) settle(sp[i][j]);
#pragma unroll
    for (int r = 0; r < 4; ++r) gate[r] = next[r];
    block_squares<1>(O, red[b & 1], wave);
    done = O[0];
    // ---- the normaliser: 16 lanes a token, by the waves that come first anyway
    const float* const n = nl[b & 1];
#pragma unroll
    for (int u = 0; u < kBlock; u += 4 * NW) {
      if (wave * 4 + u >= kBlock) continue;    // uniform
      const int t = wave * 4 + u + g, pc = min(l16, PR - 1);
      float q[8], d = 0.f;
      Vec8<BF16>::ld(st + t * dk * 2 + ((pc ^ (t & (PR - 1))) * 16), 0, q);
#pragma unroll
      for (int i = 0; i < 8; ++i) d = fmaf(q[i], n[pc * 8 + i], d);
      d = row16_sum(l16 < PR ? d : 0.f);
      const float x = fmaxf(fabsf(fmaf(aux[kInter + t], d, aux[kSum + t])) * a.q_scale, aux[kFloor + t]) + 1e-6f;
      if (l16 == 0) den[b & 1][t] = x;
    }
#pragma unroll
    for (int u = 0; u < KT; u += 4 * NW) {
      if (wave * 4 + u >= KT) continue;
      const int kt = min(wave * 4 + u + g, KT - 1);                  // channel 16 kt + l16
      float x = n[kt * 16 + l16] * keep;
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        const int r = 4 * s4 + (l16 >> 2);
        const f32x4 k4 = read_columns(ks + r * dk * 2 + (((2 * kt + ((l16 & 3) >> 1)) ^ (r & (PR - 1))) * 16) + (l16 & 1) * 8);
        const f32x4 w4 = *(const f32x4*)(aux + kWrite + 4 * s4);
#pragma unroll
        for (int i = 0; i < 4; ++i) x = fmaf(w4[i], k4[i], x);
      }
      nl[(b + 1) & 1][kt * 16 + l16] = x;
    }
  }
  wait_and_meet();
  finish(blocks - 1);
  if (!piece.last) return;
  store_state<KT, 1>(S, state, dv, col0);
  for (int c = tid; c < dk; c += blockDim.x) nstate[c] = nl[blocks & 1][c];
}

template <int KT, int NW> int launch_blocks(const RunArgs& ra, hipStream_t st) {
  constexpr int dk = 16 * KT, dv = 16 * NW;
  constexpr size_t smem = 2 * (2 * kBlock * dk * 2 + kBlock * dv * 2 + kAux * 4) + 2 * 4 * (NW * kBlock + kBlock + dk);
  const int64_t units = (int64_t)ra.d.seg.n * ra.d.heads;
  if (ra.pieces.blocks) {
    hipLaunchKernelGGL((mlstm_sums_kernel<KT, NW>), dim3((unsigned)(units * (ra.pieces.most - 1))), dim3(64 * KT), 0, st, ra);
    ZP_LAUNCH_CHECK();
    hipLaunchKernelGGL((mlstm_states_kernel<KT, NW>), dim3((unsigned)units, KT * NW / 4), dim3(256), 0, st, ra);
    ZP_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL((mlstm_blocks_kernel<KT, NW>), dim3((unsigned)(units * ra.pieces.most)), dim3(64 * NW), smem, st, ra);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}

template <int KT> int launch_runs(const RunArgs& ra, int longest, hipStream_t st) {
  const zp_mlstm& a = ra.d;
  const unsigned grid = (unsigned)((int64_t)a.seg.n * a.heads);
  const int waves = longest < 64 * kGateWaves ? (longest + 63) / 64 : kGateWaves;
  hipLaunchKernelGGL(mlstm_gates_kernel, dim3(grid), dim3(64 * waves), 0, st, ra);
  hipLaunchKernelGGL((mlstm_prepare_kernel<KT>), dim3((unsigned)((longest + kBlock - 1) / kBlock), (unsigned)((a.heads + 3) / 4), (unsigned)a.seg.n),
                     dim3(256), 0, st, ra);
  ZP_LAUNCH_CHECK();
  switch (a.dv / 32) {
    case 1: return launch_blocks<KT, 2>(ra, st);
    case 2: return launch_blocks<KT, 4>(ra, st);
    case 3: return launch_blocks<KT, 6>(ra, st);
    default: return launch_blocks<KT, 8>(ra, st);
  }
}

}  // namespace

static int64_t blocks_bytes(int64_t rows, int64_t segments, int64_t heads) {
  return ((rows / kBlock + segments) * kAux + rows * 4) * heads * 4;
}

constexpr PieceCost kCost = {1, 3, 75, 0};

// With room for the states between pieces of few heads' runs, whatever the sizes and the longest run.
extern "C" int64_t zp_mlstm_runs_workspace(int32_t rows, int32_t segments, int32_t heads) {
  if (rows < 0 || segments < 0 || heads <= 0) return -1;
  return blocks_bytes(rows, segments, heads) + most_states(rows, segments, heads, kCost) * piece_floats(128, 128) * 4;
}

extern "C" int zp_mlstm_runs(const zp_mlstm* args, int32_t first_row, int32_t longest, void* workspace,
                             int64_t workspace_bytes, int32_t dtype, void* stream) {
  ZP_REQUIRE(args, "mlstm_runs: null arguments");
  const zp_mlstm& a = *args;
  ZP_REQUIRE(a.seg.n >= 0 && a.heads > 0 && a.vdim > 0 && a.vdim <= a.dv && a.cap > 0.f && a.seg.num_slots > 0 &&
                 a.gate_stride >= 2 * a.heads && a.out_stride >= (int64_t)a.heads * a.dv && first_row >= 0 && longest >= 0 &&
                 first_row <= a.seg.num_rows, "mlstm_runs: bad dims");
  if (dtype != ZP_BF16 || (a.dk != 32 && a.dk != 64 && a.dk != 128) || a.dv % 32 || a.dv > 128 || a.in_stride % 8 || a.q_at % 8 ||
      a.k_at % 8 || a.v_at % 8 || a.in_stride >= (1 << 24) || a.out_stride >= (1 << 24) || a.heads > 65535 || a.seg.n > 65535) {
    zp_set_error("mlstm_runs: bfloat16, head sizes %d (32, 64, 128) and %d (a multiple of 32, <= 128) unsupported", a.dk, a.dv);
    return ZP_EUNSUPPORTED;
  }
  if (a.seg.n == 0 || longest == 0) return ZP_OK;
  ZP_REQUIRE(a.in && a.gates && a.i_bias && a.f_bias && a.norm && a.state && a.out && a.seg.rows && a.seg.counts &&
                 a.seg.slots && a.seg.starts && aligned16(a.in) && aligned16(a.state) && aligned16(workspace),
             "mlstm_runs: null or unaligned pointer");
  const int64_t rows = a.seg.num_rows - first_row, whole = blocks_bytes(rows, a.seg.n, a.heads);
  ZP_REQUIRE(workspace && workspace_bytes >= whole, "mlstm_runs: workspace too small");
  RunArgs ra = {a, (float*)workspace, nullptr, first_row, {}};
  ra.pieces = pieces_of(rows, a.seg.n, a.heads, longest, kCost, 1, (workspace_bytes - whole) / 4 / piece_floats(a.dk, a.dv));
  ra.pieces.states = (float*)workspace + whole / 4;
  ra.scal = (float4*)(ra.aux + ((int64_t)(a.seg.num_rows - first_row) / kBlock + a.seg.n) * a.heads * kAux);
  ra.d.seg.max_count = longest;               // no segment has more blocks than were prepared
  hipStream_t st = (hipStream_t)stream;
  switch (a.dk) {
    case 32: return launch_runs<2>(ra, longest, st);
    case 64: return launch_runs<4>(ra, longest, st);
    default: return launch_runs<8>(ra, longest, st);
  }
}
