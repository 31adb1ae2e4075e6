// Latent attention: keys and values of all heads are linear images of one cached vector c per token
// (R elements), so the cache holds c alone, or c and a rotated key part (P elements) that all heads share.
//
//   latent_norm_store   RMS norms of the two low-rank projections of a token; c, and the key part turned by
//                       the token's position, go to its slot
//   headwise            per-head product out[n, h] = W[h] in[n, h]  (q -> W_uk^T q, sum p c -> W_uv sum p c);
//                       a tail behind each head's part passes beside it, turned
//   rotate_heads        rotary positions on a part of every head, in place
//   latent_rows         attention of single tokens over the paged latents, all heads of a token on
//                       one read of its context: score = (W_uk^T q) . c + turned q . turned k, out = sum p c
//   latent_plain        float32 form of latent_rows (true fp32 products), any sizes
//
// The attention of runs of prompt tokens over expanded keys and values is in runs.hip.
//
// The bf16 attention kernels keep S^T = K Q^T and O^T = V^T P^T: in that orientation the MFMA
// result layout of S^T (column = query, four consecutive keys per lane) IS the operand layout of
// P^T once the 32 keys of a step are numbered (lane group g holds keys 4g..4g+3 and
// 16+4g..16+4g+3), so the softmax weights never leave their lane: no LDS and no barrier in the key
// loop, every wave is its own flash loop.  V^T operands are built from row-major 16-byte loads of
// eight keys x eight columns by v_perm; the column order that results (MFMA t, row m <-> column
// 8m + t) leaves eight consecutive output columns in each lane.
#include "mfma.h"
#include <algorithm>
#include <math.h>

namespace {

// ------------------------------------------------------------------ norms of the low-rank rows
struct NormStoreArgs {
  const void* in;        // (n, q_width + c_width + p_width) T
  const float* wq;       // (q_width,)
  const float* wc;       // (c_width,)
  void* q_out;           // (n, q_width) T
  void* c_out;           // (n, c_width + p_width) T or null
  void* cache;           // (num_slots, c_width + p_width) T
  const int32_t* slots;  // (n,), -1 skips
  const int32_t* positions;
  const float* freqs;    // (half,)
  int n, q_width, c_width, p_width, q_norm, c_norm, half;   // half: rotated pairs of the last part
  int64_t num_slots;
  float eps;
};
constexpr int kNormPieces = 8;   // 8-element pieces per lane: ranks up to 4096

// One wave per (token, part); without a second part, per token.
template <typename T>
__global__ __launch_bounds__(256) void latent_norm_store_kernel(NormStoreArgs a) {
  const int lane = threadIdx.x & 63;
  const int item = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int row = a.c_width ? item >> 1 : item;
  if (row >= a.n) return;
  const bool is_c = a.c_width && (item & 1);
  const int width = is_c ? a.c_width : a.q_width, held = a.c_width + a.p_width;
  const int pieces = width / 8;
  const int64_t src = (int64_t)row * (a.q_width + held) + (is_c ? a.q_width : 0);
  const float* w = is_c ? a.wc : a.wq;
  float v[kNormPieces][8];
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < kNormPieces; ++k) {
    const int pc = lane + k * 64;
    if (pc < pieces) {
      Vec8<T>::ld(a.in, src + pc * 8, v[k]);
#pragma unroll
      for (int i = 0; i < 8; ++i) ss += v[k][i] * v[k][i];
    }
  }
  ss = wave_sum(ss);
  const float rs = 1.f / sqrtf(ss / (float)(is_c ? a.c_norm : a.q_norm) + a.eps);
  int64_t slot = is_c ? a.slots[row] : -1;
  if (slot >= a.num_slots) slot = -1;
#pragma unroll
  for (int k = 0; k < kNormPieces; ++k) {
    const int pc = lane + k * 64;
    if (pc < pieces) {
      float wv[8];
      Vec8<F32>::ld(w, pc * 8, wv);
#pragma unroll
      for (int i = 0; i < 8; ++i) v[k][i] = v[k][i] * rs * wv[i];
      if (is_c) {
        if (slot >= 0) Vec8<T>::st(a.cache, slot * held + pc * 8, v[k]);
        if (a.c_out) Vec8<T>::st(a.c_out, (int64_t)row * held + pc * 8, v[k]);
      } else {
        Vec8<T>::st(a.q_out, (int64_t)row * width + pc * 8, v[k]);
      }
    }
  }
  if (!is_c) return;
  // the key part: pairs (i, half + i) turn, what follows them passes
  const int rest = a.p_width - 2 * a.half;
  for (int i = lane; i < a.half + rest; i += 64) {
    float x[2];
    int at[2] = {i, i + a.half};
    const int cnt = i < a.half ? 2 : 1;
    if (cnt == 1) at[0] = i + a.half;
    for (int k = 0; k < cnt; ++k) x[k] = Elem<T>::ld(a.in, src + width + at[k]);
    if (cnt == 2) {
      const float2 r = rotary_turn(a.positions[row], a.freqs[i]);
      const float u = x[0], w2 = x[1];
      x[0] = u * r.x - w2 * r.y;
      x[1] = w2 * r.x + u * r.y;
    }
    for (int k = 0; k < cnt; ++k) {
      if (slot >= 0) Elem<T>::st(a.cache, slot * held + width + at[k], x[k]);
      if (a.c_out) Elem<T>::st(a.c_out, (int64_t)row * held + width + at[k], x[k]);
    }
  }
}

// ------------------------------------------------------------------ rotary positions in place
struct RotateArgs {
  void* x;                  // token rows of x_st elements; head h's part at h * head + at
  const int32_t* positions;
  const float* freqs;
  int n, H, head, at, half;
  int64_t x_st;
};
constexpr int kRotTokens = 4;

template <typename T, int VEC>
__global__ __launch_bounds__(256) void rotate_heads_kernel(RotateArgs a) {
  extern __shared__ __align__(16) char lds_raw[];
  float2* cs = (float2*)lds_raw;            // [kRotTokens][half]
  const int n0 = blockIdx.x * kRotTokens;
  for (int i = threadIdx.x; i < kRotTokens * a.half; i += 256) {
    const int tok = i / a.half;
    if (n0 + tok < a.n) cs[i] = rotary_turn(a.positions[n0 + tok], a.freqs[i - tok * a.half]);
  }
  __syncthreads();
  const int per_head = a.half / VEC, items = a.H * per_head;
  for (int id = threadIdx.x; id < kRotTokens * items; id += 256) {
    const int tok = id / items, it = id - tok * items;
    if (n0 + tok >= a.n) break;
    const int h = it / per_head, p = (it - h * per_head) * VEC;
    const int64_t at = (n0 + tok) * a.x_st + (int64_t)h * a.head + a.at + p;
    float u[VEC], v[VEC];
    if constexpr (VEC == 8) { Vec8<T>::ld(a.x, at, u); Vec8<T>::ld(a.x, at + a.half, v); }
    else { u[0] = Elem<T>::ld(a.x, at); v[0] = Elem<T>::ld(a.x, at + a.half); }
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      const float2 r = cs[tok * a.half + p + i];
      const float x = u[i], y = v[i];
      u[i] = x * r.x - y * r.y;
      v[i] = y * r.x + x * r.y;
    }
    if constexpr (VEC == 8) { Vec8<T>::st(a.x, at, u); Vec8<T>::st(a.x, at + a.half, v); }
    else { Elem<T>::st(a.x, at, u[0]); Elem<T>::st(a.x, at + a.half, v[0]); }
  }
}

// ------------------------------------------------------------------ per-head product
struct HeadArgs {
  const void* in;   // (n, H, K + tail) T
  const void* w;    // (H, M, K) T
  void* out;        // (n, H, M + tail) T
  const int32_t* positions;
  const float* freqs;
  int n, H, K, M, tail, half;   // behind each head's part `tail` elements, of which 2 * half turn
};

// What lies behind head h's part in `tokens` tokens from n0 on: share `part` of `parts`, one of a workgroup (one workgroup
// for all, and the others of its head waited for it: 256 tokens, 32 heads of 128 -> 512 with 64 behind them 19.2 us, 15.1).
template <typename T>
__device__ __forceinline__ void head_tails(const HeadArgs& a, int h, int n0, int tokens, int part, int parts) {
  const int rest = a.tail - a.half;               // items of a token: the pairs, then what follows them
  for (int it = part * 256 + threadIdx.x; it < tokens * rest; it += parts * 256) {
    const int tok = it / rest, i = it - tok * rest, n = n0 + tok;
    if (n >= a.n) break;
    const int64_t from = ((int64_t)n * a.H + h) * (a.K + a.tail) + a.K, to = ((int64_t)n * a.H + h) * (a.M + a.tail) + a.M;
    if (i < a.half) {
      const float2 r = rotary_turn(a.positions[n], a.freqs[i]);
      const float u = Elem<T>::ld(a.in, from + i), v = Elem<T>::ld(a.in, from + i + a.half);
      Elem<T>::st(a.out, to + i, u * r.x - v * r.y);
      Elem<T>::st(a.out, to + i + a.half, v * r.x + u * r.y);
    } else {
      Elem<T>::st(a.out, to + i + a.half, Elem<T>::ld(a.in, from + i + a.half));
    }
  }
}

// bf16.  Workgroup: 64 outputs of one head for 16 * TT tokens; a wave has MT tiles of 16 outputs for NT of 16 tokens.
//
// Operands pass through LDS: read from memory as they are multiplied, a load touches 16 rows for 64 bytes each and keeps
// the L1 for some 70 cycles; whole rows are a quarter of that (256 tokens, 32 heads, 128 -> 512 with 64 behind: 15.1 us, now
// 7.6; 512 -> 128: 13.4, now 6.1; 2048 tokens, 16 heads 45 and 39, now 22 and 18).  Stages hold 128 elements of a row, and
// all of them are on their way at once where K is at most 512.  A row's sixteen 16-byte pieces lie in the order of
// (piece ^ row), so that no two rows of an operand meet in a bank.  W is the row operand; the rows of two tiles alternate
// by fours, so that a lane ends with eight consecutive outputs of a token.  Workgroups of a head follow one another on one
// XCD, whose L2 holds its W and its tokens.
constexpr int kHeadStage = 128, kHeadRing = 4;
template <int TT> struct HeadTile {
  static constexpr int MT = TT > 1 ? 2 : 1, NT = TT > 1 ? TT / 2 : 1;
  static constexpr int kBytes = (64 + 16 * TT) * kHeadStage * 2, kLoads = 4 + TT;     // of a stage; of a wave for one
};
template <int kLeft> __device__ __forceinline__ void wait_loads_left() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0f70 | (kLeft & 15) | (kLeft >> 4) << 14);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
template <int TT>
__global__ __launch_bounds__(256) void headwise_tile_kernel(HeadArgs a, int blocks_m, int blocks_n) {
  extern __shared__ __align__(16) char lds_raw[];
  typedef HeadTile<TT> Tile;
  constexpr int MT = Tile::MT, NT = Tile::NT;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int total = gridDim.x;
  int id = total % 8 == 0 ? (int)(blockIdx.x % 8) * (total / 8) + blockIdx.x / 8 : blockIdx.x;
  const int bm = id % blocks_m;
  id /= blocks_m;
  const int n0 = id % blocks_n * 16 * TT, h = id / blocks_n;
  const int x_row = a.H * (a.K + a.tail) * 2;                    // bytes from token to token
  const u32x4 wr = rows_from((const uint16_t*)a.w + ((int64_t)h * a.M + bm * 64) * a.K, (uint32_t)min(64, a.M - bm * 64) * a.K * 2);
  const u32x4 xr = rows_from((const uint16_t*)a.in + ((int64_t)n0 * a.H + h) * (a.K + a.tail),
                             (uint32_t)(min(16 * TT, a.n - n0) - 1) * x_row + a.K * 2);
  const int stages = (a.K + kHeadStage - 1) / kHeadStage, ring = min(stages, kHeadRing);
  // loads of a stage: four rows each, first of W, then of the tokens; what is not there has an address past the end
  int from[Tile::kLoads];
#pragma unroll
  for (int i = 0; i < Tile::kLoads; ++i) {
    const int at = wave * Tile::kLoads + i, row = at * 4 + g;
    int r = at < 16 ? row : row - 64;
    if (at < 16 && MT == 2) r = (r & 32) + ((r & 12) << 1) + ((r & 16) >> 2) + (r & 3);
    const bool there = at < 16 ? bm * 64 + r < a.M : n0 + r < a.n;
    from[i] = (there ? r * (at < 16 ? a.K * 2 : x_row) : INT_MIN) + (l16 ^ (row & 15)) * 16;
  }
  auto issue = [&](int s) {
    char* const to = lds_raw + (s % kHeadRing * Tile::kBytes + wave * Tile::kLoads * 1024);
    const bool whole = (s + 1) * kHeadStage <= a.K;
#pragma unroll
    for (int i = 0; i < Tile::kLoads; ++i) {
      int at = from[i] + s * 256;
      if (!whole) at = s * 256 + (l16 ^ ((wave * Tile::kLoads + i) * 4 + g & 15)) * 16 < a.K * 2 ? at : INT_MIN;
      load_to_lds(wave * Tile::kLoads + i < 16 ? wr : xr, to + i * 1024, at, 0);
    }
  };
  for (int s = 0; s < ring; ++s) issue(s);
  if (a.tail) head_tails<BF16>(a, h, n0, 16 * TT, bm, blocks_m);
  const int m_row = (MT == 2 ? (wave & 1) * 32 : wave * 16) + l16, x_first = (TT == 1 ? 0 : (wave >> 1) * 16 * NT) + l16;
  f32x4 acc[MT][NT] = {};
  for (int s = 0; s < stages; ++s) {
    const int behind = min(stages - 1 - s, kHeadRing - 1);       // stages on their way behind this one
    if (behind == 0) wait_loads_left<0>();
    else if (behind == 1) wait_loads_left<Tile::kLoads>();
    else if (behind == 2) wait_loads_left<2 * Tile::kLoads>();
    else wait_loads_left<3 * Tile::kLoads>();
    const char* const at = lds_raw + s % kHeadRing * Tile::kBytes;
    u32x4 wf[4][MT], xf[4][NT];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int piece = ((ks * 4 + g) ^ l16) * 16;
#pragma unroll
      for (int j = 0; j < MT; ++j) wf[ks][j] = *(const u32x4*)(at + (m_row + j * 16) * 256 + piece);
#pragma unroll
      for (int t = 0; t < NT; ++t) xf[ks][t] = *(const u32x4*)(at + (64 + x_first + t * 16) * 256 + piece);
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)                               // what lies behind the contraction's end is zero
#pragma unroll
      for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[j][t] = mfma_bf16(wf[ks][j], xf[ks][t], acc[j][t]);
    if (s + kHeadRing < stages) {
      __builtin_amdgcn_s_waitcnt(0xc07f);                        // this stage has been read
      wait_loads_left<63>();
      issue(s + kHeadRing);
    }
  }
  const int m = bm * 64 + (MT == 2 ? (wave & 1) * 32 + g * 8 : wave * 16 + g * 4);
  if (m >= a.M) return;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int n = n0 + x_first + t * 16;
    if (n >= a.n) continue;
    uint16_t* const out = (uint16_t*)a.out + ((int64_t)n * a.H + h) * (a.M + a.tail) + m;
    const f32x4 u = acc[0][t], v = acc[MT - 1][t];
    if constexpr (MT == 2) *(u32x4*)out = u32x4{pack_bf16(u[0], u[1]), pack_bf16(u[2], u[3]), pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
    else *(uint2*)out = uint2{pack_bf16(u[0], u[1]), pack_bf16(u[2], u[3])};
  }
}

// A wave owns 16 outputs of one head for 16 * kTokTiles tokens: W is the row operand, so a lane ends
// with four consecutive outputs of one token.  Token rows past the end repeat the last one.
template <typename T, int kTokTiles>
__global__ __launch_bounds__(256) void headwise_kernel(HeadArgs a) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int m0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 16;
  const int h = blockIdx.y;
  const int n0 = blockIdx.z * 16 * kTokTiles;
  if (a.tail) head_tails<T>(a, h, n0, 16 * kTokTiles, blockIdx.x, gridDim.x);
  if (m0 >= a.M) return;
  f32x4 acc[kTokTiles];
#pragma unroll
  for (int t = 0; t < kTokTiles; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int64_t wrow = ((int64_t)h * a.M + m0 + l16) * a.K;
  int64_t xrow[kTokTiles];
#pragma unroll
  for (int t = 0; t < kTokTiles; ++t)
    xrow[t] = ((int64_t)min(n0 + t * 16 + l16, a.n - 1) * a.H + h) * (a.K + a.tail);
  if constexpr (T::bytes == 2) {
    const uint16_t* w = (const uint16_t*)a.w;
    const uint16_t* x = (const uint16_t*)a.in;
    const int steps = a.K / 32;
#pragma unroll 4
    for (int ks = 0; ks < steps; ++ks) {
      const int k = ks * 32 + g * 8;
      const u32x4 wf = *(const u32x4*)(w + wrow + k);
#pragma unroll
      for (int t = 0; t < kTokTiles; ++t) acc[t] = mfma_bf16(wf, *(const u32x4*)(x + xrow[t] + k), acc[t]);
    }
  } else {
    const float* w = (const float*)a.w;
    const float* x = (const float*)a.in;
    const int steps = a.K / 4;
#pragma unroll 4
    for (int ks = 0; ks < steps; ++ks) {
      const int k = ks * 4 + g;
      const float wf = w[wrow + k];
#pragma unroll
      for (int t = 0; t < kTokTiles; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf, x[xrow[t] + k], acc[t], 0, 0, 0);
    }
  }
#pragma unroll
  for (int t = 0; t < kTokTiles; ++t) {
    const int n = n0 + t * 16 + l16;
    if (n < a.n) {
      const int64_t at = ((int64_t)n * a.H + h) * (a.M + a.tail) + m0 + g * 4;
      if constexpr (T::bytes == 2) {
        uint2 o;
        o.x = pack_bf16(acc[t][0], acc[t][1]);
        o.y = pack_bf16(acc[t][2], acc[t][3]);
        *(uint2*)((uint16_t*)a.out + at) = o;
      } else {
        *(f32x4*)((float*)a.out + at) = acc[t];
      }
    }
  }
}

// ------------------------------------------------------------------ single tokens over the pages
struct RowsArgs {
  const void* q;          // (n, H, R + P) T
  const void* cache;      // (pages, BS, R + P) T
  const int32_t* table;   // (B, NB) page ids
  const int32_t* ctx;     // (n,) tokens of the sequence up to and including this one; 0 = inert
  const int32_t* seq;     // (n,) row of table, or null: row i
  void* out;              // (n, H, R) T
  float* part;            // splits > 1: (n, H, splits, R) fp32, then (n, H, splits, 2) max and sum
  int n, H, R, P, BS, bs_shift, B, NB, num_pages;   // P: elements that only join the scores
  int window;             // a token sees the last `window` tokens including itself; 0 = all
  int splits;             // key ranges handled by different workgroups
  int lds_pages;          // narrow rows: page ids held in LDS
  float scale;
};

__device__ __forceinline__ int page_of(const RowsArgs& a, int t) {
  return a.bs_shift >= 0 ? t >> a.bs_shift : t / a.BS;
}

// Rows of at most 256 for up to 32 heads: a step of 32 keys is too little work to have the waves meet for it (256
// sequences, 16 heads: 72 us; by the kernel below 75), so every wave goes its own way.  NCB column blocks of 128 cover R.
// Workgroup: one token, one key range.  A wave computes HT tiles of 16 heads on the same keys: with two, the second tile
// costs no key or value read.
//
// A wave takes 32 keys at a time.  They come from memory once, as whole 256-byte row pieces (lane: 8
// keys x 8 columns), and stay in registers as the value operand; the key operand (lane: one key, 8
// columns per MFMA) would touch 16 cache lines per 16 lanes if it were read from memory, so the wave
// passes each half of the block through an LDS stage of its own.  The next block's pieces are
// requested as the value products free their registers.  No barrier until the waves meet at the end.
// The rotated part (PK MFMA steps) is a key only, never a value: it is read as a key operand straight from
// memory, P elements of a key per four lanes.
template <int NCB, int PK> struct RowsLds {
  static constexpr int kStride = NCB * 128 + 8;                  // elements: rows 16 bytes apart in the banks
  static constexpr int kStage = 16 * kStride * 2;                // bytes per wave: 16 keys
  static constexpr int kQStride = kStride + PK * 32;             // with 64 more: an odd number of 16 bytes still
  static constexpr int kQ = 16 * kQStride * 2;                   // bytes per 16 heads
};
__host__ __device__ inline int rows_merge_floats(int R) { return 16 * (R + 4) + 32; }   // per wave

template <int NCB, int HT, int PK, bool PAST> __device__ __forceinline__ void latent_narrow(const RowsArgs& a) {
  extern __shared__ __align__(16) char lds_raw[];
  typedef RowsLds<NCB, PK> Lds;
  int* pg = (int*)lds_raw;
  char* const shared = lds_raw + ((a.lds_pages * 4 + 15) & ~15);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  uint16_t* const stage = (uint16_t*)(shared + wave * Lds::kStage);
  uint16_t* const qlds = (uint16_t*)(shared + 4 * Lds::kStage);
  const int split = blockIdx.x % a.splits, row = blockIdx.x / a.splits;
  // queries to LDS, zeros past R and past the last head
  const int RW = a.R + a.P;
  constexpr int kQPieces = NCB * 16 + PK * 4;
  for (int it = tid; it < HT * 16 * kQPieces; it += 256) {
    const int hl = it / kQPieces, c = (it % kQPieces) * 8;
    const int p = c - NCB * 128;                                 // >= 0: of the rotated part
    u32x4 v = {0u, 0u, 0u, 0u};
    if (hl < a.H && (p < 0 ? c < a.R : p < a.P))
      v = *(const u32x4*)((const uint16_t*)a.q + ((int64_t)row * a.H + hl) * RW + (p < 0 ? c : a.R + p));
    *(u32x4*)(qlds + hl * Lds::kQStride + c) = v;
  }
  const int seq = a.seq ? min(max(a.seq[row], 0), a.B - 1) : row;
  const int n = min(a.ctx[row], a.NB * a.BS);
  const int lo = a.window > 0 ? max(0, n - a.window) : 0;
  const int p0 = lo >> a.bs_shift;
  constexpr int KS = 4 * NCB;

  // every entry gets a valid page, whatever the context length says: no address rests on it
  for (int j = tid; j < a.lds_pages; j += 256) {
    const int p = p0 + j < a.NB ? a.table[(int64_t)seq * a.NB + p0 + j] : 0;
    pg[j] = (p >= 0 && p < a.num_pages) ? p : 0;
  }
  __syncthreads();
  // R may end inside the last column block: columns past it hold the row's start again, and meet
  // zeros in q or results that are not written
  int col_off[NCB];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    const int c = cb * 128 + l16 * 8;
    col_off[cb] = (c < a.R ? c : 0) * 2;
  }
  f32x4 o[HT][NCB * 8];
  float m[HT], l[HT];
#pragma unroll
  for (int ht = 0; ht < HT; ++ht) {
    m[ht] = -INFINITY;
    l[ht] = 0.f;
#pragma unroll
    for (int i = 0; i < NCB * 8; ++i) o[ht][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float sc = a.scale * 1.44269504088896f;
  const uint16_t* const qrow = qlds + l16 * Lds::kQStride + g * 8;
  const int mask = a.BS - 1;
  u32x4 v[NCB][8], kr[2][PK ? PK : 1];
  int rot_off[PK ? PK : 1];                   // past P: the part's start again, against zeros in q
#pragma unroll
  for (int ks = 0; ks < PK; ++ks) rot_off[ks] = (a.R + (ks * 32 + g * 8 < a.P ? ks * 32 + g * 8 : 0)) * 2;

  // Page of the visible keys of block b's half (16 keys lie in one page) and the range its rows are
  // clamped to: keys outside the visible range repeat a visible row, with weight zero.
  const char* base[2];
  int from[2], upto[2];
  auto locate = [&](int b) {
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const int h0 = b * 32 + hf * 16;
      from[hf] = min(max(h0, lo), n - 1);
      upto[hf] = max(min(h0 + 15, n - 1), from[hf]);
      if (h0 + 15 < lo) upto[hf] = from[hf] = lo;
      const int page = __builtin_amdgcn_readfirstlane(pg[(from[hf] >> a.bs_shift) - p0]);
      base[hf] = (const char*)a.cache + (int64_t)page * a.BS * RW * 2;
    }
  };
  auto row_off = [&](int b, int i) {                             // bytes into the page
    const int hf = i >> 2;
    const int key = min(max(b * 32 + step_key(g, i), from[hf]), upto[hf]);
    return (uint32_t)((key & mask) * RW * 2);
  };
  auto load_rotated = [&](int b) {
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const int key = min(max(b * 32 + hf * 16 + l16, from[hf]), upto[hf]);
      const uint32_t ro = (uint32_t)((key & mask) * RW * 2);
#pragma unroll
      for (int ks = 0; ks < PK; ++ks) kr[hf][ks] = load_piece<PAST>(base[hf] + (ro + rot_off[ks]));
    }
  };

  const int b1 = n > 0 ? (n - 1) >> 5 : -1, step = a.splits * 4;
  int b = (lo >> 5) + split * 4 + wave;
  if (b <= b1) {
    locate(b);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t ro = row_off(b, i);
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) v[cb][i] = load_piece<PAST>(base[i >> 2] + (ro + col_off[cb]));
    }
    load_rotated(b);
  }
  for (; b <= b1; b += step) {
    const int k0 = b * 32;
    f32x4 s[HT][2];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          *(u32x4*)(stage + (4 * g + i) * Lds::kStride + cb * 128 + l16 * 8) = v[cb][hf * 4 + i];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      f32x4 part[HT][2];                      // even and odd steps: two chains per head tile
#pragma unroll
      for (int ht = 0; ht < HT; ++ht) part[ht][0] = part[ht][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const u32x4 kf = *(const u32x4*)(stage + l16 * Lds::kStride + ks * 32 + g * 8);
#pragma unroll
        for (int ht = 0; ht < HT; ++ht)
          part[ht][ks & 1] = mfma_bf16(kf, *(const u32x4*)(qrow + ht * 16 * Lds::kQStride + ks * 32), part[ht][ks & 1]);
      }
#pragma unroll
      for (int ks = 0; ks < PK; ++ks)
#pragma unroll
        for (int ht = 0; ht < HT; ++ht)
          part[ht][ks & 1] = mfma_bf16(kr[hf][ks], *(const u32x4*)(qrow + ht * 16 * Lds::kQStride + NCB * 128 + ks * 32),
                                       part[ht][ks & 1]);
#pragma unroll
      for (int ht = 0; ht < HT; ++ht) s[ht][hf] = part[ht][0] + part[ht][1];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();        // the stage is written again after these reads
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    u32x4 pf[HT];
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) {
      float p[8], mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 8; ++i) p[i] = s[ht][i >> 2][i & 3] * sc;
      if (k0 < lo || k0 + 31 >= n) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int key = k0 + step_key(g, i);
          if (key < lo || key >= n) p[i] = -INFINITY;
        }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) mx = fmaxf(mx, p[i]);
      mx = fmaxf(mx, lane_xor16(mx));
      mx = fmaxf(mx, lane_xor32(mx));
      const float mn = fmaxf(m[ht], mx);      // finite: every block holds a visible key
      const float f = __builtin_amdgcn_exp2f(m[ht] - mn);
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p[i] = __builtin_amdgcn_exp2f(p[i] - mn);
        sum += p[i];
      }
      l[ht] = l[ht] * f + sum;
      m[ht] = mn;
      if (__any(f != 1.f)) {
#pragma unroll
        for (int i = 0; i < NCB * 8; ++i) o[ht][i] *= f;
      }
      pf[ht] = u32x4{pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3]), pack_bf16(p[4], p[5]),
                     pack_bf16(p[6], p[7])};
    }
    const int next = min(b + step, b1);       // after the last block its own rows again, unused
    locate(next);
    uint32_t ro[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) ro[i] = row_off(next, i);
    load_rotated(next);
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const u32x4 vf = column_of(v[cb], t);
#pragma unroll
        for (int ht = 0; ht < HT; ++ht) o[ht][cb * 8 + t] = mfma_bf16(vf, pf[ht], o[ht][cb * 8 + t]);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) v[cb][i] = load_piece<PAST>(base[i >> 2] + (ro[i] + col_off[cb]));
    }
  }

  // the waves meet in LDS, one head tile of each at a time: sums, maxima and partial results per
  // wave, then all threads combine those that split the keys of a head
  const int RS = a.R + 4, per = rows_merge_floats(a.R);
  float* const merge = (float*)shared;
#pragma unroll
  for (int ht = 0; ht < HT; ++ht) {
    l[ht] += lane_xor16(l[ht]);
    l[ht] += lane_xor32(l[ht]);
    __syncthreads();                              // what the LDS held before is used up
    {
      float* const dst = merge + wave * per;
      if (g == 0) { dst[16 * RS + l16] = m[ht]; dst[16 * RS + 16 + l16] = l[ht]; }
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int col = cb * 128 + (4 * g + i) * 8;
          if (col < a.R) {
            float* d = dst + l16 * RS + col;
            const f32x4* t = o[ht] + cb * 8;
            *(f32x4*)d = f32x4{t[0][i], t[1][i], t[2][i], t[3][i]};
            *(f32x4*)(d + 4) = f32x4{t[4][i], t[5][i], t[6][i], t[7][i]};
          }
        }
    }
    __syncthreads();
    // per head: the common maximum, each key part's factor (over its maximum's place) and the sum
    if (tid < 16) {
      float* const src = merge + 16 * RS + tid;              // wave k: key part k
      float mx = src[0];
      for (int k = 1; k < 4; ++k) mx = fmaxf(mx, src[k * per]);
      const float ms = mx == -INFINITY ? 0.f : mx;
      float sum = 0.f;
      for (int k = 0; k < 4; ++k) {
        float* const at = src + k * per;
        const float f = __builtin_amdgcn_exp2f(at[0] - ms);
        sum += at[16] * f;
        at[0] = f;
      }
      const float inv = a.splits > 1 ? 1.f : (sum > 0.f ? 1.f / sum : 0.f);
      for (int k = 0; k < 4; ++k) src[k * per] *= inv;
      const int head = ht * 16 + tid;
      if (a.splits > 1 && head < a.H) {
        float* ml = a.part + (int64_t)a.n * a.H * a.splits * a.R + (((int64_t)row * a.H + head) * a.splits + split) * 2;
        ml[0] = mx;
        ml[1] = sum;
      }
    }
    __syncthreads();
#pragma unroll 1
    for (int it = tid; it < 256 * NCB; it += 256) {
      const int hl = it / (16 * NCB), c = it % (16 * NCB) * 8;
      const int head = ht * 16 + hl;
      if (head >= a.H || c >= a.R) continue;
      float r[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int k = 0; k < 4; ++k) {
        const float* part = merge + k * per;
        const float f = part[16 * RS + hl];
        float x[8];
        Vec8<F32>::ld(part, hl * RS + c, x);
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i] += x[i] * f;
      }
      const int64_t item = (int64_t)row * a.H + head;
      if (a.splits == 1) Vec8<BF16>::st(a.out, item * a.R + c, r);
      else Vec8<F32>::st(a.part, (item * a.splits + split) * a.R + c, r);
    }
  }
}

// Whether rows are asked for past the last-level cache.  How much of their tables a call's tokens use is known here alone: a workgroup
// takes all of them to see as many keys as its own does.  (May be and is not: 0.1 to 0.3 us.)
__device__ __forceinline__ bool rows_past(const RowsArgs& a, int row) {
  int keys = min(max(a.ctx[row], 0), a.NB * a.BS);
  if (a.window > 0) keys = min(keys, a.window);
  return past_cache(min((int64_t)a.n * keys, (int64_t)a.num_pages * a.BS) * (a.R + a.P) * 2);
}
// MAY: it may be (see may_pass)
template <int NCB, int HT, int PK, bool MAY>
__global__ __launch_bounds__(256, NCB * HT <= 2 ? 2 : 1) void latent_narrow_kernel(RowsArgs a) {
  if constexpr (MAY)
    if (rows_past(a, blockIdx.x / a.splits)) return latent_narrow<NCB, HT, PK, true>(a);
  latent_narrow<NCB, HT, PK, false>(a);
}

// NCB column blocks of 128 cover R; PK steps of 32 the rotated part, which is a key only, never a value.  Workgroup: one
// token, HW tiles of 16 heads, one key range.  All four waves take the same 32 keys; waves on the same head tile
// (4 / HW) share its value columns out, and its scores: two take 16 keys each, four also every other step of the contraction,
// and hand them over through LDS (each for itself read all keys: 16 heads, 256 sequences of 1800 to 2304 tokens 123 us,
// now 115; 32 heads 134, now 121; the same sums).
//
// Bound by HBM, so what counts is how much is on its way: rows go from memory into LDS without passing through
// registers, in a ring of stages of 32 keys of which all but one are in flight (108 KB per CU for rows of 576; held in
// registers between its two uses, a block left its place only when its products were done: 256 sequences of 2050 tokens,
// 32 heads 157 us, now 141; a window of 1024 76, now 60; 64 sequences, 128 heads 124, now 92).  The value operand is
// transposed by the LDS reads.  Staged rows are twice an odd number of 16-byte pieces apart: of a read of 16 bytes lanes 0 to 3,
// 12 to 15 and 20 to 27 go together, and then the two quarters of a wave have every other piece of the banks each (an odd
// number had half of the LDS cycles in conflicts; 100 to 4096 tokens, 32 heads 174 us, 167 without them).
//
// Softmax weights meet the values in two bf16 planes.  With one, results were up to 0.5 % further from 64-bit ones than those
// of waves with maxima of their own (the weight of a maximum is 1 and loses nothing, and here there are fewer); with two
// they are 2 to 3 % nearer, for 5 % of the kernel's time (141 -> 147 us of the first).
constexpr int rows_ring(int NCB) { return NCB <= 2 ? 3 : 4; }       // two workgroups per CU where rows are short
template <int NCB, int PK> struct RowsStage {
  static constexpr int kMaxPieces = NCB * 16 + PK * 4 + 2;
  static constexpr int kHalf = (kMaxPieces + 3) / 4 * 1024;           // bytes of 16 keys, whole loads
  static constexpr int kLoads = ((kMaxPieces + 3) / 4 + 1) / 2;       // of a wave for a stage
  static constexpr int kBytes = rows_ring(NCB) * 2 * kHalf;
};

template <int NCB, int HW, int PK, bool PAST>
__global__ __launch_bounds__(256, NCB <= 2 || HW <= 2 ? 2 : 1) void latent_rows_kernel(RowsArgs a) {
  extern __shared__ __align__(16) char lds_raw[];
  typedef RowsStage<NCB, PK> Stage;
  constexpr int kRing = rows_ring(NCB), KS = 4 * NCB, SH = 4 / HW, VT = NCB * 8 / SH;     // value tiles of 16 columns of a wave
  constexpr int kKeys = KS + PK, kDots = 2 * kKeys / SH, kOdd = SH == 4 ? 2 : 1;   // products of a wave for the scores of a block
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hgroups = (a.H + 16 * HW - 1) / (16 * HW);
  int id = blockIdx.x;
  const int split = id % a.splits;
  id /= a.splits;
  const int row = id / hgroups, head = (id % hgroups * HW + wave % HW) * 16 + l16;
  const int RW = a.R + a.P, pieces = RW / 8, staged = ((pieces + 1) | 3) - 1;
  const int share = wave / HW, col0 = share * VT * 16;           // of the wave's values
  const int mine = SH > 1 ? share & 1 : 0, odd = SH == 4 ? share >> 1 : 0;      // of the scores: its 16 keys, its steps

  u32x4 q[kKeys / kOdd];
#pragma unroll
  for (int i = 0; i < kKeys / kOdd; ++i) {
    const int ks = kOdd * i + odd;
    const int c = ks < KS ? ks * 32 + g * 8 : (ks - KS) * 32 + g * 8;
    const bool there = head < a.H && c < (ks < KS ? a.R : a.P);
    q[i] = u32x4{0u, 0u, 0u, 0u};
    if (there) q[i] = *(const u32x4*)((const uint16_t*)a.q + ((int64_t)row * a.H + head) * RW + (ks < KS ? c : a.R + c));
  }
  const int seq = a.seq ? min(max(a.seq[row], 0), a.B - 1) : row;
  const int n = min(a.ctx[row], a.NB * a.BS);
  const int lo = a.window > 0 ? max(0, n - a.window) : 0;
  const int b0 = (lo >> 5) + split, b1 = n > 0 ? (n - 1) >> 5 : -1;
  const int blocks = b1 >= b0 ? (b1 - b0) / a.splits + 1 : 0;

  // ---- rows into LDS: 16 keys of a page with `staged` pieces each, by loads of 64 pieces.  A wave has every other load of
  // one half of the keys; its last may come twice.
  const int half = wave & 1, loads = (staged + 3) / 4;
  int piece_at[Stage::kLoads];                                   // byte of a lane's piece in 16 rows, row in the upper bits
#pragma unroll
  for (int k = 0; k < Stage::kLoads; ++k) {
    const int p = min((wave >> 1) + 2 * k, loads - 1) * 64 + lane, r = min(p / staged, 15), pc = p - r * staged;
    piece_at[k] = (r * RW * 2 + (pc < pieces ? pc : 0) * 16) | r << 20;
  }
  const int mask = a.BS - 1;
  // page ids of the table from page0 on, one a lane; 64 are enough for a while
  int page0 = lo >> a.bs_shift, ids;
  auto fetch_ids = [&] {
    const int at = page0 + lane, id = at < a.NB ? a.table[(int64_t)seq * a.NB + at] : 0;
    ids = id >= 0 && id < a.num_pages ? id : 0;                  // whatever the table says, it is one of the cache's
  };
  fetch_ids();
  // what the loads of stage j need, then load k of them
  char* to;
  int h0, from, upto;
  bool whole;
  u32x4 rows;
  auto locate = [&](int j) {
    const bool there = j < blocks;                               // past the last block nothing is read
    h0 = (b0 + j * a.splits) * 32 + half * 16;
    to = lds_raw + (j % kRing) * (2 * Stage::kHalf) + half * Stage::kHalf;
    // keys outside the visible range repeat a visible row, with weight zero
    from = h0 + 15 < lo ? lo : min(max(h0, lo), n - 1), upto = h0 + 15 < lo ? lo : max(min(h0 + 15, n - 1), from);
    const int index = there ? from >> a.bs_shift : page0;
    if (index >= page0 + 64) {                                   // uniform
      page0 = index;
      fetch_ids();
    }
    const char* const page = (const char*)a.cache + (int64_t)__builtin_amdgcn_readlane(ids, index - page0) * a.BS * RW * 2;
    whole = from == h0 && upto == h0 + 15;
    const int first = whole ? (h0 & mask) * RW * 2 : 0;
    rows = rows_from(page + first, there ? (uint32_t)a.BS * RW * 2 - first : 0u);
  };
  auto load = [&](int k, bool all) {
    char* const at = to + min((wave >> 1) + 2 * k, loads - 1) * 1024;
    if (all) {
      load_to_lds<PAST>(rows, at, piece_at[k] & 0xfffff, 0);
    } else {
      const int r = piece_at[k] >> 20, key = min(max(h0 + r, from), upto);
      load_to_lds<PAST>(rows, at, (piece_at[k] & 0xfffff) + ((key & mask) - r) * RW * 2, 0);
    }
  };
#pragma unroll
  for (int j = 0; j < kRing - 1; ++j) {
    locate(j);
    if (whole)
#pragma unroll
      for (int k = 0; k < Stage::kLoads; ++k) load(k, true);
    else
#pragma unroll
      for (int k = 0; k < Stage::kLoads; ++k) load(k, false);
  }

  f32x4 o[VT];
#pragma unroll
  for (int i = 0; i < VT; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const float sc = a.scale * 1.44269504088896f;
  // R may end inside the last column block: columns past it are others again, against zeros in q or in results that are not
  // written
  const int key_at = mine * Stage::kHalf + l16 * staged * 16 + g * 16, value_at = (4 * g + (l16 >> 2)) * staged * 16 + (l16 & 3) * 8;
  int rot_at[PK ? PK / kOdd : 1];
#pragma unroll
  for (int i = 0; i < PK / kOdd; ++i) {
    const int ks = kOdd * i + odd;
    rot_at[i] = key_at + (a.R / 8 - g + (ks * 32 + g * 8 < a.P ? ks * 4 + g : 0)) * 16;
  }
  f32x4* const shared = (f32x4*)(lds_raw + Stage::kBytes) + wave % HW * SH * 64 + lane;     // scores of the wave's heads
#pragma unroll 1
  for (int j = 0; j < blocks; ++j) {
    // this wave's share of block j has come when at most those of the blocks behind it are on their way
    static_assert((kRing - 2) * Stage::kLoads < 64, "the counter's range");
    constexpr int kOn = (kRing - 2) * Stage::kLoads;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070 | (kOn & 15) | (kOn >> 4) << 14);      // LDS reads of the block before are done, too
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    locate(j + kRing - 1);                                       // over what the block before was in
    const int k0 = (b0 + j * a.splits) * 32;
    const char* const at = lds_raw + (j % kRing) * (2 * Stage::kHalf);
    // operands leave LDS kAhead products ahead; the barriers keep the compiler from moving a read to its use
    constexpr int kAhead = 4, kRead = kAhead + 1, kSteps = kKeys / kOdd;
    u32x4 kf[kRead];
    auto read_key = [&](int i) {                                 // of the wave's half i / kSteps, its step i % kSteps
      if (i >= kDots) return;
      const int own = i % kSteps, first = kOdd * own, ks = first + odd;
      const int c = first < KS ? key_at + (first < KS - 4 ? ks * 64 : min(ks * 64, a.R * 2 - 64))
                               : rot_at[first < KS ? 0 : own - KS / kOdd];
      kf[i % kRead] = *(const u32x4*)(at + i / kSteps * Stage::kHalf + c);
    };
    f32x4 part[2][2] = {};                                       // of both halves, even and odd steps
#pragma unroll
    for (int i = 0; i < kAhead; ++i) read_key(i);
    auto scores = [&](bool loads_too) {
#pragma unroll
      for (int i = 0; i < kDots; ++i) {
        read_key(i + kAhead);
        const int hf = i / kSteps, own = i % kSteps, chain = SH == 4 ? 0 : own & 1;
        part[hf][chain] = mfma_bf16(kf[i % kRead], q[own], part[hf][chain]);
        if (loads_too)
#pragma unroll
          for (int k = i * Stage::kLoads / kDots; k < (i + 1) * Stage::kLoads / kDots; ++k) load(k, true);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (whole) {                                                 // the loads are spread over the products
      scores(true);
    } else {
#pragma unroll
      for (int k = 0; k < Stage::kLoads; ++k) load(k, false);
      scores(false);
    }
    f32x4 s[2] = {part[0][0] + part[0][1], part[1][0] + part[1][1]};
    if constexpr (SH > 1) shared[share * 64] = SH == 4 ? part[0][0] : s[0];
    u32x4 vf[kRead];
    auto read_value = [&](int i) {
      if (i >= VT) return;
      const int c = col0 + i * 16;
      const char* const v = at + value_at + (c < a.R ? c : 0) * 2;
      const uint2 x = read_transposed((const uint16_t*)v), y = read_transposed((const uint16_t*)(v + Stage::kHalf));
      vf[i % kRead] = u32x4{x.x, x.y, y.x, y.y};
    };
#pragma unroll
    for (int i = 0; i < kRead; ++i) read_value(i);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (SH > 1) {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0xc07f);                        // in LDS; loads from memory go on
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      s[0] = shared[0], s[1] = shared[64];
      if constexpr (SH == 4) s[0] += shared[128], s[1] += shared[192];
    }
    float p[8], mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = s[i >> 2][i & 3] * sc;
    if (k0 < lo || k0 + 31 >= n) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int key = k0 + step_key(g, i);
        if (key < lo || key >= n) p[i] = -INFINITY;
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) mx = fmaxf(mx, p[i]);
    if (__any(mx > m)) {                                         // in any lane: seldom after the first keys
      mx = fmaxf(m, mx);
      mx = fmaxf(mx, lane_xor16(mx));
      mx = fmaxf(mx, lane_xor32(mx));                            // finite: every block holds a visible key
      const float f = __builtin_amdgcn_exp2f(m - mx);
      m = mx;
      l *= f;
#pragma unroll
      for (int i = 0; i < VT; ++i) o[i] *= f;
    }
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      p[i] = __builtin_amdgcn_exp2f(p[i] - m);
      sum += p[i];
    }
    l += sum;
    u32x4 pf, pl;                                                // planes
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      pf[d] = pack_bf16(p[2 * d], p[2 * d + 1]);
      pl[d] = pack_bf16(p[2 * d] - __uint_as_float(pf[d] << 16), p[2 * d + 1] - __uint_as_float(pf[d] & 0xffff0000u));
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < VT; i += 2) {                            // no product waits for the one before it
      o[i] = mfma_bf16(vf[i % kRead], pf, o[i]);
      o[i + 1] = mfma_bf16(vf[(i + 1) % kRead], pf, o[i + 1]);
      o[i] = mfma_bf16(vf[i % kRead], pl, o[i]);
      o[i + 1] = mfma_bf16(vf[(i + 1) % kRead], pl, o[i + 1]);
      read_value(i + kRead);
      read_value(i + 1 + kRead);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __builtin_amdgcn_s_waitcnt(0);                                 // no load is left on its way to LDS
  l += lane_xor16(l);
  l += lane_xor32(l);
  if (head >= a.H) return;
  const int64_t item = (int64_t)row * a.H + head;
  const float inv = a.splits > 1 ? 1.f : (l > 0.f ? 1.f / l : 0.f);
#pragma unroll
  for (int i = 0; i < VT; ++i) {
    const int c = col0 + i * 16 + 4 * g;
    if (c >= a.R) continue;
    o[i] *= inv;
    if (a.splits == 1) *(uint2*)((uint16_t*)a.out + item * a.R + c) = uint2{pack_bf16(o[i][0], o[i][1]), pack_bf16(o[i][2], o[i][3])};
    else *(f32x4*)(a.part + (item * a.splits + split) * a.R + c) = o[i];
  }
  if (a.splits > 1 && wave < HW && g == 0) {
    float* const ml = a.part + (int64_t)a.n * a.H * a.splits * a.R + (item * a.splits + split) * 2;
    ml[0] = m;
    ml[1] = l;
  }
}

__global__ __launch_bounds__(64) void latent_rows_combine_kernel(RowsArgs a) {
  const int64_t item = blockIdx.x;       // (row, head)
  const float* ml = a.part + (int64_t)a.n * a.H * a.splits * a.R + item * a.splits * 2;
  float mx = -INFINITY;
  for (int s = 0; s < a.splits; ++s) mx = fmaxf(mx, ml[2 * s]);
  if (mx == -INFINITY) mx = 0.f;
  float l = 0.f;
  for (int s = 0; s < a.splits; ++s) l += ml[2 * s + 1] * __builtin_amdgcn_exp2f(ml[2 * s] - mx);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  for (int c = threadIdx.x * 8; c < a.R; c += 512) {
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < a.splits; ++s) {
      const float f = __builtin_amdgcn_exp2f(ml[2 * s] - mx) * inv;
      float v[8];
      Vec8<F32>::ld(a.part, (item * a.splits + s) * a.R + c, v);
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] += v[i] * f;
    }
    Vec8<BF16>::st(a.out, item * a.R + c, acc);
  }
}

// One workgroup per (token, head), plain fp32 arithmetic, any R and P.
template <typename T>
__global__ __launch_bounds__(256) void latent_plain_kernel(RowsArgs a) {
  extern __shared__ __align__(16) char lds_raw[];
  float* q = (float*)lds_raw;              // R + P
  __shared__ float sc[256];
  __shared__ float red[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int row = blockIdx.x / a.H;
  const int RW = a.R + a.P;
  const int64_t qat = (int64_t)blockIdx.x * RW, oat = (int64_t)blockIdx.x * a.R;
  const int seq = a.seq ? min(max(a.seq[row], 0), a.B - 1) : row;
  const int n = min(a.ctx[row], a.NB * a.BS);
  const int lo = a.window > 0 ? max(0, n - a.window) : 0;
  for (int c = tid; c < RW; c += 256) q[c] = Elem<T>::ld(a.q, qat + c);
  auto key_at = [&](int t) -> int64_t {
    const int p = page_of(a, t);
    int page = a.table[(int64_t)seq * a.NB + p];
    if (page < 0 || page >= a.num_pages) page = 0;
    return ((int64_t)page * a.BS + (t - p * a.BS)) * RW;
  };
  constexpr int kCols = 16;                // columns per thread: R <= 4096
  float o[kCols];
#pragma unroll
  for (int i = 0; i < kCols; ++i) o[i] = 0.f;
  float m = -INFINITY, l = 0.f;
  for (int c0 = lo; c0 < n; c0 += 256) {
    const int cnt = min(256, n - c0);
    __syncthreads();                       // q is there; the last chunk's scores are used up
    for (int j = wave; j < cnt; j += 4) {
      const int64_t at = key_at(c0 + j);
      float acc = 0.f;
      for (int c = lane; c < RW; c += 64) acc = fmaf(q[c], Elem<T>::ld(a.cache, at + c), acc);
      acc = wave_sum(acc);
      if (lane == 0) sc[j] = acc * a.scale;
    }
    __syncthreads();
    float mx = tid < cnt ? sc[tid] : -INFINITY;
    mx = wave_max(mx);
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float mn = fmaxf(m, mx);
    const float f = expf(m - mn);
    __syncthreads();
    const float p = tid < cnt ? expf(sc[tid] - mn) : 0.f;
    sc[tid] = p;
    const float s = wave_sum(p);
    if (lane == 0) red[wave] = s;
    __syncthreads();
    l = l * f + red[0] + red[1] + red[2] + red[3];
    m = mn;
#pragma unroll
    for (int i = 0; i < kCols; ++i) o[i] *= f;
    for (int j = 0; j < cnt; ++j) {
      const int64_t at = key_at(c0 + j);
      const float pj = sc[j];
#pragma unroll
      for (int i = 0; i < kCols; ++i) {
        const int c = tid + i * 256;
        if (c < a.R) o[i] = fmaf(pj, Elem<T>::ld(a.cache, at + c), o[i]);
      }
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int i = 0; i < kCols; ++i) {
    const int c = tid + i * 256;
    if (c < a.R) Elem<T>::st(a.out, oat + c, o[i] * inv);
  }
}

constexpr int kMaxLdsPages = 4096, kMaxRotated = 64;

// Which rows the narrow kernel takes, with its head tiles per wave.  Past 32 heads it would take a head's keys with fewer
// waves and read a row twice (256 columns, 40 heads, a window of 300 keys: 49 us against 27), and wider rows don't fit
// its registers with two tiles; up to 32 heads of 16 to 256 columns it is ahead by 2 to 20 per cent.
bool rows_narrow(int H, int R) { return R <= 256 && H <= 32; }
int rows_ht(int H) { return H > 16 ? 2 : 1; }
// Head tiles of a workgroup of the other one.
int rows_hw(int H) { return H > 32 ? 4 : (H > 16 ? 2 : 1); }

// Key ranges per token: enough workgroups to cover the chip, at least four 32-key steps each (of the narrow kernel two per
// wave).
int rows_splits(int n, int H, int R, int window, int NB, int BS) {
  const bool narrow = rows_narrow(H, R);
  const int groups = narrow ? n : n * ((H + 16 * rows_hw(H) - 1) / (16 * rows_hw(H)));
  int64_t keys = (int64_t)NB * BS;
  if (window > 0 && window < keys) keys = window;
  const int steps = (int)((keys + 31) / 32);
  const int resident = (narrow ? (R + 127) / 128 * rows_ht(H) : (R + 127) / 128) <= 2 ? 2 : 1;       // workgroups per CU
  const int least = narrow ? 8 : 4;
  int s = 256 * resident / (groups > 0 ? groups : 1);
  s = s < steps / least ? s : steps / least;
  s = s < 32 ? s : 32;
  return s < 1 ? 1 : s;
}

template <int TT> int launch_headwise(const HeadArgs& a, hipStream_t st) {
  const int bm = (a.M + 63) / 64, bn = (a.n + 16 * TT - 1) / (16 * TT), stages = (a.K + kHeadStage - 1) / kHeadStage;
  const int smem = (stages < kHeadRing ? stages : kHeadRing) * HeadTile<TT>::kBytes;
  if (smem > 64 * 1024 &&
      hipFuncSetAttribute((const void*)headwise_tile_kernel<TT>, hipFuncAttributeMaxDynamicSharedMemorySize, smem) !=
          hipSuccess) {
    zp_set_error("headwise_linear: cannot reserve %d bytes of LDS", smem);
    return ZP_EHIP;
  }
  hipLaunchKernelGGL((headwise_tile_kernel<TT>), dim3((unsigned)bm * bn * a.H), dim3(256), smem, st, a, bm, bn);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}
int launch_combine(const RowsArgs& a, hipStream_t st) {
  if (a.splits > 1) {
    hipLaunchKernelGGL(latent_rows_combine_kernel, dim3((unsigned)a.n * a.H), dim3(64), 0, st, a);
    ZP_LAUNCH_CHECK();
  }
  return ZP_OK;
}
// Whether rows may be asked for past the last-level cache: one workgroup reads a key, in whole lines, and all that may be read do
// not fit.  256 sequences of 1800 to 2304 tokens: rows of 576, 16 heads 115 us through it and 103 past it, 32 heads 122 and
// 115, 64 heads 181 and 176; rows of 320, 32 heads 78 and 73, 16 heads 71 and 65.  With two workgroups on a token (128
// heads) 324 and 338; where rows fit, 40 sequences, 42 and 43; rows of 192, 200 MB, 42 and 47.  What may be read is as much as the
// tables hold.  Where contexts are shorter, the narrow kernel asks itself (rows of 320, 16 heads, 256 sequences of 1000 tokens
// in tables of 4096: 34 us through it, 37 past it, now 34.5); the other one goes past it all the same (rows of 576, 32
// heads, 700 tokens 47 us for 44; with both forms in one kernel 64 heads took 2 % longer wherever they are).
bool may_pass(const RowsArgs& a, int hgroups) {
  const int64_t keys = a.window > 0 ? std::min<int64_t>(a.window, (int64_t)a.NB * a.BS) : (int64_t)a.NB * a.BS;
  return hgroups == 1 && (a.R + a.P) % 64 == 0 &&
         past_cache(std::min(a.n * keys, (int64_t)a.num_pages * a.BS) * (a.R + a.P) * 2);
}
template <int NCB, int HT, int PK, bool MAY> int launch_latent_narrow(const RowsArgs& a, hipStream_t st) {
  const size_t merge = 4 * sizeof(float) * (size_t)rows_merge_floats(a.R);
  const size_t work = 4 * RowsLds<NCB, PK>::kStage + (size_t)HT * RowsLds<NCB, PK>::kQ;
  const size_t smem = (((size_t)a.lds_pages * 4 + 15) & ~(size_t)15) + (merge > work ? merge : work);
  if (smem > 64 * 1024 &&
      hipFuncSetAttribute((const void*)latent_narrow_kernel<NCB, HT, PK, MAY>, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)smem) != hipSuccess) {
    zp_set_error("latent_rows_attention: cannot reserve %zu bytes of LDS", smem);
    return ZP_EHIP;
  }
  hipLaunchKernelGGL((latent_narrow_kernel<NCB, HT, PK, MAY>), dim3((unsigned)a.n * a.splits), dim3(256), smem, st, a);
  ZP_LAUNCH_CHECK();
  return launch_combine(a, st);
}
template <int NCB, int HT, int PK> int launch_latent_narrow(const RowsArgs& a, hipStream_t st) {
  return may_pass(a, 1) ? launch_latent_narrow<NCB, HT, PK, true>(a, st) : launch_latent_narrow<NCB, HT, PK, false>(a, st);
}
template <int NCB, int HW, int PK, bool PAST> int launch_latent_rows(const RowsArgs& a, int hgroups, hipStream_t st) {
  constexpr int smem = RowsStage<NCB, PK>::kBytes + (HW < 4 ? 4096 : 0);
  static_assert(smem <= 160 * 1024, "LDS of a CU");
  if (smem > 64 * 1024 &&
      hipFuncSetAttribute((const void*)latent_rows_kernel<NCB, HW, PK, PAST>, hipFuncAttributeMaxDynamicSharedMemorySize,
                          smem) != hipSuccess) {
    zp_set_error("latent_rows_attention: cannot reserve %d bytes of LDS", smem);
    return ZP_EHIP;
  }
  hipLaunchKernelGGL((latent_rows_kernel<NCB, HW, PK, PAST>), dim3((unsigned)a.n * hgroups * a.splits), dim3(256), smem, st, a);
  ZP_LAUNCH_CHECK();
  return launch_combine(a, st);
}
template <int NCB, int HW, int PK> int launch_latent_rows(const RowsArgs& a, hipStream_t st) {
  const int hgroups = (a.H + 16 * HW - 1) / (16 * HW);
  return may_pass(a, hgroups) ? launch_latent_rows<NCB, HW, PK, true>(a, hgroups, st)
                               : launch_latent_rows<NCB, HW, PK, false>(a, hgroups, st);
}
template <int NCB, int PK> int launch_latent_rows(const RowsArgs& a, hipStream_t st) {
  if constexpr (NCB <= 2) {
    if (!rows_narrow(a.H, a.R)) return launch_latent_rows<NCB, 4, PK>(a, st);
    return rows_ht(a.H) == 2 ? launch_latent_narrow<NCB, 2, PK>(a, st) : launch_latent_narrow<NCB, 1, PK>(a, st);
  } else {
    switch (rows_hw(a.H)) {
      case 1: return launch_latent_rows<NCB, 1, PK>(a, st);
      case 2: return launch_latent_rows<NCB, 2, PK>(a, st);
      default: return launch_latent_rows<NCB, 4, PK>(a, st);
    }
  }
}

}  // namespace


extern "C" int zp_latent_norm_store(const void* in, const float* q_weight, const float* c_weight,
                                    void* q_out, void* c_out, void* cache, const int32_t* slots,
                                    const int32_t* positions, const float* freqs, int32_t n, int32_t q_width,
                                    int32_t c_width, int32_t p_width, int32_t q_norm, int32_t c_norm,
                                    int32_t rot, int64_t num_slots, float eps, int32_t dtype, void* stream) {
  ZP_REQUIRE(n >= 0 && q_width > 0 && c_width >= 0 && q_norm > 0 && q_norm <= q_width && c_norm <= c_width &&
                 (c_width ? c_norm > 0 && num_slots > 0 : p_width == 0) && p_width >= 0 && rot >= 0 && rot % 2 == 0 &&
                 rot <= p_width, "latent_norm_store: bad dims");
  ZP_MODEL_DTYPE("latent_norm_store");
  if (q_width % 8 || c_width % 8 || p_width % 8 || q_width > 512 * kNormPieces || c_width > 512 * kNormPieces) {
    zp_set_error("latent_norm_store: ranks %d, %d, rotated part %d unsupported (multiples of 8, <= %d)", q_width, c_width,
                 p_width, 512 * kNormPieces);
    return ZP_EUNSUPPORTED;
  }
  if (n == 0) return ZP_OK;
  ZP_REQUIRE(in && q_weight && q_out && (!c_width || (c_weight && cache && slots)) && (!rot || (positions && freqs)),
             "latent_norm_store: null pointer");
  ZP_REQUIRE(aligned16(in) && aligned16(q_weight) && aligned16(c_weight) && aligned16(q_out) &&
                 aligned16(c_out) && aligned16(cache), "latent_norm_store: tensors must be 16-byte aligned");
  NormStoreArgs a = {in, q_weight, c_weight, q_out, c_out, cache, slots, positions, freqs, n, q_width, c_width, p_width,
                     q_norm, c_norm, rot / 2, num_slots, eps};
  const unsigned grid = (unsigned)(((c_width ? 2 : 1) * (int64_t)n + 3) / 4);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == ZP_BF16) hipLaunchKernelGGL((latent_norm_store_kernel<BF16>), dim3(grid), dim3(256), 0, st, a);
  else hipLaunchKernelGGL((latent_norm_store_kernel<F32>), dim3(grid), dim3(256), 0, st, a);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}

extern "C" int zp_rotate_heads(void* x, const int32_t* positions, const float* freqs, int32_t n, int32_t H, int32_t head,
                               int32_t at, int32_t rot, int64_t x_stride, int32_t dtype, void* stream) {
  ZP_REQUIRE(n >= 0 && H > 0 && head > 0 && at >= 0 && rot >= 0 && rot % 2 == 0 && at + rot <= head &&
                 x_stride >= (int64_t)H * head, "rotate_heads: bad dims");
  ZP_MODEL_DTYPE("rotate_heads");
  if (rot > 2048) {
    zp_set_error("rotate_heads: %d rotated dimensions (<= 2048)", rot);
    return ZP_EUNSUPPORTED;
  }
  if (n == 0 || rot == 0) return ZP_OK;
  ZP_REQUIRE(x && positions && freqs, "rotate_heads: null pointer");
  RotateArgs a = {x, positions, freqs, n, H, head, at, rot / 2, x_stride};
  const unsigned grid = (unsigned)((n + kRotTokens - 1) / kRotTokens);
  const size_t smem = sizeof(float2) * kRotTokens * (rot / 2);
  hipStream_t st = (hipStream_t)stream;
  const bool wide = rot % 16 == 0 && head % 8 == 0 && at % 8 == 0 && x_stride % 8 == 0 && aligned16(x);
#define ZP_ROTATE(T)                                                                                          \
  do {                                                                                                        \
    if (wide) hipLaunchKernelGGL((rotate_heads_kernel<T, 8>), dim3(grid), dim3(256), smem, st, a);            \
    else hipLaunchKernelGGL((rotate_heads_kernel<T, 1>), dim3(grid), dim3(256), smem, st, a);                 \
  } while (0)
  if (dtype == ZP_BF16) ZP_ROTATE(BF16); else ZP_ROTATE(F32);
#undef ZP_ROTATE
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}

extern "C" int zp_headwise_linear(const void* in, const void* w, void* out, const int32_t* positions,
                                  const float* freqs, int32_t n, int32_t H, int32_t K, int32_t M, int32_t tail,
                                  int32_t rot, int32_t dtype, void* stream) {
  ZP_REQUIRE(n >= 0 && H > 0 && K > 0 && M > 0 && tail >= 0 && rot >= 0 && rot % 2 == 0 && rot <= tail &&
                 (rot == 0 || (positions && freqs)), "headwise_linear: bad dims");
  ZP_MODEL_DTYPE("headwise_linear");
  if (K % 32 != 0 || M % 16 != 0 || tail % 8 != 0 || H > 65535) {
    zp_set_error("headwise_linear: K %d, M %d, tail %d unsupported (multiples of 32, 16, 8)", K, M, tail);
    return ZP_EUNSUPPORTED;
  }
  if (n == 0) return ZP_OK;
  ZP_REQUIRE(in && w && out && aligned16(in) && aligned16(w) && aligned16(out),
             "headwise_linear: null or unaligned pointer");
  HeadArgs a = {in, w, out, positions, freqs, n, H, K, M, tail, rot / 2};
  // The staged kernel, except for what its 32-bit offsets don't span and for little work in one or two stages, whose set-up
  // nothing hides: from 8192 matrix products on it is ahead (us of both, the staged one second: K 160, 16 heads of M 64, 1 to
  // 200 tokens 2.9 to 3.3 and 3.5 to 3.8, 1000 tokens 5.6 and 4.5; K 128, 16 heads of M 64, 200 tokens 3.3 and 3.4, 1000 5.4
  // and 3.9; K 96, 64 heads of M 112, 17 tokens 2.9 and 3.4, 64 tokens 3.5 and 3.7, 200 6.6 and 4.5; K 64, 64 heads of M 256,
  // 17 tokens 3.1 and 3.6, 64 tokens 4.0 and 3.8; K 32, 64 heads of M 64, 200 tokens 3.2 and 3.8, 1000 6.7 and 6.3), if its
  // rows of W hold at least 3 KB (M 16, K 32, 64 heads, 4000 tokens: 10.0 and 13.3) and the tails are not most of it (K 64, M
  // 64, 64 behind them, 128 heads, 4000 tokens: 96 and 122).  K 256: 17 tokens 4.2 and 3.7; 512: 5.8 and 4.6; with M 16 3.4
  // and 3.6, 4.5 and 4.5
  const int64_t columns = (int64_t)((M + 63) / 64) * H;
  const int64_t products = (int64_t)(K / 32) * (M / 16) * H * (n < 24 ? 1 : (n + 8) / 16);
  const bool much = K >= (M < 64 ? 512 : 256) || (products >= 8192 && (M < 64 ? M : 64) * K >= 1536 && (tail < K || tail < M));
  const bool staged = dtype == ZP_BF16 && much && (int64_t)M * K * 2 < 1ll << 31 && (int64_t)64 * H * (K + tail) * 2 < 1ll << 31;
  // as many tokens per wave (W is read once for them) as still leave two workgroups per CU; of the staged kernel as many as
  // leave one (64 tokens, 32 heads of 512 -> 128: 6.9 us with 64 workgroups, 5.5 with 256), and no more than there are
  int tt = staged && n <= 32 ? (n <= 16 ? 1 : 2) : 4;
  while (tt > 1 && columns * ((n + 16 * tt - 1) / (16 * tt)) < (staged ? 256 : 512)) tt >>= 1;
  const dim3 grid((M + 63) / 64, H, (n + 16 * tt - 1) / (16 * tt));
  ZP_REQUIRE(grid.z <= 65535, "headwise_linear: too many tokens");
  hipStream_t st = (hipStream_t)stream;
  if (staged && columns * grid.z < 1ll << 31)
    return tt == 4 ? launch_headwise<4>(a, st) : (tt == 2 ? launch_headwise<2>(a, st) : launch_headwise<1>(a, st));
#define ZP_HEADWISE(T)                                                                            \
  do {                                                                                            \
    if (tt == 4) hipLaunchKernelGGL((headwise_kernel<T, 4>), grid, dim3(256), 0, st, a);          \
    else if (tt == 2) hipLaunchKernelGGL((headwise_kernel<T, 2>), grid, dim3(256), 0, st, a);     \
    else hipLaunchKernelGGL((headwise_kernel<T, 1>), grid, dim3(256), 0, st, a);                  \
  } while (0)
  if (dtype == ZP_BF16) ZP_HEADWISE(BF16);
  else ZP_HEADWISE(F32);
#undef ZP_HEADWISE
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}

extern "C" int64_t zp_latent_rows_workspace(int32_t n, int32_t H, int32_t R, int32_t window,
                                            int32_t NB, int32_t BS, int32_t dtype) {
  if (n < 0 || H <= 0 || R <= 0 || NB <= 0 || BS <= 0) return -1;
  if (dtype != ZP_BF16 || R > 512) return 0;
  const int s = rows_splits(n, H, R, window, NB, BS);
  return s == 1 ? 0 : (int64_t)n * H * s * (R + 2) * 4;
}

extern "C" int zp_latent_rows_attention(const void* q, const void* cache, const int32_t* table,
                                        const int32_t* context_lens, const int32_t* table_rows,
                                        void* out, int32_t n, int32_t H, int32_t R, int32_t P, int32_t BS,
                                        int32_t B, int32_t NB, int32_t num_pages, int32_t window,
                                        float scale, int32_t dtype, void* workspace,
                                        int64_t workspace_bytes, void* stream) {
  ZP_REQUIRE(n >= 0 && H > 0 && R > 0 && P >= 0 && BS > 0 && B > 0 && NB > 0 && num_pages > 0 && window >= 0,
             "latent_rows_attention: bad dims");
  ZP_MODEL_DTYPE("latent_rows_attention");
  if (R % 32 != 0 || R > 4096 || P % 8 != 0 || P > 4096) {
    zp_set_error("latent_rows_attention: latent size %d, rotated part %d unsupported (multiples of 32 and 8, <= 4096)", R, P);
    return ZP_EUNSUPPORTED;
  }
  if (n == 0) return ZP_OK;
  ZP_REQUIRE(q && cache && table && context_lens && out, "latent_rows_attention: null pointer");
  ZP_REQUIRE(table_rows || n <= B, "latent_rows_attention: more tokens than table rows");
  ZP_REQUIRE(aligned16(q) && aligned16(cache) && aligned16(out) && aligned16(workspace),
             "latent_rows_attention: tensors must be 16-byte aligned");
  RowsArgs a = {};
  a.q = q; a.cache = cache; a.table = table; a.ctx = context_lens; a.seq = table_rows; a.out = out;
  a.part = (float*)workspace; a.n = n; a.H = H; a.R = R; a.P = P; a.BS = BS; a.B = B; a.NB = NB;
  a.num_pages = num_pages; a.window = window; a.scale = scale; a.bs_shift = -1;
  if ((BS & (BS - 1)) == 0)
    for (a.bs_shift = 0; (1 << a.bs_shift) < BS; ++a.bs_shift) {}
  hipStream_t st = (hipStream_t)stream;
  int64_t pages = NB;
  if (window > 0 && (window - 1) / BS + 2 < pages) pages = (window - 1) / BS + 2;
  if (dtype == ZP_F32 || R > 512 || P > kMaxRotated || a.bs_shift < 4 || (rows_narrow(H, R) && pages > kMaxLdsPages) ||
      (int64_t)BS * (R + P) * 2 >= 1ll << 31) {   // bs_shift -1: not a power of two
    const size_t smem = sizeof(float) * (R + P);
    if (dtype == ZP_BF16)
      hipLaunchKernelGGL((latent_plain_kernel<BF16>), dim3((unsigned)n * H), dim3(256), smem, st, a);
    else
      hipLaunchKernelGGL((latent_plain_kernel<F32>), dim3((unsigned)n * H), dim3(256), smem, st, a);
    ZP_LAUNCH_CHECK();
    return ZP_OK;
  }
  a.lds_pages = (int)pages;
  a.splits = rows_splits(n, H, R, window, NB, BS);
  ZP_REQUIRE(a.splits == 1 || (workspace && workspace_bytes >= zp_latent_rows_workspace(n, H, R, window, NB, BS, dtype)),
             "latent_rows_attention: workspace too small");
#define ZP_LATENT_ROWS(NCB) (P ? launch_latent_rows<NCB, 2>(a, st) : launch_latent_rows<NCB, 0>(a, st))
  switch ((R + 127) / 128) {
    case 1: return ZP_LATENT_ROWS(1);
    case 2: return ZP_LATENT_ROWS(2);
    case 3: return ZP_LATENT_ROWS(3);
    default: return ZP_LATENT_ROWS(4);
  }
#undef ZP_LATENT_ROWS
}
